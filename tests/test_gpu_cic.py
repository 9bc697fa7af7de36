"""HIP CIC kernels vs the float64 oracle (the reference's Pallas-vs-JAX gate,
tests/test_pallas_cic.py:31-154, restated: rtol/atol 2e-6, 3e-5 for explicit cell sizes)."""

import numpy as np
import pytest
import torch

from oracle import cic
from pmpp_amd.cic import hip_gather, hip_gather_bwd, hip_scatter, hip_scatter_bwd

pytestmark = pytest.mark.gpu


def _t(x, dev, dtype=torch.float32):
    return torch.as_tensor(np.asarray(x), device=dev).to(dtype)


def _np(t):
    return t.detach().cpu().numpy().astype(np.float64)


CASES = [
    # (mesh spatial, global, channels, offset, mesh_cell, particle_cell, n, valid)
    ((4, 4, 4), (4, 4, 4), (), 0.0, None, 1.0, 4, False),
    ((4, 4, 4), (4, 4, 4), (2,), 0.0, None, 1.0, 5, False),
    ((4, 4, 4), (4, 4, 4), (3,), 0.0, None, 1.0, 5, True),
    ((16, 8, 32), (16, 8, 32), (), [0.3, -0.7, 0.1], None, 0.5, 3000, True),
    ((8, 8, 8), (4, 4, 4), (), [1.0, 0.0, 0.0], 0.5, 1.0, 50, False),
    ((6, 4, 4), (8, 4, 4), (), 0.0, None, 1.0, 200, False),  # local mesh smaller than global: drops
]


def _inputs(case, seed):
    ls, gs, chan, off, mcell, pcell, n, use_valid = case
    rng = np.random.default_rng(seed)
    pmid = rng.integers(0, min(gs), (n, 3)).astype(np.int16)
    disp = rng.uniform(-0.45, 0.45, (n, 3)).astype(np.float32) * np.float32(pcell)
    mesh = rng.normal(size=ls + chan).astype(np.float32)
    val = rng.normal(size=(n,) + chan).astype(np.float32)
    valid = (rng.random(n) > 0.3) if use_valid else None
    return pmid, disp, mesh, val, valid


@pytest.mark.parametrize("ci", range(len(CASES)))
def test_forward_and_adjoints_match_oracle(device, ci):
    case = CASES[ci]
    ls, gs, chan, off, mcell, pcell, n, _ = case
    pmid, disp, mesh, val, valid = _inputs(case, 17 + ci)
    tol = dict(rtol=3e-5, atol=3e-5) if mcell is not None else dict(rtol=2e-6, atol=2e-6)
    kw = dict(offset=off, particle_cell_size=pcell, cell_size=mcell, global_shape=gs)
    okw = dict(cell_size=pcell, mesh_shape=gs, offset=off, mesh_cell_size=mcell, valid=valid)
    vm = None if valid is None else _t(valid, device, torch.bool)
    P, D, M, V = _t(pmid, device, torch.int16), _t(disp, device), _t(mesh, device), _t(val, device)

    g = hip_gather(P, D, M, valid_mask=vm, **kw)
    np.testing.assert_allclose(_np(g), cic.gather(pmid, disp, mesh, **okw), **tol)

    base = np.ones(ls + chan, np.float32)
    s = hip_scatter(P, D, V, _t(base, device), valid_mask=vm, **kw)
    np.testing.assert_allclose(_np(s), cic.scatter(pmid, disp, val, base, **okw), **tol)

    vc = np.random.default_rng(5).normal(size=(n,) + chan).astype(np.float32)
    dcot, mcot = hip_gather_bwd(P, D, M, _t(vc, device), valid_mask=vm, **kw)
    dref, mref = cic.gather_adj(pmid, disp, mesh, vc, **okw)
    np.testing.assert_allclose(_np(dcot), dref, **tol)
    np.testing.assert_allclose(_np(mcot), mref, **tol)

    dcot, vcot = hip_scatter_bwd(P, D, V, M, valid_mask=vm, **kw)
    dref, vref = cic.scatter_adj(pmid, disp, val, mesh, **okw)
    np.testing.assert_allclose(_np(dcot), dref, **tol)
    np.testing.assert_allclose(_np(vcot), vref, **tol)

    # scalar value: scatter and the summed value cotangent
    s = hip_scatter(P, D, 1.7, _t(np.zeros(ls), device), valid_mask=vm, offset=off, particle_cell_size=pcell,
                    cell_size=mcell, global_shape=gs) if not chan else None
    if s is not None:
        np.testing.assert_allclose(_np(s), cic.scatter(pmid, disp, 1.7, np.zeros(ls), **okw), **tol)
        m0 = mesh if not chan else mesh[..., 0]
        _, vcs = hip_scatter_bwd(P, D, 1.7, _t(m0, device), valid_mask=vm, **kw)
        _, vref = cic.scatter_adj(pmid, disp, 1.7, m0, **okw)
        assert float(vcs) == pytest.approx(float(vref), rel=2e-5, abs=2e-5)


def test_empty_and_single_particle_edge_cases(device):
    kw = dict(offset=0.0, particle_cell_size=1.0, global_shape=(4, 4, 4))
    P = torch.zeros((0, 3), dtype=torch.int16, device=device)
    D = torch.zeros((0, 3), dtype=torch.float32, device=device)
    M = torch.ones((4, 4, 4), device=device)
    assert hip_gather(P, D, M, **kw).shape == (0,)
    assert torch.equal(hip_scatter(P, D, 1.0, M, **kw), M)
    # a particle exactly on a node puts all its mass there; gradients use sign(0) = 0
    P1 = torch.tensor([[1, 2, 3]], dtype=torch.int16, device=device)
    D1 = torch.zeros((1, 3), device=device)
    s = hip_scatter(P1, D1, 2.0, torch.zeros((4, 4, 4), device=device), **kw)
    assert float(s[1, 2, 3]) == 2.0 and float(s.sum()) == 2.0
    # periodic wrap: a particle at the last node spreads into node 0
    D2 = torch.tensor([[0.5, 0.0, 0.0]], device=device)
    P2 = torch.tensor([[3, 0, 0]], dtype=torch.int16, device=device)
    s = hip_scatter(P2, D2, 1.0, torch.zeros((4, 4, 4), device=device), **kw)
    assert float(s[3, 0, 0]) == pytest.approx(0.5) and float(s[0, 0, 0]) == pytest.approx(0.5)


def test_bad_arguments_raise(device):
    P = torch.zeros((3, 3), dtype=torch.int16, device=device)
    D = torch.zeros((3, 3), dtype=torch.float32, device=device)
    with pytest.raises(RuntimeError, match="float32"):
        hip_gather(P, D, torch.zeros((4, 4, 4), dtype=torch.float64, device=device), offset=0,
                   particle_cell_size=1.0, global_shape=(4, 4, 4))
    with pytest.raises(ValueError, match="valid_mask"):
        hip_gather(P, D, torch.zeros((4, 4, 4), device=device), offset=0, particle_cell_size=1.0,
                   global_shape=(4, 4, 4), valid_mask=torch.ones(2, dtype=torch.bool, device=device))
    with pytest.raises(ValueError, match="channel shape mismatch"):
        hip_scatter(P, D, torch.ones((3, 2), device=device), torch.zeros((4, 4, 4, 3), device=device), offset=0,
                    particle_cell_size=1.0, global_shape=(4, 4, 4))


# the tiled path: (mesh, n, spread in cells, invalid share, value kind); small bricks (8, 8, 16) up to
# 2^21 cells, (16, 16, 32) above; axes that are and are not powers of two; the smallest n
TILED = [
    ((48, 32, 64), 1 << 18, 0.4, 0.0, "normal"),
    ((8, 8, 16), (1 << 18) + 5, 3.0, 0.3, "normal"),
    ((24, 16, 48), (1 << 18) + 77, 9.0, 0.2, "scalar"),
    ((144, 128, 128), (1 << 18) + 1, 1.5, 0.1, "normal"),
    ((64, 32, 32), 1 << 18, 1.5, 0.0, "wide"),  # values 10^12 apart: the smaller ones take the atomics
    ((64, 32, 32), 1 << 18, 1.5, 0.1, "zero"),
]


@pytest.mark.parametrize("mesh_shape,n,spread,invalid,kind", TILED)
def test_tiled_scatter_and_gather_adjoint_match_oracle(device, mesh_shape, n, spread, invalid, kind):
    rng = np.random.default_rng(n + mesh_shape[0])
    cell = 0.75
    pmid = np.stack([rng.integers(-3, m + 3, n) for m in mesh_shape], 1).astype(np.int16)
    disp = (rng.uniform(-spread, spread, (n, 3)) * cell).astype(np.float32)
    val = (rng.choice([-1.0, 1.0], n) * rng.uniform(0.01, 2.0, n)).astype(np.float32)
    if kind == "wide":
        val[::1000] *= 1e12
    if kind == "zero":
        val[:] = 0
        val[::3] = 0.5
    valid = (rng.random(n) >= invalid) if invalid else None
    if valid is not None:
        val[~valid] = np.nan  # never read
    mesh = rng.normal(size=mesh_shape).astype(np.float32)
    v = 1.7 if kind == "scalar" else val
    okw = dict(cell_size=cell, mesh_shape=mesh_shape, valid=valid)
    kw = dict(offset=0.0, particle_cell_size=cell, global_shape=mesh_shape,
              valid_mask=None if valid is None else _t(valid, device, torch.bool))
    P, D, M = _t(pmid, device, torch.int16), _t(disp, device), _t(mesh, device)
    V = v if kind == "scalar" else _t(v, device)
    from pmpp_amd import _lib
    from pmpp_amd.cic.kernels import _geom, hip_scatter_new

    g = _geom(mesh_shape, mesh_shape, 0.0, cell, None)
    assert _lib.size_query("pm_cic_tiled_workspace", n, 1, g) > 0

    # a deposit's error: 3 axes x (fraction: 2^-24 (1 + |t|), weight and products: 2^-23) of |v|, atomics
    # another 2^-24 of the partial sum each; bounded through the sum of |v| over the touching particles
    ok = np.ones(n, bool) if valid is None else valid
    av = np.where(ok, np.abs(np.nan_to_num(v) if kind != "scalar" else np.full(n, v)), 0.0)
    t = disp.astype(np.float64) / cell
    base = pmid.astype(np.int64) + np.floor(disp / np.float32(cell)).astype(np.int64)
    touch = np.zeros(mesh_shape)
    cnt = np.zeros(mesh_shape)
    for c in range(8):
        ix = tuple((base[:, a] + ((c >> a) & 1)) % mesh_shape[a] for a in range(3))
        np.add.at(touch, ix, av)
        np.add.at(cnt, ix, av > 0)
    per = 3 * (2.0 ** -24 * (1 + spread) + 2.0 ** -23)
    bound = touch * (per + (cnt * 2.0 ** -24 if kind == "wide" else 0)) + 1e-30

    vo = np.nan_to_num(v) if kind != "scalar" else v
    ref = cic.scatter(pmid, disp, vo, np.zeros(mesh_shape), **okw)
    s0 = _np(hip_scatter_new(P, D, V, mesh_shape, **kw))
    assert np.all(np.abs(s0 - ref) <= bound + 2.0 ** -24 * np.abs(ref))
    s1 = _np(hip_scatter(P, D, V, M, **kw))
    assert np.all(np.abs(s1 - (ref + mesh)) <= bound + 2.0 ** -23 * (np.abs(ref) + np.abs(mesh)))
    if kind == "scalar":
        return
    dcot, mcot = hip_gather_bwd(P, D, M, V, **kw)
    dref, mref = cic.gather_adj(pmid, disp, mesh, vo, **okw)
    assert np.all(np.abs(_np(mcot) - mref) <= bound + 2.0 ** -24 * np.abs(mref))
    # eight mesh values of at most max|mesh| with weights of error per, over the cell size
    assert np.all(np.abs(_np(dcot) - dref) <= av[:, None] * np.abs(mesh).max() * 8 * per / cell + 1e-30)


def test_tiled_path_refuses_and_falls_back(device):
    from pmpp_amd import _lib
    from pmpp_amd.cic.kernels import _geom

    n = 1 << 18

    def need(n=n, c=1, ls=(64, 32, 32), gs=None, off=0.0, cell=None):
        return _lib.size_query("pm_cic_tiled_workspace", n, c, _geom(ls, gs or ls, off, 0.5, cell))

    assert need() > 0
    for kw in (dict(n=n - 1), dict(ls=(512, 512, 160)), dict(c=2), dict(ls=(64, 32, 24)), dict(ls=(60, 32, 32)), dict(gs=(128, 32, 32)),
               dict(off=[0.1, 0, 0]), dict(cell=0.5), dict(ls=(256, 256, 48))):
        assert need(**kw) == 0, kw

    # a value or a position that is not finite: the atomics' results, on the cells it touches only
    rng = np.random.default_rng(3)
    pmid = rng.integers(0, 32, (n, 3)).astype(np.int16)
    disp = rng.uniform(-0.4, 0.4, (n, 3)).astype(np.float32)
    val = rng.uniform(0.5, 1.0, n).astype(np.float32)
    kw = dict(offset=0.0, particle_cell_size=1.0, global_shape=(64, 32, 32))
    P, M = _t(pmid, device, torch.int16), torch.ones((64, 32, 32), device=device)
    for what in ("nan value", "inf value", "nan position"):
        d, v = disp.copy(), val.copy()
        if what == "nan position":
            d[11, 1] = np.nan
        else:
            v[11] = np.nan if what == "nan value" else np.inf
        D, V = _t(d, device), _t(v, device)
        plain = M.clone()
        g = _geom((64, 32, 32), (64, 32, 32), 0.0, 1.0, None)
        from pmpp_amd._torch import ptr, stream_handle
        _lib.call("pm_cic_scatter", ptr(P), ptr(D), None, ptr(V), 0.0, n, 1, g, ptr(plain), stream_handle(device))
        s = hip_scatter(P, D, V, M, **kw)
        # sums of at most ~100 float32 additions of values up to 1, in another order
        assert torch.equal(torch.isnan(s), torch.isnan(plain)), what
        assert torch.allclose(s, plain, rtol=100 * 2.0 ** -24, atol=100 * 2.0 ** -24, equal_nan=True), what
        dcot, mcot = hip_gather_bwd(P, D, M, V, **kw)
        bad = torch.isnan(dcot).any(1).nonzero().flatten().tolist()
        assert bad in ([], [11]) and not torch.isfinite(mcot).all(), what
    for vs in (0.0, float("inf"), 1e30):
        D = _t(disp, device)
        s = hip_scatter(P, D, vs, M, **kw)
        if vs == 0.0:
            assert torch.equal(s, M)
        else:
            assert not torch.isnan(s).any() and float(s.max()) > 1e29


@pytest.mark.parametrize("mesh_shape", [(128, 128, 128), (256, 128, 128)])  # small and large bricks
@pytest.mark.parametrize("outlier", [1.0, 2.0 ** 16, 2.0 ** 24, 2.0 ** 100])
def test_tiled_deposits_keep_their_own_precision(device, mesh_shape, outlier):
    """Every cell as good as the deposits in it, whatever the other values and however small its
    weights: against the float64 sum of the float32 deposits v W, to the roundings of the stored
    sum and of the three column planes a cell may get, 2^-24 of the sum of |v W| each."""
    rng = np.random.default_rng(int(np.log2(outlier)) + mesh_shape[0])
    n = 1 << 18
    pmid = np.stack(np.meshgrid(*[np.arange(0, m, 2) for m in mesh_shape], indexing="ij"), -1).reshape(-1, 3)
    pmid = pmid[rng.permutation(len(pmid))[:n]].astype(np.int16)
    disp = (0.05 * rng.normal(size=(n, 3))).astype(np.float32)
    val = (rng.choice([-1.0, 1.0], n) * rng.uniform(0.5, 1.0, n)).astype(np.float32)
    val[n // 3] *= np.float32(outlier)
    one = np.float32(1)
    lo = np.floor(disp)
    f = disp - lo
    w = (one - np.abs(f), one - np.abs(f - one))
    ref, absum = np.zeros(mesh_shape), np.zeros(mesh_shape)
    for c in range(8):
        b = [(c >> a) & 1 for a in range(3)]
        dep = val * (w[b[0]][:, 0] * w[b[1]][:, 1] * w[b[2]][:, 2])
        assert dep.dtype == np.float32
        ix = tuple((pmid[:, a] + lo[:, a].astype(np.int64) + b[a]) % mesh_shape[a] for a in range(3))
        np.add.at(ref, ix, dep.astype(np.float64))
        np.add.at(absum, ix, np.abs(dep).astype(np.float64))
    bound = 4 * 2.0 ** -24 * absum + 1e-44  # and of subnormal sums
    P, D, V = _t(pmid, device, torch.int16), _t(disp, device), _t(val, device)
    kw = dict(offset=0.0, particle_cell_size=1.0, global_shape=mesh_shape)
    M = torch.zeros(mesh_shape, device=device)
    for got in (hip_scatter(P, D, V, M, **kw), hip_gather_bwd(P, D, M, V, **kw)[1]):
        assert np.all(np.abs(_np(got) - ref) <= bound)
    if outlier == 1.0:
        s = _np(hip_scatter(P, D, float(val[0]), M, **kw))
        assert np.all(s[absum == 0] == 0) and s.sum() == pytest.approx(n * float(val[0]), rel=1e-6)


def test_calls_whose_tiled_workspace_does_not_fit_take_the_atomics(device, monkeypatch):
    from pmpp_amd.cic import kernels

    shape, n = (64, 32, 32), 1 << 18
    rng = np.random.default_rng(7)
    P = _t(rng.integers(0, 32, (n, 3)), device, torch.int16)
    D, V, M = (_t(rng.uniform(0.25, 0.75, s), device) for s in ((n, 3), (n,), shape))
    kw = dict(offset=0.0, particle_cell_size=1.0, global_shape=shape)

    def outputs():
        return (hip_scatter(P, D, V, M, **kw), kernels.hip_scatter_new(P, D, V, shape, **kw),
                kernels.hip_scatter_new(P, D, 0.5, shape, **kw), *hip_gather_bwd(P, D, M, V, **kw))

    tiled = outputs()

    def full(nbytes, dev):
        raise torch.cuda.OutOfMemoryError("no room for %d bytes" % nbytes)

    monkeypatch.setattr(kernels, "workspace", full)
    for a, b in zip(outputs(), tiled):
        # up to about 100 float32 additions of positive values in another order
        assert torch.allclose(a, b, rtol=100 * 2.0 ** -24, atol=1e-6)


@pytest.mark.parametrize("n,invalid", [((1 << 19) + 3, 0.0), ((1 << 19) + 3, 0.2), ((1 << 21) + 5, 0.1)])
def test_tiles_of_particles_in_no_grid_equal_the_plain_entry_points(device, n, invalid):
    """Particle counts that are no cube at the second and the largest chunk of the binning (index
    ranges), against the same float32 deposits added one by one with float atomics."""
    from pmpp_amd import _lib
    from pmpp_amd._torch import ptr, stream_handle
    from pmpp_amd.cic.kernels import _geom

    shape = (128, 144, 128)
    g = torch.Generator(device=device).manual_seed(n)
    P = torch.randint(0, 128, (n, 3), device=device, generator=g, dtype=torch.int16)
    D = torch.randn((n, 3), device=device, generator=g)
    V = torch.rand(n, device=device, generator=g) + 0.5
    M = torch.rand(shape, device=device, generator=g)
    ok = torch.rand(n, device=device, generator=g) >= invalid
    geo = _geom(shape, shape, 0.0, 1.0, None)
    assert _lib.size_query("pm_cic_tiled_workspace", n, 1, geo) > 0
    kw = dict(offset=0.0, particle_cell_size=1.0, global_shape=shape, valid_mask=ok)
    u8 = ok.to(torch.uint8)
    s = stream_handle(device)
    plain, mc, dc = M.clone(), torch.zeros_like(M), torch.empty_like(D)
    _lib.call("pm_cic_scatter", ptr(P), ptr(D), ptr(u8), ptr(V), 0.0, n, 1, geo, ptr(plain), s)
    _lib.call("pm_cic_gather_bwd", ptr(P), ptr(D), ptr(u8), n, 1, geo, ptr(M), ptr(V), ptr(dc), ptr(mc), s)
    got = hip_scatter(P, D, V, M, **kw)
    gdc, gmc = hip_gather_bwd(P, D, M, V, **kw)
    # positive sums of up to about 100 deposits, one rounding each
    assert torch.allclose(got, plain, rtol=100 * 2.0 ** -24, atol=0)
    assert torch.allclose(gmc, mc, rtol=100 * 2.0 ** -24, atol=0)
    # eight products of mesh values up to 1, weights of sum 4 and a cotangent up to 1.5, in another order
    assert torch.allclose(gdc, dc, rtol=0, atol=32 * 1.5 * 2.0 ** -24)


@pytest.mark.parametrize("mesh_shape,brick", [((128, 64, 64), (8, 8, 16)), ((256, 128, 128), (16, 16, 32))])
def test_tiled_gather_adjoint_of_bricks_of_every_count(device, mesh_shape, brick):
    """Bricks of no, one, and around 256, 512, 1024 and 2048 particles (a workgroup's threads and the
    rounds of four per thread), the rest anywhere: the displacement cotangent of the plain entry point."""
    from pmpp_amd import _lib
    from pmpp_amd._torch import ptr, stream_handle
    from pmpp_amd.cic.kernels import _geom

    rng = np.random.default_rng(mesh_shape[0])
    n, counts = 1 << 18, [0, 1, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4097]
    nb = [m // b for m, b in zip(mesh_shape, brick)]
    ids = np.repeat(np.arange(len(counts)) * 3, counts)  # every third brick of the first columns
    ids = np.concatenate([ids, rng.integers(3 * len(counts), np.prod(nb), n - len(ids))])
    corner = np.stack(np.unravel_index(ids, nb), 1) * np.array(brick)
    pmid = (corner + rng.integers(0, brick, (n, 3))).astype(np.int16)
    disp = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    order = rng.permutation(n)
    P, D = _t(pmid[order], device, torch.int16), _t(np.minimum(disp, np.float32(0.999))[order], device)
    V, M = _t(rng.normal(size=n), device), _t(rng.normal(size=mesh_shape), device)
    geo = _geom(mesh_shape, mesh_shape, 0.0, 1.0, None)
    assert _lib.size_query("pm_cic_tiled_workspace", n, 1, geo) > 0
    dc, mc = torch.empty_like(D), torch.zeros_like(M)
    _lib.call("pm_cic_gather_bwd", ptr(P), ptr(D), None, n, 1, geo, ptr(M), ptr(V), ptr(dc), ptr(mc),
              stream_handle(device))
    got, _ = hip_gather_bwd(P, D, M, V, offset=0.0, particle_cell_size=1.0, global_shape=mesh_shape)
    # eight products of a mesh value, two weights (sum 4 over the corners) and a cotangent, in another order
    scale = float(M.abs().max()) * V.abs()[:, None]
    assert torch.all((got - dc).abs() <= 32 * 2.0 ** -24 * scale)
