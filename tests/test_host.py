"""Host-side logic: configuration geometry and spectral caches vs the oracle."""

import numpy as np
import pytest

from oracle import spectral
from pmpp_amd import Configuration


def test_configuration_geometry_and_validation():
    conf = Configuration(1000 / 512, (512,) * 3, mesh_shape=2)
    assert conf.mesh_shape == (1024,) * 3
    assert conf.cell_size == pytest.approx(1000 / 1024)
    assert conf.mesh_size == 1024 ** 3 and conf.ptcl_num == 512 ** 3
    assert conf.brick == (16, 16, 32)
    with pytest.raises(ValueError, match="cannot be smaller"):
        Configuration(1.0, (8, 8, 8), mesh_shape=(4, 8, 8))
    with pytest.raises(ValueError, match="aspect ratios"):
        Configuration(1.0, (8, 8, 8), mesh_shape=(16, 8, 8))
    with pytest.raises(ValueError, match="symplectic"):
        Configuration(1.0, (8, 8, 8), symp_splits=((0, 0.5), (1, 0.6)))


@pytest.mark.parametrize("ratio", [1, 2, 4])
def test_spectral_caches_match_oracle(ratio):
    conf = Configuration(2.0, (8, 8, 8), mesh_shape=ratio)
    for a, k in enumerate(conf.kvec):
        np.testing.assert_allclose(k, spectral.kvec(conf.mesh_shape, conf.cell_size)[a].astype(np.float32))
    masks = spectral.particle_nyquist_masks(conf.mesh_shape, conf.ptcl_grid_shape, conf.ptcl_spacing,
                                            conf.cell_size)
    assert len(conf.particle_nyquist_masks) == len(masks)
    for m, mo in zip(conf.particle_nyquist_masks, masks):
        np.testing.assert_array_equal(m, mo)
    for a, nik in enumerate(conf.neg_ik):
        np.testing.assert_allclose(nik.imag, spectral.neg_k(conf.mesh_shape, conf.cell_size)[a], rtol=1e-6)


def test_nbody_schedule():
    conf = Configuration(2.0, (8, 8, 8), a_start=1 / 64, a_stop=1.0, a_nbody_maxstep=(1 - 1 / 64) / 10)
    a = conf.a_nbody
    assert len(a) == 11 and a[0] == pytest.approx(1 / 64) and a[-1] == pytest.approx(1.0)


def test_step_factors_match_the_oracle():
    # host float64 growth table (Dormand-Prince) vs the oracle's (scipy DOP853), same nodes
    import numpy as np
    from oracle import cosmology as oc
    from pmpp_amd import Configuration
    from pmpp_amd.initial_conditions import LCDM
    from pmpp_amd.nbody import integrator

    conf = Configuration(2.0, (8, 8, 8), mesh_shape=2)
    for cos in (LCDM(), LCDM(Omega_m=0.25, Omega_k=0.05, w_0=-0.9, w_a=0.1)):
        kw = dict(Ok=cos.Omega_k, w0=cos.w_0, wa=cos.w_a)
        t = oc.growth_table(conf.growth_a, cos.Omega_m, conf.a_lpt_step, **kw)
        for a0, a1 in zip(conf.a_nbody[:-1], conf.a_nbody[1:]):
            am = 0.5 * (a0 + a1)
            d = oc.drift_factor(am, a0, a1, t, conf.growth_a, cos.Omega_m, **kw)
            k = oc.kick_factor(a0, a0, am, t, conf.growth_a, cos.Omega_m, **kw)
            assert integrator.drift_factor(am, a0, a1, cos, conf) == pytest.approx(d, rel=1e-9)
            assert integrator.kick_factor(a0, a0, am, cos, conf) == pytest.approx(k, rel=1e-9)
    assert np.isclose(integrator._factor_dOm("kick_factor", 0.5, 0.5, 0.55, LCDM(), conf),
                      (integrator.kick_factor(0.5, 0.5, 0.55, LCDM(Omega_m=0.30001), conf)
                       - integrator.kick_factor(0.5, 0.5, 0.55, LCDM(Omega_m=0.29999), conf)) / 2e-5, rtol=1e-5)


def test_correction_parameter_layout_and_initialisation():
    import math

    import torch

    from pmpp_amd.corrections.mesh_cnn import initial_params, param_layout

    for depth, block, nconv in [(1, "residual", 2), (2, "residual", 4), (4, "residual", 8), (2, "plain", 3),
                                (4, "plain", 5)]:
        layers, gain, total = param_layout(depth, block)
        assert [L.name for L in layers][0] == "stem" and layers[-1].name == "out"
        assert len(layers) == nconv
        ends = [L.offset + L.size for L in layers]
        # 64-element alignment (16-byte aligned bf16 weights and float32 biases), no overlap
        assert all(L.offset % 64 == 0 for L in layers) and gain % 64 == 0
        assert all(e <= nxt.offset for e, nxt in zip(ends, layers[1:])) and ends[-1] <= gain
        assert total >= gain + 4
    layers, gain, total = param_layout(2)
    p = initial_params(seed=3, depth=2)
    assert p.shape == (total,)
    out = layers[-1]
    assert torch.all(p[out.offset:out.offset + out.size] == 0)  # zero output layer: zero residual
    stem = p[:layers[0].nweights].view(27, 16, 8)
    assert torch.all(stem[:, :, 4:] == 0)  # padding input channels
    std = math.sqrt(1 / (27 * 4)) / 0.87962566103423978
    assert stem[:, :, :4].abs().max() <= 2 * std + 1e-7
    assert abs(float(stem[:, :, :4].std()) - math.sqrt(1 / (27 * 4))) < 0.1 * math.sqrt(1 / (27 * 4))
    conv1 = p[layers[1].offset:layers[1].offset + layers[1].nweights]
    assert abs(float(conv1.std()) - math.sqrt(1 / (27 * 16))) < 0.05 * math.sqrt(1 / (27 * 16))
    assert torch.all(p[layers[0].nweights:layers[0].size] == 0)  # zero biases
    assert 0 < float(p[gain:gain + 3].abs().max()) < 0.05 and p[gain + 3] == 0


def test_validity_mask_is_converted_once_per_mask_and_follows_in_place_changes():
    """The force step's uint8 validity mask (1 = valid) is the negation of ``unused_index``; it
    is converted once while the same mask tensor is passed unchanged (an N-body run carries one
    mask through every step), again after an in-place change, and separately for another mask."""
    import gc
    from types import SimpleNamespace

    import torch

    from pmpp_amd.nbody.gravity import _VALID_MASKS, _valid_u8

    ui = torch.tensor([False, True, False, False])
    p = SimpleNamespace(unused_index=ui, pmid=torch.zeros(4, 3, dtype=torch.int16))
    first = _valid_u8(p)
    assert first.dtype == torch.uint8 and first.tolist() == [1, 0, 1, 1]
    assert _valid_u8(p) is first
    ui[3] = True
    changed = _valid_u8(p)
    assert changed is not first and changed.tolist() == [1, 0, 1, 0]
    other = SimpleNamespace(unused_index=ui.clone(), pmid=p.pmid)
    assert _valid_u8(other) is not changed and _valid_u8(other).tolist() == [1, 0, 1, 0]
    assert _valid_u8(SimpleNamespace(unused_index=None, pmid=p.pmid)) is None
    with pytest.raises(ValueError, match="unused_index has shape"):
        _valid_u8(SimpleNamespace(unused_index=ui[:2], pmid=p.pmid))
    n = len(_VALID_MASKS)
    del p, other, ui, first, changed
    gc.collect()
    assert len(_VALID_MASKS) < n  # entries go with their masks


@pytest.mark.parametrize("kw", [{}, dict(Omega_k=0.05, w_0=-0.9, w_a=0.2), dict(w_a=-0.3)])
def test_step_factors_of_floats_equal_the_array_functions(kw):
    from pmpp_amd.cosmology import LCDM, GrowthTable

    conf = Configuration(1.0, (8,) * 3)
    t = GrowthTable(LCDM(Omega_m=0.3, **kw), conf.growth_a, conf.a_lpt_step)
    nodes = t.growth_a
    scales = np.concatenate((nodes[1:], 0.5 * (nodes[1:-1] + nodes[2:]), [1.5 * nodes[-1], 0.3 * nodes[1]]))
    for a in scales:
        for b in (a + 0.01, 1.1 * a):
            v = 0.5 * (a + b)
            d = (t.growth(b) - t.growth(a)) / t.G_D(v)
            k = (t.G_D(b) - t.G_D(a)) / t.G_K(v)
            # differences of numbers up to (a, a^2) / (b - a) times larger, each to a few 2^-52
            tol = 64 * 2.0 ** -52 * b / (b - a)
            assert t.drift_factor(v, a, b) == pytest.approx(float(d), rel=tol)
            assert t.kick_factor(v, a, b) == pytest.approx(float(k), rel=tol)
            assert np.float32(t.drift_factor(v, a, b)) == pytest.approx(np.float32(d), rel=2.0 ** -23)
    with np.errstate(all="ignore"):  # a scale factor that Python's arithmetic refuses: as the arrays have it
        assert np.isnan(t.drift_factor(0.0, 0.0, 0.1)) and np.isnan(t.kick_factor(0.1, 0.0, 0.1))


def test_growth_tables_are_kept_per_schedule():
    from pmpp_amd.cosmology import LCDM
    from pmpp_amd.nbody.integrator import growth_table

    cosmo = LCDM(Omega_m=0.31)
    a, b = (Configuration(1.0, (8,) * 3, a_nbody_maxstep=s) for s in (1 / 8, 1 / 16))
    assert growth_table(cosmo, a) is growth_table(cosmo, a.replace(ptcl_spacing=2.0))
    assert growth_table(cosmo, a) is not growth_table(cosmo, b)
    for c in (a, b, a.replace(a_custom=(0.1, 0.4, 1.0))):
        assert np.array_equal(growth_table(cosmo, c).growth_a, c.growth_a)


def test_particles_replace_converts_and_refuses_as_the_constructor():
    import torch

    from pmpp_amd import Particles

    p = Particles(None, torch.zeros(4, 3, dtype=torch.int16), torch.zeros(4, 3))
    q = p.replace(vel=torch.ones(4, 3, dtype=torch.float64), unused_index=torch.ones(4, dtype=torch.uint8))
    assert q.vel.dtype == torch.float32 and q.unused_index.dtype == torch.bool
    assert q.pmid is p.pmid and q.disp is p.disp and p.vel is None
    assert q.replace(vel=None, pmid=torch.zeros(4, 3)).vel is None
    with pytest.raises(TypeError):
        p.replace(velocity=q.vel)


def test_lazy_views_are_written_out_for_the_kernels(monkeypatch):
    import ctypes

    import torch

    from pmpp_amd import _torch

    monkeypatch.setattr(_torch, "require_device", lambda t, name: t)
    z = torch.complex(torch.arange(6.0).view(2, 3), 1.0 + torch.arange(6.0).view(2, 3))
    for t, dtype in ((z.conj(), torch.complex64), (z.conj().T, torch.complex64), (z, torch.complex64),
                     (torch._neg_view(z.real.clone()), torch.float32), (z.conj().imag, torch.float32)):
        got = _torch.as_contig(t, dtype, "t")
        want = t.resolve_conj().resolve_neg().contiguous()
        # what a kernel reads through the pointer
        raw = ctypes.string_at(got.data_ptr(), got.numel() * got.element_size())
        assert raw == want.numpy().tobytes()
    assert _torch.as_contig(z, torch.complex64, "z") is z  # nothing to do: no copy


def test_the_particle_grid_is_made_on_the_device_it_is_asked_for(monkeypatch):
    # a default stream's handle is 0 on every device, so the launch goes to the current one
    import torch

    from pmpp_amd import Particles, _lib, _torch

    current, launched = ["cuda:0"], []

    class Device:
        def __init__(self, dev):
            self.dev = str(dev)

        def __enter__(self):
            current.append(self.dev)

        def __exit__(self, *exc):
            current.pop()

    def on_cpu(f):
        return lambda *a, device=None, **kw: f(*a, **kw)

    for name in ("empty", "zeros"):
        monkeypatch.setattr(torch, name, on_cpu(getattr(torch, name)))
    monkeypatch.setattr(torch.cuda, "device", Device)
    monkeypatch.setattr(_torch, "stream_handle", lambda dev: None)
    monkeypatch.setattr(_lib, "call", lambda name, *a: launched.append((name, current[-1])))
    p = Particles.gen_grid(Configuration(1.0, (4, 4, 4)), vel=True, device="cuda:1")
    assert len(p) == 64 and launched == [("pm_ic_lpt_particles", "cuda:1")] and current == ["cuda:0"]
