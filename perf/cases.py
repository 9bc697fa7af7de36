"""What a program built on this framework spends its time on: the cases its speed is measured on.

Every case is one call (or the forward and backward of one call) of a public entry point, with the
inputs such a program holds on the GPU when it makes it:

* ``force``      ``gravity``: the PM force on particles, once per stage of a run.  The hot path.
* ``force_vjp``  ``gravity`` and its reverse: the gradient of a loss on accelerations.
* ``nbody``      ``nbody``: a whole KDK run from early displacements and velocities.
* ``corrected``  ``gravity`` with the shipped learned correction, its potential channel included.
* ``network``    one pass of the correction's training: the network on a density mesh with its
                 activations kept, and the gradient of its parameters.
* ``pk``         ``density_to_pk`` / ``density_to_cross_correlation``: the run's measurement.
* ``cic``        ``scatter`` and ``gather`` with their gradients: the building blocks of a
                 program with a loss of its own.
* ``lpt``        ``lpt``: particles from linear modes, the start of every run.

Particles are a Lagrangian grid in its own order, displaced by a random field with a cold-dark-matter
like spectrum whose rms is ``growth`` particle spacings per axis: about 0.05 when a run starts, 1 to 3
when it ends.  ``slots`` says what the particles carry: no validity mask, one that is all valid (what
``Particles.gen_grid`` and so every run carries), or one with every 16th slot unused.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

DEV = "cuda"
OMEGA_M = 0.3


def _case(name, path, grid, mesh, cell, growth=1.0, slots="all", **more):
    c = {"name": name, "path": path, "g0": grid[0], "g1": grid[1], "g2": grid[2],
         "n0": mesh[0], "n1": mesh[1], "n2": mesh[2], "cell": cell, "growth": growth, "slots": slots}
    c.update(more)
    return c


def listed():
    return [
        # interactive and unit-test sized forces: launches and latency are what counts
        _case("force 32^3 on 64^3", "force", (32,) * 3, (64,) * 3, 1.0, growth=1.0),
        # the ordinary force of a small production run, mid-run state
        _case("force 128^3 on 256^3", "force", (128,) * 3, (256,) * 3, 1.0, growth=1.0),
        # a particle grid that is no power of two, with padding slots, as from an external catalogue
        _case("force 180^3 on 256^3", "force", (180,) * 3, (256,) * 3, 0.9765625, growth=2.0, slots="some"),
        # the headline workload: 512^3 particles, 1024^3 mesh, 1000 Mpc/h, final state
        _case("force 512^3 on 1024^3", "force", (512,) * 3, (1024,) * 3, 0.9765625, growth=3.0),
        # the gradient of a loss on accelerations, at the gradient workloads' small and large sizes
        _case("force vjp 64^3 on 128^3", "force_vjp", (64,) * 3, (128,) * 3, 1.0, growth=1.0),
        _case("force vjp 256^3 on 512^3", "force_vjp", (256,) * 3, (512,) * 3, 0.5, growth=2.0, slots="none"),
        # a whole run: 64^3 particles, 128^3 mesh, 128 Mpc/h, 10 KDK steps from a = 1/64 to 1
        _case("run 64^3 on 128^3", "nbody", (64,) * 3, (128,) * 3, 1.0, growth=0.03, steps=10),
        # the learned correction: the force of a corrected run, and a pass of its training
        _case("corrected 128^3 on 256^3", "corrected", (128,) * 3, (256,) * 3, 0.9765625, growth=1.0),
        _case("network 128^3", "network", (64,) * 3, (128,) * 3, 0.9765625),
        # the power spectrum of a run's final density
        _case("pk 256^3", "pk", (128,) * 3, (256,) * 3, 1.0, cross=False),
        # mass assignment and interpolation with their gradients
        _case("cic 128^3 on 256^3", "cic", (128,) * 3, (256,) * 3, 1.0, growth=1.0),
        # initial conditions of a run
        _case("lpt 128^3", "lpt", (128,) * 3, (256,) * 3, 1.0),
    ]


def draw(rng):
    path = rng.choice(["force", "force", "force", "force_vjp", "force_vjp", "nbody", "corrected", "network", "pk",
                       "cic", "lpt"])
    top = {"force": 9, "force_vjp": 8, "nbody": 8, "corrected": 8, "network": 7, "pk": 8, "cic": 8, "lpt": 8}[path]
    low = {"corrected": 6, "network": 6}.get(path, 5)
    e = rng.randint(low, top)
    mesh = [2 ** e] * 3
    if rng.random() < 0.4:  # a slab or a beam instead of a cube
        for a in range(3):
            mesh[a] = 2 ** max(low, e - rng.randint(0, 1))
    ratio = rng.choice([1, 2, 2, 4])
    grid = [m // ratio for m in mesh]
    # a particle grid of any size on a cubic mesh; the initial conditions are on power-of-two grids
    if len(set(mesh)) == 1 and path in ("force", "force_vjp", "cic") and rng.random() < 0.5:
        grid = [rng.randint(mesh[0] // 4, mesh[0])] * 3
    cell = rng.choice([0.5, 1.0, 2.0])
    slots = rng.choice(["none", "all", "all", "some"])
    growth = math.exp(rng.uniform(math.log(0.05), math.log(3.0)))
    more = {}
    if path == "nbody":
        more["steps"] = rng.randint(2, 10)
        growth, slots = 0.03, "all"
    if path == "pk":
        more["cross"] = rng.random() < 0.5
    c = _case("", path, grid, mesh, cell, growth, slots, **more)
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs ----


def _grid(c):
    return c["g0"], c["g1"], c["g2"]


def _mesh(c):
    return c["n0"], c["n1"], c["n2"]


def _spacing(c):
    return c["cell"] * c["n0"] / c["g0"]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _freq(shape):
    k = [2 * math.pi * torch.fft.fftfreq(n, device=DEV) for n in shape[:2]]
    k.append(2 * math.pi * torch.fft.rfftfreq(shape[2], device=DEV))
    return k[0][:, None, None], k[1][None, :, None], k[2][None, None, :]


def _modes(shape, gen):
    """Random modes of a density contrast with a cold-dark-matter like spectrum (grid units)."""
    k = _freq(shape)
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    amp = torch.sqrt(torch.sqrt(k2) / (1 + 64 * k2) ** 1.3)
    return torch.fft.rfftn(torch.randn(shape, generator=gen, device=DEV)) * amp, k, k2


def _displacements(shape, gen, rms):
    """(N, 3) displacements: the gradient of the inverse Laplacian of such a density, with that rms."""
    d, k, k2 = _modes(shape, gen)
    d = d / torch.where(k2 == 0, torch.ones_like(k2), k2)
    out = torch.empty(tuple(shape) + (3,), device=DEV)
    for a in range(3):
        out[..., a] = torch.fft.irfftn(1j * k[a] * d, s=shape)
    out = out.reshape(-1, 3)
    return out * (rms / out.square().mean().sqrt().clamp_min(1e-30))


def _lattice(c):
    """The particle grid's anchors (nearest mesh cells, int16) and what is left over, as displacements."""
    grid, mesh = _grid(c), _mesh(c)
    pm, dp = [], []
    for g, m in zip(grid, mesh):
        i = torch.arange(g, device=DEV, dtype=torch.float64)
        p = torch.round(i * m / g)
        pm.append(p.to(torch.int16))
        dp.append(((i * m - p * g) * (c["cell"] / g)).to(torch.float32))
    return [torch.stack(torch.meshgrid(*v, indexing="ij"), -1).reshape(-1, 3) for v in (pm, dp)]


def _inputs(c, seed):
    """pmid, disp and the unused slots (or None) of the particles."""
    gen = _gen(seed)
    pmid, disp = _lattice(c)
    disp = disp + _displacements(_grid(c), gen, c["growth"] * _spacing(c))
    unused = None
    if c["slots"] != "none":
        unused = torch.zeros(pmid.shape[0], dtype=torch.bool, device=DEV)
        if c["slots"] == "some":
            unused[::16] = True
    return pmid, disp.contiguous(), unused, gen


def _density(shape, gen, sigma=1.0):
    """A positive density mesh of mean 1: the exponential of a random field of that rms."""
    f = torch.fft.irfftn(_modes(shape, gen)[0], s=shape)
    f = torch.exp(f * (sigma / f.square().mean().sqrt()))
    return (f / f.mean()).contiguous()


def _conf(c, **more):
    from pmpp_amd import Configuration

    return Configuration(_spacing(c), _grid(c), mesh_shape=_mesh(c), **more)


def _mesh_inputs(c, seed):
    gen = _gen(seed)
    rho = _density(_mesh(c), gen)
    return rho, torch.randn(_mesh(c), generator=gen, device=DEV) / rho.numel() ** 0.5


def _lpt_modes(c, seed):
    d = _modes(_grid(c), _gen(seed))[0]
    psi = c["growth"] * _spacing(c)  # about that rms of displacement at a = 1
    vol = _spacing(c) ** 3
    return (d * (vol * psi / d.abs().square().mean().sqrt() * d.numel() ** 0.5 / 8)).contiguous()


def prepare(case, seed):
    from pmpp_amd import Particles
    from pmpp_amd.cosmology import LCDM

    c, path = case, case["path"]
    s = {"path": path, "case": c}
    if path in ("force", "force_vjp", "nbody", "corrected", "cic"):
        pmid, disp, unused, gen = _inputs(c, seed)
    if path == "nbody":
        a0 = 1 / 64
        s["conf"] = _conf(c, a_start=a0, a_nbody_maxstep=(1 - a0) / c["steps"])
        # velocities of the growing mode in matter domination: a^2 H dD/dlna = sqrt(Omega_m a)
        vel = disp * math.sqrt(OMEGA_M * a0)
        s["cosmo"] = LCDM(Omega_m=OMEGA_M)
        s["ptcl"] = Particles(s["conf"], pmid, disp, vel=vel, unused_index=unused)
        return s
    s["conf"] = _conf(c)
    if path in ("force", "corrected"):
        s["ptcl"] = Particles(s["conf"], pmid, disp, unused_index=unused)
        if path == "corrected":
            from pmpp_amd.corrections import load_correction

            s["model"] = load_correction(device=DEV)
    elif path == "force_vjp":
        s["disp"] = disp.requires_grad_(True)
        s["omega"] = torch.tensor(OMEGA_M, device=DEV, requires_grad=True)
        s["ptcl"] = Particles(s["conf"], pmid, s["disp"], unused_index=unused)
        s["cot"] = torch.randn(disp.shape, generator=gen, device=DEV)
    elif path == "cic":
        s["disp"] = disp.requires_grad_(True)
        s["ptcl"] = Particles(s["conf"], pmid, s["disp"], unused_index=unused)
        s["field"] = _density(_mesh(c), gen).requires_grad_(True)
        s["mesh_cot"] = torch.randn(_mesh(c), generator=gen, device=DEV)
        s["val_cot"] = torch.randn(disp.shape[0], generator=gen, device=DEV)
    elif path == "network":
        from pmpp_amd.corrections import load_correction

        s["model"] = load_correction(device=DEV)
        s["rho"], s["rho_cot"] = _mesh_inputs(c, seed)
    elif path == "pk":
        gen = _gen(seed)
        s["rho"] = _density(_mesh(c), gen)
        if c["cross"]:
            s["other"] = (0.8 * s["rho"] + 0.2 * _density(_mesh(c), gen)).contiguous()
    elif path == "lpt":
        s["cosmo"] = LCDM(Omega_m=OMEGA_M)
        s["modes"] = _lpt_modes(c, seed)
    return s


def run(state):
    path, conf = state["path"], state["conf"]
    if path == "force":
        from pmpp_amd import gravity

        return gravity(1.0, state["ptcl"], OMEGA_M, conf)
    if path == "force_vjp":
        from pmpp_amd import gravity

        acc = gravity(1.0, state["ptcl"], state["omega"], conf)
        disp_cot, omega_cot = torch.autograd.grad(acc, (state["disp"], state["omega"]), state["cot"])
        return acc.detach(), disp_cot, omega_cot
    if path == "nbody":
        from pmpp_amd.nbody.solver import nbody

        out = nbody(state["ptcl"], state["cosmo"], conf)
        return out.disp, out.vel, out.acc
    if path == "corrected":
        from pmpp_amd import gravity

        return gravity(0.5, state["ptcl"], OMEGA_M, conf, correction=state["model"])
    if path == "network":
        from pmpp_amd.corrections.mesh_cnn import evaluate_residual, residual_backward

        rho_add, tape = evaluate_residual(state["model"], state["rho"], 0.5, OMEGA_M, keep=True, conf=conf)
        return rho_add, residual_backward(state["model"], tape, state["rho_cot"])
    if path == "pk":
        from pmpp_amd.analysis import density_to_cross_correlation, density_to_pk

        if "other" in state:
            return density_to_cross_correlation(state["rho"], state["other"], conf)
        return density_to_pk(state["rho"], conf)
    if path == "cic":
        from pmpp_amd.cic import gather, scatter

        mesh = scatter(state["ptcl"], conf)
        vals = gather(state["ptcl"], conf, state["field"])
        grads = torch.autograd.grad((mesh, vals), (state["disp"], state["field"]), (state["mesh_cot"], state["val_cot"]))
        return (mesh.detach(), vals.detach()) + grads
    from pmpp_amd.initial_conditions import lpt

    p = lpt(state["modes"], state["cosmo"], conf)
    return p.pmid, p.disp, p.vel


def work(case):
    """Bytes: inputs read and outputs written once.  Operations: 2.5 N log2 N per real transform,
    about 60 per particle and interpolated field, 2 x 27 x inputs x outputs per cell and layer."""
    c, path = case, case["path"]
    n, m = math.prod(_grid(c)), math.prod(_mesh(c))
    mask = 0 if c["slots"] == "none" else 1
    fft = 2.5 * m * math.log2(m)
    part = n * (18 + mask)
    force = 4 * fft + 4 * 60 * n
    net = 2 * 27 * m * (2 * 16 + 16 * 16 + 16)
    if path == "force":
        return {"bytes": part + 12 * n, "flops": force}
    if path == "force_vjp":
        return {"bytes": part + 12 * n * 3, "flops": 2 * force}
    if path == "nbody":
        return {"bytes": part + 12 * n * 4, "flops": (c["steps"] + 1) * force}
    if path == "corrected":
        return {"bytes": part + 12 * n, "flops": force + 2 * fft + net}
    if path == "network":
        return {"bytes": 12 * m, "flops": 2 * fft + 3 * net}
    if path == "pk":
        k = 2 if c["cross"] else 1
        return {"bytes": 4 * m * k, "flops": k * fft + 10 * m}
    if path == "cic":
        return {"bytes": part + 12 * n + 8 * n + 4 * m * 4, "flops": 4 * 60 * n}
    g = math.prod(_grid(c))
    return {"bytes": 8 * g // 2 + 30 * g, "flops": 13 * 2.5 * g * math.log2(g)}


# ------------------------------------------------- the same in 64 bits ----

_CHUNK = 1 << 23


def _corners(pmid, disp, cell, mesh, grad=False):
    """For each of a chunk's 8 corners: flat cell index, weight and, with grad, d weight / d disp."""
    t = disp.double() / cell
    fl = torch.floor(t)
    base, f = pmid.long() + fl.long(), t - fl
    for b in range(8):
        bits = [(b >> a) & 1 for a in range(3)]
        idx = [torch.remainder(base[:, a] + bits[a], mesh[a]) for a in range(3)]
        w = [f[:, a] if bits[a] else 1 - f[:, a] for a in range(3)]
        flat = (idx[0] * mesh[1] + idx[1]) * mesh[2] + idx[2]
        g = None
        if grad:
            # d(1 - |f - b|) / df, 0 where a particle sits exactly on its cell
            sg = [1.0 if bits[a] else -(f[:, a] > 0).double() for a in range(3)]
            g = torch.stack((sg[0] * w[1] * w[2], sg[1] * w[0] * w[2], sg[2] * w[0] * w[1]), 1) / cell
        yield flat, w[0] * w[1] * w[2], g


def _chunks(n):
    return [slice(lo, min(n, lo + _CHUNK)) for lo in range(0, n, _CHUNK)]


def _scatter64(pmid, disp, val, cell, mesh):
    out = torch.zeros(math.prod(mesh), dtype=torch.float64, device=DEV)
    for s in _chunks(pmid.shape[0]):
        for flat, w, _ in _corners(pmid[s], disp[s], cell, mesh):
            out.index_add_(0, flat, w * val[s])
    return out.reshape(mesh)


def _gather64(pmid, disp, field, cell, mesh, grad=False):
    f = field.reshape(-1)
    out = torch.zeros((pmid.shape[0], 3) if grad else (pmid.shape[0],), dtype=torch.float64, device=DEV)
    for s in _chunks(pmid.shape[0]):
        for flat, w, g in _corners(pmid[s], disp[s], cell, mesh, grad):
            out[s] += f[flat][:, None] * g if grad else f[flat] * w
    return out


def _spectral64(c):
    """(mask * -1/k^2, the three -k with the Nyquist derivative zeroed) on the mesh's half spectrum."""
    mesh, cell, sp = _mesh(c), c["cell"], _spacing(c)
    k = [torch.fft.fftfreq(n, d=cell, dtype=torch.float64, device=DEV) * 2 * math.pi for n in mesh[:2]]
    k.append(torch.fft.rfftfreq(mesh[2], d=cell, dtype=torch.float64, device=DEV) * 2 * math.pi)
    shapes = ((-1, 1, 1), (1, -1, 1), (1, 1, -1))
    k2 = sum(x.reshape(s) ** 2 for x, s in zip(k, shapes))
    green = torch.where(k2 == 0, torch.zeros_like(k2), -1 / torch.where(k2 == 0, torch.ones_like(k2), k2))
    del k2
    if _grid(c) != mesh:
        lim = math.pi / sp * (1 + 8 * 1.2e-7)
        for x, s in zip(k, shapes):
            green *= (x.abs() <= lim).double().reshape(s)
    nyq = math.pi / cell
    neg = [torch.where((x.abs() - nyq).abs() <= 1e-6 * nyq, torch.zeros_like(x), -x).reshape(s)
           for x, s in zip(k, shapes)]
    return green, neg


def _valid64(c, n, unused):
    v = torch.ones(n, dtype=torch.float64, device=DEV)
    return v if unused is None else v * (~unused).double()


def _force64(c, pmid, disp, valid, rho_add=None, keep=False):
    mesh, cell = _mesh(c), c["cell"]
    val = valid * (math.prod(mesh) / math.prod(_grid(c)))
    rho = _scatter64(pmid, disp, val, cell, mesh)
    src = rho - 1 if rho_add is None else rho + rho_add(rho) - 1
    green, neg = _spectral64(c)
    pot = torch.fft.rfftn(src * (1.5 * OMEGA_M)) * green
    acc, comps = torch.empty((pmid.shape[0], 3), dtype=torch.float64, device=DEV), []
    for a in range(3):
        f = torch.fft.irfftn(1j * neg[a] * pot, s=mesh)
        acc[:, a] = _gather64(pmid, disp, f, cell, mesh) * valid
        if keep:
            comps.append(f)
    return acc, src, comps, green, neg


def _vjp64(c, pmid, disp, valid, cot):
    mesh, cell = _mesh(c), c["cell"]
    acc, src, comps, green, neg = _force64(c, pmid, disp, valid, keep=True)
    cot = cot.double() * valid[:, None]
    spec, out = 0, 0
    for a in range(3):
        out = out + _gather64(pmid, disp, comps[a], cell, mesh, grad=True) * cot[:, a:a + 1]
        spec = spec - 1j * neg[a] * green * torch.fft.rfftn(_scatter64(pmid, disp, cot[:, a], cell, mesh))
    src_cot = torch.fft.irfftn(spec, s=mesh)
    omega = 1.5 * (src_cot * src).sum()
    val = valid * (math.prod(mesh) / math.prod(_grid(c)))
    out = out + _gather64(pmid, disp, src_cot * (1.5 * OMEGA_M), cell, mesh, grad=True) * val[:, None]
    return acc, out, omega


_OFFSETS = [(dx, dy, dz) for dx in (-1, 0, 1) for dy in (-1, 0, 1) for dz in (-1, 0, 1)]


def _shift(x, off):
    return torch.roll(x, shifts=tuple(-o for o in off), dims=(0, 1, 2))


def _conv64(x, w, b):
    return sum(_shift(x, o) @ w[t].T for t, o in enumerate(_OFFSETS)) + b


def _gelu64(x, grad=False):
    u = math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)
    th = torch.tanh(u)
    if not grad:
        return 0.5 * x * (1 + th)
    return 0.5 * (1 + th) + 0.5 * x * (1 - th * th) * math.sqrt(2 / math.pi) * (1 + 3 * 0.044715 * x * x)


def _network64(c, rho, rho_cot=None, a=0.5):
    """rho_add of the shipped correction and, for rho_cot, its parameters' gradient (the layout of its
    parameter vector: per layer 27 x 16 x inputs weights, 16 biases, padded to 64; then the gain)."""
    import os

    import pmpp_amd

    where = os.path.join(os.path.dirname(pmpp_amd.__file__), "corrections", "weights", "mesh_cnn_2x_from_4x.npz")
    with np.load(where, allow_pickle=False) as z:
        p = torch.from_numpy(np.ascontiguousarray(z["params"])).to(DEV).double()
        big, s8 = float(z["max_residual"]), float(z["sigma8_value"])
    off, layers = 0, []
    for cin in (8, 16, 16):
        nw = 27 * 16 * cin
        layers.append((off, cin, p[off:off + nw].view(27, 16, cin), p[off + nw:off + nw + 16]))
        off = (off + nw + 16 + 63) // 64 * 64
    rho = rho.double()
    coef = 1.5 * OMEGA_M
    src = coef * (rho - 1)
    green, _ = _spectral64(c)
    phi = torch.fft.irfftn(torch.fft.rfftn(src) * green, s=_mesh(c))
    del green
    sigma, sp = (src.square().mean() + 1e-6).sqrt(), (phi.square().mean() + 1e-6).sqrt()
    x0 = torch.zeros(_mesh(c) + (8,), dtype=torch.float64, device=DEV)
    x0[..., 0], x0[..., 1] = src / sigma, phi / sp
    x0[..., 2], x0[..., 3], x0[..., 4] = a, OMEGA_M, s8
    cond = torch.tensor([a, OMEGA_M, s8, 1.0], dtype=torch.float64, device=DEV)
    th = torch.tanh((p[off:off + 4] * cond).sum())
    z1 = _conv64(x0, layers[0][2], layers[0][3])
    x1 = _gelu64(z1)
    z2 = _conv64(x1, layers[1][2], layers[1][3])
    x2 = _gelu64(z2)
    o = _conv64(x2, layers[2][2][:, :1], layers[2][3][:1])[..., 0]
    t = torch.tanh(o)
    amp = big * sigma / coef
    rho_add = big * th * (rho - 1) + amp * t
    if rho_cot is None:
        return rho_add
    rc = rho_cot.double()
    grads = torch.zeros_like(p)
    grads[off:off + 4] = cond * (big * (1 - th * th) * (rc * (rho - 1)).sum())
    dz = torch.zeros(_mesh(c) + (16,), dtype=torch.float64, device=DEV)
    dz[..., 0] = rc * amp * (1 - t * t)
    for (lo, cin, w, _), x, pre in zip(reversed(layers), (x2, x1, x0), (z2, z1, None)):
        flat = dz.reshape(-1, 16)
        gw = torch.stack([flat.T @ _shift(x, f).reshape(-1, cin) for f in _OFFSETS])
        grads[lo:lo + gw.numel()] = gw.reshape(-1)
        grads[lo + gw.numel():lo + gw.numel() + 16] = flat.sum(0)
        if pre is not None:
            dx = sum(_shift(dz, tuple(-q for q in f)) @ w[k] for k, f in enumerate(_OFFSETS))
            dz = dx * _gelu64(pre, grad=True)
    return rho_add, grads


def _pk64(c, rho, other=None):
    mesh, dim = _mesh(c), c["n0"]
    m = [torch.fft.fftfreq(n, 1 / n, dtype=torch.float64, device=DEV) for n in mesh[:2]]
    m.append(torch.fft.rfftfreq(mesh[2], 1 / mesh[2], dtype=torch.float64, device=DEV))
    m = [x.reshape(s) for x, s in zip(m, ((-1, 1, 1), (1, -1, 1), (1, 1, -1)))]
    mag = torch.sqrt(m[0] ** 2 + m[1] ** 2 + m[2] ** 2)
    shell = torch.floor(mag + 1e-6).long().reshape(-1)
    mult = torch.full_like(mag, 2.0)
    mult[..., 0] = mult[..., -1] = 1.0
    win = torch.sinc(m[0] / mesh[0]) * torch.sinc(m[1] / mesh[1]) * torch.sinc(m[2] / mesh[2])
    n = int(shell.max()) + 1
    top = math.floor(math.sqrt(3) * (dim // 2)) + 1  # shells of the measurement; the last takes the rest

    def sums(x, k=n):
        return torch.zeros(k, dtype=torch.float64, device=DEV).index_add_(0, shell.clamp_max(k - 1), x.reshape(-1))

    nmodes = sums(mult)
    k = (sums(mag * mult) / nmodes.clamp_min(1) * (2 * math.pi / (dim * c["cell"])))[1:]
    count = min(n - 1, top - 1)

    def finish(x):
        return sums(x * mult / win ** 4, top)[1:1 + count] / nmodes[1:1 + count] * (c["cell"] ** 3 / math.prod(mesh))

    a = torch.fft.rfftn(rho.double() / rho.double().mean())
    pa = finish(a.abs() ** 2)
    if other is None:
        return k[:count], pa, None
    b = torch.fft.rfftn(other.double() / other.double().mean())
    pb, pab = finish(b.abs() ** 2), finish((a * b.conj()).real)
    return k[:count], pab / torch.sqrt((pa * pb).clamp_min(1e-30)), pab, pa, pb, None


def _growth64(a):
    """D_m and a^2 H dD_m / dln a at a, m = 1, 2, of a flat universe with Omega_m (Runge-Kutta in ln a)."""
    def e2(x):
        return OMEGA_M * x ** -3 + 1 - OMEGA_M

    def f(t, g):
        x = math.exp(t)
        h, om = -1.5 * OMEGA_M * x ** -3 / e2(x), 1.5 * OMEGA_M * x ** -3 / e2(x)
        return np.array([g[1], -(3 + h - om) * g[0] - (4 + h) * g[1],
                         g[3], om * g[0] ** 2 - (8 + 2 * h - om) * g[2] - (6 + h) * g[3]])

    t, g, steps = math.log(3e-6), np.array([1.0, 0.0, 3 / 7, 0.0]), 2000
    h = (math.log(a) - t) / steps
    for _ in range(steps):
        k1 = f(t, g)
        k2 = f(t + h / 2, g + h / 2 * k1)
        k3 = f(t + h / 2, g + h / 2 * k2)
        k4 = f(t + h, g + h * k3)
        g, t = g + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4), t + h
    return [(a ** m * g[2 * m - 2], a ** 2 * math.sqrt(e2(a)) * a ** m * (m * g[2 * m - 2] + g[2 * m - 1]))
            for m in (1, 2)]


def _lpt64(c, modes):
    grid, sp = _grid(c), _spacing(c)
    k = [torch.fft.fftfreq(n, d=sp, dtype=torch.float64, device=DEV) * 2 * math.pi for n in grid[:2]]
    k.append(torch.fft.rfftfreq(grid[2], d=sp, dtype=torch.float64, device=DEV) * 2 * math.pi)
    k = [x.reshape(s) for x, s in zip(k, ((-1, 1, 1), (1, -1, 1), (1, 1, -1)))]
    nyq = math.pi / sp
    kz = [torch.where((x.abs() - nyq).abs() <= 1e-6 * nyq, torch.zeros_like(x), x) for x in k]
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    inv = torch.where(k2 == 0, torch.zeros_like(k2), -1 / torch.where(k2 == 0, torch.ones_like(k2), k2))
    back = functools.partial(torch.fft.irfftn, s=grid)
    pot = modes.to(torch.complex128) / sp ** 3 * inv
    d = [back(-k[i] ** 2 * pot) for i in range(3)]
    src = d[0] * d[1] + d[0] * d[2] + d[1] * d[2]
    for i, j in ((0, 1), (0, 2), (1, 2)):
        src -= back(-kz[i] * kz[j] * pot) ** 2
    pots = [pot, torch.fft.rfftn(src) * inv]
    pmid, disp = _lattice(c)
    disp, vel = disp.double(), torch.zeros(disp.shape, dtype=torch.float64, device=DEV)
    for p, (dm, vm) in zip(pots, _growth64(1 / 64)):
        for i in range(3):
            g = back(-1j * kz[i] * p).reshape(-1)
            disp[:, i] += dm * g
            vel[:, i] += vm * g
    return None, disp, vel


def exact(case, seed):
    """What ``run`` returns, in 64 bits.  A whole run has no such value here: its step factors are
    interpolated from a growth table of the framework's own."""
    c, path = case, case["path"]
    if path == "nbody":
        return None
    with torch.no_grad():
        if path in ("force", "force_vjp", "corrected", "cic"):
            pmid, disp, unused, gen = _inputs(c, seed)
            valid = _valid64(c, pmid.shape[0], unused)
        if path == "force":
            return _force64(c, pmid, disp, valid)[0]
        if path == "force_vjp":
            return _vjp64(c, pmid, disp, valid, torch.randn(disp.shape, generator=gen, device=DEV))
        if path == "corrected":
            return _force64(c, pmid, disp, valid, rho_add=lambda rho: _network64(c, rho))[0]
        if path == "cic":
            mesh, cell = _mesh(c), c["cell"]
            val = valid * (math.prod(mesh) / math.prod(_grid(c)))
            field = _density(mesh, gen).double()
            mc = torch.randn(mesh, generator=gen, device=DEV).double()
            vc = torch.randn(disp.shape[0], generator=gen, device=DEV).double() * valid
            dg = (_gather64(pmid, disp, mc, cell, mesh, grad=True) * val[:, None]
                  + _gather64(pmid, disp, field, cell, mesh, grad=True) * vc[:, None])
            return (_scatter64(pmid, disp, val, cell, mesh), _gather64(pmid, disp, field, cell, mesh) * valid, dg,
                    _scatter64(pmid, disp, vc, cell, mesh))
        if path == "network":
            return _network64(c, *_mesh_inputs(c, seed))
        if path == "pk":
            gen = _gen(seed)
            rho = _density(_mesh(c), gen)
            other = (0.8 * rho + 0.2 * _density(_mesh(c), gen)).contiguous() if c["cross"] else None
            return _pk64(c, rho, other)
        return _lpt64(c, _lpt_modes(c, seed))
