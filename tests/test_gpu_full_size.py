"""512^3 particles on a 1024^3 mesh against operators that neither bin nor tile.

The force step, its VJP and the tiled CIC entry points share the binning and the brick tiles, so here
the reference side scatters and gathers through the plain entry points: one thread per particle in the
caller's order, float atomics.
"""

import numpy as np
import pytest
import torch

from pmpp_amd import Configuration, _lib, gravity
from pmpp_amd._torch import ptr, stream_handle
from pmpp_amd.cic.kernels import _geom, hip_gather, hip_gather_bwd, hip_scatter, hip_scatter_bwd
from pmpp_amd.initial_conditions import LCDM, particles_2lpt
from pmpp_amd.nbody.gravity import gravity_desc, gravity_vjp
from pmpp_amd.numerics import irfftn, rfftn, spectral_force_multiply

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a - b).norm() / b.norm())


def test_step_vjp_and_tiled_cic_against_the_plain_cic(device):
    conf = Configuration(1000.0 / 512, (512,) * 3, mesh_shape=2)
    cos = LCDM()
    omega, shape = cos.Omega_m, tuple(conf.mesh_shape)
    ptcl = particles_2lpt(conf, cos, seed=0, jitter_seed=1, device=device, a=1.0)
    n, val = len(ptcl), float(conf.mesh_size / conf.ptcl_num)
    P, D = ptcl.pmid, ptcl.disp
    geo = _geom(shape, shape, 0.0, conf.cell_size, None)
    kw = dict(offset=0.0, particle_cell_size=conf.cell_size, global_shape=shape)
    s = stream_handle(device)
    desc = gravity_desc(conf, omega)
    assert _lib.size_query("pm_cic_tiled_workspace", n, 1, geo) > 0

    rho = torch.zeros(shape, device=device)
    _lib.call("pm_cic_scatter", ptr(P), ptr(D), None, None, val, n, 1, geo, ptr(rho), s)
    tiled = hip_scatter(P, D, val, torch.zeros(shape, device=device), **kw)
    # an addition per particle that touches the cell, 2^-24 of the sum each; a few hundred at most in rms
    print(f"tiled vs plain scatter {_rel(tiled, rho):.2e}", flush=True)
    assert _rel(tiled, rho) < 1e-6
    del tiled

    shat = rfftn((rho - 1.0) * np.float32(1.5 * omega))
    comps = [irfftn(spectral_force_multiply(shat, desc, i), s=shape) for i in range(3)]
    del shat
    acc = torch.stack([hip_gather(P, D, f, **kw) for f in comps], dim=1)
    err = _rel(gravity(1.0, ptcl, omega, conf), acc)
    print(f"force vs the plain chain {err:.2e}", flush=True)
    assert err < 1e-5
    del acc

    cot = torch.randn(D.shape, device=device, generator=torch.Generator(device=device).manual_seed(3))
    d_fused, o_fused = gravity_vjp(ptcl, cos, conf, cot)
    d_ref, src = torch.zeros_like(D), torch.zeros(shape, device=device)
    for i in range(3):
        c = cot[:, i].contiguous()
        dc, mc = torch.empty_like(D), torch.zeros(shape, device=device)
        _lib.call("pm_cic_gather_bwd", ptr(P), ptr(D), None, n, 1, geo, ptr(comps[i]), ptr(c), ptr(dc), ptr(mc), s)
        if i == 0:
            tdc, tmc = hip_gather_bwd(P, D, comps[i], c, **kw)
            print(f"tiled vs plain gather adjoint {_rel(tmc, mc):.2e} {_rel(tdc, dc):.2e}", flush=True)
            assert _rel(tmc, mc) < 1e-6 and _rel(tdc, dc) < 1e-6
            del tdc, tmc
        d_ref += dc
        src += irfftn(spectral_force_multiply(rfftn(mc), desc, i, adjoint=True), s=shape)
        del dc, mc
    del comps
    o_ref = 1.5 * float((src.double() * (rho.double() - 1.0)).sum())
    d_ref += hip_scatter_bwd(P, D, val, src * np.float32(1.5 * omega), **kw)[0]
    err = _rel(d_fused, d_ref)
    print(f"VJP vs the plain chain {err:.2e}, Omega_m {o_fused:.6e} {o_ref:.6e}", flush=True)
    assert err < 1e-5 and o_fused == pytest.approx(o_ref, rel=1e-5)
