"""Entry points of the C interface that the Python package itself does not call."""

import math

import numpy as np
import pytest
import torch

from pmpp_amd import _lib
from pmpp_amd._torch import ensure_init, ptr, stream_handle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 2, 2), (16, 8, 64), (4, 64, 1024)])
def test_inverse_transform_that_overwrites_its_input(device, shape):
    ensure_init(device)
    x = np.random.default_rng(sum(shape)).normal(size=shape)
    X = np.fft.rfftn(x).astype(np.complex64)
    spec, out = torch.from_numpy(X).to(device), torch.empty(shape, device=device)
    _lib.call("pm_irfft3d", ptr(spec), ptr(out), _lib.int3(shape), None, 0, stream_handle(device))
    ref = np.fft.irfftn(X.astype(np.complex128), s=shape, axes=(0, 1, 2))
    np.testing.assert_allclose(out.cpu().numpy(), ref, atol=3e-6 * math.log2(x.size))  # values of order one


@pytest.mark.parametrize("n,vel", [(1, True), (1000, False), (70001, True)])
def test_lpt_accumulate_adds_one_component(device, n, vel):
    rng = np.random.default_rng(n)
    d, v, g = (rng.normal(size=s).astype(np.float32) for s in ((n, 3), (n, 3), (n,)))
    for axis in range(3):
        D, V = torch.from_numpy(d).to(device), torch.from_numpy(v).to(device)
        G = torch.from_numpy(g).to(device)
        _lib.call("pm_ic_lpt_accumulate", ptr(D), ptr(V) if vel else None, ptr(G), n, axis, 0.7, -1.3,
                  stream_handle(device))
        for got, old, f in ((D, d, 0.7), (V, v, -1.3 if vel else 0.0)):
            want = old.astype(np.float64)
            want[:, axis] += np.float64(np.float32(f)) * g
            # a product and a sum in float32
            bound = 2.0 ** -23 * (np.abs(old) + abs(f) * np.abs(g)[:, None])
            assert np.all(np.abs(got.cpu().numpy() - want) <= bound)


@pytest.mark.parametrize("n", [512, 4096 + 8])
def test_residual_gradient_in_sixteen_channels_is_the_one_channel_one_padded(device, n):
    g = torch.Generator().manual_seed(n)
    rc, out, rho = (torch.randn(n, generator=g).to(device) for _ in range(3))
    stats = torch.tensor([1.3, 0.4, 0.2, 0.9], device=device)
    ws = torch.empty(_lib.size_query("pm_correction_workspace"), dtype=torch.uint8, device=device)
    res = []
    for ch in (1, 16):
        dz, gain = torch.full((n, ch), 7.0, device=device), torch.empty(4, device=device)
        _lib.call("pm_correction_residual_bwd", ptr(rc), ptr(out), ptr(rho), n, 0.3, 0.5, 0.8, 0.25, ptr(stats),
                  ptr(dz), ch, ptr(gain), ptr(ws), ws.numel(), stream_handle(device))
        res.append((dz, gain))
    (d1, g1), (d16, g16) = res
    assert torch.equal(d16[:, 0], d1[:, 0]) and torch.equal(g16, g1)
    assert float(d1.abs().max()) > 0 and not d16[:, 1:].any()
