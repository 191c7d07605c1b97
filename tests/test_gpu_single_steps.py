"""Calls of one step, whose state ends in the workspace and is copied back:
four of them give the bits of one call of four steps, which needs no copy.

Sizes on both sides of the copy kernel's limit of 65,536 points, lines of one
workgroup and of many.
"""
import numpy as np
import pytest

from nls_amd import native
from test_gpu_march import generic_coeffs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("bc,dyn", [("periodic", True), ("periodic", False), ("ref", True), ("ref", False)])
@pytest.mark.parametrize("dim,n", [(1, 5), (1, 255), (1, 1000), (1, 1921), (1, 4096), (1, 65536), (1, 65537), (2, 41),
                                   (2, 64), (2, 65), (2, 256), (2, 257)])
def test_four_calls_equal_one(gpu, dim, n, dtype, bc, dyn):
    import torch
    rng = np.random.default_rng(n)
    shape = (n,) * dim
    psi0 = 0.3 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
    rt, ct = (torch.float64, torch.complex128) if dtype == "f64" else (torch.float32, torch.complex64)
    d = native.ProblemDesc.make(dim, n, 5, 5e-4, 0.1, generic_coeffs(dyn), bc=bc, dtype=dtype)
    P = torch.from_numpy(1.0 + rng.random(shape)).to(gpu, rt)
    n0 = torch.from_numpy(rng.random(shape)).to(gpu, rt)
    ws = torch.empty(max(1, native.workspace_bytes(d)), dtype=torch.uint8, device=gpu)
    out = []
    for calls in (1, 4):
        psi, nres = torch.from_numpy(psi0).to(gpu, ct), n0.clone() if dyn else None
        for _ in range(calls):
            native.advance(d, 4 // calls, P, psi, nres, ws)
        out.append((psi.cpu().numpy(), nres.cpu().numpy() if dyn else None))
    assert np.isfinite(out[0][0]).all()
    np.testing.assert_array_equal(out[1][0], out[0][0])
    if dyn:
        np.testing.assert_array_equal(out[1][1], out[0][1])
