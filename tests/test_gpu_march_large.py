"""The marching kernel past 2048 points a side, up to the largest grids whose
byte offsets it takes (11585 in double and 16383 in single precision): the same
bits as the tile kernel."""
import pytest

from nls_amd import native
from test_gpu_march import generic_coeffs, with_form

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dtype,dyn", [(4100, "f32", True), (4100, "f64", False), (11585, "f64", True),
                                         (16383, "f32", False)])
def test_equals_tiles(gpu, n, dtype, dyn):
    import torch
    torch.manual_seed(n)
    rt, ct = (torch.float64, torch.complex128) if dtype == "f64" else (torch.float32, torch.complex64)
    d = native.ProblemDesc.make(2, n, 5, 1e-4, 0.1, generic_coeffs(dyn), bc="periodic", dtype=dtype, engine="fused")
    P = torch.rand((n, n), dtype=rt, device=gpu)
    psi0 = torch.randn((n, n), dtype=ct, device=gpu)
    n0 = torch.rand((n, n), dtype=rt, device=gpu) if dyn else None

    def run():
        psi, nres = psi0.clone(), n0.clone() if dyn else None
        ws = torch.empty(native.workspace_bytes(d), dtype=torch.uint8, device=gpu)
        native.advance(d, 2, P, psi, nres, ws)
        return psi, nres

    march, tall = with_form(dtype, "auto", run), with_form(dtype, "tall", run)
    assert torch.isfinite(torch.view_as_real(march[0])).all()
    assert torch.equal(march[0], tall[0])
    if dyn:
        assert torch.equal(march[1], tall[1])
