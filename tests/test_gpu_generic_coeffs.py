"""Lines in pieces, tiles of each form and several steps a launch against the
double-precision oracle, with coefficients none of which is 1 and no two equal:
equal bits of two kernels do not show a factor that both leave out.

Sizes: lines of one workgroup and of many; grids of one tile and of several,
below, at and past the largest that steps several times a launch.
"""
import numpy as np
import pytest

from nls_amd import native
from test_gpu_march import fields, generic_coeffs, with_form
from test_gpu_resident import TOL, check

pytestmark = pytest.mark.gpu
STEPS = 5
CASES = [(order, bc, dtype, dyn) for order in (3, 5, 7) for bc in ("periodic", "ref")
         for dtype in ("f32", "f64") for dyn in (True, False)]


def rounded(P, psi0, n0):
    """Inputs that single precision holds."""
    return P.astype(np.float32).astype(float), psi0.astype(np.complex64).astype(complex), \
        n0.astype(np.float32).astype(float)


@pytest.mark.parametrize("order,bc,dtype,dyn", CASES)
def test_lines(gpu, oracle, order, bc, dtype, dyn):
    for n in (order, 48, 385, 1000, 5000, 30011):
        rng = np.random.default_rng(n)
        r = 0.1 * np.arange(n)
        P, psi0, n0 = rounded(2.0 + np.sin(3.0 * r), 0.3 * np.cos(r) + 0.1j * rng.standard_normal(n),
                              0.2 + 0.1 * np.cos(r))
        c, n0 = generic_coeffs(dyn), n0 if dyn else None
        d = native.ProblemDesc.make(1, n, order, 5e-4, 0.1, c, bc=bc, dtype=dtype)
        check(native.solve_host(d, STEPS, P, psi0, n0),
              oracle.rk4(1, n, order, native.BC[bc], 5e-4, 0.1, STEPS, P, c, psi0, n0), dtype, n)


@pytest.mark.parametrize("order,bc,dtype,dyn", CASES)
def test_grids(gpu, oracle, order, bc, dtype, dyn):
    for n in (order, 40, 64, 65, 130, 180, 185, 256, 257):
        h, P, psi0, n0 = fields(n, n)
        P, psi0, n0 = rounded(P, psi0, n0)
        c, n0 = generic_coeffs(dyn), n0 if dyn else None
        want = oracle.rk4(2, n, order, native.BC[bc], 5e-4, h, STEPS, P, c, psi0, n0)
        d = native.ProblemDesc.make(2, n, order, 5e-4, h, c, bc=bc, dtype=dtype, engine="fused")
        for form in ("auto", "tall", "short", "half", "tall512"):
            check(with_form(dtype, form, lambda: native.solve_host(d, STEPS, P, psi0, n0)), want, dtype, (n, form))
        d = native.ProblemDesc.make(2, n, order, 5e-4, h, c, bc=bc, dtype=dtype, engine="stage")
        check(native.solve_host(d, STEPS, P, psi0, n0), want, dtype, (n, "stage"))
