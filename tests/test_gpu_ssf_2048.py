"""Split-step at 2048^2, whose row, column, first and last passes have kernels
of their own: several steps in one call and in two against the oracle.

Tolerances: a step rounds each value about 3 log2 n times in double precision
(2 transforms and the pointwise part), so 4 steps stay within 4 * 36 * 2^-53 <
2e-14 of its scale; single-precision storage rounds once a pass, 2 passes a
step: 8 * 2^-24 < 5e-7; both are given a factor of 10 for the norm's spread.
"""
import numpy as np
import pytest

from oracle import ssf_oracle as S
from test_gpu_march import generic_coeffs
from test_ssf import rel, ssf_case

pytestmark = pytest.mark.gpu
STEPS = 4
TOL = {"f64": 2e-13, "f32": 5e-6}


@pytest.mark.parametrize("dyn", [True, False])
def test_general_field(gpu, dyn):
    from nls_amd import native
    n, dt = 2048, 2e-3
    h, P, psi0, n0, _ = ssf_case(2, n, dyn)
    c = generic_coeffs(dyn)
    opsi, onres = S.ssf(2, n, h, dt, STEPS, P, c, psi0, n0)
    for dtype in ("f64", "f32"):
        desc = native.ProblemDesc.make(2, n, 5, dt, h, c, bc="periodic", dtype=dtype, scheme="ssf")
        whole = native.solve_host(desc, STEPS, P, psi0, n0)
        first = native.solve_host(desc, 1, P, psi0, n0)
        for psi, nres in (whole, native.solve_host(desc, STEPS - 1, P, *first)):
            assert rel(psi, opsi) <= TOL[dtype]
            if dyn:
                assert rel(nres, onres) <= TOL[dtype]
