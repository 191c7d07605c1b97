"""Split-step lines in registers: every line length of both dimensions, so
every number of points a thread, lines a workgroup and remainder stage, against
the double-precision oracle; and several advances of a few steps against one of
their sum (first and last row passes).  Tolerances: a step rounds each value
about 3 log2 n times in double precision (2 transforms and the pointwise part),
so 4 steps stay within 4 * 36 * 2^-53 < 2e-14 of its scale; single-precision
storage rounds once a pass, 2 passes a step: 8 * 2^-24 < 5e-7; both are given a
factor of 10 for the norm's spread.
"""
import numpy as np
import pytest

from oracle import ssf_oracle as S
from test_ssf import rel, ssf_case

pytestmark = pytest.mark.gpu
STEPS = 4
TOL = {"f64": 2e-13, "f32": 5e-6}


@pytest.mark.parametrize("dtype,dyn", [("f64", True), ("f64", False), ("f32", True), ("f32", False)])
@pytest.mark.parametrize("dim,log2n", [(1, k) for k in range(4, 13)] + [(2, k) for k in range(4, 11)])
def test_every_length(gpu, dim, log2n, dtype, dyn):
    from nls_amd import native
    n, dt = 1 << log2n, 2e-3
    h, P, psi0, n0, c = ssf_case(dim, n, dyn)
    desc = native.ProblemDesc.make(dim, n, 5, dt, h, c, bc="periodic", dtype=dtype, scheme="ssf")
    psi, nres = native.solve_host(desc, STEPS, P, psi0, n0)
    opsi, onres = S.ssf(dim, n, h, dt, STEPS, P, c, psi0, n0)
    assert rel(psi, opsi) <= TOL[dtype], rel(psi, opsi)
    if dyn:
        assert rel(nres, onres) <= TOL[dtype]
    first = native.solve_host(desc, 1, P, psi0, n0)
    again = native.solve_host(desc, STEPS - 1, P, *first)
    assert rel(again[0], opsi) <= TOL[dtype]
    assert np.all(np.isfinite(again[0]))
