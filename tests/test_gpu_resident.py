"""The resident engine in 2-D (one workgroup per grid of up to 64 points a
side) against the double-precision oracle, with coefficients none of which is 1
and no two equal.

Sizes: the stencil width, and the first and last grid of each number of points
a thread (1, 2, 3 and 4 in single precision, 1, 2, 5, 6 and 8 in double), alone
and in batches of more grids than the device has compute units.
"""
import numpy as np
import pytest

from nls_amd import native
from nls_amd.batch import Batch
from test_gpu_march import fields, generic_coeffs

pytestmark = pytest.mark.gpu
STEPS = 5
# A step rounds a value some 60 times at its scale: 5 steps stay within 300 *
# 2^-53 and 300 * 2^-24; double precision is given a factor of 10 for the growth
# of earlier errors.
TOL = {"f64": 3.3e-13, "f32": 1.8e-5}
CASES = [(order, bc, dtype, dyn) for order in (3, 5, 7) for bc in ("periodic", "ref")
         for dtype in ("f32", "f64") for dyn in (True, False) if not (dtype == "f64" and order == 7)]


class Member(object):
    def __init__(self, n, seed, dyn):
        self.n, self.dt, self.coeffs = n, 5e-4, generic_coeffs(dyn) * (1.0 + 0.01 * (seed % 5))
        self.dx, P, psi0, n0 = fields(n, seed)
        self.P, self.psi0, self.n0 = (a.astype(t).astype(w) for a, t, w in (
            (P, np.float32, float), (psi0, np.complex64, complex), (n0, np.float32, float)))

    def oracle(self, oracle, order, bc):
        dyn = self.coeffs[10] != 0.0
        return oracle.rk4(2, self.n, order, native.BC[bc], self.dt, self.dx, STEPS, self.P, self.coeffs, self.psi0,
                          self.n0 if dyn else None)


def check(got, want, dtype, n):
    for a, b in zip(got, want):
        if b is not None:
            assert np.linalg.norm(a - b) <= TOL[dtype] * np.linalg.norm(b), n


@pytest.mark.parametrize("order,bc,dtype,dyn", CASES)
def test_alone(gpu, oracle, order, bc, dtype, dyn):
    for n in (order, 16, 31, 32, 33, 44, 45, 46, 50, 51, 53, 54, 55, 63, 64):
        m = Member(n, n, dyn)
        d = native.ProblemDesc.make(2, n, order, m.dt, m.dx, m.coeffs, bc=bc, dtype=dtype, engine="resident")
        check(native.solve_host(d, STEPS, m.P, m.psi0, m.n0 if dyn else None), m.oracle(oracle, order, bc), dtype, n)


@pytest.mark.parametrize("order,bc,dtype,dyn", CASES)
def test_many(gpu, oracle, order, bc, dtype, dyn):
    """More grids than compute units: each as it is alone, whatever the largest is."""
    for sides in ([16] * 290, [24, 31] * 150, [33, 9] * 145, [50, 20] * 145, [54, 12] * 145, [64, 17] * 145):
        ms = [Member(n, i % 6, dyn) for i, n in enumerate(sides)]
        b = Batch(ms, dim=2, order=order, bc=bc, dtype=dtype, engine="resident")
        b.advance(STEPS)
        out = [b.member(i) for i in range(len(ms))]
        b.close()
        for i in (0, 1, 2, 3, 4, 5):
            check(out[i], ms[i].oracle(oracle, order, bc), dtype, sides[i])
        for i in range(6, len(ms)):
            np.testing.assert_array_equal(out[i][0], out[i % 6][0])
            if dyn:
                np.testing.assert_array_equal(out[i][1], out[i % 6][1])
