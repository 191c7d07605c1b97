"""The resident engine's lines against the double-precision oracle, with
coefficients none of which is 1 and no two equal, in batches of fewer and of more
lines than the device has compute units (zero-outside lines of order 3 with a
reservoir take another variant of the kernel for more, in single precision).

Sizes: the stencil width, one point a thread and the next, the largest line.
"""
import numpy as np
import pytest

from nls_amd import native
from nls_amd.batch import Batch
from test_gpu_generic_coeffs import rounded
from test_gpu_march import generic_coeffs
from test_gpu_resident import STEPS, check

pytestmark = pytest.mark.gpu


class Line(object):
    def __init__(self, n, seed, dyn):
        rng = np.random.default_rng(n)
        r = 0.1 * np.arange(n)
        self.n, self.dt, self.dx, self.coeffs = n, 5e-4, 0.1, generic_coeffs(dyn) * (1.0 + 0.01 * seed)
        self.P, self.psi0, self.n0 = rounded(2.0 + np.sin(3.0 * r), 0.3 * np.cos(r) + 0.1j * rng.standard_normal(n),
                                             0.2 + 0.1 * np.cos(r))


@pytest.mark.parametrize("order,bc,dtype,dyn", [(order, bc, dtype, dyn) for order in (3, 5, 7)
                                                for bc in ("periodic", "ref") for dtype in ("f32", "f64")
                                                for dyn in (True, False)])
def test_few_and_many(gpu, oracle, order, bc, dtype, dyn):
    sides = [order, 256, 1024, 1025, 3073, 4096]
    for count in (1, 50):
        ms = [Line(n, i, dyn) for i, n in enumerate(sides)] * count
        b = Batch(ms, dim=1, order=order, bc=bc, dtype=dtype, engine="resident")
        b.advance(STEPS)
        out = [b.member(i) for i in range(len(ms))]
        b.close()
        for i, m in enumerate(ms[:6]):
            check(out[i], oracle.rk4(1, m.n, order, native.BC[bc], m.dt, m.dx, STEPS, m.P, m.coeffs, m.psi0,
                                     m.n0 if dyn else None), dtype, m.n)
        for i in range(6, len(ms)):
            np.testing.assert_array_equal(out[i][0], out[i % 6][0])
            if dyn:
                np.testing.assert_array_equal(out[i][1], out[i % 6][1])
