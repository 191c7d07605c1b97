"""Single-precision 2-D kernels step with the caller's coefficients and dt: over
many points their rounding errors average out, and what is left along the step's
increment is a coefficient or a step that is rounded once for all points, a drift
that grows with the steps.

One step of random fields, with little of the Laplacian (a wide spacing, at which
the coefficients in units of the stencil's first weight round unluckily) and a dt
whose sixth is exact: the error's component along the increment, against the
double-precision oracle.  A new value rounds at 3e-8 of its size (root mean
square) and the increment is a tenth of it, so over 90,000 points the component
is known to 1e-9, over 16 grids of 48^2 to 2e-9; 1.5e-8 is eight times that.  Tiles
of order 5 take the coefficients in units of the first weight, one rounding each:
2^-24 more.
"""
import numpy as np
import pytest

from nls_amd import native

pytestmark = pytest.mark.gpu
SPACING = {3: 9.4, 5: 12.9, 7: 13.6}


@pytest.mark.parametrize("bc", ["periodic", "ref"])
@pytest.mark.parametrize("n,order,engine", [(48, 3, "auto"), (48, 5, "auto"), (48, 7, "auto"), (48, 3, "resident"),
                                            (48, 5, "resident"), (48, 7, "resident"), (160, 3, "fused"),
                                            (300, 3, "fused"), (300, 5, "fused"), (300, 7, "fused"),
                                            (700, 7, "fused")])
def test_step_is_unbiased(gpu, oracle, n, order, engine, bc):
    c = np.zeros(23)
    c[4], c[12] = 6.0, 1.0
    dt, dx = 6.0 / 512.0, SPACING[order]
    along = whole = 0.0
    for seed in range(16 if n == 48 else 4 if n == 160 else 1):
        rng = np.random.default_rng(seed)
        psi0 = (rng.uniform(0.4, 1.2, (n, n)) * np.exp(2j * np.pi * rng.random((n, n)))).astype(np.complex64)
        d = native.ProblemDesc.make(2, n, order, dt, dx, c, bc=bc, dtype="f32", engine=engine)
        psi, _ = native.solve_host(d, 1, np.zeros((n, n)), psi0, None)
        exact, _ = oracle.rk4(2, n, order, native.BC[bc], dt, dx, 1, np.zeros((n, n)), c, psi0.astype(complex), None)
        step = exact - psi0
        along += np.vdot(step, psi - exact).real
        whole += np.vdot(step, step).real
    assert abs(along / whole) <= 1.5e-8 + (2.0 ** -24 if order == 5 and n > 64 else 0.0)
