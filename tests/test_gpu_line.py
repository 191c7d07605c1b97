"""The line kernel (plain 1-D solves): pieces of a line stepped in registers,
one workgroup or many, against the per-stage engine bit for bit (the 1-D
engines share one arithmetic) and against the FP64 oracle.

Sizes at the edges of its pieces: the stencil width, one wave's own points
(48 of 64 at order 5, 56 at order 3, 40 at order 7) and its neighbours, the
largest one-workgroup line and past it, lines of several hundred workgroups.
"""
import numpy as np
import pytest

from nls_amd import configs, native

pytestmark = pytest.mark.gpu


def solve(n, order, bc, dtype, dyn, steps, engine, seed=3):
    rng = np.random.default_rng(seed)
    h = 0.1
    r = h * np.arange(n)
    psi0 = 0.3 * np.exp(-(r - 0.3 * n * h) ** 2 / (0.01 + (0.1 * n * h) ** 2)) + configs.noise(rng, (n,), 1e-2)
    P = 2.0 + np.sin(3.0 * r)
    n0 = 0.2 + 0.1 * np.cos(r)
    c = configs.model_coeffs(dynamic=dyn)
    d = native.ProblemDesc.make(1, n, order, 5e-4, h, c, bc=bc, dtype=dtype, engine=engine)
    out = native.solve_host(d, steps, P, psi0, n0 if dyn else None)
    return out, (h, P, psi0, n0, c)


CASES = [(order, bc, dtype, dyn) for order in (3, 5, 7) for bc in ("periodic", "ref")
         for dtype, dyn in (("f32", True), ("f64", False))]


@pytest.mark.parametrize("order,bc,dtype,dyn", CASES)
def test_line_equals_stage_engine(gpu, order, bc, dtype, dyn):
    own = 64 - 4 * (order - 1)
    for n, steps in ((order, 9), (own - 1, 5), (own, 64), (own + 1, 33), (2 * own, 13), (8 * own + 1, 65), (700, 1),
                     (1000, 130), (4097, 24), (30011, 17)):
        (psi, nres), _ = solve(n, order, bc, dtype, dyn, steps, "auto")
        (psi_s, nres_s), _ = solve(n, order, bc, dtype, dyn, steps, "stage")
        assert np.isfinite(psi).all()
        np.testing.assert_array_equal(psi, psi_s, err_msg="n=%d steps=%d" % (n, steps))
        if dyn:
            np.testing.assert_array_equal(nres, nres_s, err_msg="n=%d steps=%d" % (n, steps))


@pytest.mark.parametrize("bc,dyn", [("periodic", True), ("ref", False)])
def test_line_matches_oracle(gpu, oracle, bc, dyn):
    for n, steps in ((50, 4100), (385, 200), (5000, 60)):
        (psi, nres), (h, P, psi0, n0, c) = solve(n, 5, bc, "f64", dyn, steps, "auto")
        opsi, onres = oracle.rk4(1, n, 5, native.BC[bc], 5e-4, h, steps, P, c, psi0, n0)
        assert np.linalg.norm(psi - opsi) <= 1e-10 * np.linalg.norm(opsi)
        if dyn:
            assert np.linalg.norm(nres - onres) <= 1e-10 * np.linalg.norm(onres)
