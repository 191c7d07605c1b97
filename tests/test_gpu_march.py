"""The marching kernel (large order-5 periodic grids and batches): the same
bits as the tile kernel, which a forced tile form runs on the same problem.

Sizes at its edges: strips that do not divide the grid, rows that are not a
multiple of a piece, whole rows of 64 to 256 points (one to four pieces side
by side, 65 and 255 with idle lanes), 257 (the first cut into strips), odd
step counts and budgets that end inside a call.
"""
import numpy as np
import pytest

from nls_amd import configs, native
from nls_amd.batch import Batch

pytestmark = pytest.mark.gpu


def fields(n, seed):
    rng = np.random.default_rng(seed)
    X, Y, h = configs.grid_2d(n, 0.1 * n)
    psi0 = 0.3 * np.exp(-(X ** 2 + Y ** 2) / (0.04 * n) ** 2) + configs.noise(rng, (n, n), 1e-2)
    return h, 2.0 + np.sin(3.0 * X) * np.cos(2.0 * Y), psi0, 0.2 + 0.1 * np.cos(X + Y)


def with_form(dtype, form, run):
    native.fused_form(dtype, form)
    try:
        return run()
    finally:
        native.fused_form(dtype, "auto")


@pytest.mark.parametrize("n,dtype,dyn", [(1801, "f32", True), (2048, "f32", False), (1279, "f64", True),
                                         (1442, "f64", False)])
def test_plain_grid_equals_tiles(gpu, n, dtype, dyn):
    h, P, psi0, n0 = fields(n, n)
    d = native.ProblemDesc.make(2, n, 5, 5e-4, h, configs.model_coeffs(dynamic=dyn), bc="periodic", dtype=dtype,
                                engine="fused")
    run = lambda: native.solve_host(d, 5, P, psi0, n0 if dyn else None)
    march, tall = with_form(dtype, "auto", run), with_form(dtype, "tall", run)
    assert np.isfinite(march[0]).all()
    np.testing.assert_array_equal(march[0], tall[0])
    if dyn:
        np.testing.assert_array_equal(march[1], tall[1])


class M(object):
    def __init__(self, n, seed, dyn):
        self.n, self.dt, self.coeffs = n, 5e-4, configs.model_coeffs(dynamic=dyn)
        self.dx, self.P, self.psi0, self.n0 = fields(n, seed)


@pytest.mark.parametrize("dtype,dyn", [("f32", True), ("f64", True), ("f32", False), ("f64", False)])
def test_batch_equals_tiles(gpu, dtype, dyn):
    sides = [64, 65, 100, 128, 171, 200, 255, 256, 257, 300] * 10
    ms = [M(n, 7 * i + n, dyn) for i, n in enumerate(sides)]
    steps = [9 - i % 4 for i in range(len(ms))]

    def run():
        b = Batch(ms, dim=2, order=5, bc="periodic", dtype=dtype, engine="fused")
        b.set_steps(steps)
        b.advance(7)                             # odd, and past some members' budgets
        out = b.psi.cpu().numpy(), b.nres.cpu().numpy() if dyn else None
        b.close()
        return out

    march, tall = with_form(dtype, "auto", run), with_form(dtype, "tall", run)
    assert np.isfinite(march[0]).all()
    np.testing.assert_array_equal(march[0], tall[0])
    if dyn:
        np.testing.assert_array_equal(march[1], tall[1])


def generic_coeffs(dyn):
    """No coefficient 1 and no two equal, so that none drops out of a kernel unseen."""
    c = configs.model_coeffs(dynamic=dyn)
    c[2:6] = 0.6, 0.45, 1.2, 3.1
    c[10:14] = 0.8 if dyn else 0.0, 1.3, 0.9, 1.7
    return c


# Against double precision: a step rounds a value some 60 times at its scale,
# so 5 steps stay within 300 * 2^-53 = 3.3e-14 and 300 * 2^-24 = 1.8e-5; double
# precision is given a factor of 10 for the growth of earlier errors.
TOL = {"f64": 3.3e-13, "f32": 1.8e-5}


def close(got, want, dtype):
    assert np.linalg.norm(got - want) <= TOL[dtype] * np.linalg.norm(want)


@pytest.mark.parametrize("n,dtype,dyn", [(1500, "f32", True), (1500, "f32", False), (1279, "f64", True),
                                         (1279, "f64", False)])
def test_plain_grid_generic_coefficients(gpu, oracle, n, dtype, dyn):
    h, P, psi0, n0 = fields(n, n)
    P, psi0, n0 = (a.astype(t).astype(w) for a, t, w in
                   ((P, np.float32, float), (psi0, np.complex64, complex), (n0, np.float32, float)))
    c = generic_coeffs(dyn)
    d = native.ProblemDesc.make(2, n, 5, 5e-4, h, c, bc="periodic", dtype=dtype, engine="fused")
    run = lambda: native.solve_host(d, 5, P, psi0, n0 if dyn else None)
    march, tall = with_form(dtype, "auto", run), with_form(dtype, "tall", run)
    np.testing.assert_array_equal(march[0], tall[0])
    opsi, onres = oracle.rk4(2, n, 5, 1, 5e-4, h, 5, P, c, psi0, n0 if dyn else None)
    close(march[0], opsi, dtype)
    if dyn:
        np.testing.assert_array_equal(march[1], tall[1])
        close(march[1], onres, dtype)


@pytest.mark.parametrize("dtype,dyn", [("f32", True), ("f64", True), ("f32", False), ("f64", False)])
def test_batch_generic_coefficients(gpu, oracle, dtype, dyn):
    sides = [64, 100, 171, 255, 256, 257, 300] * 30
    ms = [M(n, 7 * i + n, dyn) for i, n in enumerate(sides)]
    for i, m in enumerate(ms):
        m.coeffs = generic_coeffs(dyn) * (1.0 + 0.01 * (i % 5))
        m.P, m.psi0, m.n0 = (a.astype(t).astype(w) for a, t, w in
                             ((m.P, np.float32, float), (m.psi0, np.complex64, complex), (m.n0, np.float32, float)))

    def run():
        b = Batch(ms, dim=2, order=5, bc="periodic", dtype=dtype, engine="fused")
        b.advance(5)
        out = b.psi.cpu().numpy(), b.nres.cpu().numpy() if dyn else None, [b.member(i) for i in range(len(ms))]
        b.close()
        return out

    march, tall = with_form(dtype, "auto", run), with_form(dtype, "tall", run)
    np.testing.assert_array_equal(march[0], tall[0])
    if dyn:
        np.testing.assert_array_equal(march[1], tall[1])
    for i in range(7):
        m = ms[i]
        opsi, onres = oracle.rk4(2, m.n, 5, 1, m.dt, m.dx, 5, m.P, m.coeffs, m.psi0, m.n0 if dyn else None)
        close(march[2][i][0], opsi, dtype)
        if dyn:
            close(march[2][i][1], onres, dtype)
