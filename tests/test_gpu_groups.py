"""The group kernel (tall tiles of order 7, and of order 5 in double
precision): the same bits as the short tiles, whose threads own single points.

Sizes at its edges: grids smaller than a tile and its halo (every wrap), one
row more or less than the tiles' 24 or 32, a last column of one point, and
sizes that the form rule itself sends to tall tiles; single-precision fields
under double-precision arithmetic; and batches of mixed sizes with budgets
that end inside a call.
"""
import numpy as np
import pytest

from nls_amd import configs, native
from nls_amd.batch import Batch
from test_gpu_march import M, fields, with_form

pytestmark = pytest.mark.gpu
KINDS = [(7, "f32"), (7, "f64"), (5, "f64")]


@pytest.mark.parametrize("order,dtype", KINDS)
@pytest.mark.parametrize("bc,dyn", [("ref", False), ("ref", True), ("periodic", False), ("periodic", True)])
@pytest.mark.parametrize("n", [25, 33, 65, 71, 97, 127, 193])
def test_tall_equals_short(gpu, n, order, dtype, bc, dyn):
    h, P, psi0, n0 = fields(n, n)
    d = native.ProblemDesc.make(2, n, order, 5e-4, h, configs.model_coeffs(dynamic=dyn), bc=bc, dtype=dtype,
                                engine="fused")
    run = lambda: native.solve_host(d, 3, P, psi0, n0 if dyn else None)
    tall, short = with_form(dtype, "tall", run), with_form(dtype, "short", run)
    assert np.isfinite(tall[0]).all()
    np.testing.assert_array_equal(tall[0], short[0])
    if dyn:
        np.testing.assert_array_equal(tall[1], short[1])


@pytest.mark.parametrize("n,dtype,bc", [(777, "f64", "ref"), (1024, "f32", "periodic")])
def test_rule_equals_short(gpu, n, dtype, bc):
    h, P, psi0, n0 = fields(n, n)
    d = native.ProblemDesc.make(2, n, 7, 5e-4, h, configs.model_coeffs(dynamic=True), bc=bc, dtype=dtype,
                                engine="fused")
    run = lambda: native.solve_host(d, 2, P, psi0, n0)
    auto, short = with_form(dtype, "auto", run), with_form(dtype, "short", run)
    np.testing.assert_array_equal(auto[0], short[0])
    np.testing.assert_array_equal(auto[1], short[1])


@pytest.mark.parametrize("order", [5, 7])
@pytest.mark.parametrize("dyn", [False, True])
def test_wide_arithmetic_equals_short(gpu, order, dyn):
    n = 101
    h, P, psi0, n0 = fields(n, n)
    d = native.ProblemDesc.make(2, n, order, 5e-4, h, configs.model_coeffs(dynamic=dyn), bc="periodic", dtype="f32",
                                f64_arith=True)
    run = lambda: native.solve_host(d, 3, P, psi0, n0 if dyn else None)
    tall, short = with_form("f64", "tall", run), with_form("f64", "short", run)
    np.testing.assert_array_equal(tall[0], short[0])
    if dyn:
        np.testing.assert_array_equal(tall[1], short[1])


@pytest.mark.parametrize("order,dtype", KINDS)
@pytest.mark.parametrize("bc", ["ref", "periodic"])
def test_batch_tall_equals_short(gpu, order, dtype, bc):
    ms = [M(n, 7 * i + n, True) for i, n in enumerate([24, 65, 48, 130, 90])]

    def run():
        b = Batch(ms, dim=2, order=order, bc=bc, dtype=dtype, engine="fused")
        b.set_steps([5 - i % 3 for i in range(len(ms))])
        b.advance(4)
        out = b.psi.cpu().numpy(), b.nres.cpu().numpy()
        b.close()
        return out

    tall, short = with_form(dtype, "tall", run), with_form(dtype, "short", run)
    np.testing.assert_array_equal(tall[0], short[0])
    np.testing.assert_array_equal(tall[1], short[1])
