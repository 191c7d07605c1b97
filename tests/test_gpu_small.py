"""Small 2-D grids: several steps per launch (plain solves) and one workgroup
per grid (the resident engine), the same bits as the tile kernel, which a
forced tile form runs.

In single precision, up to 64 points a side, the resident kernel and what AUTO
picks sum the stencil from the centre and agree with each other.

Sizes at the edges: the stencil width (the halo wraps several times), one tile
and past it, grids not a multiple of a tile or of a thread's strip, the
largest of each shape and one past it; step counts that leave steps over.
"""
import numpy as np
import pytest

from nls_amd import configs, native

pytestmark = pytest.mark.gpu


def solve(n, order, bc, dtype, dyn, steps, engine, form):
    rng = np.random.default_rng(n)
    X, Y, h = configs.grid_2d(n, 0.1 * n)
    psi0 = 0.3 * np.exp(-(X ** 2 + Y ** 2) / (0.04 * n + 0.1) ** 2) + configs.noise(rng, (n, n), 1e-2)
    P = 2.0 + np.sin(3.0 * X) * np.cos(2.0 * Y)
    n0 = 0.2 + 0.1 * np.cos(X + Y)
    d = native.ProblemDesc.make(2, n, order, 5e-4, h, configs.model_coeffs(dynamic=dyn), bc=bc, dtype=dtype,
                                engine=engine)
    native.fused_form(dtype, form)
    try:
        return native.solve_host(d, steps, P, psi0, n0 if dyn else None)
    finally:
        native.fused_form(dtype, "auto")


CASES = [(order, bc, dtype, dyn) for order in (3, 5, 7) for bc in ("periodic", "ref")
         for dtype, dyn in (("f32", True), ("f64", True), ("f32", False), ("f64", False))]


@pytest.mark.parametrize("order,bc,dtype,dyn", CASES)
def test_small_grids_equal_tiles(gpu, order, bc, dtype, dyn):
    for n, steps in ((order, 9), (16, 8), (17, 7), (40, 6), (61, 5), (63, 4), (64, 3), (65, 5), (128, 4), (180, 3),
                     (185, 2), (256, 5), (257, 3)):
        ref = solve(n, order, bc, dtype, dyn, steps, "fused", "tall")
        small = n <= 64 and not (dtype == "f64" and order == 7)
        # up to 64 points a side the resident kernel, and what AUTO picks, sum
        # single precision from the centre: the same bits as each other
        groups = [(ref, ["fused"] + (["resident"] if small and dtype == "f64" else []))]
        if n <= 64 and dtype == "f32":
            groups.append((solve(n, order, bc, dtype, dyn, steps, "resident", "auto"), ["auto"]))
        for want, engines in groups:
            for engine in engines:
                out = solve(n, order, bc, dtype, dyn, steps, engine, "auto")
                assert np.isfinite(out[0]).all()
                np.testing.assert_array_equal(out[0], want[0], err_msg="n=%d %s" % (n, engine))
                if dyn:
                    np.testing.assert_array_equal(out[1], want[1], err_msg="n=%d %s" % (n, engine))
