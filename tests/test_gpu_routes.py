"""Which kernel the library's own choice runs, by the kernels' names in a trace,
for the problems on which other tests compare that choice with a forced form: a
cost estimate that moves would have them compare a kernel with itself.

The marching kernel is also compared here, with the tiles bit for bit and with
the double-precision oracle, at problems for which the trace shows it in each
precision and reservoir mode, strips and whole rows.
"""
import numpy as np
import pytest

from nls_amd import native
from nls_amd.batch import Batch
from test_gpu_march import close, fields, generic_coeffs, with_form
from test_gpu_generic_coeffs import rounded

pytestmark = pytest.mark.gpu
STEPS = 5


def kernels(run):
    """Names of the kernels that run() launches."""
    import torch
    run()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        run()
        torch.cuda.synchronize()
    names = {e.name.split("(")[0].split("::")[-1] for e in p.events() if "nls::k_" in e.name}
    if not names:
        pytest.skip("no kernel trace on this system")
    return names


def advance(gpu, dim, n, order, bc, dtype, dyn, steps, engine="auto", scheme="rk4"):
    import torch
    rt, ct = (torch.float64, torch.complex128) if dtype == "f64" else (torch.float32, torch.complex64)
    d = native.ProblemDesc.make(dim, n, order, 1e-5, 0.1, generic_coeffs(dyn), bc=bc, dtype=dtype, engine=engine,
                                scheme=scheme, graphs=False)
    psi = torch.full((n,) * dim, 0.1, dtype=ct, device=gpu)
    P = torch.ones((n,) * dim, dtype=rt, device=gpu)
    nres = torch.zeros_like(P) if dyn else None
    ws = torch.empty(max(1, native.workspace_bytes(d)), dtype=torch.uint8, device=gpu)
    return lambda: native.advance(d, steps, P, psi, nres, ws)


@pytest.mark.parametrize("kernel,problem", [
    ("k_line<float, 5, 0, false,", (1, 1000, 5, "ref", "f32", False, 9)),
    ("k_line<double, 7, 1, true,", (1, 30011, 7, "periodic", "f64", True, 17)),
    ("k_multi<float, 3,", (2, 61, 3, "ref", "f32", False, 8)),
    ("k_multi<float, 5,", (2, 256, 5, "periodic", "f32", True, 6)),
    ("k_multi<double, 7,", (2, 180, 7, "ref", "f64", True, 4)),
    ("k_resident_2d<float, 5,", (2, 40, 5, "periodic", "f32", True, 4)),
    ("k_fused_groups_2d<double, 7,", (2, 777, 7, "ref", "f64", True, 2)),
    ("k_fused_groups_2d<float, 7,", (2, 1024, 7, "periodic", "f32", True, 2)),
    ("k_fused_pairs_2d<", (2, 300, 5, "ref", "f32", False, 2)),
    ("k_copy_state<", (1, 5000, 5, "periodic", "f64", True, 1)),
    ("k_copy_state<", (2, 64, 5, "periodic", "f32", True, 1)),
    ("k_march<float, true, false>", (2, 4100, 5, "periodic", "f32", True, 2)),
    ("k_march<double, false, false>", (2, 4100, 5, "periodic", "f64", False, 2)),
    ("k_ssf_rows2048<float,", (2, 2048, 5, "periodic", "f32", True, 3, "auto", "ssf")),
])
def test_route(gpu, kernel, problem):
    names = kernels(advance(gpu, *problem))
    assert any(n.startswith(kernel) for n in names), names


@pytest.mark.parametrize("n,dtype,dyn", [(1801, "f32", True), (2300, "f32", False), (1279, "f64", True),
                                         (1442, "f64", False)])
def test_marching_grid(gpu, oracle, n, dtype, dyn):
    h, P, psi0, n0 = fields(n, n)
    P, psi0, n0 = rounded(P, psi0, n0)
    c, n0 = generic_coeffs(dyn), n0 if dyn else None
    d = native.ProblemDesc.make(2, n, 5, 5e-4, h, c, bc="periodic", dtype=dtype)
    run = lambda: native.solve_host(d, STEPS, P, psi0, n0)
    names = kernels(run)
    assert len(names) == 1 and next(iter(names)).startswith("k_march<"), names
    march, tall = run(), with_form(dtype, "tall", run)
    np.testing.assert_array_equal(march[0], tall[0])
    opsi, onres = oracle.rk4(2, n, 5, 1, 5e-4, h, STEPS, P, c, psi0, n0)
    close(march[0], opsi, dtype)
    if dyn:
        np.testing.assert_array_equal(march[1], tall[1])
        close(march[1], onres, dtype)


class M(object):
    def __init__(self, n, seed, dyn):
        self.n, self.dt, self.coeffs = n, 5e-4, generic_coeffs(dyn) * (1.0 + 0.01 * (seed % 5))
        self.dx, P, psi0, n0 = fields(n, seed)
        self.P, self.psi0, self.n0 = rounded(P, psi0, n0)


@pytest.mark.parametrize("sides,dtype,dyn,full", [
    ([64, 100, 171, 255, 256, 65] * 35, "f32", True, True), ([257, 300, 401] * 20, "f32", True, False),
    ([256, 255, 128, 171] * 40, "f32", False, True), ([400, 700, 401] * 30, "f32", False, False),
    ([64, 100, 171, 255, 256, 65] * 35, "f64", True, True), ([257, 300, 401] * 30, "f64", True, False),
    ([64, 100, 171, 255, 256, 65] * 35, "f64", False, True), ([257, 300, 401] * 30, "f64", False, False)])
def test_marching_batch(gpu, oracle, sides, dtype, dyn, full):
    k = len(set(sides))
    few = [M(n, n, dyn) for n in sides[:k]]
    ms = [few[i % k] for i in range(len(sides))]

    def run():
        b = Batch(ms, dim=2, order=5, bc="periodic", dtype=dtype, engine="fused")
        b.advance(STEPS)
        out = b.psi.cpu().numpy(), b.nres.cpu().numpy() if dyn else None, [b.member(i) for i in range(k)]
        b.close()
        return out

    names = kernels(run)
    assert "k_march<%s, %s, %s>" % ({"f32": "float", "f64": "double"}[dtype], str(dyn).lower(), str(full).lower()) in names
    march, tall = run(), with_form(dtype, "tall", run)
    np.testing.assert_array_equal(march[0], tall[0])
    if dyn:
        np.testing.assert_array_equal(march[1], tall[1])
    for m, out in zip(few, march[2]):
        opsi, onres = oracle.rk4(2, m.n, 5, 1, m.dt, m.dx, STEPS, m.P, m.coeffs, m.psi0, m.n0 if dyn else None)
        close(out[0], opsi, dtype)
        if dyn:
            close(out[1], onres, dtype)


@pytest.mark.parametrize("count,many", [(64, "false"), (300, "true")])
def test_lines_of_order_3(gpu, count, many):
    class Line(object):
        n, dt, dx, coeffs = 100, 1e-5, 0.1, generic_coeffs(True)
        P, psi0, n0 = np.ones(100), np.full(100, 0.1 + 0j), np.zeros(100)
    b = Batch([Line()] * count, dim=1, order=3, bc="ref", dtype="f32", engine="resident")
    names = kernels(lambda: b.advance(4))
    b.close()
    assert "k_resident<float, 3, 0, true, %s>" % many in names, names
