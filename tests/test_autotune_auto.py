"""The autotuner times the library's own choice beside the engines and tile
forms that have names: it runs kernels that no name reaches (1-D lines in
pieces, marching strips, several steps a launch)."""
import json

import pytest

from nls_amd import autotune, configs, native


def timer(table, calls):
    def t(cand, _setup):
        if cand[1] not in table:
            raise KeyError(cand[1])
        calls.append(cand[1])
        return table[cand[1]]
    return t


def line(n=1000):
    return native.ProblemDesc.make(1, n, 5, 1e-3, 0.1, configs.model_coeffs())


@pytest.mark.parametrize("n", [1000, 5000])
def test_lines_may_stay_on_the_librarys_choice(n):
    calls = []
    T = autotune.Tuner(path=None, reps=1, timer=timer({"resident": 3.0, "stage": 2.0, "auto": 1.0}, calls),
                       device_name="dev")
    assert T.plain_engine(line(n)) == "auto" and "auto" in T.last
    assert T.tuned(line(n)).engine == native.ENGINE["auto"]
    T = autotune.Tuner(path=None, reps=1, timer=timer({"resident": 3.0, "stage": 2.0, "auto": 4.0}, calls),
                       device_name="dev")
    assert T.plain_engine(line(n)) == "stage"


def test_stored_choice_without_it_is_measured_again(tmp_path):
    path = str(tmp_path / "tune.json")
    d = line()
    old = "dev|plain|" + "|".join("%s=%s" % kv for kv in sorted(
        dict(dim=1, n=d.n, dtype=d.dtype, order=d.order, bc=d.bc, dyn=1).items()))
    json.dump({old: {"best": "resident", "seconds_per_step": {"resident": 1.0, "stage": 2.0}}}, open(path, "w"))
    T = autotune.Tuner(path=path, reps=1, timer=timer({"resident": 3.0, "stage": 2.0, "auto": 1.0}, []),
                       device_name="dev")
    assert T.plain_engine(d) == "auto"


@pytest.mark.parametrize("order", [5, 7])
def test_form_is_asked_for_only_where_it_is_faster(order):
    ms = configs.sweep512(count=4, steps=10)
    d = native.ProblemDesc.make(2, 2048, order, 1e-4, 0.05, configs.model_coeffs(), bc="periodic", dtype="f64")
    slow = {"tall": 2.0, "short": 1.9, "half": 2.5, "tall512": 2.5, "auto": 1.5}
    T = autotune.Tuner(path=None, reps=1, timer=timer(slow, []), device_name="dev")
    assert T.fused_form(ms, order=order) == "auto"
    assert T.plain_fused_form(d) == "auto"
    T = autotune.Tuner(path=None, reps=1, timer=timer(dict(slow, auto=1.9), []), device_name="dev")
    assert T.fused_form(ms, order=order) == "short"              # no gain in leaving it
    assert T.plain_fused_form(d) == "short"


def test_order_7_has_two_forms():
    calls = []
    ms = configs.sweep512(count=4, steps=10)
    T = autotune.Tuner(path=None, reps=1, timer=timer({"tall": 2.0, "short": 1.0}, calls), device_name="dev")
    assert T.fused_form(ms, order=7) == "short"
    assert set(calls) == {"tall", "short"}
