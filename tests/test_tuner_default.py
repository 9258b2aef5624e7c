"""The tuner's default is a default handle, by the library's own rules: timed,
kept by the gate and chosen as one. No GPU."""
import numpy as np
import pytest

import gpuprefixsums_amd as gps
from gpuprefixsums_amd.tuner import Tuner
from gpuprefixsums_amd.tuner.harness import Runner
from gpuprefixsums_amd.tuner.space import Config, Workload, candidates, default_config

SIZES = [1 << 12, 1 << 19, 1 << 21, (1 << 23) + 5, 1 << 24, 1 << 27]


def workload(dtype, segments, n):
    return Workload(0, n, dtype, segments, np.linspace(0, n, segments + 1).astype(np.uint64))


@pytest.mark.parametrize("dtype", ["u32", "f32", "bf16"])
@pytest.mark.parametrize("segments", [1, 100])
def test_default_handle(dtype, segments):
    for n in SIZES:
        d = default_config(dtype, segments, n)
        assert d.handle_args() == (gps.ALGO_CSDL, {})
        alike = next(c for c in candidates(dtype) if c == d)  # under its name, but run by that shape
        assert alike.name == d.name and alike.handle_args()[1]["block_threads"] == d.block


class Model:
    """Predicts one candidate the fastest, by 1%, or by a factor of 4."""
    margin = 0.05

    def __init__(self, cands, best, gain):
        self.pred = np.array([0.0 if c != best else -gain for c in cands])

    def predict(self, X):
        return self.pred


def test_gate_and_exhaustive_choice():
    w = workload("u32", 100, 1 << 21)
    cands, d = candidates("u32"), default_config("u32", 100, 1 << 21)
    other = next(c for c in cands if c != d)
    t = Tuner(model_path=None)
    for best, gain, args in ((other, 2.0, other.handle_args()), (other, 0.01, (gps.ALGO_CSDL, {})), (d, 2.0, (gps.ALGO_CSDL, {}))):
        t.model = Model(cands, best, gain)
        assert t.choose(w).handle_args() == args
    t.model = None
    for best, args in ((other, other.handle_args()), (d, (gps.ALGO_CSDL, {}))):
        t._runner = type("R", (), {"time_all": lambda self, w: {c.name: 1.0 if c == best else 2.0 for c in cands}})()
        assert t.choose(w).handle_args() == args
        assert t.choose(w, fallback="default").handle_args() == (gps.ALGO_CSDL, {})


def test_harness_times_a_default_handle():
    w = workload("f32", 100, 1 << 21)
    seen = []
    r = Runner.__new__(Runner)
    r.handles = {}
    r.stage = lambda w: None
    r.time = lambda w, c, best: seen.append(c) or 1.0
    times = r.time_all(w, passes=1)
    assert list(times) == [c.name for c in candidates("f32")]
    assert [c.name for c in seen if c.plain] == [default_config("f32", 100, 1 << 21).name]
    assert Config("batched_fp", 1024, 4).handle_args()[1] != {}
