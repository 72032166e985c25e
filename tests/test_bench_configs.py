"""The optimized product quantizer's benchmark takes the same route timed and when its parity is recorded."""
import numpy as np

import bench_configs


class _Array:
    def download(self):
        return np.zeros((2, 2), np.float32)


class _Context:
    """Writes down the calls; arrays stand for nothing."""

    def __init__(self):
        self.calls = []

    def empty(self, shape, dtype):
        return _Array()

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return np.zeros((2, 2))
        return call


def test_the_recorded_fit_makes_the_calls_of_the_timed_one():
    timed, recorded, trace = _Context(), _Context(), []
    for ctx, t in ((timed, None), (recorded, trace)):
        bench_configs.opq_fit_device(ctx, _Array(), 4, 2, 1, 2, 3, 3, (None, None), 1, trace=t)
    assert timed.calls.count("opq_rotation") == 3 and len(trace) == 3
    assert [c for c in recorded.calls if c != "cross_cov"] == timed.calls
