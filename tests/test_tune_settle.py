"""A launch that one timing among many showed as fastest replaces the present
one only if it is faster when the two are timed again (no GPU: an engine with
given times per step)."""
import pytest


class _Engine:
    dims = (64, 64)

    def __init__(self, times, two=None):
        self.times, self.two, self.k, self.launch = times, two or {}, {}, None

    def set_launch(self, *launch):
        self.launch = launch
        self.k[launch] = self.k.get(launch, -1) + 1

    def run(self, a, b, nsteps):
        t = self.times[self.launch]
        self.t = 5.0 + nsteps * t[min(self.k[self.launch], len(t) - 1)]
        if nsteps == 2:
            self.t = self.two.get(self.launch, self.t)

    def last_run_ms(self):
        return self.t


OLD, NEW = (256, 1, 8, 10), (64, 1, 128, 10)


@pytest.mark.parametrize('old,new,keep', [
    ([1.0], [1.0], OLD),                      # equal, however the first timing fell
    ([1.0, 1.02, 1.0], [1.0, 0.97, 1.0], OLD),  # one of three off either way
    ([1.0], [0.9], NEW), ([1.0], [0.995], OLD), ([1.0], [1.2], OLD)])
def test_the_present_launch_stays_unless_another_is_faster_again(old, new, keep):
    from idmx import tune
    eng = _Engine({OLD: old, NEW: new})
    assert tune.settle(eng, None, None, 10, OLD, NEW) == keep
    assert tune.settle(eng, None, None, 10, OLD, OLD) == OLD


@pytest.mark.parametrize('two,keep', [(1.0, NEW), (1.1, OLD), (0.9, NEW)])
def test_equal_long_runs_are_told_apart_by_single_steps(two, keep):
    """Two launches of variant 10 whose long runs differ by chance."""
    from idmx import tune
    eng = _Engine({OLD: [1.0], NEW: [0.985]}, {OLD: 1.0, NEW: two})
    assert tune.settle(eng, None, None, 10, OLD, NEW) == keep
    other = NEW[:3] + (9,)      # another variant takes single steps throughout
    eng = _Engine({OLD: [1.0], other: [0.985]}, {OLD: 1.0, other: two})
    assert tune.settle(eng, None, None, 10, OLD, other) == other
