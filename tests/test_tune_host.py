"""The single-domain tuner's timing and cache key without a GPU, on an engine
that models the run times of the launches."""
import types

import pytest


class _Engine:
    """Run times in units of 1: a conversion before and after the steps (pull
    form), and `per` steps per launch, an even number of such launches, where
    a launch of `per` steps takes `many` and a single step takes `one`."""

    def __init__(self, per, many, one, convert=0.0):
        self.per, self.many, self.one, self.convert, self.t = per, many, one, convert, 0.0

    def run(self, a, b, nsteps):
        k = nsteps // self.per & ~1 if self.per > 1 else 0
        self.t = 5.0 + self.convert + k * self.many + (nsteps - k * self.per) * self.one

    def last_run_ms(self):
        return self.t


@pytest.mark.parametrize('steps', [1, 3, 5, 10, 17])
def test_step_time_is_that_of_the_launches_a_long_run_takes(steps):
    from idmx import tune
    for per, many, one, convert in ((1, 0.0, 2.0, 0.0), (1, 0.0, 2.0, 3.0), (2, 3.0, 2.5, 0.0),
                                    (2, 3.0, 40.0, 0.0), (4, 7.0, 5.0, 0.0), (4, 7.0, 90.0, 0.0)):
        want = many / per if per > 1 else one
        got = tune.step_ms(_Engine(per, many, one, convert), None, None, steps)
        assert abs(got - want) < 1e-12, (per, many, one, convert)


def test_sim_cache_key_is_not_that_of_earlier_launch_tables():
    """Picks cached when variant 10 took single steps stay unused."""
    from idmx import tune
    eng = types.SimpleNamespace(tenet=types.SimpleNamespace(GetDeviceName=lambda: 'gpu'),
                                xi_name='D2Q9', e_name='D2E8', dims=(4096, 4096),
                                precision='fp64', is_mrt=False)
    assert tune.sim_key(eng) != 'sim|gpu|D2Q9|D2E8|4096x4096|fp64|bgk'
    assert tune.sim_key(eng).split('|')[1:] == ['gpu', 'D2Q9', 'D2E8', '4096x4096', 'fp64', 'bgk']
