"""Tuning a simulation leaves it no slower than it was created, whatever run
length the tuner is asked to time, and trying (apply=False) leaves its launch
in place. Times are minima of several runs."""
import pytest

from test_gpu_launch_restore import _sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('xi,es,dims,mrt', [('D2Q9', 'D2E4', (128, 128), False),
                                            ('D2Q9', 'D2E8', (620, 620), False),
                                            ('D3Q19', 'D3E4', (24, 24, 24), True)])
@pytest.mark.parametrize('steps', [3, 5, 10])
def test_tuned_launch_is_not_slower_than_the_default(tenet, xi, es, dims, mrt, steps):
    from idmx import tune
    eng, ms, close = _sim(tenet, xi, es, dims, mrt)
    at_creation, t0 = eng.get_launch(), ms(200)
    best, timings = tune.tune_sim(eng, steps=steps, use_cache=False, apply=False)
    assert eng.get_launch() == at_creation and ms(200) < 1.2 * t0
    assert ','.join(map(str, at_creation)) in timings
    eng.set_launch(*best)
    print(xi, es, dims, steps, 'default', at_creation, t0 / 200, 'tuned', best, ms(200) / 200,
          flush=True)
    assert ms(200) < 1.2 * t0
    close()
