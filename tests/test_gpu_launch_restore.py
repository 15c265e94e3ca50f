"""Asking whether a launch is possible, and setting another one and going back,
leave a simulation no slower than it was created: the launch chosen at creation
includes a step that no variant names (small 3D lattices), and setting that
launch again selects it again. Times are minima of several runs; what is told
apart differs by a third and more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sim(tenet, xi, es, dims, mrt):
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM import hermite
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    kw = {'mrt': hermite.mrt_kernel_tables(xi, np.diag(np.linspace(0.7, 1.5, 19)))} if mrt else {}
    eng = SCEngine(tenet, xi, es, dims, 'exp', -5.0 / 3.0, 1.0, **kw)
    n = IdpyMemory.OnDevice(1.0 + 1e-3 * np.sin(np.arange(eng.V) * 0.37), tenet)
    u = IdpyMemory.Zeros(eng.D * eng.V, np.float64, tenet)
    a, b = PopArray(eng, tenet), PopArray(eng, tenet)
    eng.init_pop(a, n, u)

    def ms(steps, runs=7):
        t = []
        for _ in range(runs):
            eng.run(a, b, steps)
            t.append(eng.last_run_ms())
        return min(t)

    def close():
        for x in (a, b, n, u):
            x.Free()
        eng.close()
    return eng, ms, close


def test_small_3d_launch_survives_a_query_and_a_round_trip(tenet):
    eng, ms, close = _sim(tenet, 'D3Q19', 'D3E4', (24, 24, 24), True)
    at_creation, t0 = eng.get_launch(), ms(200)
    assert eng.launch_ok(32, 8, 2, 1) and not eng.launch_ok(256, 2, 8, 9)
    assert eng.get_launch() == at_creation and ms(200) < 1.2 * t0
    eng.set_launch(32, 8, 2, 1)
    assert ms(200) > 1.2 * t0     # the march
    eng.set_launch(*at_creation)
    assert ms(200) < 1.2 * t0
    close()
