"""Single steps on the x-shifted storage on large 2D lattices, where the
default launch takes pairs of steps: runs with per-step times, which take
single steps, and lattices too narrow for a pair's blocks, against variant 9.
Every site sees the same arithmetic: equal in FP64."""
import numpy as np
import pytest

from helpers import droplet_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('es,dims,coll,profiled', [
    ('D2E4', (1000, 527), 'bgk', True), ('D2E8', (517, 1021), 'mrt', True),
    ('D2E4', (257, 2051), 'mrt', True), ('D2E4', (63, 8323), 'bgk', False),
    ('D2E8', (37, 10701), 'bgk', False), ('D2E6', (50, 8001), 'mrt', True),
    ('D2E4', (59, 8999), 'sc', False)])
@pytest.mark.parametrize('steps,wf', [(1, True), (2, False), (4, True), (7, False), (8, True)])
def test_single_steps_equal_variant_9(tenet, es, dims, coll, profiled, steps, wf):
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM import hermite
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    kw = {'mrt': hermite.mrt_kernel_tables('D2Q9', np.diag(np.linspace(0.7, 1.5, 9)))} \
        if coll == 'mrt' else {'forcing': 'sc'} if coll == 'sc' else {}
    out = []
    for default in (True, False):
        eng = SCEngine(tenet, 'D2Q9', es, dims, 'exp', -5.0 / 3.0, 1.0, **kw)
        assert eng.get_launch()[3] == 10
        if not default:
            eng.set_launch(64, 1, 7, 9)
        V = eng.V
        n = IdpyMemory.OnDevice(droplet_field(dims, seed=3), tenet)
        psi = IdpyMemory.Zeros(V, np.float64, tenet)
        u = IdpyMemory.Zeros(2 * V, np.float64, tenet)
        a, b = PopArray(eng, tenet), PopArray(eng, tenet)
        eng.init_pop(a, n, u)
        ms = np.zeros(2 * steps, dtype=np.float32) if profiled and default else None
        swapped = eng.run(a, b, steps, n=n, psi=psi, u=u, write_fields=wf, step_ms=ms,
                          two_pass=not default and coll == 'sc')
        assert swapped == (steps % 2 == 1)
        if ms is not None:
            assert (ms[1::2] > 0).all()
        out.append([(b if swapped else a).RawD2H()]
                   + ([n.D2H(), psi.D2H(), u.D2H()] if wf else []))
        for x in (a, b, n, psi, u):
            x.Free()
        eng.close()
    for g, r in zip(*out):
        assert np.isfinite(g).all() and np.array_equal(r, g)
