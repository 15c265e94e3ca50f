"""Lattices of 2^19 sites and more with wall flags that are neither 0 nor 1
(not updated, no bounce-back: what streams out of such a site is whatever its
slot in the target buffer holds, of two steps before) against the two-pass
step, from two buffers that differ: pairs, single steps on lattices where
pairs do not run, and 3D. Same arithmetic in the same order on the fluid
sites."""
import numpy as np
import pytest

from helpers import droplet_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dims,other', [((1024, 520), True), ((1024, 520), False),
                                        ((63, 8400), True), ((96, 80, 70), True),
                                        ((96, 80, 70), False)])
@pytest.mark.parametrize('steps,wf', [(1, False), (1, True), (2, False), (3, True), (4, False),
                                      (5, True), (8, False), (9, True)])
def test_large_walls_with_other_flags_equal_two_pass(tenet, dims, other, steps, wf):
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    rng = np.random.default_rng(17)
    D, Q, V = len(dims), 9 if len(dims) == 2 else 19, int(np.prod(dims))
    w = np.where(rng.random(V) < 0.02, 0, 1).astype(np.uint8)
    w[:dims[0]] = 0
    if other:
        w[rng.integers(0, V, 50)] = 2
        w[V // 2:V // 2 + 3] = 255
    psi_w = np.where(w != 1, rng.uniform(0.3, 0.7, size=V), 0.0)
    n0, fl = droplet_field(dims, seed=2), w == 1
    wd = IdpyMemory.OnDevice(w, tenet)
    out = []
    for two_pass in (True, False):
        eng = SCEngine(tenet, 'D%dQ%d' % (D, Q), 'D%dE4' % D, dims, 'exp', -5.0 / 3.0, 1.0)
        eng.set_walls(wd)
        n = IdpyMemory.OnDevice(1.1 * n0, tenet)
        psi = IdpyMemory.OnDevice(psi_w, tenet)
        u = IdpyMemory.Zeros(D * V, np.float64, tenet)
        a, b = PopArray(eng, tenet), PopArray(eng, tenet)
        eng.init_pop(b, n, u)
        n.H2D(n0)
        eng.init_pop(a, n, u)
        swapped = eng.run(a, b, steps, n=n, psi=psi, u=u, write_fields=wf, two_pass=two_pass)
        assert swapped == (steps % 2 == 1)
        got = [eng.pop_to_host_soa(b if swapped else a).reshape(Q, V)[:, fl], psi.D2H()[~fl]]
        if wf:
            got += [n.D2H()[fl], psi.D2H()[fl], u.D2H().reshape(D, V)[:, fl]]
        out.append(got)
        for x in (n, psi, u, a, b):
            x.Free()
        eng.close()
    wd.Free()
    for r, t in zip(*out):
        assert np.isfinite(t).all() and np.array_equal(r, t)
