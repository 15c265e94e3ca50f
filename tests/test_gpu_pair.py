"""Two steps per launch (k_pair2d, 2D lattices of at least 2^19 sites, with E6
/ E8 in FP64 3 * 2^17, on variant 10 and with the Shan-Chen forcing or the isotropy filter) against
single steps: variant 9, or the two-pass step for the forcing and the filter.
Every site sees the same arithmetic, so FP64 results are equal and FP32 ones
may differ by the contraction of a few operations per step. Sizes lie at the
edges of the tiles (250 / 246 and 122 / 118 columns written per block), with
rows that leave a remainder; runs of 4 to 7 steps have 2 pairs and 0 to 3
single steps, and 3 steps none."""
import numpy as np
import pytest

from helpers import droplet_field, rel_err

pytestmark = pytest.mark.gpu

CASES = [('D2E4', (500, 787), 'fp64', 'bgk'), ('D2E4', (251, 1571), 'fp64', 'mrt'),
         ('D2E8', (493, 801), 'fp64', 'bgk'), ('D2E6', (4099, 97), 'fp64', 'dense'),
         ('D2E4', (123, 3201), 'fp64', 'bgk'), ('D2E4', (1499, 263), 'fp64', 'sc'),
         ('D2E8', (613, 643), 'fp64', 'iso'), ('D2E4', (749, 526), 'fp32s', 'bgk'),
         ('D2E8', (640, 615), 'fp32s', 'mrt'), ('D2E4', (500, 1051), 'fp64', 'bgk'),
         ('D2E4', (251, 2091), 'fp64', 'mrt'), ('D2E4', (123, 4301), 'fp64', 'bgk'),
         ('D2E4', (1499, 351), 'fp64', 'sc'), ('D2E4', (749, 702), 'fp32s', 'bgk'),
         ('D2E8', (640, 821), 'fp32s', 'mrt')]


def _run(tenet, es, dims, prec, coll, single, steps, wf):
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM import hermite
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    S = np.diag(np.linspace(0.7, 1.5, 9))
    if coll == 'dense':
        S[3, 4] = 0.05
    kw = {'mrt': hermite.mrt_kernel_tables('D2Q9', S)} if coll in ('mrt', 'dense') else \
        {'forcing': 'sc'} if coll == 'sc' else {'iso_filter': True} if coll == 'iso' else {}
    eng = SCEngine(tenet, 'D2Q9', es, dims, 'exp', -5.0 / 3.0, 1.0, precision=prec, rho0=1.0,
                   **kw)
    assert eng.get_launch()[3] == 10
    if single:
        eng.set_launch(64, 1, 8, 9)
    V = eng.V
    n = IdpyMemory.OnDevice(droplet_field(dims, seed=21), tenet)
    psi = IdpyMemory.Zeros(V, np.float64, tenet)
    u = IdpyMemory.Zeros(2 * V, np.float64, tenet)
    a, b = PopArray(eng, tenet), PopArray(eng, tenet)
    eng.init_pop(a, n, u)
    swapped = eng.run(a, b, steps, n=n, psi=psi, u=u, write_fields=wf,
                      two_pass=single and coll in ('sc', 'iso'))
    out = [(b if swapped else a).RawD2H()]
    if wf:
        out += [n.D2H(), psi.D2H(), u.D2H()]
    for x in (a, b, n, psi, u):
        x.Free()
    eng.close()
    return swapped, out


@pytest.mark.parametrize('es,dims,prec,coll', CASES)
@pytest.mark.parametrize('steps,wf', [(3, True), (4, True), (5, False), (6, True), (7, True),
                                      (8, False)])
def test_two_steps_per_launch_equal_single_steps(tenet, es, dims, prec, coll, steps, wf):
    sw1, ref = _run(tenet, es, dims, prec, coll, True, steps, wf)
    sw2, got = _run(tenet, es, dims, prec, coll, False, steps, wf)
    assert sw1 == sw2      # the state ends in the buffer where single steps leave it
    for r, g in zip(ref, got):
        assert np.isfinite(g).all()
        if prec == 'fp64':
            assert np.array_equal(r, g)
        else:
            # ~10 roundings of 6e-8 of the largest value per step
            assert np.abs(r - g).max() <= steps * 10 * 6e-8 * np.abs(r).max()


@pytest.mark.parametrize('dims,g', [((1024, 520), 1e-5), ((613, 643), 0.0), ((251, 1571), 2e-5),
                                    ((251, 2091), 1e-5), ((613, 857), 0.0)])
@pytest.mark.parametrize('steps,wf', [(3, True), (4, True), (5, False), (8, True), (11, False)])
def test_two_steps_per_launch_with_walls(tenet, dims, g, steps, wf):
    """The walls step (plates, blocks across the periodic edges, lone solid
    and lone fluid sites) against the two-pass step on the fluid sites: the
    same arithmetic in the same order."""
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    rng = np.random.default_rng(5)
    w = np.ones(dims[::-1], dtype=np.uint8)
    w[0] = w[-1] = 0
    w[dims[1] // 3:dims[1] // 3 + 5, :3] = 0
    w[dims[1] // 3:dims[1] // 3 + 5, -2:] = 0
    w[dims[1] // 2:dims[1] // 2 + 40, dims[0] // 2:dims[0] // 2 + 60] = 0
    w[dims[1] // 2 + 7, dims[0] // 2 + 9] = 1
    w[rng.integers(0, dims[1], 4000), rng.integers(0, dims[0], 4000)] = 0
    psi_w = np.where(w == 0, rng.uniform(0.3, 0.7, size=w.shape), 0.0).ravel()
    w = w.ravel()
    fl, V, n0 = w == 1, w.size, droplet_field(dims, seed=8)
    wd = IdpyMemory.OnDevice(w, tenet)
    out = []
    for two_pass in (True, False):
        eng = SCEngine(tenet, 'D2Q9', 'D2E4', dims, 'exp', -5.0 / 3.0, 1.0)
        eng.set_walls(wd)
        if g:
            eng.set_body_force(0.0, g, 0.0)
        n = IdpyMemory.OnDevice(n0, tenet)
        psi = IdpyMemory.OnDevice(psi_w, tenet)
        u = IdpyMemory.Zeros(2 * V, np.float64, tenet)
        a, b = PopArray(eng, tenet), PopArray(eng, tenet)
        eng.init_pop(a, n, u)
        swapped = eng.run(a, b, steps, n=n, psi=psi, u=u, write_fields=wf, two_pass=two_pass)
        assert swapped == (steps % 2 == 1)
        out.append((eng.pop_to_host_soa(b if swapped else a).reshape(9, V)[:, fl], n.D2H()[fl],
                    psi.D2H(), u.D2H().reshape(2, V)[:, fl]))
        for x in (n, psi, u, a, b):
            x.Free()
        eng.close()
    wd.Free()
    (f1, n1, p1, u1), (f2, n2, p2, u2) = out
    assert np.isfinite(f2).all() and rel_err(f2.ravel(), f1.ravel()) <= 1e-15
    assert np.array_equal(p2[~fl], psi_w[~fl])
    if wf:
        assert rel_err(n2, n1) <= 1e-15 and rel_err(p2[fl], p1[fl]) <= 1e-15
        assert rel_err(u2.ravel(), u1.ravel()) <= 1e-14
