"""Two or four steps per launch on small 2D lattices (k_tile2d, below 2^19
sites, with E6 / E8 in FP64 3 * 2^17, the default launch) against single steps with the populations
in registers (variant 1), or against the two-pass step for the Shan-Chen
forcing and the isotropy filter: the same arithmetic per site, equal in FP64
and, contraction being the same in every launch, to rounding in FP32. Lattices
smaller than a tile and its ring, edges of the 8, 16, 22 and 24 wide tiles, and
runs that leave single steps over. Likewise one step of a small 3D lattice
without a march (k_tile3d), on lattices shorter than its 16 x 4 x 4 tile and
its halo and ones that leave partial tiles."""
import numpy as np
import pytest

from helpers import droplet_field

pytestmark = pytest.mark.gpu

CASES = [((3, 3), 'fp64', 'bgk'), ((5, 70), 'fp64', 'mrt'), ((128, 128), 'fp64', 'bgk'),
         ((127, 129), 'fp64', 'bgk'), ((129, 145), 'fp64', 'dense'), ((17, 300), 'fp64', 'sc'),
         ((8, 16), 'fp64', 'iso'), ((301, 47), 'fp64', 'bgk'), ((627, 627), 'fp64', 'mrt'),
         ((95, 64), 'fp32s', 'bgk'), ((161, 200), 'fp32s', 'mrt'),
         ((385, 313), 'fp64', 'bgk'), ((337, 361), 'fp64', 'sc'), ((400, 300), 'fp64', 'iso'),
         ((500, 401), 'fp32s', 'bgk')]
CASES = [c + ('D2E4',) for c in CASES] + [
    ((5, 5), 'fp64', 'bgk', 'D2E8'), ((5, 70), 'fp64', 'mrt', 'D2E6'),
    ((127, 129), 'fp64', 'bgk', 'D2E8'), ((301, 47), 'fp64', 'iso', 'D2E8'),
    ((161, 200), 'fp64', 'dense', 'D2E6'), ((627, 627), 'fp64', 'bgk', 'D2E6'),
    ((95, 64), 'fp32s', 'bgk', 'D2E8'), ((463, 440), 'fp32s', 'bgk', 'D2E8'),
    ((463, 440), 'fp32s', 'mrt', 'D2E6')]


def _run(tenet, dims, prec, coll, single, steps, wf, es='D2E4'):
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM import hermite
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    S = np.diag(np.linspace(0.7, 1.5, 9))
    if coll == 'dense':
        S[3, 4] = 0.05
    kw = {'mrt': hermite.mrt_kernel_tables('D2Q9', S)} if coll in ('mrt', 'dense') else \
        {'forcing': 'sc'} if coll == 'sc' else {'iso_filter': True} if coll == 'iso' else {}
    eng = SCEngine(tenet, 'D2Q9', es, dims, 'exp', -5.0 / 3.0, 1.0, precision=prec,
                   rho0=1.0, **kw)
    assert eng.get_launch()[3] == 10
    if single:
        eng.set_launch(64, 1, 3, 1)
    V = eng.V
    n0 = droplet_field(dims, seed=4) if min(dims) > 20 else \
        1.0 + 0.3 * np.sin(2 * np.pi * np.arange(V) / max(dims) + 0.3)
    n = IdpyMemory.OnDevice(n0, tenet)
    psi = IdpyMemory.Zeros(V, np.float64, tenet)
    u = IdpyMemory.Zeros(2 * V, np.float64, tenet)
    a, b = PopArray(eng, tenet), PopArray(eng, tenet)
    eng.init_pop(a, n, u)
    swapped = eng.run(a, b, steps, n=n, psi=psi, u=u, write_fields=wf,
                      two_pass=single and coll in ('sc', 'iso'))
    out = [(b if swapped else a).RawD2H()]
    if wf:
        out += [n.D2H(), psi.D2H()] + ([u.D2H()] if prec == 'fp64' else [])
    for x in (a, b, n, psi, u):
        x.Free()
    eng.close()
    return swapped, out


@pytest.mark.parametrize('dims,prec,coll,es', CASES)
@pytest.mark.parametrize('steps,wf', [(3, True), (7, True), (8, True), (8, False), (13, True), (18, False)])
def test_four_steps_per_launch_equal_single_steps(tenet, dims, prec, coll, es, steps, wf):
    sw1, ref = _run(tenet, dims, prec, coll, True, steps, wf, es)
    sw2, got = _run(tenet, dims, prec, coll, False, steps, wf, es)
    assert sw1 == sw2      # the state ends in the buffer where single steps leave it
    for r, g in zip(ref, got):
        assert np.isfinite(g).all()
        if prec == 'fp64':
            assert np.array_equal(r, g)
        else:
            # ~10 roundings of 6e-8 of the largest value per step
            assert np.abs(r - g).max() <= steps * 10 * 6e-8 * np.abs(r).max()


CASES3 = [('D3E4', (3, 3, 3), 'fp64', 'bgk'), ('D3E8', (5, 5, 5), 'fp64', 'mrt'),
          ('D3E4', (17, 5, 9), 'fp64', 'mrt'), ('D3E4', (48, 44, 40), 'fp64', 'mrt'),
          ('D3E6', (31, 9, 6), 'fp64', 'bgk'), ('D3E8', (33, 29, 31), 'fp64', 'bgk'),
          ('D3E4', (18, 6, 40), 'fp64', 'dense'), ('D3E4', (16, 70, 5), 'fp64', 'sc'),
          ('D3E4', (40, 41, 42), 'fp32s', 'mrt'), ('D3E8', (21, 22, 23), 'fp32s', 'bgk')]


@pytest.mark.parametrize('es,dims,prec,coll', CASES3)
@pytest.mark.parametrize('wf', [True, False])
def test_small_3d_step_equals_march(tenet, es, dims, prec, coll, wf):
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM import hermite
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    S = np.diag(np.linspace(0.7, 1.5, 19))
    if coll == 'dense':
        S[5, 6] = 0.05
    kw = {'mrt': hermite.mrt_kernel_tables('D3Q19', S)} if coll in ('mrt', 'dense') else \
        {'forcing': 'sc'} if coll == 'sc' else {}
    V = int(np.prod(dims))
    n0 = 1.0 + 0.3 * np.sin(2 * np.pi * np.arange(V) / 17 + 0.3)
    out = []
    for march in (False, True):
        eng = SCEngine(tenet, 'D3Q19', es, dims, 'exp', -5.0 / 3.0, 1.0, precision=prec,
                       rho0=1.0, **kw)
        if march:
            eng.set_launch(32, 8, 2, 1)
        n = IdpyMemory.OnDevice(n0, tenet)
        psi = IdpyMemory.Zeros(V, np.float64, tenet)
        u = IdpyMemory.Zeros(3 * V, np.float64, tenet)
        a, b = PopArray(eng, tenet), PopArray(eng, tenet)
        eng.init_pop(a, n, u)
        swapped = eng.run(a, b, 5, n=n, psi=psi, u=u, write_fields=wf,
                          two_pass=march and coll == 'sc')
        out.append([(b if swapped else a).RawD2H()]
                   + ([n.D2H(), psi.D2H()] + ([u.D2H()] if prec == 'fp64' else []) if wf else []))
        for x in (a, b, n, psi, u):
            x.Free()
        eng.close()
    for g, r in zip(*out):
        assert np.isfinite(g).all()
        if prec == 'fp64':
            assert np.array_equal(r, g)
        else:
            # ~10 roundings of 6e-8 of the largest value per step
            assert np.abs(r - g).max() <= 5 * 10 * 6e-8 * np.abs(r).max()


@pytest.mark.parametrize('dims,g,other', [((5, 7), 0.0, False), ((40, 9), 1e-5, False),
                                          ((123, 130), 2e-5, False), ((250, 131), 0.0, False),
                                          ((61, 50), 1e-5, True), ((700, 640), 1e-5, False),
                                          ((700, 640), 0.0, True)])
@pytest.mark.parametrize('steps,wf', [(7, True), (8, False), (11, True), (17, False)])
def test_small_2d_walls_equal_two_pass(tenet, dims, g, other, steps, wf):
    """Walls on the tiles: solid sites across the periodic edges and between
    tiles; with a flag that is neither 0 nor 1 the run stays on the two-pass
    step. Same arithmetic in the same order on the fluid sites."""
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    rng = np.random.default_rng(6)
    V = int(np.prod(dims))
    w = np.where(rng.random(V) < 0.2, 0, 1).astype(np.uint8)
    w[:dims[0]] = 0
    if other:
        w[V // 2:V // 2 + 3] = 2
    psi_w = np.where(w != 1, rng.uniform(0.3, 0.7, size=V), 0.0)
    n0 = 1.0 + 0.3 * np.sin(2 * np.pi * np.arange(V) / 17 + 0.3)
    fl = w == 1
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
        eng.init_pop(b, n, u)
        swapped = eng.run(a, b, steps, n=n, psi=psi, u=u, write_fields=wf, two_pass=two_pass)
        assert swapped == (steps % 2 == 1)
        out.append((eng.pop_to_host_soa(b if swapped else a).reshape(9, V)[:, fl], n.D2H()[fl],
                    psi.D2H(), u.D2H().reshape(2, V)[:, fl]))
        for x in (n, psi, u, a, b):
            x.Free()
        eng.close()
    wd.Free()
    for r, t in zip(*out):
        assert np.isfinite(t).all() and np.array_equal(r, t)
