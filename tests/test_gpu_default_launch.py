"""The launch a 3D simulation starts with (the LDS-staged step on the
x-shifted storage, its tile and march length by the lattice; registers on
small lattices, for reach-2 stencils in FP64 and for the dense MRT) against
the register launch of every lattice, on sizes at the edges of the rule: the
same arithmetic per site, equal in FP64."""
import numpy as np
import pytest

from helpers import droplet_field

pytestmark = pytest.mark.gpu

CASES = [('D3E4', (59, 59, 58), 'fp64', 'bgk', True), ('D3E4', (53, 61, 61), 'fp64', 'mrt', False),
         ('D3E4', (129, 33, 47), 'fp64', 'sc', True), ('D3E4', (33, 129, 48), 'fp64', 'mrt', True),
         ('D3E4', (7, 5, 6001), 'fp64', 'bgk', True), ('D3E4', (70, 69, 49), 'fp64', 'dense', False),
         ('D3E8', (66, 61, 53), 'fp64', 'bgk', False), ('D3E6', (97, 75, 69), 'fp32s', 'bgk', True),
         ('D3E4', (81, 77, 81), 'fp32s', 'mrt', True), ('D3E4', (79, 79, 80), 'fp32s', 'mrt', False)]


@pytest.mark.parametrize('es,dims,prec,coll,staged', CASES)
def test_default_launch_equals_register_launch(tenet, es, dims, prec, coll, staged):
    from idmx.IdpyCode import IdpyMemory
    from idmx.LBM import hermite
    from idmx.LBM._base import PopArray
    from idmx.LBM._engine import SCEngine
    S = np.diag(np.linspace(0.7, 1.5, 19))
    if coll == 'dense':
        S[5, 6] = 0.05
    kw = {'mrt': hermite.mrt_kernel_tables('D3Q19', S)} if coll in ('mrt', 'dense') else \
        {'forcing': 'sc'} if coll == 'sc' else {}
    n0 = droplet_field(dims, seed=9) if min(dims) > 8 else \
        1.0 + 0.3 * np.sin(2 * np.pi * np.arange(int(np.prod(dims))) / 4000)
    out = []
    for default in (True, False):
        eng = SCEngine(tenet, 'D3Q19', es, dims, 'exp', -5.0 / 3.0, 1.0, precision=prec,
                       rho0=1.0, **kw)
        assert (eng.get_launch()[3] == 10) == staged
        if not default:
            eng.set_launch(32, 8, 5, 1)
        V = eng.V
        n = IdpyMemory.OnDevice(n0, tenet)
        psi = IdpyMemory.Zeros(V, np.float64, tenet)
        u = IdpyMemory.Zeros(3 * V, np.float64, tenet)
        a, b = PopArray(eng, tenet), PopArray(eng, tenet)
        eng.init_pop(a, n, u)
        swapped = eng.run(a, b, 5, n=n, psi=psi, u=u, write_fields=True,
                          two_pass=not default and coll == 'sc')
        out.append([(b if swapped else a).RawD2H(), n.D2H(), psi.D2H()])
        for x in (a, b, n, psi, u):
            x.Free()
        eng.close()
    for r, g in zip(out[1], out[0]):
        assert np.isfinite(g).all()
        if prec == 'fp64':
            assert np.array_equal(r, g)
        else:
            # ~10 roundings of 6e-8 of the largest value per step
            assert np.abs(r - g).max() <= 5 * 10 * 6e-8 * np.abs(r).max()
