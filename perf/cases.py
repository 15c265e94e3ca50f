"""The work that users of this package have it do, as timed cases.

A case is a dict of plain values. Three kinds, each through the package's
Python surface:

  loop   ShanChenMultiPhase: one checkpoint interval of MainLoop,
         MainLoopMRT, MainLoopSimpleSC or MainLoopSimpleWallsGravity on a
         droplet field, as a notebook runs it between two looks at the
         fields (optionally with the velocity-convergence callback)
  sweep  Batch: one check interval of a batched (G, R, L) sweep (200 steps
         and the residual check, as run_sweep does) and the read-out of the
         relaxed fields
  net    the warm-start U-Net: a forward pass over a batch of sweep points,
         or one training step (forward, loss, backward, Adam)

Simulations use the library's default launch: the classes and run_sweep call
no autotuner. Sizes are those of the package's workloads (the 128^2 droplet,
the 4096^2 field of 64 droplets, the 256^3 sphere, sweeps of 64^2 to 256^2
domains, batches of 64 x 64 images) and ragged ones between them.
"""
import math
import os
import random  # noqa: F401  (draw takes a random.Random)
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'idea.deploy_amd')
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

N_G, N_L, WIDTH = 0.1, 2.0, 2.0
SC_G = -5.0 / 3.0

XIS = {2: ((0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)),
       3: ((0, 0, 0), (1, 0, 0), (0, 1, 0), (-1, 0, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1),
           (1, 1, 0), (-1, 1, 0), (-1, -1, 0), (1, -1, 0),
           (1, 0, 1), (-1, 0, 1), (-1, 0, -1), (1, 0, -1),
           (0, 1, 1), (0, -1, 1), (0, -1, -1), (0, 1, -1))}
XI_W = {2: {0: 4 / 9, 1: 1 / 9, 2: 1 / 36}, 3: {0: 1 / 3, 1: 1 / 18, 2: 1 / 36}}
# isotropic-gradient weights by squared length of the vector
E_W = {(2, 4): {1: 1 / 3, 2: 1 / 12},
       (2, 6): {1: 4 / 15, 2: 1 / 10, 4: 1 / 120},
       (2, 8): {1: 4 / 21, 2: 4 / 45, 4: 1 / 60, 5: 2 / 315, 8: 1 / 5040},
       (3, 4): {1: 1 / 6, 2: 1 / 12},
       (3, 6): {1: 2 / 15, 2: 1 / 15, 3: 1 / 60, 4: 1 / 120},
       (3, 8): {1: 4 / 45, 2: 1 / 21, 3: 2 / 105, 4: 5 / 504, 5: 1 / 315, 6: 1 / 630, 8: 1 / 5040}}

# the U-Net's layers: (name, input channels, output channels, image size / 64)
NET = (('c1a', 8, 16, 1), ('c1b', 16, 16, 1), ('c2a', 16, 32, 2), ('c2b', 32, 32, 2),
       ('c3a', 32, 64, 4), ('c3b', 64, 64, 4), ('c4a', 64, 64, 8), ('c4b', 64, 64, 8),
       ('d3a', 128, 32, 4), ('d3b', 32, 32, 4), ('d2a', 64, 16, 2), ('d2b', 16, 16, 2),
       ('d1a', 32, 16, 1), ('d1b', 16, 16, 1), ('head', 16, 1, 1))


def _loop(name, dims, e, coll, steps, prec='fp64', tau=1.0, droplets=1, check=False):
    c = {'kind': 'loop', 'dim': len(dims), 'L0': dims[0], 'L1': dims[1],
         'L2': dims[2] if len(dims) == 3 else 1, 'e': e, 'coll': coll, 'steps': steps,
         'prec': prec, 'tau': tau, 'droplets': droplets, 'check': check}
    if name:
        c['name'] = name
    return c


def listed():
    return [
        # the smallest work: the 128^2 droplet between two looks at it;
        # a step is a few microseconds, so launches and latency count
        _loop('droplet_128', (128, 128), 4, 'bgk', 200),
        # a parameter point of a study: mid-size, ragged, Shan-Chen forcing
        _loop('forcing_sc_ragged', (1000, 613), 4, 'sc', 50, tau=0.9),
        # a channel with solid walls and gravity, wetting by the walls' psi
        _loop('walls_gravity', (1024, 768), 4, 'walls', 40),
        # many droplets on a large 2D lattice, eighth-order isotropy
        _loop('droplets_4096_e8', (4096, 4096), 8, 'bgk', 20, droplets=64),
        # a small 3D droplet, MRT: latency-bound in 3D
        _loop('droplet3d_small_mrt', (48, 44, 40), 4, 'mrt', 100, tau=0.9),
        # a mid-size ragged 3D run that watches its velocity converge
        _loop('droplet3d_ragged_check', (150, 101, 93), 4, 'bgk', 20, check=True),
        # 3D with the 92-vector stencil
        _loop('droplet3d_e8', (96, 96, 96), 8, 'bgk', 20),
        # the large 3D sphere, MRT, in both population precisions
        _loop('sphere_256_mrt', (256, 256, 256), 4, 'mrt', 20),
        _loop('sphere_256_mrt_fp32s', (256, 256, 256), 4, 'mrt', 20, prec='fp32s'),
        # a sweep's check interval with all its domains live
        {'name': 'sweep_64_domains', 'kind': 'sweep', 'domains': 64, 'Lmin': 64, 'Lmax': 256,
         'e': 4, 'steps': 200},
        # warm starts predicted for a 128-point sweep
        {'name': 'net_predict_128', 'kind': 'net', 'batch': 128, 'train': False},
        # one training step of the warm-start network
        {'name': 'net_train_32', 'kind': 'net', 'batch': 32, 'train': True},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    k = rng.random()
    if k < 0.12:
        return {'kind': 'net', 'batch': int(round(_log(rng, 4, 128))),
                'train': False} if rng.random() < 0.5 else \
            {'kind': 'net', 'batch': int(round(_log(rng, 4, 64))), 'train': True}
    if k < 0.27:
        lmin = 32 * rng.randint(2, 4)
        return {'kind': 'sweep', 'domains': rng.randint(3, 64), 'Lmin': lmin,
                'Lmax': lmin + 32 * rng.randint(0, 4), 'e': rng.choice((4, 4, 8)),
                'steps': 200}
    dim = rng.choice((2, 3))
    sites = _log(rng, 16e3, 12e6)
    coll = rng.choice(('bgk', 'bgk', 'mrt', 'sc', 'walls'))
    e = 4 if coll in ('sc', 'walls') else rng.choice((4, 4, 6, 8))
    side = sites ** (1.0 / dim)
    dims = [max(24, int(side * _log(rng, 0.6, 1.67))) for _ in range(dim - 1)]
    dims.append(max(24, int(sites / math.prod(dims))))
    if rng.random() < 0.3:      # sizes that are multiples of a tile
        dims = [max(32, 32 * round(d / 32)) for d in dims]
    V = math.prod(dims)
    cost = 250.0 if (dim, e) == (3, 8) else 120.0 if dim == 3 else 60.0
    steps = max(6, min(200, int(20 * 16.7e6 * 60 / (V * cost))))
    prec = 'fp32s' if coll in ('bgk', 'mrt') and rng.random() < 0.25 else 'fp64'
    check = coll in ('bgk', 'mrt') and prec == 'fp64' and rng.random() < 0.25
    return _loop('', tuple(dims), e, coll, steps, prec, rng.choice((0.9, 1.0, 1.1)),
                 rng.choice((1, 1, 8)) if dim == 2 and V > 200000 else 1, check)


# -- inputs ---------------------------------------------------------------------
def _dims(case):
    return (case['L0'], case['L1'], case['L2'])[:case['dim']]


def _density(case, seed):
    """Tanh droplets of liquid in gas plus uniform noise of 1e-4: the
    simulation's initial density, float64 on the GPU, slowest axis first."""
    dims = _dims(case)
    rng = np.random.default_rng(seed)
    g = torch.Generator(device='cuda').manual_seed(seed)
    axes = [torch.arange(L, dtype=torch.float64, device='cuda') for L in dims]
    n = torch.full(dims[::-1], N_G, dtype=torch.float64, device='cuda')
    count = case['droplets']
    rmax = 0.25 * min(dims) if count == 1 else 60.0 / 4096 * min(dims) * 8 / math.sqrt(count)
    for k in range(count):
        R = rmax * rng.uniform(0.7, 1.0)
        r2 = 0
        for d, (x, L) in enumerate(zip(axes, dims)):
            c = L / 2 + rng.uniform(-2, 2)
            if count > 1:   # one droplet per cell of a grid of cells
                m = math.ceil(math.sqrt(count))
                c = L * ((k % m, k // m)[d] + 0.5 + rng.uniform(-0.1, 0.1)) / m
            dx = x - c
            dx = dx - L * torch.round(dx / L)
            r2 = r2 + (dx * dx).reshape([L if j == len(dims) - 1 - d else 1
                                         for j in range(len(dims))])
        n += (N_L - N_G) * 0.5 * (1.0 - torch.tanh((r2.sqrt() - R) / WIDTH))
    n.clamp_(N_G, N_L)
    n += 1e-4 * (2 * torch.rand(n.shape, dtype=torch.float64, device='cuda', generator=g) - 1)
    return n


def _channel(case, seed):
    """Plates at both ends of the last axis and a solid block inside, with
    the psi that the solid sites carry."""
    dims = _dims(case)
    rng = np.random.default_rng(seed + 1)
    w = np.ones(dims[::-1], dtype=np.uint8)
    w[0] = w[-1] = 0
    lo = [int(L * rng.uniform(0.05, 0.15)) for L in dims]
    w[tuple(slice(a, a + max(2, L // 10)) for a, L in zip(lo[::-1], dims[::-1]))] = 0
    return w, np.where(w == 0, rng.uniform(0.3, 0.7), 0.0)


def _net_inputs(case, seed):
    """Images of random sweep points (x, y, r over L, cold tanh droplet, G,
    R / L, L / 512 and a zero channel) and correction targets."""
    N, S = case['batch'], 64
    rng = np.random.default_rng(seed)
    g = torch.Generator(device='cuda').manual_seed(seed)
    L = torch.tensor(rng.choice(np.arange(64, 513, 32), N), dtype=torch.float32, device='cuda')
    G = torch.tensor(rng.uniform(-5.5, -4.2, N) / 3, dtype=torch.float32, device='cuda')
    R = L * torch.tensor(rng.uniform(0.1, 0.35, N), dtype=torch.float32, device='cuda')
    one = torch.ones((N, S, S), device='cuda')
    c = (torch.arange(S, device='cuda') + 0.5)[None] * L[:, None] / S - 0.5 - L[:, None] / 2
    dx, dy = c[:, None, :] * one, c[:, :, None] * one
    r = (dx * dx + dy * dy).sqrt()
    col = lambda v: v[:, None, None] * one  # noqa: E731
    base = 0.5 * (N_G + N_L) - 0.5 * (N_L - N_G) * torch.tanh((r - col(R)) / WIDTH)
    x = torch.stack([dx / col(L), dy / col(L), r / col(L), base, col(G) * 0.6 + 1.0, col(R / L),
                     col(L / 512), 0 * one], -1)
    tgt = 0.3 * torch.exp(-((r - col(R)) / (0.1 * col(L))) ** 2) \
        + 0.01 * torch.randn((N, S, S), device='cuda', generator=g)
    return x.to(torch.bfloat16), tgt


def _net_weights(seed):
    """Float32 weights and biases, and the moments of a training that runs."""
    rng = np.random.default_rng(seed + 2)
    out = {}
    for name, ci, co, _ in NET:
        w = (rng.standard_normal((co, 9 * ci)) * math.sqrt(2.0 / (9 * ci))).astype(np.float32)
        w *= 0.3 if name == 'head' else 1.0
        out[name] = {'w': w, 'b': (0.05 * rng.standard_normal(co)).astype(np.float32)}
        for k, sh in (('', (co, 9 * ci)), ('b', (co,))):
            out[name]['m' + k] = (1e-3 * rng.standard_normal(sh)).astype(np.float32)
            out[name]['v' + k] = (1e-4 * rng.uniform(0.5, 1.5, sh)).astype(np.float32)
    return out


NET_STEP, NET_LR = 400, 2.5e-4   # late in a training


def _points(case, seed):
    """(L, G, R) of the sweep's domains: sizes in steps of 32, evenly used."""
    rng = np.random.default_rng(seed)
    sizes = list(range(case['Lmin'], case['Lmax'] + 1, 32))
    out = []
    for i in range(case['domains']):
        L = sizes[i % len(sizes)]
        out.append((L, float(rng.uniform(-5.4, -4.8)) / 3.0, float(rng.uniform(0.12, 0.35) * L)))
    return out


# -- the cases ------------------------------------------------------------------
class _View:
    """A device buffer of the library as an array that torch can share."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {'data': (int(ptr), False), 'shape': tuple(shape),
                                         'typestr': typestr, 'version': 2}


def _view(buf, shape, typestr='<f8'):
    return torch.as_tensor(_View(buf.ptr.value, shape, typestr), device='cuda')


def prepare(case, seed):
    return {'loop': _prepare_loop, 'sweep': _prepare_sweep, 'net': _prepare_net}[
        case['kind']](case, seed)


def _prepare_loop(case, seed):
    import sympy as sp
    from idmx.IdpyCode import HIP_T
    from idmx.LBM.MultiPhase import FStencils, ShanChenMultiPhase, XIStencils
    dims = _dims(case)
    D, Q = len(dims), len(XIS[len(dims)])
    sim = ShanChenMultiPhase(
        lang=HIP_T, dim_sizes=dims, xi_stencil=XIStencils['D%dQ%d' % (D, Q)],
        f_stencil=FStencils['D%dE%d' % (D, case['e'])], psi_code='1. - exp(-ln_0)',
        psi_sym=1 - sp.exp(-sp.Symbol('n')), SC_G=SC_G, tau=case['tau'],
        precision=case['prec'], set_ordering='gpu')
    sim.SetDensityField(_density(case, seed).cpu().numpy())
    m = sim.sims_idpy_memory
    s = {'case': case, 'sim': sim, 'times': [0, case['steps']]}
    shape, t = dims[::-1], '<f8' if case['prec'] == 'fp64' else '<f4'
    if case['coll'] == 'walls':
        sim.GetWalls(*_channel(case, seed))
    elif case['coll'] == 'mrt':
        s['S'] = np.eye(Q) / case['tau']
    s['views'] = {m[k].ptr.value: _view(m[k], (Q,) + shape, t) for k in ('pop', 'pop_swap')}
    s['fields'] = {k: _view(m[k], shape) for k in ('n', 'psi')}
    s['fields']['u'] = _view(m['u'], (D,) + shape)
    if case['check']:
        from idmx.LBM.MultiPhaseLoopChecks import CheckUConvergenceSCMP
        s['checks'] = [CheckUConvergenceSCMP]
    sim.tenet.Sync()
    return s


def _prepare_sweep(case, seed):
    from idmx.IdpyCode import Tenet
    from idmx.sweep import Batch, SweepPoint, cold_start
    pts = [SweepPoint(L=L, G=G, R=R) for L, G, R in _points(case, seed)]
    tenet = Tenet(0)
    b = Batch(tenet, pts, 'fp64', 'E%d' % case['e'])
    for i, p in enumerate(pts):
        b.set_density(i, cold_start(p))
    b.check()
    tenet.Sync()
    return {'case': case, 'tenet': tenet, 'batch': b}


def _prepare_net(case, seed):
    from idmx.IdpyCode import Tenet
    from idmx.warmstart import UNet
    tenet = Tenet(0)
    net = UNet(tenet, case['batch'], seed=seed)
    x, tgt = _net_inputs(case, seed)
    ws = _net_weights(seed)
    net.set_weights({k: (w['w'], w['b']) for k, w in ws.items()})
    net.set_input(x.view(torch.int16).cpu().numpy())
    s = {'case': case, 'tenet': tenet, 'net': net}
    if case['train']:
        net.tgt.h2d(tgt.cpu().numpy())
        for k, w in ws.items():
            for f in ('m', 'v', 'mb', 'vb'):
                net.layers[k][f].h2d(w[f])
        net.step = NET_STEP
        s['out'] = {k: {f: _view(net.layers[k][f], ws[k][f].shape, '<f4')
                        for f in ('w', 'b', 'm', 'v')} for k in ws}
    else:
        s['out'] = _view(net.out32, (case['batch'], 64, 64), '<f4')
    tenet.Sync()
    return s


def run(s):
    c = s['case']
    if c['kind'] == 'net':
        net = s['net']
        net.forward()
        if not c['train']:
            return s['out']
        loss = net.loss_and_grad()
        net.backward()
        net.adam(lr=NET_LR)
        return {'loss': loss, 'state': s['out']}
    if c['kind'] == 'sweep':
        b = s['batch']
        b.run(c['steps'])
        dn = b.check()
        return {'dn': dn, 'n': np.concatenate([b.get_density(i).ravel() for i in range(b.n)])}
    sim, f = s['sim'], s['fields']
    if c['coll'] == 'mrt':
        sim.MainLoopMRT(s['times'], relaxation_matrix=s['S'], omega_syms_vals=[],
                        convergence_functions=s.get('checks', []))
    elif c['coll'] == 'sc':
        sim.MainLoopSimpleSC(s['times'])
    elif c['coll'] == 'walls':
        # the solid sites' populations are not defined: the fields are
        sim.MainLoopSimpleWallsGravity(s['times'], g=1e-5)
        return f
    else:
        sim.MainLoop(s['times'], convergence_functions=s.get('checks', []))
    pop = s['views'][sim.sims_idpy_memory['pop'].ptr.value]
    if c['prec'] == 'fp32s':
        return {'pop': pop}     # n and psi are float32 sums of these, kept in float64 arrays
    out = {'pop': pop, 'n': f['n'], 'psi': f['psi']}
    if c['coll'] == 'sc' or c['check']:
        out['u'] = f['u']
    if c['check']:
        out['u_conv'] = float(sim.sims_vars['u_conv'][-1])
        out['max_u'] = float(sim.sims_vars['max_u'][-1])
    return out


def work(case):
    """One pass. A step of a loop or sweep reads and writes every population
    once (a step is the unit of the method: its result is the next one's
    input), a pass also writes the fields; the network reads its input and
    weights and writes its output, in training each layer's output once and
    reads it once."""
    if case['kind'] == 'net':
        N = case['batch']
        flops = sum(2.0 * 9 * ci * co * N * (64 // r) ** 2 for _, ci, co, r in NET)
        params = sum(9 * ci * co + co for _, ci, co, _ in NET)
        nbytes = N * 4096 * (8 * 2 + 4) + 2.0 * params
        if case['train']:
            first = 2.0 * 9 * 8 * 16 * N * 4096     # no gradient for the images
            flops = 3 * flops - first
            nbytes += sum(4.0 * co * N * (64 // r) ** 2 for _, _, co, r in NET) + 28.0 * params
        return {'bytes': nbytes, 'flops': flops}
    if case['kind'] == 'sweep':
        V = sum(L * L for L, _, _ in _points(case, 0))
        D, Q, s, fields = 2, 9, 8, 2 * 8
    else:
        V = math.prod(_dims(case))
        D, Q = case['dim'], len(XIS[case['dim']])
        s = 8 if case['prec'] == 'fp64' else 4
        fields = 8 * (2 + (D if case['coll'] in ('sc', 'walls') or case['check'] else 0))
    e = len(_stencil(D, case['e']))
    flops = Q * 20.0 + e * 2 * D + 40      # moments, equilibrium, forcing; gradient; psi
    return {'bytes': V * (case['steps'] * 2.0 * Q * s + fields), 'flops': V * case['steps'] * flops}


# -- 64-bit values ----------------------------------------------------------------
def _stencil(D, e):
    w = E_W[(D, e)]
    r = range(-2, 3)
    pts = [(a, b) for a in r for b in r] if D == 2 else \
        [(a, b, c) for a in r for b in r for c in r]
    return [(p, w[sum(v * v for v in p)]) for p in pts if sum(v * v for v in p) in w]


def _shift(a, c, D):
    """a(x - c) on the last D axes (x is the last)."""
    return torch.roll(a, shifts=tuple(c), dims=tuple(-1 - d for d in range(D)))


class _Lattice:
    """The Shan-Chen step in 64 bits on [.., z, y, x] arrays."""

    def __init__(self, D, e, G, tau, coll='bgk', fluid=None, psi_w=None, g=0.0):
        self.D, self.G, self.om, self.coll = D, G, 1.0 / tau, coll
        self.xi, self.E = XIS[D], _stencil(D, e)
        self.w = [XI_W[D][sum(v * v for v in c)] for c in self.xi]
        self.opp = [self.xi.index(tuple(-v for v in c)) for c in self.xi]
        self.fluid, self.psi_w, self.g = fluid, psi_w, g
        if fluid is not None:
            self.from_solid = [~_shift(fluid, c, D) for c in self.xi]

    def start(self, n):
        return [w * n for w in self.w]

    def fields(self, f):
        n = sum(f)
        psi = 1.0 - torch.exp(-n)
        if self.fluid is not None:
            psi = torch.where(self.fluid, psi, self.psi_w)
        F = [0.0] * self.D
        for c, w in self.E:
            v = _shift(psi, [-a for a in c], self.D) * w
            for d in range(self.D):
                if c[d]:
                    F[d] = F[d] + c[d] * v
        F = [-self.G * psi * a for a in F]
        F[1] = F[1] + self.g
        j = [sum(c[d] * a for c, a in zip(self.xi, f) if c[d]) for d in range(self.D)]
        return n, psi, F, j

    def step(self, f):
        """(populations after the step; n, psi and u of the step)"""
        n, psi, F, j = self.fields(f)
        om, D = self.om, self.D
        if self.coll == 'sc':
            u0 = [a / n for a in j]
            u = [a + b / n / om for a, b in zip(u0, F)]
        else:
            u = [(a + 0.5 * b) / n for a, b in zip(j, F)]
        uu = sum(a * a for a in u)
        Fu = sum(a * b for a, b in zip(F, u))
        out = []
        for c, w, a in zip(self.xi, self.w, f):
            cu = sum(v * b for v, b in zip(c, u) if v) if any(c) else torch.zeros_like(n)
            b = (1 - om) * a + om * w * n * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * uu)
            if self.coll != 'sc':
                cF = sum(v * e for v, e in zip(c, F) if v) if any(c) else torch.zeros_like(n)
                b = b + (1 - 0.5 * om) * w * (3 * cF + 9 * cF * cu - 3 * Fu)
            out.append(b)
        if self.coll == 'sc':
            j1 = [sum(c[d] * a for c, a in zip(self.xi, out) if c[d]) for d in range(D)]
            u = [0.5 * (a + b / n) for a, b in zip(u0, j1)]
        new = [_shift(a, c, D) for c, a in zip(self.xi, out)]
        if self.fluid is not None:
            new = [torch.where(s, out[o], a)
                   for s, o, a in zip(self.from_solid, self.opp, new)]
        return new, n, psi, u


def exact(case, seed):
    return {'loop': _exact_loop, 'sweep': _exact_sweep, 'net': _exact_net}[
        case['kind']](case, seed)


def _exact_loop(case, seed):
    n0 = _density(case, seed)
    kw = {}
    if case['coll'] == 'walls':
        w, psi_w = _channel(case, seed)
        kw = {'fluid': torch.from_numpy(w).cuda() == 1, 'psi_w': torch.from_numpy(psi_w).cuda(),
              'g': 1e-5}
    # all rates equal: the MRT collision is the BGK one
    lat = _Lattice(case['dim'], case['e'], SC_G, case['tau'],
                   'sc' if case['coll'] == 'sc' else 'bgk', **kw)
    f = lat.start(n0)
    for _ in range(case['steps']):
        f, n, psi, u = lat.step(f)
    if case['coll'] == 'walls':
        fl = kw['fluid']
        u = torch.stack([torch.where(fl, a, torch.zeros_like(a)) for a in u])
        return {'n': torch.where(fl, n, n0), 'psi': psi, 'u': u}
    if case['prec'] == 'fp32s':
        return {'pop': torch.stack([a - w for a, w in zip(f, lat.w)])}
    if case['check']:
        n, psi, F, j = lat.fields(f)
        u = [(a + 0.5 * b) / n for a, b in zip(j, F)]
    out = {'pop': torch.stack(f), 'n': n, 'psi': psi}
    if case['coll'] == 'sc' or case['check']:
        out['u'] = torch.stack(u)
    if case['check']:
        out['u_conv'] = float(out['u'].abs().sum() / n.numel())
        out['max_u'] = math.sqrt(float(sum(a * a for a in u).max()) * 3.0)
    return out


def _exact_sweep(case, seed):
    pts = _points(case, seed)
    n_out, dn = [None] * len(pts), np.zeros(len(pts))
    for L in sorted({p[0] for p in pts}):
        idx = [i for i, p in enumerate(pts) if p[0] == L]
        x = torch.arange(L, dtype=torch.float64, device='cuda') - L // 2
        r = (x[None, :] ** 2 + x[:, None] ** 2).sqrt()[None]
        R, G = (torch.tensor([pts[i][k] for i in idx], dtype=torch.float64,
                             device='cuda')[:, None, None] for k in (2, 1))
        n0 = 0.5 * (N_G + N_L) - 0.5 * (N_L - N_G) * torch.tanh((r - R) / WIDTH)
        lat = _Lattice(2, case['e'], G, 1.0)
        f = lat.start(n0)
        for _ in range(case['steps']):
            f = lat.step(f)[0]
        n = sum(f)
        d = (n - n0).abs().amax(dim=(1, 2)).cpu().numpy()
        for k, i in enumerate(idx):
            n_out[i], dn[i] = n[k].reshape(-1).cpu().numpy(), d[k]
    return {'dn': dn, 'n': np.concatenate(n_out)}


def _bf(a):
    """Rounded to bf16, the network's storage of activations and weights."""
    return a.to(torch.bfloat16).to(torch.float64)


def _conv(x, w, co):
    """3x3 convolution, zero padding, of [N, H, W, C] by [co, 9 C]."""
    N, H, W, C = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    cols = torch.cat([p[:, a:a + H, b:b + W] for a in range(3) for b in range(3)], -1)
    return (cols.reshape(-1, 9 * C) @ w.t()).reshape(N, H, W, co)


class _Round(torch.autograd.Function):
    """bf16 storage of a value and of its gradient."""

    @staticmethod
    def forward(ctx, a):
        return _bf(a)

    @staticmethod
    def backward(ctx, g):
        return _bf(g)


def _exact_net(case, seed):
    x, tgt = _net_inputs(case, seed)
    ws = _net_weights(seed)
    par = {k: {f: torch.from_numpy(v).cuda().double() for f, v in w.items()}
           for k, w in ws.items()}
    rnd = _Round.apply
    leaf = {k: (_bf(p['w']).requires_grad_(case['train']),
                p['b'].clone().requires_grad_(case['train'])) for k, p in par.items()}

    def layer(name, a):
        y = _conv(a, leaf[name][0], leaf[name][1].numel()) + leaf[name][1]
        return y if name == 'head' else rnd(torch.relu(y))

    def pool(a):
        N, H, W, C = a.shape
        return rnd(a.reshape(N, H // 2, 2, W // 2, 2, C).mean(dim=(2, 4)))

    def up(a):
        return a.repeat_interleave(2, 1).repeat_interleave(2, 2)

    c1 = layer('c1b', layer('c1a', x.double()))
    c2 = layer('c2b', layer('c2a', pool(c1)))
    c3 = layer('c3b', layer('c3a', pool(c2)))
    c4 = layer('c4b', layer('c4a', pool(c3)))
    d3 = layer('d3b', layer('d3a', torch.cat([up(c4), c3], -1)))
    d2 = layer('d2b', layer('d2a', torch.cat([up(d3), c2], -1)))
    d1 = layer('d1b', layer('d1a', torch.cat([up(d2), c1], -1)))
    y = layer('head', d1)[..., 0]
    if not case['train']:
        return y
    loss = ((y - tgt.double()) ** 2).mean()
    loss.backward()
    b1, b2, eps, t = 0.9, 0.999, 1e-8, NET_STEP + 1
    out = {}
    for k, p in par.items():
        o = out[k] = {}
        for f, g in zip(('w', 'b'), leaf[k]):
            q = '' if f == 'w' else 'b'
            m = b1 * p['m' + q] + (1 - b1) * g.grad
            v = b2 * p['v' + q] + (1 - b2) * g.grad ** 2
            o[f] = p[f] - NET_LR * (m / (1 - b1 ** t)) / ((v / (1 - b2 ** t)).sqrt() + eps)
            if f == 'w':
                o['m'], o['v'] = m, v
    return {'loss': float(loss.detach()), 'state': out}
