"""The work that is timed: IB steps, their transfers and their pressure
solves, each through a public entry point, over the sizes of this
repository's benchmark, its many-instance mixes and its tests.

``listed`` names the cases, ``draw`` gives more of the same ranges,
``prepare`` makes what a program has in hand before the call, ``run`` makes
one pass, ``work`` states what the pass cannot do without, ``tolerance`` how
far another correct implementation may be off, and ``exact`` the same
results from plain torch in FP64 without this package (dense index sums for
the transfers, separable eigenvector solves for the pressure).

Every pass solves its pressure from zero and the time steps are tiny: a pass
repeated many times on one state then does the work of the first, with the
points where the case puts them.
"""
from functools import lru_cache
from math import exp, log, pi, prod

import numpy as np
import torch

from afsi_gpu_amd import workloads
from afsi_gpu_amd.batch import BatchedIBStep
from afsi_gpu_amd.mac import MACFlow, MACGrid, MGOptions, cuda_ib
from afsi_gpu_amd.mac.assembled import AssembledTransfer
from afsi_gpu_amd.mac.fe import FEGeometry, FETransfer
from afsi_gpu_amd.mac.multigrid import MIXED_INNER_CYCLES, MIXED_RELAX
from afsi_gpu_amd.mac.transfer import Binner, TiledTransfer, from_points
from afsi_gpu_amd.mac2d import ChannelGrid, ChannelIBStep
from afsi_gpu_amd.mac2d.batch import BatchedChannelStep
from afsi_gpu_amd.step import IBStep

GPU = torch.device('cuda:0')
CHANNEL_DT = 1e-6
STEP_DT = 2e-8
MIX_3D = ('32x32x32:10000,48x48x48:17000,64x64x64:30000,96x96x96:52000,32x32x32:90000,64x64x64:155000,'
          '96x96x96:270000,48x48x48:12000')
MIX_2D = ('128x32:10000,256x64:17000,512x128:30000,128x32:52000,256x64:90000,512x128:155000,'
          '256x64:270000,128x32:12000')


def listed():
    return [
        # one immersed curve pair in a 256x64 channel: the smallest workload
        # of the benchmark set, a chain of small launches
        dict(name='channel_256x64', kind='channel', nx=256, ny=64, points=4096, periodic=True, smoother='rbgs'),
        # the largest served channel, as the inlet/outlet channel with the
        # reference's Jacobi V(4,4) cycle (the default options)
        dict(name='channel_512x128_jacobi', kind='channel', nx=512, ny=128, points=20000, periodic=False,
             smoother='jacobi'),
        # the closed-box flow step (transport screen, predictor, projection)
        # with the default Jacobi V(4,4) options, as the reference's 64^3 runs
        dict(name='flow_closed_64', kind='flow', nx=64, ny=64, nz=64, smoother='jacobi'),
        # the transfer alone on a small, odd point count and a ragged closed
        # box: binning, spread and interpolation of a small body
        dict(name='transfer_40x56x48', kind='transfer', nx=40, ny=56, nz=48, points=30011, periodic=False,
             cloud='shell'),
        # the same at the benchmark's size: 1.5M clustered points
        dict(name='transfer_128_1p5M', kind='transfer', nx=128, ny=128, nz=128, points=1_500_000, periodic=True,
             cloud='clustered'),
        # the reference's own transfer calls on point stencils, 64^3 closed
        dict(name='compact_64_200k', kind='compact', nx=64, ny=64, nz=64, points=200_000, cloud='shell'),
        # an ordinary FP64 step: 64^3 with 200k points
        dict(name='step_fp64_64_200k', kind='step', nx=64, ny=64, nz=64, points=200_000, periodic=True,
             cloud='shell', precision='fp64', graphs=False),
        # the headline step: 128^3, 1.5M clustered points, mixed precision,
        # as HIP graphs
        dict(name='step_mixed_128_1p5M', kind='step', nx=128, ny=128, nz=128, points=1_500_000, periodic=True,
             cloud='clustered', precision='mixed', graphs=True),
        # the P2 left-ventricle wall in a 64^3 box through the fused transfer
        # with both mass solves: 3.87M interaction points
        dict(name='fe_p2_lv_fused', kind='fe', mesh='lv_p2', nt=3, ntheta=48, nphi=70, n=64, mode='fused'),
        # a P1 wall whose operator is assembled to CSR, then applied once in
        # each direction
        dict(name='fe_p1_lv_assembled', kind='fe', mesh='lv_p1', nt=2, ntheta=30, nphi=45, n=96, mode='assembled'),
        # a batch of uneven 3D instances, one launch per phase (mixed)
        dict(name='batch_3d_8', kind='batch3', mix=MIX_3D),
        # a batch of uneven channels
        dict(name='batch_2d_8', kind='batch2', mix=MIX_2D),
    ]


def _log(rng, lo, hi):
    return int(round(exp(rng.uniform(log(lo), log(hi)))))


def _box(rng, largest=128):
    """Cell counts base * 2^m, base 4..8 per axis: coarsenable to <= 512."""
    m = rng.choice((3, 3, 4)) if largest > 64 else 3
    return tuple(rng.randint(4, 8) * 2 ** m for _ in range(3))


def draw(rng):
    kind = rng.choice(('channel', 'flow', 'transfer', 'compact', 'step', 'fe', 'batch3', 'batch2'))
    if kind == 'channel':
        m = rng.choice((3, 4, 5))
        return dict(kind=kind, nx=rng.randint(8, 16) * 2 ** m, ny=4 * 2 ** m, points=_log(rng, 2000, 20000) | 1,
                    periodic=rng.random() < .5, smoother=rng.choice(('rbgs', 'jacobi')))
    if kind == 'batch2':
        shapes = [workloads.GRIDS_2D[rng.randrange(3)] for _ in range(rng.randint(3, 8))]
        return dict(kind=kind, mix=','.join(f'{a}x{b}:{_log(rng, 1e4, 1.5e5)}' for a, b in shapes))
    if kind == 'batch3':
        shapes = [workloads.GRIDS_3D[rng.randrange(4)] for _ in range(rng.randint(3, 8))]
        return dict(kind=kind, mix=','.join(f'{a}x{b}x{c}:{_log(rng, 1e4, 2e5)}' for a, b, c in shapes))
    if kind == 'fe':
        mode = rng.choice(('fused', 'assembled', 'tiled'))
        mesh = 'lv_p2' if mode == 'fused' else 'lv_p1' if mode == 'assembled' else 'sphere'
        if mesh == 'sphere':
            return dict(kind=kind, mesh=mesh, level=rng.randint(4, 7), n=rng.choice((64, 96, 128)), mode=mode)
        most = 2 if mesh == 'lv_p2' else 1
        return dict(kind=kind, mesh=mesh, nt=rng.randint(1, 1 + most), ntheta=rng.randint(12, 16 + 16 * most),
                    nphi=rng.randint(18, 24 + 20 * most), n=rng.choice((48, 64, 80)), mode=mode)
    nx, ny, nz = _box(rng)
    base = dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind == 'flow':
        return dict(base, smoother=rng.choice(('jacobi', 'rbgs')))
    points = _log(rng, 1e4, 1e6 if kind != 'compact' else 4e5) | 1
    cloud = rng.choice(('shell', 'clustered'))
    if kind == 'compact':
        return dict(base, points=points, cloud=cloud)
    base = dict(base, points=points, periodic=rng.random() < .6, cloud=cloud)
    if kind == 'step':
        return dict(base, precision=rng.choice(('fp64', 'mixed')), graphs=rng.random() < .5)
    return base


# ---------------------------------------------------------------------------
# inputs

def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(int(seed) % (1 << 62))


def _uniform(gen, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, generator=gen, device='cuda', dtype=torch.float64)


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device='cuda', dtype=torch.float64)


def _on_ellipsoid(gen, axes, count, thickness=.02, tip=None):
    """``count`` points uniform in area on the ellipsoid about the centre of
    the unit cube, spread over ``thickness`` along the normal; ``tip`` keeps
    those within that distance of the +x tip."""
    a = torch.tensor(axes, device='cuda', dtype=torch.float64)
    weight = torch.stack((a[1] * a[2], a[0] * a[2], a[0] * a[1]))
    kept, have = [], 0
    while have < count:
        m = max(4 * (count - have), 4096)
        if tip is None:
            d = _normal(gen, m, 3)
        else:
            top = min(pi, 2.5 * tip / min(axes[1], axes[2]))
            c = _uniform(gen, float(np.cos(top)), 1., m)
            s, p = (1 - c * c).sqrt(), _uniform(gen, 0., 2 * pi, m)
            d = torch.stack((c, s * p.cos(), s * p.sin()), 1)
        d = d / d.norm(dim=1, keepdim=True)
        keep = _uniform(gen, 0., 1., m) < (d * weight).norm(dim=1) / weight.max()
        surface = d * a
        if tip is not None:
            keep &= (surface - torch.tensor((axes[0], 0., 0.), device='cuda', dtype=torch.float64)).norm(dim=1) <= tip
        surface = surface[keep]
        normal = surface / a ** 2
        normal = normal / normal.norm(dim=1, keepdim=True)
        kept.append(.5 + surface + _uniform(gen, -thickness / 2, thickness / 2, len(surface), 1) * normal)
        have += len(surface)
    return torch.cat(kept)[:count].contiguous()


def _cloud(gen, cloud, count):
    """Positions and forces: one random shell with N(0,1) forces, or the
    benchmark's two nested shells with a tenth of the points in a patch and
    lognormal magnitudes."""
    if cloud == 'shell':
        axes = [float(v) for v in _uniform(gen, .15, .35, 3)]
        return _on_ellipsoid(gen, axes, count), _normal(gen, count, 3)
    outer, inner = (.35, .25, .25), (.3, .2, .2)
    patch = count // 10
    ao, ai = workloads.ellipsoid_area(outer), workloads.ellipsoid_area(inner)
    n_outer = int(round((count - patch) * ao / (ao + ai)))
    x = torch.cat((_on_ellipsoid(gen, outer, n_outer), _on_ellipsoid(gen, inner, count - patch - n_outer),
                   _on_ellipsoid(gen, outer, patch, tip=.05)))
    d = _normal(gen, count, 3)
    return x.contiguous(), _normal(gen, count, 1).exp() * (d / d.norm(dim=1, keepdim=True))


def _curves(gen, count, shape):
    """Two sinusoidal curves along a 4 x 1 channel, kept clear of its ends."""
    hx = 4. / shape[0]
    half = count // 2
    amp, phase = float(_uniform(gen, .05, .15, 1)), float(_uniform(gen, 0., 2 * pi, 1))
    parts = []
    for sign, m in ((1, half), (-1, count - half)):
        x = 3 * hx + (4. - 6 * hx) * (torch.arange(m, device='cuda', dtype=torch.float64) + .5) / m
        parts.append(torch.stack((x, .5 + sign * amp * (2 * pi * x / 4. + phase).sin()), 1))
    x = torch.cat(parts)
    return x + _uniform(gen, -.05 * hx, .05 * hx, *x.shape), _normal(gen, count, 2)


def _faces(gen, grid):
    """A smooth face velocity of a few modes, zero on the walls' normal
    faces of a closed box, of magnitude up to about 1."""
    out = []
    for c in range(3):
        at = grid.coordinates(c, device='cuda')
        if grid.periodic:
            u = torch.zeros(grid.face_shape(c), device='cuda', dtype=torch.float64)
            for _ in range(2):
                k = torch.randint(1, 4, (3,), generator=gen, device='cuda').double() * 2 * pi
                u += .4 * (at @ k + float(_uniform(gen, 0., 6., 1))).sin()
        else:
            amp = float(_uniform(gen, .3, .9, 1))
            u = amp * torch.ones(grid.face_shape(c), device='cuda', dtype=torch.float64)
            for a in range(3):
                u = u * ((pi * at[..., a]).sin() if a == c else (pi * at[..., a]).cos())
            u.narrow(c, 0, 1).zero_()
            u.narrow(c, u.shape[c] - 1, 1).zero_()
        out.append(u.contiguous())
    return tuple(out)


@lru_cache(maxsize=8)
def _mesh(mesh, *shape):
    if mesh == 'sphere':
        return workloads.fe_sphere(shape[0])
    make = workloads.lv_p2 if mesh == 'lv_p2' else workloads.lv_p1
    return make(nt=shape[0], ntheta=shape[1], nphi=shape[2])


def _case_mesh(case):
    if case['mesh'] == 'sphere':
        return _mesh('sphere', case['level'])
    return _mesh(case['mesh'], case['nt'], case['ntheta'], case['nphi'])


def _fe_inputs(case, seed):
    """The mesh in its reference shape, nodes moved by a seeded smooth
    motion, smooth nodal forces of the mass-weighted kind and a velocity."""
    gen = _gen(seed)
    nodes, cells, values, weights = _case_mesh(case)
    t = lambda a, dtype=torch.float64: torch.tensor(a, device='cuda', dtype=dtype)
    geometry = FEGeometry(t(cells, torch.int64), t(values), t(weights), len(nodes))
    X = t(nodes)
    k = _uniform(gen, 2., 6., 3, 3)
    x = .5 + (X - .5) * (1 - .04 * torch.rand((), generator=gen, device='cuda', dtype=torch.float64))
    x = x + .004 * (X @ k).sin()
    density = (X @ _uniform(gen, 2., 12., 3, 3)).cos() + .3 * _normal(gen, *X.shape)
    lump = torch.zeros(len(nodes), device='cuda', dtype=torch.float64).index_add_(
        0, geometry.cells.reshape(-1), (geometry.weights @ geometry.values).reshape(-1))
    grid = MACGrid((case['n'],) * 3, (1., 1., 1.))
    return grid, geometry, x.contiguous(), (density * lump[:, None].abs()).contiguous(), _faces(gen, grid)


def _grid(case):
    return MACGrid((case['nx'], case['ny'], case['nz']), (1., 1., 1.), periodic=bool(case.get('periodic', False)))


def _flow_dt(case):
    return 1e-3 * min(1., (64 / max(case['nx'], case['ny'], case['nz'])) ** 2)


def _options(smoother):
    return MGOptions() if smoother == 'jacobi' else MGOptions(smooth=2, smoother='rbgs')


def _mix(case):
    """[(shape, points)] of a batch."""
    items = []
    for part in case['mix'].split(','):
        shape, points = part.split(':')
        items.append((tuple(int(n) for n in shape.split('x')), int(points)))
    return items


def _channel_inputs(case, seed):
    gen = _gen(seed)
    shape = (case['nx'], case['ny'])
    grid = ChannelGrid(shape, (4., 1.), bool(case['periodic']))
    x, F = _curves(gen, case['points'], shape)
    # a through-flow with a swirl; the wall-normal faces are zero
    u, v = grid.zeros(device='cuda')
    y = grid.coordinates(0, device='cuda')
    u += .1 * y[..., 1] * (1 - y[..., 1]) * (1 + .2 * (2 * pi * y[..., 0] / 4 + float(_uniform(gen, 0., 6., 1))).sin())
    y = grid.coordinates(1, device='cuda')
    v += .02 * (pi * y[..., 1]).sin() * (2 * pi * y[..., 0] / 4 + float(_uniform(gen, 0., 6., 1))).cos()
    v[:, 0] = 0
    v[:, -1] = 0
    return grid, x, F, (u, v)


def _batch_inputs(case, seed):
    gen = _gen(seed)
    items = _mix(case)
    if case['kind'] == 'batch3':
        grids = [MACGrid(s, (1., 1., 1.), periodic=True) for s, _ in items]
        clouds = [_cloud(gen, 'shell', p) for _, p in items]
    else:
        grids = [ChannelGrid(s, (4., 1.), periodic=True) for s, _ in items]
        clouds = [_curves(gen, p, s) for s, p in items]
    return grids, [c[0] for c in clouds], [c[1] for c in clouds]


def _points_inputs(case, seed):
    gen = _gen(seed)
    grid = _grid(case)
    x, F = _cloud(gen, case['cloud'], case['points'])
    return grid, x, F, _faces(gen, grid)


def _flow_inputs(case, seed):
    gen = _gen(seed)
    grid = _grid(case)
    u = _faces(gen, grid)
    return grid, u, tuple(5 * f + .5 * _normal(gen, *f.shape) for f in _faces(gen, grid))


def prepare(case, seed):
    kind = case['kind']
    if kind == 'channel':
        grid, x, F, u = _channel_inputs(case, seed)
        stepper = ChannelIBStep(grid, dt=CHANNEL_DT, device=GPU, options=_options(case['smoother']))
        return dict(kind=kind, stepper=stepper, x=x, F=F, u=u)
    if kind == 'flow':
        grid, u, f = _flow_inputs(case, seed)
        flow = MACFlow(grid, dt=_flow_dt(case), mu=.01, device=GPU, options=_options(case['smoother']))
        return dict(kind=kind, flow=flow, u=u, f=f)
    if kind == 'transfer':
        grid, x, F, u = _points_inputs(case, seed)
        return dict(kind=kind, binner=Binner(grid, len(x), GPU), transfer=TiledTransfer(grid, GPU), x=x, F=F, u=u)
    if kind == 'compact':
        grid, x, F, u = _points_inputs(case, seed)
        return dict(kind=kind, grid=grid, x=x, F=F, u=u)
    if kind == 'step':
        grid, x, F, _ = _points_inputs(case, seed)
        stepper = IBStep(grid, len(x), dt=STEP_DT, device=GPU, precision=case['precision'],
                         resident_pressure=case['graphs'], graphs=case['graphs'])
        return dict(kind=kind, stepper=stepper, x=x, F=F, u=grid.zeros(device='cuda'))
    if kind == 'fe':
        grid, geometry, x, F, u = _fe_inputs(case, seed)
        if case['mode'] == 'assembled':
            transfer = AssembledTransfer(grid, geometry)
        else:
            transfer = FETransfer(grid, geometry, fused=case['mode'] == 'fused')
        return dict(kind=kind, transfer=transfer, x=x, F=F, u=u)
    grids, xs, Fs = _batch_inputs(case, seed)
    counts = [len(x) for x in xs]
    if kind == 'batch3':
        options = MGOptions(smooth=2, smoother='rbgs', relax=MIXED_RELAX, inner_cycles=MIXED_INNER_CYCLES)
        batch = BatchedIBStep(grids, counts, dt=STEP_DT, device=GPU, options=options)
        return dict(kind=kind, batch=batch, x=xs, F=Fs, u=[g.zeros(device='cuda') for g in grids])
    batch = BatchedChannelStep(grids, counts, dt=CHANNEL_DT, device=GPU)
    for i, (x, F) in enumerate(zip(xs, Fs)):
        batch.x[i].copy_(x)
        batch.force[i].copy_(F)
    return dict(kind=kind, batch=batch)


def run(s):
    kind = s['kind']
    if kind == 'channel':
        u, p, U, _ = s['stepper'].step(s['x'], s['F'], s['u'])
        return dict(u=list(u), p=p, U=U, x=s['x'])
    if kind == 'flow':
        r = s['flow'].step(s['u'], s['f'])
        return dict(u=list(r.velocity), p=r.pressure)
    if kind == 'transfer':
        bins = s['binner'](s['x'])
        f = s['transfer'].spread(s['x'], s['F'], bins)
        return dict(f=list(f), U=s['transfer'].interpolate(s['x'], s['u'], bins))
    if kind == 'compact':
        stencil = from_points(s['x'], s['grid'])
        f = cuda_ib.compact_spread(s['grid'], s['F'], stencil)
        return dict(f=list(f), U=cuda_ib.compact_gather(s['grid'], s['u'], stencil))
    if kind == 'step':
        u, p, U, _ = s['stepper'].step(s['x'], s['F'], s['u'])
        return dict(u=list(u), p=p, U=U, x=s['x'])
    if kind == 'fe':
        t = s['transfer']
        stencil = t.prepare(s['x'])
        f, _ = t.spread(s['F'], stencil)
        U, _ = t.interpolate(s['u'], stencil)
        return dict(f=list(f), U=U)
    if kind == 'batch3':
        u, p, U, _ = s['batch'].step(s['x'], s['F'], s['u'])
        return dict(u=[torch.cat([c.reshape(-1) for c in v]) for v in u], p=list(p), U=list(U), x=list(s['x']))
    b = s['batch']
    b.reset()
    U, _ = b.step()
    return dict(u=b.u, v=b.v, p=[b.pressure(i) for i in range(len(b.grids))], U=U, x=b.x_all)


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _solve_flops(cells, cycles, sweeps, points):
    """V-cycles of ``sweeps`` sweeps of a ``points``-point operator per
    level, residual, restriction and prolongation included."""
    return cycles * cells * (2 * points * (sweeps + 1) + 20) * (8 / 7 if points == 7 else 4 / 3)


def work(case):
    kind = case['kind']
    if kind in ('batch3', 'batch2'):
        total = dict(bytes=0., flops=0.)
        for shape, points in _mix(case):
            if kind == 'batch3':
                w = work(dict(kind='step', nx=shape[0], ny=shape[1], nz=shape[2], points=points, precision='mixed'))
            else:
                w = work(dict(kind='channel', nx=shape[0], ny=shape[1], points=points, smoother='rbgs'))
            total = {k: total[k] + w[k] for k in total}
        return total
    if kind == 'channel':
        cells, P = case['nx'] * case['ny'], case['points']
        sweeps, cycles = (4, 10) if case['smoother'] == 'rbgs' else (8, 10)
        # positions, forces, velocities in; positions, velocities, pressure out
        return dict(bytes=8. * (8 * P + 5 * cells), flops=_solve_flops(cells, cycles, sweeps, 5) + P * 400.)
    if kind == 'fe':
        nodes, cells, values, weights = _case_mesh(case)
        P, V, Q = weights.size, len(nodes), case['n'] ** 3
        # the tables of the interaction points stay internal: nodal fields,
        # cells and weights in, face fields in and out
        return dict(bytes=8. * (12 * V + cells.size + P + 6 * Q), flops=P * (2. * 2 * 3 * 64 + 9 * 2 * cells.shape[1]))
    cells = case['nx'] * case['ny'] * case['nz']
    if kind == 'flow':
        sweeps, cycles = (8, 8) if case['smoother'] == 'jacobi' else (4, 10)
        return dict(bytes=8. * 10 * cells, flops=_solve_flops(cells, cycles, sweeps, 7) + 200. * cells)
    P = case['points']
    transfer = P * 2. * 3 * (64 + 16 + 4) * 2
    if kind in ('transfer', 'compact'):
        return dict(bytes=8. * (9 * P + 6 * cells), flops=transfer)
    sweeps, cycles = (4, 6) if case['precision'] == 'mixed' else (4, 10)
    return dict(bytes=8. * (12 * P + 7 * cells), flops=transfer + _solve_flops(cells, cycles, sweeps, 7))


def tolerance(case):
    """About four times the distance from ``exact``. The FP64 transfers differ
    by the order of their sums and the spread's fixed-point rounding (2.3e-14).
    Pressure solves stop at a residual of 1e-10 of the right-hand side (4.1e-10
    in the pressure). Mass solves stop at 1e-13 absolute, which on these small
    nodal volumes leaves 3.9e-9 in the nodal velocity."""
    kind = case['kind']
    if kind in ('transfer', 'compact'):
        return dict(rel=1e-13, max=1e-11)
    if kind == 'fe':
        return dict(rel=2e-8, max=8e-7)
    return dict(rel=2e-9, max=1e-7)


# ---------------------------------------------------------------------------
# the same results in plain FP64 torch

def _phi(r):
    r = r.abs()
    a, b = r.clamp(max=1.), r.clamp(1., 2.)
    inner = (3 - 2 * a + (1 + 4 * a - 4 * a * a).clamp(min=0).sqrt()) / 8
    outer = (5 - 2 * b - (-7 + 12 * b - 4 * b * b).clamp(min=0).sqrt()) / 8
    return torch.where(r < 1, inner, torch.where(r < 2, outer, torch.zeros_like(r)))


CHUNK = 131072


def _links(x, grid, c):
    """Flat face ids and weights (P, 64) of component c."""
    d = len(grid.shape)
    h = x.new_tensor(grid.spacing)
    start = x.new_tensor([0. if a == c else .5 for a in range(d)])
    s = x / h - start
    nodes = torch.floor(s - 1).long()[..., None] + torch.arange(4, device=x.device)
    w = _phi(s[..., None] - nodes.double())
    if d == 2:
        nx, ny = grid.shape
        j = nodes[:, 1]
        low, high = (-j - 1, 2 * ny - 1 - j) if c == 0 else (-j, 2 * ny - j)
        top = ny if c == 0 else ny + 1
        outside = (j < 0) | (j >= top)
        j = torch.where(j < 0, low, torch.where(j >= top, high, j))
        i = nodes[:, 0] % nx if grid.periodic else nodes[:, 0]
        wy = torch.where(outside, -w[:, 1], w[:, 1])
        ids = i[:, :, None] * grid.face_shape(c)[1] + j[:, None, :]
        return ids.reshape(len(x), 16), (w[:, 0, :, None] * wy[:, None, :]).reshape(len(x), 16)
    shape = grid.face_shape(c)
    if grid.periodic:
        nodes = nodes % torch.tensor(shape, device=x.device)[:, None]
    ids = (nodes[:, 0, :, None, None] * shape[1] + nodes[:, 1, None, :, None]) * shape[2] + nodes[:, 2, None, None, :]
    w = w[:, 0, :, None, None] * w[:, 1, None, :, None] * w[:, 2, None, None, :]
    return ids.reshape(len(x), 64), w.reshape(len(x), 64)


def _spread(x, F, grid):
    out = []
    for c in range(len(grid.shape)):
        f = torch.zeros(prod(grid.face_shape(c)), device=x.device, dtype=torch.float64)
        for a in range(0, len(x), CHUNK):
            ids, w = _links(x[a:a + CHUNK], grid, c)
            f.index_add_(0, ids.reshape(-1), (w * F[a:a + CHUNK, c, None]).reshape(-1))
        out.append((f / grid.volume).view(grid.face_shape(c)))
    return out


def _gather(x, u, grid):
    out = torch.empty_like(x)
    for c, uc in enumerate(u):
        flat = uc.reshape(-1)
        for a in range(0, len(x), CHUNK):
            ids, w = _links(x[a:a + CHUNK], grid, c)
            out[a:a + CHUNK, c] = (flat[ids] * w).sum(1)
    return out


def _axis_operator(n, h, periodic, outlet=False):
    A = np.zeros((n, n))
    for i in range(n if periodic else n - 1):
        j = (i + 1) % n
        A[i, i] += 1
        A[j, j] += 1
        A[i, j] -= 1
        A[j, i] -= 1
    if outlet:
        A[n - 1, n - 1] += 2
    lam, V = np.linalg.eigh(A / h ** 2)
    return torch.tensor(lam, device='cuda'), torch.tensor(V, device='cuda')


def _along(V, t, axis):
    """V applied along an axis."""
    return torch.movedim((V @ torch.movedim(t, axis, 0).reshape(t.shape[axis], -1)).view(
        V.shape[0], *[n for a, n in enumerate(t.shape) if a != axis]), 0, axis)


def _poisson(b, grid):
    """-Laplacian p = b by the axes' eigenvectors; zero mean where the
    constant is in the null space."""
    d = b.dim()
    channel = d == 2
    ops = []
    for a, (n, h) in enumerate(zip(grid.shape, grid.spacing)):
        wraps = grid.periodic and (a == 0 or not channel)
        ops.append(_axis_operator(n, h, wraps, channel and a == 0 and not wraps))
    t = b
    for a, (_, V) in enumerate(ops):
        t = _along(V.T.contiguous(), t, a)
    lam = sum(l.view([-1 if a == c else 1 for c in range(d)]) for a, (l, _) in enumerate(ops))
    null = lam.abs() < 1e-9 * float(lam.max())
    t = torch.where(null, torch.zeros_like(t), t / torch.where(null, torch.ones_like(lam), lam))
    for a, (_, V) in enumerate(ops):
        t = _along(V, t, a)
    return t.contiguous()


def _project(star, grid, dt):
    """Velocity and pressure of the projection (rho = 1)."""
    div = 0.
    for c, (u, h) in enumerate(zip(star, grid.spacing)):
        wraps = u.shape[c] == grid.shape[c]
        div = div + ((u.roll(-1, c) - u) if wraps else u.diff(dim=c)) / h
    p = _poisson(-div / dt, grid)
    out = []
    for c, (u, h) in enumerate(zip(star, grid.spacing)):
        if u.shape[c] == grid.shape[c]:
            out.append(u - dt * (p - p.roll(1, c)) / h)
            continue
        v = u.clone()
        v.narrow(c, 1, p.shape[c] - 1).sub_(dt * p.diff(dim=c) / h)
        if p.dim() == 2 and c == 0:
            v[-1] += dt * 2 * p[-1] / h
        out.append(v)
    return out, p


def _exact_step(x, F, u, grid, dt):
    f = _spread(x, F, grid)
    star = [a + dt * b for a, b in zip(u, f)]
    if len(grid.shape) == 2:
        if not grid.periodic:
            star[0][0] = u[0][0]
        star[1][:, 0] = 0
        star[1][:, -1] = 0
    v, p = _project(star, grid, dt)
    U = _gather(x, v, grid)
    return v, p, U, x + dt * U


def _pad(u, axis, odd):
    sign = -1 if odd else 1
    return torch.cat((sign * u.narrow(axis, 0, 1), u, sign * u.narrow(axis, u.shape[axis] - 1, 1)), axis)


def _predict(u, f, grid, dt, nu):
    """u + dt (-N(u) + nu L u + f) with odd ghosts across the walls; the
    walls' normal faces stay zero."""
    out = []
    for c, uc in enumerate(u):
        total = f[c].clone()
        for a, h in enumerate(grid.spacing):
            padded = _pad(uc, a, True)
            n = uc.shape[a]
            total += nu * (padded.narrow(a, 0, n) - 2 * uc + padded.narrow(a, 2, n)) / h ** 2
            if a == c:
                flux = (.5 * (uc.narrow(c, 1, n - 1) + uc.narrow(c, 0, n - 1))) ** 2
                total.narrow(c, 1, n - 2).sub_(flux.diff(dim=c) / h)
            else:
                other = _pad(u[a], c, True)
                m = other.shape[c] - 1
                advector = .5 * (other.narrow(c, 1, m) + other.narrow(c, 0, m))
                carried = .5 * (padded.narrow(a, 1, n + 1) + padded.narrow(a, 0, n + 1))
                total -= (advector * carried).diff(dim=a) / h
        star = uc + dt * total
        star.narrow(c, 0, 1).zero_()
        star.narrow(c, star.shape[c] - 1, 1).zero_()
        out.append(star)
    return out


def _mass_solve(geometry, b):
    """Conjugate gradients on the consistent mass to rounding."""
    cells, N, W = geometry.cells, geometry.values, geometry.weights
    local = torch.matmul(N.t() * W[:, None, :], N)
    A = cells.shape[1]
    apply = lambda v: torch.zeros_like(v).index_add_(0, cells.reshape(-1),
                                                     torch.matmul(local, v[cells]).reshape(-1, 3))
    diag = torch.zeros(len(b), device=b.device, dtype=b.dtype).index_add_(
        0, cells.reshape(-1), local[:, range(A), range(A)].reshape(-1))[:, None]
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz = z.clone(), (r * z).sum(0)
    for _ in range(140):
        q = apply(p)
        alpha = rz / (p * q).sum(0)
        x += alpha * p
        r -= alpha * q
        z = r / diag
        rz, old = (r * z).sum(0), rz
        if float((rz / (b * b / diag).sum(0)).max()) < 1e-32:
            break
        p = z + (rz / old) * p
    return x


def exact(case, seed):
    kind = case['kind']
    if kind == 'channel':
        grid, x, F, u = _channel_inputs(case, seed)
        v, p, U, x = _exact_step(x, F, u, grid, CHANNEL_DT)
        return dict(u=v, p=p, U=U, x=x)
    if kind == 'flow':
        grid, u, f = _flow_inputs(case, seed)
        dt = _flow_dt(case)
        f = [a.clone() for a in f]
        v, p = _project(_predict(u, f, grid, dt, .01), grid, dt)
        return dict(u=v, p=p)
    if kind in ('transfer', 'compact'):
        grid, x, F, u = _points_inputs(case, seed)
        return dict(f=_spread(x, F, grid), U=_gather(x, u, grid))
    if kind == 'step':
        grid, x, F, _ = _points_inputs(case, seed)
        v, p, U, x = _exact_step(x, F, grid.zeros(device='cuda'), grid, STEP_DT)
        return dict(u=v, p=p, U=U, x=x)
    if kind == 'fe':
        grid, g, x, F, u = _fe_inputs(case, seed)
        points = torch.matmul(g.values, x[g.cells]).reshape(-1, 3)
        C = _mass_solve(g, F)
        Fq = (g.weights[..., None] * torch.matmul(g.values, C[g.cells])).reshape(-1, 3)
        Uq = _gather(points, u, grid).view(*g.weights.shape, 3) * g.weights[..., None]
        rhs = torch.zeros_like(F).index_add_(0, g.cells.reshape(-1),
                                             torch.matmul(g.values.t().contiguous(), Uq).reshape(-1, 3))
        return dict(f=_spread(points, Fq, grid), U=_mass_solve(g, rhs))
    grids, xs, Fs = _batch_inputs(case, seed)
    if kind == 'batch3':
        steps = [_exact_step(x, F, g.zeros(device='cuda'), g, STEP_DT) for g, x, F in zip(grids, xs, Fs)]
        return dict(u=[torch.cat([c.reshape(-1) for c in s[0]]) for s in steps], p=[s[1] for s in steps],
                    U=[s[2] for s in steps], x=[s[3] for s in steps])
    steps = [_exact_step(x, F, g.zeros(device='cuda'), g, CHANNEL_DT) for g, x, F in zip(grids, xs, Fs)]
    return dict(u=torch.cat([s[0][0].reshape(-1) for s in steps]), v=torch.cat([s[0][1].reshape(-1) for s in steps]),
                p=[s[1] for s in steps], U=torch.cat([s[2] for s in steps]), x=torch.cat([s[3] for s in steps]))
