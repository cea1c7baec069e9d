"""The tiled smoothing stages of the 3D V-cycle against the oracle's cycle
where tiles, halos and phase chunks can go wrong: extents that are no multiple
of the tile, axes shorter than a tile with its halo, stages that need several
launches, both smoothers and boundary types, and a level large enough for the
two-phase launches."""
import numpy as np
import pytest
import torch

from afsi_gpu_amd.mac import MACGrid, MGOptions
from afsi_gpu_amd.mac.multigrid import GeometricMultigrid
from oracle import mac3d

pytestmark = pytest.mark.gpu
LENGTHS = (1., 1.3, .9)
CYCLES = 60  # more than Jacobi cycles take to stagnate in FP64


def check(gpu, shape, periodic, smoother, nu):
    h = tuple(L / n for L, n in zip(LENGTHS, shape))
    ref = mac3d.Multigrid(shape, h, mac3d.MGOptions(smooth=nu, smoother=smoother), periodic)
    gen = np.random.default_rng(5)
    start, rhs = gen.normal(size=shape), gen.normal(size=shape) / min(h) ** 2
    start -= start.mean()
    rhs -= rhs.mean()
    want = ref.cycle(0, start, rhs)
    want -= want.mean()
    # Some 45 roundings of 2^-53 along a path of the cycle; an FP32 cycle rounds 2^29 times as coarsely.
    # Measured: at most 1.4e-15 (FP32: 7.4e-7) in the norm, 1.9e-15 (1.1e-6) in a cell.
    for dtype, bound in ((torch.float64, 5e-15), (torch.float32, 5e-15 * 2. ** 29)):
        mg = GeometricMultigrid(MACGrid(shape, LENGTHS, periodic=periodic), device=gpu, dtype=dtype,
                                options=MGOptions(smooth=nu, smoother=smoother), backend='workspace')
        mg.initialize(torch.tensor(start, device=gpu, dtype=dtype), torch.tensor(rhs, device=gpu, dtype=dtype))
        got = mg.cycle().double().cpu().numpy()
        got -= got.mean()
        assert np.linalg.norm(got - want) <= bound * np.linalg.norm(want), (shape, dtype)
        # cell by cell too: a few wrong cells at a tile's edge would vanish in the norm
        assert abs(got - want).max() <= bound * abs(want).max(), (shape, dtype)


@pytest.mark.parametrize('periodic', [False, True], ids=['closed', 'periodic'])
@pytest.mark.parametrize('smoother,nu', [('rbgs', 1), ('rbgs', 2), ('rbgs', 3), ('jacobi', 4), ('jacobi', 5)])
@pytest.mark.parametrize('shape', [(24, 40, 48), (128, 16, 16), (12, 40, 40), (40, 56, 24)])
def test_cycle_matches_oracle(gpu, shape, smoother, nu, periodic):
    check(gpu, shape, periodic, smoother, nu)


@pytest.mark.parametrize('periodic', [False, True], ids=['closed', 'periodic'])
@pytest.mark.parametrize('smoother,nu', [('rbgs', 2), ('jacobi', 3)])
def test_two_phase_level_matches_oracle(gpu, smoother, nu, periodic):
    check(gpu, (128, 80, 112), periodic, smoother, nu)


@pytest.mark.parametrize('periodic', [False, True], ids=['closed', 'periodic'])
@pytest.mark.parametrize('shape', [(16, 16, 16), (32, 24, 40)])
def test_jacobi_stagnates_no_higher_than_the_oracle(gpu, shape, periodic):
    """Where Jacobi cycles stop converging (the coarse kernel alone; tiled levels
    above it), the residual is what the rounding of the stored iterate leaves
    plus that of one update. The oracle's update p + omega (rhs - A p) / diag
    rounds a small correction; (rhs + sum w p) / diag would stagnate 1.6 to 1.8
    times higher. The mean over five cycles varies by a few percent."""
    h = tuple(L / n for L, n in zip(LENGTHS, shape))
    options = dict(smooth=4, smoother='jacobi')
    ref = mac3d.Multigrid(shape, h, mac3d.MGOptions(**options), periodic)
    rhs = np.random.default_rng(6).normal(size=shape)
    rhs -= rhs.mean()
    p, floor = np.zeros(shape), []
    for i in range(CYCLES):
        p = ref.cycle(0, p, rhs)
        if i >= CYCLES - 5:
            floor.append(np.linalg.norm(rhs - mac3d.negative_laplacian(p, h, periodic)))
    assert floor[-1] > .5 * floor[0]  # stagnated
    for dtype, unit in ((torch.float64, 1.), (torch.float32, 2. ** 29)):
        mg = GeometricMultigrid(MACGrid(shape, LENGTHS, periodic=periodic), device=gpu, dtype=dtype,
                                options=MGOptions(**options), backend='workspace')
        mg.initialize(torch.zeros(shape, device=gpu, dtype=dtype), torch.tensor(rhs, device=gpu, dtype=dtype))
        got = []
        for i in range(CYCLES):
            mg.advance(1)
            got.append(float(mg.results[0, 1].sqrt()))
        print(shape, periodic, dtype, np.mean(got[-5:]) / (np.mean(floor) * unit))
        assert np.mean(got[-5:]) <= 1.2 * np.mean(floor) * unit


class DividingMultigrid(mac3d.Multigrid):
    """The oracle with Gauss-Seidel values (b + sum w p) / diag, the neighbours
    added one by one: the rounding of the sweeps for rows longer than 128."""

    def rbgs(self, level, p, rhs):
        w = [1 / h ** 2 for h in self.spacings[level]]
        parity = np.indices(p.shape).sum(0) % 2
        p = p.copy()
        for colour in (0, 1):
            s, diag = np.zeros_like(p), np.zeros_like(p)
            for axis in range(3):
                for step in (-1, 1):
                    there = np.ones(p.shape, bool)
                    if not self.periodic:
                        there[(slice(None),) * axis + (-1 if step < 0 else 0,)] = False
                    s += np.where(there, w[axis] * np.roll(p, step, axis), 0)
                    diag += np.where(there, w[axis], 0)
            p = np.where(parity == colour, (rhs + s) / diag, p)
        return p


@pytest.mark.parametrize('periodic', [False, True], ids=['closed', 'periodic'])
@pytest.mark.parametrize('shape', [(16, 24, 32), (32, 32, 160)])
def test_red_black_stagnates_no_higher_than_by_division(gpu, shape, periodic):
    """The residual where red-black cycles stop converging, on rows shorter and
    longer than 128 cells, against values rounded as by a sum and a division.
    A product with the rounded reciprocal stagnates up to 1.2 times higher; the
    mean over ten cycles varies by less than 3 percent."""
    h = (1 / 32,) * 3
    lengths = tuple(n / 32 for n in shape)
    options = dict(smooth=2, smoother='rbgs')
    ref = DividingMultigrid(shape, h, mac3d.MGOptions(**options), periodic)
    rhs = np.random.default_rng(6).normal(size=shape)
    rhs -= rhs.mean()
    p, floor = np.zeros(shape), []
    for i in range(35):
        p = ref.cycle(0, p, rhs)
        if i >= 25:
            floor.append(np.linalg.norm(rhs - mac3d.negative_laplacian(p, h, periodic)))
    assert floor[-1] > .5 * floor[0]  # stagnated
    for dtype, unit in ((torch.float64, 1.), (torch.float32, 2. ** 29)):
        mg = GeometricMultigrid(MACGrid(shape, lengths, periodic=periodic), device=gpu, dtype=dtype,
                                options=MGOptions(**options), backend='workspace')
        mg.initialize(torch.zeros(shape, device=gpu, dtype=dtype), torch.tensor(rhs, device=gpu, dtype=dtype))
        got = []
        for i in range(35):
            mg.advance(1)
            got.append(float(mg.results[0, 1].sqrt()))
        print(shape, periodic, dtype, np.mean(got[25:]) / (np.mean(floor) * unit))
        assert np.mean(got[25:]) <= 1.05 * np.mean(floor) * unit
