"""ChannelIBStep with inputs a caller may pass: velocities of any stride order."""
import pytest
import torch

from afsi_gpu_amd.mac2d import ChannelGrid, ChannelIBStep

pytestmark = pytest.mark.gpu


def setup(gpu, periodic, backend='workspace', seed=3):
    grid = ChannelGrid((64, 16), (4., 1.), periodic)
    stepper = ChannelIBStep(grid, dt=1e-3, device=gpu, pressure_backend=backend)
    gen = torch.Generator(device='cpu').manual_seed(seed)
    rand = lambda *shape: torch.rand(shape, generator=gen, dtype=torch.float64)
    x = (rand(37, 2) * torch.tensor([2., .6]) + torch.tensor([1., .2])).to(gpu)
    force = (rand(37, 2) - .5).to(gpu)
    velocity = [(rand(*grid.face_shape(c)) - .5).to(gpu) for c in range(2)]
    velocity[1][:, 0] = velocity[1][:, -1] = 0
    if periodic:
        velocity[1].zero_()
        velocity[0] -= velocity[0].mean(0, keepdim=True)
    return grid, stepper, x, force, velocity


@pytest.mark.parametrize('periodic', [False, True], ids=['closed', 'periodic'])
@pytest.mark.parametrize('which', [(0,), (1,), (0, 1)], ids=['u', 'v', 'uv'])
def test_velocity_strides_do_not_matter(gpu, periodic, which):
    grid, stepper, x, force, velocity = setup(gpu, periodic)
    strided = [u.t().contiguous().t() if c in which else u for c, u in enumerate(velocity)]
    assert any(not u.is_contiguous() for u in strided)
    kept = [u.clone() for u in velocity]
    xa, xb = x.clone(), x.clone()
    va, pa, Ua, _ = stepper.step(xa, force, tuple(velocity))
    vb, pb, Ub, _ = stepper.step(xb, force, tuple(strided))
    # the same operations on the same numbers
    assert torch.equal(pa, pb) and torch.equal(Ua, Ub) and torch.equal(xa, xb)
    assert all(torch.equal(a, b) and b.is_contiguous() for a, b in zip(va, vb))
    assert all(torch.equal(a, b) for a, b in zip(velocity, kept))
