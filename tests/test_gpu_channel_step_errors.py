"""ChannelIBStep reads its checks at the pressure solve's first
synchronisation: the errors stay those of the parts, and the caller's
positions and velocities are untouched by a step that raises."""
import pytest
import torch

from afsi_gpu_amd.mac2d import ChannelGrid, ChannelIBStep

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('periodic', [False, True], ids=['closed', 'periodic'])
@pytest.mark.parametrize('bad,message', [('support', 'support region'), ('force', 'finite tentative velocity'),
                                         ('velocity', 'finite tentative velocity'),
                                         ('pressure', 'initial guess required')])
def test_errors_and_untouched_state(gpu, periodic, bad, message):
    grid = ChannelGrid((64, 16), (4., 1.), periodic)
    stepper = ChannelIBStep(grid, dt=1e-3, device=gpu)
    gen = torch.Generator(device='cpu').manual_seed(3)
    x = (torch.rand((37, 2), generator=gen, dtype=torch.float64) * torch.tensor([2., .6]) + torch.tensor([1., .2])).to(gpu)
    force = torch.randn((37, 2), generator=gen, dtype=torch.float64).to(gpu)
    velocity = grid.zeros(device=gpu)
    pressure = torch.zeros(grid.shape, device=gpu, dtype=torch.float64)
    stepper.step(x.clone(), force, velocity, pressure)  # the sound step runs
    if bad == 'support':
        x[5, 1] = -1.
    elif bad == 'force':
        force[7, 0] = float('nan')
    elif bad == 'velocity':
        velocity[0][9, 4] = float('inf')
    else:
        pressure[3, 3] = float('nan')
    before = [t.clone() for t in (x, *velocity)]
    with pytest.raises(ValueError, match=message):
        stepper.step(x, force, velocity, pressure)
    assert all(torch.equal(a.nan_to_num(9.), b.nan_to_num(9.)) for a, b in zip(before, (x, *velocity)))
