"""ChannelIBStep with inputs a caller may pass: velocities of any stride order,
several faults at once (the support of the points is reported first, whatever
else is wrong), and one stepper called from several streams."""
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


@pytest.mark.parametrize('other', ['pressure shape', 'pressure dtype', 'velocity shape', 'force', 'force shape'])
def test_support_is_reported_first(gpu, other):
    grid, stepper, x, force, velocity = setup(gpu, False)
    pressure = torch.zeros(grid.shape, device=gpu, dtype=torch.float64)
    if other == 'pressure shape':
        pressure = pressure[:-1]
    elif other == 'pressure dtype':
        pressure = pressure.float()
    elif other == 'velocity shape':
        velocity[0] = velocity[0][:, :-1]
    elif other == 'force':
        force = torch.full_like(force, float('nan'))
    else:
        force = force[:-1]
    for inside in (False, True):
        if not inside:
            x[5, 1] = -1.
        else:
            x[5, 1] = .5
        with pytest.raises((ValueError, RuntimeError)) as error:
            stepper.step(x, force, velocity, pressure)
        assert ('support region' in str(error.value)) == (not inside)


def test_one_stepper_on_two_streams(gpu):
    """A step returns with its last launches queued; the next call on another
    stream works in the same solver buffers."""
    grid, stepper, x, force, velocity = setup(gpu, True)
    _, _, x2, force2, velocity2 = setup(gpu, True, seed=8)
    want = [stepper.step(a.clone(), f, tuple(v))[:3] for a, f, v in ((x, force, velocity), (x2, force2, velocity2))]
    torch.cuda.synchronize()
    solver = stepper.flow.pressure_solver
    sub_mean = solver._sub_mean
    slow = [False]

    def late(t, slot):  # the mean removals of a solve, held back on their stream
        if slow[0] and t is solver.p[0]:
            torch.cuda._sleep(20_000_000)
        sub_mean(t, slot)

    solver._sub_mean = late
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    args = [(x.clone(), force, tuple(velocity)), (x2.clone(), force2, tuple(velocity2))]
    got = []
    torch.cuda.synchronize()
    for stream, a, delay in zip(streams, args, (True, False)):
        slow[0] = delay
        with torch.cuda.stream(stream):
            got.append(stepper.step(*a)[:3])
    torch.cuda.synchronize()
    for (va, pa, Ua), (vb, pb, Ub) in zip(want, got):
        assert torch.equal(pa, pb) and torch.equal(Ua, Ub)
        assert all(torch.equal(a, b) for a, b in zip(va, vb))
