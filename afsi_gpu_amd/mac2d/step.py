"""One IB time step on the channel (the ordering of mac2d/coupling.py:66-109
with the point force given): prepare -> spread -> u* = u + (dt/rho) f with
the wall normal faces kept at zero and the inlet face kept at its value
(the boundary() of mac2d/grid.py:74-79) -> project -> gather -> x += dt U.

The checks of the parts (support of the points, finite tentative velocity)
are made on the device and read at the pressure solve's first
synchronisation, before anything of the caller's is changed.
"""
import torch

from . import transfer
from .flow import ChannelFlow, ChannelResult, correct, divergence


class ChannelIBStep:
    def __init__(self, grid, *, dt, rho=1., device='cuda', options=None, pressure_backend='graph'):
        self.grid, self.dt, self.rho = grid, float(dt), float(rho)
        self.flow = ChannelFlow(grid, dt=dt, rho=rho, device=device, options=options,
                                pressure_backend=pressure_backend)
        self._done = torch.cuda.Event()

    @torch.no_grad()
    def step(self, x, force, velocity, pressure=None, *, advance=True):
        """Returns (velocity, pressure, point_velocity, info); x advances in
        place. The step returns with its last launches queued on the current
        stream. Calls may come on different streams, one after the other (the
        solver's buffers are shared, so not from two threads at once)."""
        flags = torch.zeros((), dtype=torch.int32, device=x.device)  # this call's own device word
        stencil = transfer.prepare(self.grid, x, flags=flags)
        host = torch.empty((), dtype=torch.int32, pin_memory=True)
        host.copy_(flags, non_blocking=True)
        read = []

        def precheck():  # after the solve's first synchronisation: the copy has arrived
            read.append(int(host))
            if read[0] & 1:
                raise ValueError(transfer.SUPPORT_MESSAGE)

        try:
            density = transfer.spread(self.grid, force, stencil, check=False)
            coef = self.dt / self.rho
            # row-major whatever the caller's strides: the projection passes pointers
            u = torch.add(velocity[0], density[0], alpha=coef).contiguous()
            v = torch.add(velocity[1], density[1], alpha=coef).contiguous()
            if not self.grid.periodic:
                u[0] = velocity[0][0]
            v[:, 0] = 0
            v[:, -1] = 0
            torch.cuda.current_stream(x.device).wait_event(self._done)  # the last step's use of the solver
            result = self._project((u, v), pressure, precheck)
            self._done.record(torch.cuda.current_stream(x.device))
        except Exception:
            # a point outside the support comes before any other fault
            if int(read[0] if read else flags) & 1:
                raise ValueError(transfer.SUPPORT_MESSAGE) from None
            raise
        U = transfer.gather(self.grid, result.velocity, stencil, check=False)
        if advance:
            x.add_(U, alpha=self.dt)
        return result.velocity, result.pressure, U, result.diagnostics

    def _project(self, tentative, pressure, precheck):
        """ChannelFlow.project of velocities that are this step's own (corrected
        in place, wall faces already zero), its checks deferred: a nonfinite
        face makes the right-hand side nonfinite, which the solve rejects."""
        flow = self.flow
        self.grid.check_velocity(tentative)
        rhs = divergence(tentative, self.grid, -flow.rho / flow.dt, out=flow._rhs)
        try:
            p, info = flow.pressure_solver.solve(rhs, pressure, precheck=precheck)
        except ValueError:
            if any(not torch.isfinite(t).all() for t in tentative):
                raise ValueError('finite tentative velocity required') from None
            raise
        velocity = correct(tentative, p, self.grid, flow.dt / flow.rho)
        return ChannelResult(velocity, p, dict(pressure=info))
