"""Differentiable homogenized matrices and solution fields: torch.autograd.Function over the
HIP solve.

Forward: for a voxel field theta (torch float64, shape N), a(x) = exp(theta(x)), solve
the d unit-load GaNi problems on the GPU and return the primal matrix AH (the upper
bound, ffthompy/postprocess.py:53-70). Backward: the solution fields e_i minimise the
energy, so with the fields held fixed dAH_ij/da(x) = e_i(x).e_j(x)/n (envelope
theorem, also for i != j by polarisation); the hand-written kernel fh_energy_gradient
evaluates sum_ij W_ij e_i.e_j a(x)/n for W = dL/dAH in one pass over the stored
fields. No adjoint solve is needed for losses on AH.

SolutionFields returns the unit-load fields e_i = E_i + x_i themselves; a loss on them needs
one adjoint CG per load: lam_i solves G(a lam_i) = G dL/de_i (the same operator, fp64), and
dL/da(x) = -sum_i lam_i(x) . e_i(x) (kernel fh_field_gradient).
"""
import numpy as np
import torch

from . import _native as nat


class _Buffers:
    """Where a call's float64 arrays live. For a theta on the library's GPU they are torch tensors lent to the
    library (nothing travels through host memory, and torch's allocator gives the memory that a fresh
    hipMalloc and hipFree per array would map and unmap): at 99^3 with gradient the four copies of 7.8 MB
    to or from pageable memory and ten 23 MB allocations took 8 ms beside 25 ms of solves, what is left
    takes 3 ms. Otherwise device arrays, filled and read through the host.

    The library works on a stream of its own and every call has finished on return; sync() orders the
    current torch stream (what filled an array, or used its memory before) ahead of such a call."""

    def __init__(self, theta):
        self.device = theta.device
        self.lent = theta.is_cuda and theta.device.index == 0

    def sync(self):
        if self.lent:
            torch.cuda.current_stream(self.device).synchronize()

    def lend(self, t):
        """A contiguous float64 tensor on the GPU as a device array that keeps it alive."""
        v = nat.DeviceArray.borrow(t.data_ptr(), tuple(t.shape))
        v._owner = t
        return v

    def array(self, shape, zero=False):
        if self.lent:
            return self.lend((torch.zeros if zero else torch.empty)(shape, dtype=torch.float64, device=self.device))
        return nat.DeviceArray.zeros(shape) if zero else nat.DeviceArray(shape)

    def put(self, t):
        """The values of a tensor."""
        if self.lent:
            return self.lend(t.detach().to(self.device, torch.float64, copy=True).contiguous())
        return nat.DeviceArray.from_host(t.detach().to('cpu', torch.float64).numpy())

    def tensor(self, arr):
        """An array of this call as a tensor on theta's device."""
        return arr._owner if self.lent else torch.from_numpy(arr.to_host()).to(self.device)


def _solve_unit_loads(theta, Y, tol, maxiter, precision):
    """(buffers, plan, a, fields, iteration counts) of the d unit-load problems for a = exp(theta)."""
    N = tuple(int(n) for n in theta.shape)
    d = len(N)
    buf = _Buffers(theta)
    a = buf.put(torch.exp(theta.detach()))
    plan = nat.Plan(N, np.asarray(Y, dtype=np.float64), 'scalar', 'primal')
    B = buf.array((d,) + N)
    EN = buf.array((d,) + N, zero=True)
    fields = [buf.array((d,) + N, zero=True) for _ in range(d)]
    buf.sync()
    plan.set_coeff('iso', a)
    kits = []
    for iL, x in enumerate(fields):
        E = np.zeros(d)
        E[iL] = 1.
        nat.add_constant(EN, -E)
        plan.matvec(EN, B)
        nat.add_constant(EN, E)  # back to exact zeros
        info = plan.cg_solve(B, x, tol=tol, maxiter=maxiter, mode=precision)
        if info['status'] != nat.FH_CG_OK:
            raise FloatingPointError('CG breakdown')
        nat.add_constant(x, E)
        kits.append(info['kit'])
    return buf, plan, a, fields, kits


class UpperBound(torch.autograd.Function):
    """AH(theta) with a = exp(theta), scalar conductivity on an N grid of cell Y."""

    @staticmethod
    def forward(ctx, theta, Y, tol, maxiter, precision):
        ctx.buf, ctx.plan, ctx.a_dev, ctx.fields, ctx.kits = _solve_unit_loads(theta, Y, tol, maxiter, precision)
        return torch.from_numpy(ctx.plan.energy_matrix(ctx.fields)).to(theta.device)

    @staticmethod
    def backward(ctx, gAH):
        W = gAH.detach().to('cpu', torch.float64).numpy()
        out = ctx.buf.array(ctx.plan.N)
        ctx.buf.sync()
        g = ctx.plan.energy_gradient(ctx.fields, W, chain=ctx.a_dev, out=out)
        return ctx.buf.tensor(g), None, None, None, None


def upper_bound(theta, Y=None, tol=1e-10, maxiter=5000, precision='fp64'):
    """Differentiable primal homogenized matrix AH(theta), a = exp(theta)."""
    if Y is None:
        Y = np.ones(theta.dim())
    return UpperBound.apply(theta, Y, tol, maxiter, precision)


class SolutionFields(torch.autograd.Function):
    """e (d, d) + N: e[i] = E_i + x_i for a = exp(theta); backward by adjoint CG solves."""

    @staticmethod
    def forward(ctx, theta, Y, tol, maxiter):
        ctx.buf, ctx.plan, ctx.a_dev, ctx.fields, _ = _solve_unit_loads(theta, Y, tol, maxiter, 'fp64')
        ctx.tol, ctx.maxiter = tol, maxiter
        return torch.stack([ctx.buf.tensor(f) for f in ctx.fields])  # a copy: the caller may write to it

    @staticmethod
    def backward(ctx, g):
        plan, buf = ctx.plan, ctx.buf
        g = g.detach()
        rhs = buf.array(ctx.fields[0].shape)
        adj = []
        for i, f in enumerate(ctx.fields):  # one load's gradient and right-hand side at a time
            v = buf.put(g[i])
            lam = buf.array(f.shape, zero=True)
            buf.sync()
            plan.project(v, rhs)
            info = plan.cg_solve(rhs, lam, tol=ctx.tol, maxiter=ctx.maxiter, mode='fp64')
            if info['status'] != nat.FH_CG_OK:
                raise FloatingPointError('adjoint CG breakdown')
            adj.append(lam)
        v = rhs = None
        out = buf.array(plan.N)
        buf.sync()
        grad = plan.field_gradient(ctx.fields, adj, chain=ctx.a_dev, out=out)
        return buf.tensor(grad), None, None, None


def solution_fields(theta, Y=None, tol=1e-10, maxiter=5000):
    """Differentiable unit-load solution fields e (d, d)+N for a = exp(theta) (fp64)."""
    if Y is None:
        Y = np.ones(theta.dim())
    return SolutionFields.apply(theta, Y, tol, maxiter)
