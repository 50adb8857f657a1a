"""The potential formulation's passes of any smooth length (fh_rt_pot.hpp) where they can go wrong: odd and
even axes, a padding row, planes compiled and schedule-driven, row mode with and without the strided pass
along axis 1, one point per tile, a band; the fused iteration (deferred scalars, graph batches, reliable
updates) against the operator form on the generic kernels.

The iterates after 4 and 9 iterations are compared (even axes converge slowly, so converged solutions of
two roundings differ by the condition number): unit rounding (1.1e-16, 6e-8) times 20 for the transforms of
an application, doubled by every iteration at most: 9 iterations stay below 1e-11 and 1e-3 of the largest
entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')

SHAPES = [(2, 3), (3, 2), (45, 45), (60, 50), (7, 130), (3, 3, 3), (2, 4, 2), (4, 27, 27), (15, 9, 21), (3, 20, 20),
          (33, 28, 30), (5, 140, 150), (12, 3, 256)]


def solve(plan, N, generic, mode, maxiter):
    plan.use_generic(generic)
    X = nat.DeviceArray((len(N),) + N)
    Fu, info = plan.potential_solve(np.linspace(1., 0.5, len(N)), 1e-11, maxiter, X=X, mode=mode)
    return Fu.to_host(), X.to_host(), info


@pytest.mark.parametrize('kind', ['iso', 'full'])
@pytest.mark.parametrize('N', SHAPES, ids=[str(s) for s in SHAPES])
def test_iterates_match_generic_kernels(N, kind):
    print('case rt potential', N, kind, flush=True)
    d = len(N)
    plan = nat.Plan(N, np.linspace(1., 2., d))
    a = np.exp(0.5 * np.random.default_rng(71).standard_normal(N))
    plan.set_coeff(kind, a if kind == 'iso' else np.einsum('ij,...->ij...', np.eye(d) + 0.1, a))
    for mode, tol in (('fp64', 1e-11), ('mixed', 1e-3)):
        for maxiter in (4, 9):
            ref, Xr, ir = solve(plan, N, True, mode, maxiter)
            Fu, X, info = solve(plan, N, False, mode, maxiter)
            assert info['status'] == ir['status'] and info['kit'] == ir['kit']
            assert np.abs(Fu - ref).max() <= tol * np.abs(ref).max()
            assert np.abs(X - Xr).max() <= tol * np.abs(Xr).max()


@pytest.mark.parametrize('mode', ['fp64', 'mixed'])
def test_stops(mode):
    """The iteration limit stops exactly, with the step of the last iteration in the solution."""
    N = (27, 27, 27)
    print('case rt potential stops', mode, flush=True)
    plan = nat.Plan(N, np.ones(3))
    rng = np.random.default_rng(72)
    plan.set_coeff('iso', np.exp(rng.standard_normal(N)))
    E = np.array([1., 0., 0.])
    for maxiter in (0, 1, 7, 8, 9):
        plan.set_cg_variant(True)
        Fu, info = plan.potential_solve(E, 1e-12, maxiter, mode=mode)
        plan.set_cg_variant(False)
        ref, iref = plan.potential_solve(E, 1e-12, maxiter, mode=mode)
        assert info['kit'] == iref['kit'] == maxiter
        f, r = Fu.to_host(), ref.to_host()
        assert np.abs(f - r).max() <= (1e-11 if mode == 'fp64' else 1e-4) * max(np.abs(r).max(), 1.)
