"""A breakdown of the fused fp64 iterations after they have made steps: the solution holds every finished
step once, as in the operator form, whose solution takes a step in the iteration that makes it.

The coefficients have a few negative values; with the seeds below <p, A p> / <p, p> is above 0.2 in every
iteration before the one where it is negative (float64 CG on the host). Two iterations of the two forms
differ by rounding (1.1e-16 times 20 for the transforms, times at most 1 / 0.2 per step): 1e-11 of the
largest entry holds, a step too many is of its order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')

CASES = [((9, 9, 9), 0.003, 2), ((15, 12, 14), 0.003, 2), ((27, 27), 0.003, 1)]  # grid, fraction, finished steps


def indefinite(N, frac):
    rng = np.random.default_rng(3)
    a = np.exp(0.5 * rng.standard_normal(N))
    a.reshape(-1)[rng.choice(a.size, int(frac * a.size), replace=False)] = -3.
    return a


@pytest.mark.parametrize('N,frac,steps', CASES, ids=[str(c[0]) for c in CASES])
def test_potential_breakdown_keeps_the_last_iterate(N, frac, steps):
    print('case potential breakdown', N, flush=True)
    d = len(N)
    plan = nat.Plan(N, np.ones(d))
    plan.set_coeff('iso', indefinite(N, frac))
    out = []
    for fused in (True, False):
        plan.set_cg_variant(fused)
        X = nat.DeviceArray((d,) + N)
        Fu, info = plan.potential_solve(np.eye(d)[0], 1e-10, 50, X=X, mode='fp64')
        assert info['status'] == nat.FH_CG_BREAKDOWN and info['kit'] == steps
        out.append((Fu.to_host(), X.to_host()))
    for f, o in zip(*out):
        assert np.abs(f - o).max() <= 1e-11 * np.abs(o).max()


@pytest.mark.parametrize('N,frac,steps', CASES, ids=[str(c[0]) for c in CASES])
def test_cg_breakdown_keeps_the_last_iterate(N, frac, steps):
    print('case cg breakdown', N, flush=True)
    d = len(N)
    plan = nat.Plan(N, np.ones(d), 'scalar', 'primal')
    plan.set_coeff('iso', indefinite(N, frac))
    EN = nat.DeviceArray.zeros((d,) + N)
    nat.add_constant(EN, -np.eye(d)[0])
    B = plan.matvec(EN, nat.DeviceArray((d,) + N))
    out = []
    for fused in (True, False):
        plan.set_cg_variant(fused)
        x = nat.DeviceArray.zeros((d,) + N)
        info = plan.cg_solve(B, x, tol=1e-10, maxiter=50, mode='fp64')
        assert info['status'] == nat.FH_CG_BREAKDOWN and info['kit'] >= 1
        out.append((info['kit'], x.to_host()))
    assert out[0][0] == out[1][0]
    assert np.abs(out[0][1] - out[1][1]).max() <= 1e-11 * np.abs(out[1][1]).max()
