"""Mixed CG on one plan, several solves in a row: iterations replayed from captured batches of 8, 4, 2 and 1
against the same iterations launched one by one, equal to the bit. The iteration limits make each length
follow a batch of 8 without a synchronisation between them, first on a plan that has captured it and
then on one that has only captured 8. Grids: ragged ones of fixed lengths, which stay on the fixed-length
passes (alpha and beta inside the passes), and the passes of any smooth length."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')

CASES = [('scalar', 'iso', (99, 9, 15)), ('elasticity', 'lame', (45, 9, 15)), ('scalar', 'iso', (45, 45)),
         ('scalar', 'full', (20, 24, 18)), ('elasticity', 'lame', (27, 27, 27)), ('elasticity', 'full', (10, 9, 8)),
         ('scalar', 'iso', (66, 40, 50))]


@pytest.mark.parametrize('physics,kind,N', CASES, ids=['%s-%s-%s' % c for c in CASES])
def test_captured_batches_equal_launched_iterations(physics, kind, N):
    print('case graph batches', physics, kind, N, flush=True)
    rng = np.random.default_rng(67)
    plan = nat.Plan(N, np.ones(len(N)), physics, 'primal')
    nc = plan.ncomp
    a = np.where(rng.random(N) < 0.3, 100., 1.)
    if kind == 'lame':
        a = np.stack([0.6 * a, 0.4 * a])
    elif kind == 'full':
        a = np.einsum('ij,...->ij...', np.eye(nc) + 0.1, a)
    rhs = []
    for load in range(2):
        plan.set_coeff(kind, a)
        EN = nat.DeviceArray.zeros((nc,) + N)
        nat.add_constant(EN, -np.eye(nc)[load])
        rhs.append(plan.matvec(EN, nat.DeviceArray((nc,) + N)))
    out = {}
    for graphs in (False, True):
        plan.use_graphs(graphs)
        out[graphs] = []
        for maxiter in (24, 26, 25, 28, 31, 400):
            for B in rhs:
                x = nat.DeviceArray.zeros((nc,) + N)
                info = plan.cg_solve(B, x, tol=1e-7, maxiter=maxiter, mode='mixed', hist_len=401)
                out[graphs].append((maxiter, info['kit'], info['norm_res'], info['res_log'], x.to_host()))
    for g, w in zip(out[True], out[False]):
        assert g[1:3] == w[1:3], (g[:3], w[:3])
        assert np.array_equal(g[3], w[3]) and np.array_equal(g[4], w[4]), g[:3]
