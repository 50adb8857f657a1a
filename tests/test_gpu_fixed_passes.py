"""The fixed-length passes (fh_fixed*.hpp) on grids whose operator runs them: three axes of fixed lengths and
planes that do not fit LDS, or ragged planes in more than 256 workgroups. Every length on each axis as far as
such grids have it, every coefficient kind and every number of components, against the generic kernels, and the
schedule variants against each other to the bit.

Tolerances as in test_gpu_kernels.py: float64 1e-12, float32 2e-5 of the largest entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')

# (n0, n1, n2) with 3 n0 > 256 and n1 != n2, and planes beyond LDS (225 x 243) for the short first axes
SCALAR = [(99, 5, 9), (99, 15, 5), (105, 9, 15), (105, 27, 25), (125, 25, 27), (125, 45, 63), (135, 63, 45), (99, 81, 75),
          (99, 75, 81), (105, 9, 99), (99, 99, 105), (125, 105, 9), (99, 15, 125), (99, 125, 15), (99, 9, 135),
          (225, 135, 5), (243, 9, 225), (243, 5, 243), (5, 225, 243), (9, 243, 225), (15, 243, 243), (25, 225, 225),
          (27, 225, 243), (45, 225, 243), (63, 225, 225), (75, 225, 243), (81, 243, 225)]
SIX = [(45, 9, 15), (63, 15, 9), (75, 27, 25), (81, 25, 27), (99, 5, 45), (105, 45, 5), (125, 9, 63), (135, 15, 81),
       (225, 5, 9), (243, 9, 5), (45, 27, 99), (45, 9, 105), (45, 25, 125), (45, 15, 135), (45, 5, 225), (45, 9, 243),
       (63, 105, 9), (45, 75, 45), (63, 27, 225)]  # the last three: one round of workgroups with more rows each


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def plan_of(N, physics, kind, rng):
    plan = nat.Plan(N, np.linspace(1., 1.3, 3), physics, 'primal')
    nc = plan.ncomp
    if kind == 'iso':
        vals = 1. + rng.random(N)
    elif kind == 'lame':
        vals = np.stack([1. + rng.random(N), 0.5 + rng.random(N)])
    else:
        A = 0.2 * rng.standard_normal((nc, nc) + N)
        vals = A + np.swapaxes(A, 0, 1) + 3. * np.eye(nc).reshape((nc, nc, 1, 1, 1))
    plan.set_coeff(kind, vals)
    return plan


@pytest.mark.parametrize('physics,kind,N', [('scalar', k, N) for N in SCALAR + [(99, 63, 45)] for k in ('iso', 'full')
                                               if k == 'iso' or np.prod(N) < 4e5]
                         + [('elasticity', 'lame', N) for N in SIX] + [('elasticity', 'full', N) for N in SIX[:4]])
def test_matvec_matches_generic_kernels(physics, kind, N):
    print('case fixed passes', physics, kind, N, flush=True)
    rng = np.random.default_rng(22)
    plan = plan_of(N, physics, kind, rng)
    x = rng.standard_normal((plan.ncomp,) + N)
    for dt, tol in ((np.float64, 1e-12), (np.float32, 2e-5)):
        dx, dy = nat.DeviceArray.from_host(x.astype(dt)), nat.DeviceArray((plan.ncomp,) + N, dt)
        plan.use_generic(True)
        ref = plan.matvec(dx, dy).to_host()
        plan.use_generic(False)
        assert rel(plan.matvec(dx, dy).to_host(), ref) < tol, dt


def test_transform_matches_numpy():
    """Single components, in double precision with the larger of two row counts."""
    N = (243, 99, 45)
    print('case fixed transform', N, flush=True)
    plan = nat.Plan(N, np.ones(3))
    x = np.random.default_rng(26).standard_normal(N)
    ref = np.fft.rfftn(x)
    for dt, ct, tol in ((np.float64, np.complex128, 1e-12), (np.float32, np.complex64, 2e-5)):
        X = plan.rfftn(nat.DeviceArray.from_host(x.astype(dt)[None]), nat.DeviceArray((1,) + ref.shape, ct), 1)
        assert rel(X.to_host()[0], ref) < tol
        z = plan.irfftn(X, nat.DeviceArray((1,) + N, dt), 1)
        assert rel(z.to_host()[0], x) < tol


@pytest.mark.parametrize('physics,kind,N', [('scalar', 'iso', (99, 45, 135)), ('scalar', 'iso', (105, 81, 105)),
                                            ('scalar', 'full', (135, 63, 75)), ('scalar', 'iso', (25, 225, 243)),
                                            ('elasticity', 'lame', (45, 27, 99))])
def test_schedule_variants_are_equal(physics, kind, N):
    """All 24 schedules transform each pencil alike: the same bits."""
    print('case fixed schedules', physics, kind, N, flush=True)
    rng = np.random.default_rng(23)
    plan = plan_of(N, physics, kind, rng)
    x = rng.standard_normal((plan.ncomp,) + N)
    for dt in (np.float64, np.float32):
        dx, dy = nat.DeviceArray.from_host(x.astype(dt)), nat.DeviceArray((plan.ncomp,) + N, dt)
        ref = plan.matvec(dx, dy).to_host()
        for v in np.ndindex(4, 2, 3):
            plan.set_schedule(dt, *v)
            assert np.array_equal(plan.matvec(dx, dy).to_host(), ref), (dt, v)


@pytest.mark.parametrize('physics,kind,N', [('scalar', 'iso', (99, 27, 135)), ('scalar', 'iso', (25, 225, 243)),
                                            ('elasticity', 'lame', (45, 27, 99))])
@pytest.mark.parametrize('mode', ['fp64', 'mixed'])
def test_solve_matches_generic_kernels(physics, kind, N, mode):
    """The same energy to 1e-10 and, at tol 1e-10, the same number of iterations within 2 (mixed: 4)."""
    print('case fixed solve', physics, kind, N, mode, flush=True)
    rng = np.random.default_rng(24)
    plan = plan_of(N, physics, kind, rng)
    nc = plan.ncomp
    E = np.eye(nc)[0]
    EN = nat.DeviceArray.zeros((nc,) + N)
    nat.add_constant(EN, -E)
    B = plan.matvec(EN, nat.DeviceArray((nc,) + N))
    out = []
    for generic in (True, False):
        plan.use_generic(generic)
        x = nat.DeviceArray.zeros((nc,) + N)
        info = plan.cg_solve(B, x, tol=1e-10, maxiter=500, mode=mode)
        assert info['status'] == nat.FH_CG_OK and info['norm_res'] <= 1e-10
        out.append((info['kit'], x.to_host()))
    assert abs(out[0][0] - out[1][0]) <= (2 if mode == 'fp64' else 4)
    assert rel(out[1][1], out[0][1]) < 1e-8
