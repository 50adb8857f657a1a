"""The passes with the radix schedule as data or compiled per length (fh_rt.hpp) at the sizes where they
can go wrong: every radix, single- and multi-stage axes, odd and even rows and planes (padding row,
Nyquist slots), compiled and schedule-driven planes, row mode with a last workgroup of fewer rows,
planes of more than half of the LDS; and the fused double-precision CG against the operator form.

Tolerances as in test_gpu_kernels.py: float64 1e-12, float32 2e-5 relative to the largest entry."""
import numpy as np
import pytest

from oracle import projections
from oracle.fields import DFT, Field, Operator

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


# radices 2..16 alone and in pairs; planes compiled (16, 20, 48, 64, 81) and not (others); more than 256
# plane workgroups (130 x ..) take row mode; 144 x 144 double planes exceed half of the LDS
SHAPES = [(2, 3), (7, 15), (45, 16), (22, 26), (48, 169), (600, 11), (3, 1001),
          (2, 2, 2), (3, 2, 4), (2, 26, 22), (4, 13, 11), (2, 16, 16), (3, 20, 20), (2, 15, 14), (3, 121, 7),
          (2, 12, 10), (6, 5, 64), (64, 48, 48), (130, 4, 6), (260, 3, 5), (2, 144, 144), (3, 81, 81),
          (2, 156, 154), (9, 200, 210)]


@pytest.mark.parametrize('N', SHAPES, ids=[str(s) for s in SHAPES])
def test_transforms_match_numpy(N):
    print('case rt transforms', N, flush=True)
    rng = np.random.default_rng(60)
    nc = 3  # more components than a 2-D plan holds: the inverse runs in two groups
    plan = nat.Plan(N, np.ones(len(N)))
    Nh = N[:-1] + (N[-1] // 2 + 1,)
    axes = tuple(range(1, len(N) + 1))
    x = rng.standard_normal((nc,) + N)
    ref = np.fft.rfftn(x, axes=axes)
    Z = rng.standard_normal((nc,) + Nh) + 1j * rng.standard_normal((nc,) + Nh)
    for dt, ct, tol in ((np.float64, np.complex128, 1e-12), (np.float32, np.complex64, 2e-5)):
        dX = plan.rfftn(nat.DeviceArray.from_host(x.astype(dt)), nat.DeviceArray((nc,) + Nh, ct), nc)
        assert rel(dX.to_host(), ref) < tol, (dt, rel(dX.to_host(), ref))
        Zc = Z.astype(ct)
        dz = plan.irfftn(nat.DeviceArray.from_host(Zc), nat.DeviceArray((nc,) + N, dt), nc)
        zref = np.fft.irfftn(Zc.astype(np.complex128), s=N, axes=axes)
        assert rel(dz.to_host(), zref) < tol, (dt, rel(dz.to_host(), zref))


def _coef(rng, kind, nc, N):
    if kind == 'iso':
        a = 1. + rng.random(N)
        return a, np.einsum('ij,...->ij...', np.eye(nc), a)
    if kind == 'lame':
        lam, mu = 1. + rng.random(N), 0.5 + rng.random(N)
        m = np.zeros(nc)
        m[:3 if nc == 6 else 2] = 1.
        return np.stack([lam, mu]), (np.einsum('i,j,...->ij...', m, m, lam)
                                     + 2 * np.einsum('ij,...->ij...', np.eye(nc), mu))
    A = 0.2 * rng.standard_normal((nc, nc) + N)
    A = A + np.swapaxes(A, 0, 1) + 3. * np.eye(nc).reshape((nc, nc) + (1,) * len(N))
    return A, A


def _hG(physics, N, pd):
    if physics == 'scalar':
        _, G1, G2 = projections.scalar(N, np.ones(len(N)))
        return (G1 if pd == 'primal' else G2).val
    _, G1h, G1s, G2h, G2s = projections.elasticity(N, np.ones(len(N)))
    return G1h.val + G1s.val if pd == 'primal' else G2h.val + G2s.val


MATVEC = [('scalar', 'iso', (7, 16, 16), 'primal'), ('scalar', 'full', (6, 13, 10), 'dual'),
          ('scalar', 'iso', (22, 26), 'dual'), ('scalar', 'full', (15, 33), 'primal'),
          ('elasticity', 'lame', (5, 20, 20), 'primal'), ('elasticity', 'full', (4, 9, 14), 'dual'),
          ('elasticity', 'lame', (50, 8, 6), 'dual'), ('elasticity', 'lame', (30, 22), 'primal'),
          ('elasticity', 'full', (16, 21), 'dual')]


@pytest.mark.parametrize('physics,kind,N,pd', MATVEC, ids=['%s-%s-%s-%s' % c for c in MATVEC])
def test_operator_matches_oracle_and_generic_kernels(physics, kind, N, pd):
    print('case rt operator', physics, kind, N, pd, flush=True)
    rng = np.random.default_rng(61)
    plan = nat.Plan(N, np.ones(len(N)), physics, pd)
    nc = plan.ncomp
    vals, A = _coef(rng, kind, nc, N)
    plan.set_coeff(kind, vals)
    x = rng.standard_normal((nc,) + N)
    ref = Operator([[DFT(N, inverse=True), Field(val=_hG(physics, N, pd), order=2, N=N, multype=21, Fourier=True),
                     DFT(N), Field(val=A, order=2, multype=21)]])(Field(val=x, order=1)).val
    for dt, tol in ((np.float64, 1e-12), (np.float32, 2e-5)):
        dx = nat.DeviceArray.from_host(x.astype(dt))
        for generic in (False, True):
            plan.use_generic(generic)
            y = plan.matvec(dx, nat.DeviceArray((nc,) + N, dt)).to_host()
            assert rel(y, ref) < tol, (dt, generic, rel(y, ref))
        # in place: the forward pass has read all of x before the inverse one writes it
        plan.use_generic(False)
        assert rel(plan.matvec(dx, dx).to_host(), ref) < tol


SOLVES = [('scalar', 'iso', (45, 45), 30.), ('scalar', 'iso', (20, 24, 18), 30.), ('scalar', 'full', (9, 12, 15), 1.),
          ('elasticity', 'lame', (27, 27, 27), 5.), ('elasticity', 'lame', (33, 20), 5.),
          ('scalar', 'iso', (90, 100, 77), 10.), ('elasticity', 'full', (10, 9, 8), 1.)]


@pytest.mark.parametrize('physics,kind,N,spread', SOLVES, ids=['%s-%s-%s' % c[:3] for c in SOLVES])
@pytest.mark.parametrize('x0', ['zero', 'random'])
def test_fused_fp64_cg_matches_operator_form(physics, kind, N, spread, x0):
    """The fused iteration (denominator <p, A p>, solution one step late, alpha and beta in the passes)
    against the operator form: the same iteration count and, at tol 1e-10, the same solution to 1e-8;
    the true residual of the returned x is the norm reported; repeated solves are equal to the bit."""
    print('case fused fp64', physics, kind, N, x0, flush=True)
    rng = np.random.default_rng(62)
    plan = nat.Plan(N, np.ones(len(N)), physics, 'primal')
    nc = plan.ncomp
    vals, _ = _coef(rng, kind, nc, N)
    if kind != 'full':
        vals = np.where(rng.random(N) < 0.3, spread, 1.) * vals
    plan.set_coeff(kind, vals)
    EN = nat.DeviceArray.zeros((nc,) + N)
    nat.add_constant(EN, -np.eye(nc)[nc - 1])
    B = plan.matvec(EN, nat.DeviceArray((nc,) + N))
    start = np.zeros((nc,) + N) if x0 == 'zero' else 0.1 * rng.standard_normal((nc,) + N)
    out = []
    for fused in (True, False, True):
        plan.set_cg_variant(fused)
        x = nat.DeviceArray.from_host(start)
        info = plan.cg_solve(B, x, tol=1e-10, maxiter=2000, mode='fp64', hist_len=100)
        assert info['status'] == nat.FH_CG_OK and info['norm_res'] <= 1e-10
        r = B.to_host() - plan.matvec(x, nat.DeviceArray((nc,) + N)).to_host()
        assert abs(np.sqrt(np.sum(r * r) / np.prod(N)) - info['norm_res']) < 1e-12
        out.append((info['kit'], x.to_host(), info['res_log']))
    assert abs(out[0][0] - out[1][0]) <= 1, (out[0][0], out[1][0])
    assert rel(out[0][1], out[1][1]) < 1e-8
    k = min(len(out[0][2]), len(out[1][2])) // 2
    assert np.allclose(out[0][2][:k], out[1][2][:k], rtol=1e-6)
    assert out[0][0] == out[2][0] and np.array_equal(out[0][1], out[2][1])


def test_right_hand_side_outside_the_range_keeps_the_operator_form():
    """b with a part outside the range of G: the solve takes the operator form (the fused denominator would
    differ), bit for bit the result of the plan with the fused iteration switched off."""
    print('case rhs outside range', flush=True)
    N = (20, 24, 18)
    rng = np.random.default_rng(63)
    plan = nat.Plan(N, np.ones(3), 'scalar', 'primal')
    plan.set_coeff('iso', 1. + 9. * rng.random(N))
    b = nat.DeviceArray.from_host(rng.standard_normal((3,) + N))
    out = []
    for fused in (True, False):
        plan.set_cg_variant(fused)
        x = nat.DeviceArray.zeros((3,) + N)
        info = plan.cg_solve(b, x, tol=1e-8, maxiter=12, mode='fp64')
        out.append((info['kit'], info['norm_res'], x.to_host()))
    assert out[0][:2] == out[1][:2] and np.array_equal(out[0][2], out[1][2])


def test_maxiter_and_zero_right_hand_side():
    print('case fused fp64 limits', flush=True)
    N = (15, 15, 15)
    rng = np.random.default_rng(64)
    plan = nat.Plan(N, np.ones(3), 'scalar', 'primal')
    plan.set_coeff('iso', 1. + 99. * (rng.random(N) < 0.3))
    EN = nat.DeviceArray.zeros((3,) + N)
    nat.add_constant(EN, [1., 0., 0.])
    B = plan.matvec(EN, nat.DeviceArray((3,) + N))
    ref = {}
    for fused in (True, False):
        plan.set_cg_variant(fused)
        for maxiter in (0, 1, 7, 8, 9):
            x = nat.DeviceArray.zeros((3,) + N)
            info = plan.cg_solve(B, x, tol=1e-12, maxiter=maxiter, mode='fp64')
            assert info['kit'] == maxiter
            xh = x.to_host()
            if fused:
                ref[maxiter] = xh
            else:
                assert np.abs(xh - ref[maxiter]).max() <= 1e-11 * max(np.abs(xh).max(), 1.), maxiter
        x = nat.DeviceArray.zeros((3,) + N)
        info = plan.cg_solve(nat.DeviceArray.zeros((3,) + N), x, tol=1e-8, maxiter=5, mode='fp64')
        assert info['kit'] == 0 and not x.to_host().any()
