"""Thin grids of fixed lengths (few planes): the passes of any smooth length run them in rows although the
planes fit LDS. Operator, transforms and solves on both sides of the rule, against the generic kernels; tolerances
as in test_gpu_kernels.py (operator) and test_gpu_rt_potential.py (iterates)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')

# rows: too few planes, ragged or square (125: three stages, single precision); planes: (5, 25, 9), (15, 27, 45)
SHAPES = [(5, 27, 45), (5, 45, 27), (5, 225, 75), (15, 135, 99), (27, 243, 45), (5, 99, 99), (15, 135, 135), (27, 125, 125),
          (5, 25, 9), (15, 27, 45), (15, 99, 99)]


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize('N', SHAPES, ids=[str(s) for s in SHAPES])
def test_thin_grids_match_generic_kernels(N):
    print('case thin grid', N, flush=True)
    rng = np.random.default_rng(25)
    plan = nat.Plan(N, np.linspace(1., 1.3, 3), 'scalar', 'primal')
    x = rng.standard_normal((3,) + N)
    Nh = (3,) + N[:-1] + (N[-1] // 2 + 1,)
    for kind in ('iso', 'full'):
        a = 1. + rng.random(N)
        plan.set_coeff(kind, a if kind == 'iso' else np.einsum('ij,...->ij...', np.eye(3) + 0.1, a))
        for dt, ct, tol in ((np.float64, np.complex128, 1e-12), (np.float32, np.complex64, 2e-5)):
            dx, dy = nat.DeviceArray.from_host(x.astype(dt)), nat.DeviceArray((3,) + N, dt)
            out = []
            for generic in (True, False):
                plan.use_generic(generic)
                X = plan.rfftn(dx, nat.DeviceArray(Nh, ct), 3)
                out.append((plan.matvec(dx, dy).to_host(), X.to_host(),
                            plan.irfftn(X, nat.DeviceArray((3,) + N, dt), 3).to_host()))
            for g, f in zip(*out):
                assert rel(f, g) < tol, (kind, dt)
        EN = nat.DeviceArray.zeros((3,) + N)
        nat.add_constant(EN, -np.eye(3)[1])
        B = plan.matvec(EN, nat.DeviceArray((3,) + N))
        for mode, tol in (('fp64', 1e-11), ('mixed', 1e-3)):
            out = []
            for generic in (True, False):
                plan.use_generic(generic)
                s = nat.DeviceArray.zeros((3,) + N)
                info = plan.cg_solve(B, s, tol=1e-12, maxiter=6, mode=mode)
                Fu, pinfo = plan.potential_solve(np.array([1., 0.5, 0.2]), 1e-11, 4, mode=mode)
                assert info['kit'] == 6 and pinfo['kit'] == 4
                out.append((s.to_host(), Fu.to_host()))
            for g, f in zip(*out):
                assert rel(f, g) <= tol, (kind, mode)
