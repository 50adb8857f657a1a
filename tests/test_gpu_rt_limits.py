"""The passes of any smooth length (fh_rt.hpp) at their limits: more components than the plan has, with a
spectrum above 2 GiB in all (lanes without work are put out of a buffer resource by offsets from 2 GiB on)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def part(arr, c, shape):
    """Component c of a device array."""
    n = int(np.prod(shape)) * arr.dtype.itemsize
    return nat.DeviceArray.borrow(arr.ptr.value + c * n, shape, arr.dtype)


@pytest.mark.parametrize('dt,ct,nc', [(np.float64, np.complex128, 36), (np.float32, np.complex64, 68)])
def test_transform_of_more_than_two_gib(dt, ct, nc):
    """200^3, a 6 x 6 tensor field (double precision, 2.33 GB of spectrum) and 68 components in single precision
    (2.2 GB): every component bitwise equal to its own transform, the first also to numpy's. 101 columns are
    no multiple of the tiles."""
    N = (200, 200, 200)
    print('case transform above 2 GiB', N, dt.__name__, nc, flush=True)
    rng = np.random.default_rng(68)
    plan = nat.Plan(N, np.ones(3))
    Nh = N[:-1] + (N[-1] // 2 + 1,)
    base = rng.standard_normal(N).astype(dt)
    x, X = nat.DeviceArray((nc,) + N, dt), nat.DeviceArray((nc,) + Nh, ct)
    one = nat.DeviceArray((1,) + Nh, ct)
    for c in range(nc):
        v = nat.DeviceArray.from_host(np.roll(base, c, axis=0))
        nat.call('fh_memcpy_dtod', part(x, c, N).ptr, v.ptr, v.nbytes)
    plan.rfftn(x, X, nc)
    tol = 1e-12 if dt is np.float64 else 2e-5
    assert rel(part(X, 0, Nh).to_host(), np.fft.rfftn(base.astype(np.float64))) < tol
    for c in range(nc):
        plan.rfftn(part(x, c, (1,) + N), one, 1)
        assert np.array_equal(part(X, c, Nh).to_host(), one.to_host()[0]), c


@pytest.mark.parametrize('N,nc', [((2, 2000, 2000), 1), ((2, 2000, 2000), 3), ((16, 1500, 1500), 1)])
def test_transforms_of_flat_grids(N, nc):
    """More tiles along the outermost axis (125125 of 16 points in double, 62563 of 32 in single precision at
    2 x 2000 x 2000) than a multiply-high alone splits into slabs."""
    print('case flat transforms', N, nc, flush=True)
    rng = np.random.default_rng(65)
    plan = nat.Plan(N, np.ones(len(N)))
    Nh = N[:-1] + (N[-1] // 2 + 1,)
    x = rng.standard_normal((nc,) + N)
    ref = np.fft.rfftn(x, axes=tuple(range(1, x.ndim)))
    for dt, ct, tol in ((np.float64, np.complex128, 1e-12), (np.float32, np.complex64, 2e-5)):
        X = plan.rfftn(nat.DeviceArray.from_host(x.astype(dt)), nat.DeviceArray((nc,) + Nh, ct), nc)
        assert rel(X.to_host(), ref) < tol, dt
        z = plan.irfftn(X, nat.DeviceArray((nc,) + N, dt), nc)
        assert rel(z.to_host(), x) < tol, dt


def test_potential_solve_of_a_flat_grid():
    """Iterates of the fp64 solve against the generic kernels (tolerance as in test_gpu_rt_potential.py)."""
    N = (2, 2000, 2000)
    print('case flat potential', N, flush=True)
    plan = nat.Plan(N, np.ones(3))
    plan.set_coeff('iso', np.exp(0.5 * np.random.default_rng(66).standard_normal(N)))
    out = []
    for generic in (True, False):
        plan.use_generic(generic)
        Fu, info = plan.potential_solve(np.array([1., 0.5, 0.2]), 1e-11, 4, mode='fp64')
        out.append((Fu.to_host(), info['kit'], info['status']))
    assert out[0][1:] == out[1][1:] == (4, nat.FH_CG_OK)
    assert rel(out[1][0], out[0][0]) <= 1e-11
