"""Little free device memory: calls that took less of it in an earlier form still run in that form. All but a known
amount is reserved (allocations that nothing writes to), and released again before the test ends."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')

MB = 1 << 20


def reserve(left):
    """Reserve device memory in pieces down to 64 MB; release pieces of 64 MB worth `left` bytes."""
    held = []
    for piece in (8192 * MB, 1024 * MB, 64 * MB):
        while True:
            try:
                held.append(nat.DeviceArray((piece // 8,)))
            except nat.FhError:
                break
        if piece == 1024 * MB:
            held.pop()  # enough pieces of 64 MB
    for _ in range(-(-left // (64 * MB))):
        assert held[-1].nbytes == 64 * MB
        held.pop()
    return held


def test_fp64_solve_without_memory_for_the_fused_iteration():
    """A coupled coefficient: four work vectors (472 MB) for the fused iteration, three for the operator form."""
    print('case little memory: solve', flush=True)
    N, nc = (135, 135, 135), 6
    rng = np.random.default_rng(69)
    a = np.where(rng.random(N) < 0.3, 10., 1.)
    plan = nat.Plan(N, np.ones(3), 'elasticity', 'primal')
    plan.set_coeff('lame', np.stack([0.6 * a, 0.4 * a]))
    EN = nat.DeviceArray.zeros((nc,) + N)
    nat.add_constant(EN, -np.eye(nc)[0])
    B = plan.matvec(EN, nat.DeviceArray((nc,) + N))
    x = nat.DeviceArray.zeros((nc,) + N)
    held = reserve(448 * MB)
    try:
        info = plan.cg_solve(B, x, tol=1e-6, maxiter=30, mode='fp64')
    finally:
        held.clear()
    plan.set_cg_variant(False)
    y = nat.DeviceArray.zeros((nc,) + N)
    ref = plan.cg_solve(B, y, tol=1e-6, maxiter=30, mode='fp64')
    assert (info['kit'], info['norm_res']) == (ref['kit'], ref['norm_res'])
    assert np.array_equal(x.to_host(), y.to_host())


def test_batch_without_memory_for_its_solutions():
    """1000 samples of 135 x 135: 1.2 GB of solutions where a task is one load, none where it is both."""
    print('case little memory: batch', flush=True)
    a = np.exp(0.3 * np.random.default_rng(70).standard_normal((135, 135)))
    out = []
    for held, S in ((reserve(1280 * MB), 1000), ([], 4)):
        try:
            b = nat.Batch([a.shape] * S)
            b.set_coeff([a] * S)
            b.set_schedule(1, 0)
            out.append([np.asarray(v)[:4] for v in b.solve(tol=1e-6, maxiter=20, mode='mixed')])
        finally:
            held.clear()
    assert all(np.array_equal(u, v) for u, v in zip(*out))
