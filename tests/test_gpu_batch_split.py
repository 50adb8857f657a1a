"""Batched solves with one load per task (up to 2048 samples) against two loads per task (beyond): the same
operations in the same order per load, so every result is the same bit for bit, whichever workgroup finishes
a sample last; and the fused iteration's ends (no iteration, one, a stop in the middle)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')


def batch(samples):
    b = nat.Batch([a.shape for a in samples])
    b.set_coeff(samples)
    b.set_schedule(1, 0)
    return b


@pytest.mark.parametrize('mode', ['fp64', 'mixed'])
def test_split_tasks_match_whole_tasks(mode):
    print('case batch split', mode, flush=True)
    rng = np.random.default_rng(91)
    few = [np.exp(rng.standard_normal(d)) for d in [(27, 27), (45, 27), (27, 63), (81, 45), (135, 27), (105, 135)]]
    small, large = batch(few), batch(few + [np.exp(rng.standard_normal((27, 27)))] * 2043)
    for maxiter in (0, 1, 7, 400):
        r, q = (b.solve(tol=1e-8, maxiter=maxiter, mode=mode) for b in (small, large))
        again = small.solve(tol=1e-8, maxiter=maxiter, mode=mode)
        for x, y, z in zip(r, q, again):
            assert np.array_equal(np.asarray(x), np.asarray(y)[:len(few)]) and np.array_equal(x, z), (maxiter, mode)
    assert np.all(np.asarray(r[3]) == 0) and np.all(np.asarray(r[2]) < 400)
