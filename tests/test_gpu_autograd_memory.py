"""Device memory of the backward of solution_fields: the adjoint solves go load by load, so beside the d
adjoint solutions and the gradient one load's gradient and right-hand side are held, not those of all loads.
In a fresh interpreter, which loads torch before the library (one HIP runtime for both)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def case():
    import torch
    from ffthompy_amd.autograd import solution_fields
    N = (32, 36, 40)
    gen = torch.Generator(device='cuda').manual_seed(5)
    theta = (0.3 * torch.randn(N, dtype=torch.float64, device='cuda', generator=gen)).requires_grad_(True)
    e = solution_fields(theta, tol=1e-8)
    g = torch.randn(e.shape, dtype=torch.float64, device='cuda', generator=gen)
    field = 3 * 8 * theta.numel()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    e.backward(g)
    held = (torch.cuda.max_memory_allocated() - before) / field
    print('backward held %.2f fields' % held, flush=True)
    # 3 solutions, the right-hand side, at most two copies of a load's gradient, a third for the result
    assert held < 6.5, held


def test_backward_goes_load_by_load():
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-2000:])
    assert r.returncode == 0 and 'backward held' in r.stdout


if __name__ == '__main__':
    sys.path.insert(0, ROOT)
    case()
