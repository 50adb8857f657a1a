"""The autograd functions on GPU tensors (lent to the library) against the same on CPU tensors (through host
memory): the same kernels on the same values, so results differ by the rounding of exp alone (1e-16, amplified
by the solves to less than 1e-9; single-precision input 6e-8, to less than 1e-5); strided input, a stream of
the caller's own, and inputs overwritten between forward and backward.

torch and the library share one HIP runtime only where torch is loaded first, as in a program that hands it
GPU tensors, so the cases run in a fresh interpreter."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(torch, theta, fn):
    t = theta.clone(memory_format=torch.preserve_format).requires_grad_(True)
    out = fn(t, tol=1e-10)
    kept = out.detach().clone()
    loss = ((out - 0.5) ** 2).sum()
    with torch.no_grad():
        t.mul_(0.).add_(7.)  # the backward works on the values of the forward
    loss.backward()
    return kept.cpu().numpy(), t.grad.cpu().numpy()


def cases():
    import torch
    from ffthompy_amd.autograd import solution_fields, upper_bound
    v = torch.from_numpy(0.5 * np.random.default_rng(95).standard_normal((9, 15, 14)))
    for fn in (upper_bound, solution_fields):
        for how in ('plain', 'strided', 'float32', 'stream'):
            print('case autograd device', how, fn.__name__, flush=True)
            x = v.transpose(0, 2) if how == 'strided' else v
            ref = run(torch, x, fn)
            g = (x.to(torch.float32) if how == 'float32' else x).cuda()
            side = torch.cuda.Stream() if how == 'stream' else torch.cuda.current_stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                got = run(torch, g, fn)
            side.synchronize()
            tol = 1e-5 if how == 'float32' else 1e-9
            for a, b in zip(got, ref):
                assert a.shape == b.shape
                assert np.abs(a - b).max() <= tol * np.abs(b).max(), (how, np.abs(a - b).max())


def test_gpu_tensors_match_cpu_tensors():
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-2000:])
    assert r.returncode == 0 and r.stdout.count('case') == 8


if __name__ == '__main__':
    sys.path.insert(0, ROOT)
    cases()
