"""The autograd functions on GPU tensors (lent to the library) against the same on CPU tensors (through host
memory): the same kernels on the same values, so results differ by the rounding of exp alone (1e-16, amplified
by the solves to less than 1e-9); strided and single
-precision inputs, a stream of the caller's own, and inputs and outputs overwritten afterwards."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip('torch')
nat = pytest.importorskip('ffthompy_amd._native')
from ffthompy_amd.autograd import solution_fields, upper_bound  # noqa: E402


def run(theta, fn):
    t = theta.clone(memory_format=torch.preserve_format).requires_grad_(True)
    out = fn(t, tol=1e-10)
    kept = out.detach().clone()
    loss = ((out - 0.5) ** 2).sum()
    with torch.no_grad():
        t.mul_(0.).add_(7.)  # the backward works on the values of the forward
    loss.backward()
    return kept.cpu().numpy(), t.grad.cpu().numpy()


@pytest.mark.parametrize('fn', [upper_bound, solution_fields], ids=['upper_bound', 'solution_fields'])
@pytest.mark.parametrize('how', ['plain', 'strided', 'float32', 'stream'])
def test_gpu_tensors_match_cpu_tensors(how, fn):
    print('case autograd device', how, fn.__name__, flush=True)
    nat.init()
    rng = np.random.default_rng(95)
    v = torch.from_numpy(0.5 * rng.standard_normal((9, 15, 14)))
    if how == 'strided':
        v = v.transpose(0, 2)
    if how == 'float32':
        v = v.to(torch.float32).exp().log()
    ref = run(v, fn)
    g = v.cuda()
    if how == 'float32':  # exp in single precision differs between the devices: the host values decide
        ref = run(v.double(), fn)
        g = v.double().cuda()
        got32 = run(v.cuda(), fn)
        assert all(np.abs(a - b).max() <= 1e-5 * np.abs(b).max() for a, b in zip(got32, ref))
    if how == 'stream':
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            got = run(g, fn)
        side.synchronize()
    else:
        got = run(g, fn)
    for a, b in zip(got, ref):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert np.abs(a - b).max() <= 1e-9 * np.abs(b).max()
