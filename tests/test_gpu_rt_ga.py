"""The padded passes of the Ga energies (fh_rt_ga.hpp) against the generic kernels: odd and even coarse axes
(split Nyquist coefficients), quadrature lengths compiled and schedule-driven, grids larger than 2N - 1, an
odd number of rows, one-stage axes, every number of components.

The two paths differ by rounding: interpolation multiplies sums of at most 45^3 terms of order one by unit
roundings of 1.1e-16 times the depth of the transforms, so 1e-12 of the largest entry holds for both."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

nat = pytest.importorskip('ffthompy_amd._native')

SHAPES = [((2, 3), None), ((5, 7), None), ((6, 4), (13, 8)), ((45, 45), None), ((33, 2), (70, 3)),
          ((2, 2, 2), None), ((3, 3, 3), (6, 5, 7)), ((4, 6, 2), None), ((9, 15, 7), None), ((27, 45, 14), (54, 90, 28)),
          ((14, 3, 25), (27, 5, 50))]


@pytest.mark.parametrize('physics', ['scalar', 'elasticity'])
@pytest.mark.parametrize('N,M', SHAPES, ids=[str(s) for s in SHAPES])
def test_padded_passes_match_generic(N, M, physics):
    print('case rt ga', N, M, physics, flush=True)
    rng = np.random.default_rng(81)
    plan = nat.Plan(N, np.linspace(1., 2., len(N)), physics)
    nc = plan.ncomp
    fields = [rng.standard_normal((nc,) + N) for _ in range(nc)]
    dev = [nat.DeviceArray.from_host(f) for f in fields]
    ga = nat.Ga(plan, M)
    kinds = [('iso', 1 + rng.random(N))]
    A = rng.standard_normal((nc, nc) + N)
    kinds.append(('full', A + np.swapaxes(A, 0, 1)))
    if physics == 'elasticity':
        kinds.append(('lame', 1 + rng.random((2,) + N)))
    for kind, vals in kinds:
        ga.set_grid_coeff(0, N, kind, vals)
        out = {}
        for generic in (True, False):
            plan.use_generic(generic)
            out[generic] = ga.energy_matrix(dev), ga.interpolate(dev[0]).to_host()
        plan.use_generic(False)
        for a, b in zip(out[False], out[True]):
            assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max(), (kind, np.abs(a - b).max(), np.abs(b).max())
