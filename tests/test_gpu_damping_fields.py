"""Implicit damping given cell by cell divides by the field itself, the IEEE
quotient, down to the smallest tracer values, where a quotient formed through
the divisor's reciprocal can be one unit in the last place off: tracers of
1e-308 to 1e-302, and a flow of that size started from rest, against the oracle
bit for bit, in a domain alone (default tiles, and those of a domain large
enough to split off its all-ocean tiles) and in a batch."""
import numpy as np
import pytest

import oracle
from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


def setup(nx, ny, tracers, seed):
    rng = np.random.default_rng(seed)
    s = configs.basin(nx, ny, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=1.0, dt=5.0, Ah=10.0, lateral_mixing=True)
    for _ in range(tracers):
        C = 2.0 ** rng.uniform(-1021.0, -1003.0, s.shape) * rng.choice([-1.0, 1.0], s.shape)
        host.add_tracer(s, C, kappa_h=50.0, cons=2e-3 * rng.random(s.shape))
    s.eta0 = 1e-3 * rng.standard_normal(s.shape)
    return host.finalize(s)


@pytest.mark.parametrize("nx,ny,tracers", [(130, 70, 1), (130, 70, 2), (1025, 650, 1)])
def test_tiny_tracers_are_divided_by_the_damping_field(gpu_lib, nx, ny, tracers):
    s = setup(nx, ny, tracers, seed=nx + tracers)
    o = oracle.Oracle(s)
    o.step(4)
    want = [o.get("CH", k) for k in range(tracers)]
    o.close()
    alone = gpu.SwmGpu(s).init_from_setup()
    alone.step(4)
    m = gpu.SwmGpu(s).init_from_setup()
    with gpu.SwmBatch() as b:
        b.attach(m, 4)
        b.step(4)
        for k in range(tracers):
            assert 1e-308 < np.nanmedian(np.abs(want[k])) < 1e-302
            assert same(alone.get("CH", k), want[k]), k
            assert same(m.get("CH", k), want[k]), k
        b.detach(m)
    alone.close()
    m.close()


@pytest.mark.parametrize("nx,ny", [(130, 70), (1025, 650)])
@pytest.mark.parametrize("tiny", [True, False])
def test_flow_is_divided_by_the_damping_field(gpu_lib, nx, ny, tiny):
    """Forced from rest, a flow's first increments carry no other quotient; at
    ordinary sizes it goes on for some steps."""
    rng = np.random.default_rng(nx)
    s = configs.basin(nx, ny, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=1.0, dt=1.0)
    s.impl_u, s.impl_v, s.impl_eta = (1.0 + 1e-2 * rng.random(s.shape) for _ in range(3))
    size = lambda: 2.0 ** (rng.uniform(-1021.0, -1003.0, s.shape) if tiny else -10.0) * rng.choice([-1.0, 1.0], s.shape)
    s.F_x_const, s.F_y_const, s.F_eta_const = size(), size(), size()
    s = host.finalize(s)
    steps = 2 if tiny else 9
    o = oracle.Oracle(s)
    o.step(steps)
    with gpu.SwmGpu(s).init_from_setup() as alone, gpu.SwmGpu(s).init_from_setup() as m, gpu.SwmBatch() as b:
        alone.step(steps)
        b.attach(m, steps)
        b.step(steps)
        for n in ("u", "v", "eta"):
            want = o.get(n)
            assert not tiny or 1e-308 < np.median(np.abs(want)) < 1e-302
            assert same(alone.get("SWM_" + n.upper()), want), n
            assert same(m.get("SWM_" + n.upper()), want), n
        b.detach(m)
    o.close()
