"""FP64 batches of more than 2560 tiles split off the tiles that are all ocean;
each member alone has fewer and steps without the split: the same bits, at one
tile above and below the line, without, with one and with two tracers."""
import numpy as np
import pytest

from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [40, 41])   # 80 x 31 tiles and 2 x 40 or 2 x 41: 2560 or 2562
@pytest.mark.parametrize("tracers", [[0, 0, 0], [1, 0, 0], [2, 1, 0]])
def test_members_equal_alone(gpu_lib, cols, tracers):
    rng = np.random.default_rng(cols)
    setups = []
    for (nx, ny), n in zip([(31 * 32 - 5, 80 * 8 - 3), (cols * 32, 8), (cols * 32 - 9, 7)], tracers):
        s = configs.basin(nx, ny, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=500.0, dt=5.0, Ah=100.0, f0=1e-4,
                          beta=2e-11, lateral_mixing=True)
        for _ in range(n):
            host.add_tracer(s, 2.0 + rng.random(s.shape), kappa_h=50.0, gamma_C=1e-6, cons=1e-7)
        for g in s.grids.values():
            g.ocean = np.ones(s.shape, np.int8)
            g.ocean[: ny // 3, : nx // 3] = rng.random((ny // 3, nx // 3)) < 0.7
        s.u0, s.v0, s.eta0 = (0.1 * rng.standard_normal(s.shape) for _ in range(3))
        setups.append(host.finalize(s))
    names = [[("SWM_U", -1), ("SWM_V", -1), ("SWM_ETA", -1)] + [("CH", k) for k in range(n)] for n in tracers]
    members = [gpu.SwmGpu(s).init_from_setup() for s in setups]
    with gpu.SwmBatch() as b:
        for m in members:
            b.attach(m, 5)
        b.step(5)
        for s, m, ns in zip(setups, members, names):
            with gpu.SwmGpu(s).init_from_setup() as alone:
                alone.step(5)
                for n in ns:
                    assert same(m.get(*n), alone.get(*n)), n
            b.detach(m)
            m.close()
