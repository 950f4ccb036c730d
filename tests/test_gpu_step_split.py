"""FP64 domains of more than 2560 tiles split off the tiles that are all ocean:
with land in one corner only, so that both kinds occur, at partial tiles on
either edge and just below and above the line, the default kernel steps to the
same bits as the one without the split (shape 1)."""
import numpy as np
import pytest

from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1638, 394), (1664, 393), (64 * 32, 40 * 8), (2561 * 32, 5)])
@pytest.mark.parametrize("tracers", [0, 1, 2])
def test_split_equals_unsplit(gpu_lib, nx, ny, tracers):
    rng = np.random.default_rng(nx)
    s = configs.basin(nx, ny, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=500.0, dt=5.0, Ah=100.0, f0=1e-4, beta=2e-11,
                      lateral_mixing=True)
    for _ in range(tracers):
        host.add_tracer(s, 2.0 + rng.random(s.shape), kappa_h=50.0, gamma_C=1e-6, cons=1e-7)
    for g in s.grids.values():
        g.ocean = np.ones(s.shape, np.int8)
        g.ocean[: ny // 3, : nx // 3] = rng.random((ny // 3, nx // 3)) < 0.7
    s.u0, s.v0, s.eta0 = (0.1 * rng.standard_normal(s.shape) for _ in range(3))
    s = host.finalize(s)
    names = [("SWM_U", -1), ("SWM_V", -1), ("SWM_ETA", -1), ("G_U", -1)] + [("CH", k) for k in range(tracers)]
    out = {}
    for shape in (1, 11):
        with gpu.SwmGpu(s).init_from_setup() as g:
            g.set_kernel_shape(shape)
            g.step(3)
            out[shape] = [g.get(*n) for n in names]
    for n, x, y in zip(names, out[11], out[1]):
        assert same(x, y), n
