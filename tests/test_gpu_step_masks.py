"""The tile kernels form every masked term and select by the bits of per-cell
codes; the marching kernel (shape 6) branches on the mask bytes themselves.
With land strewn at random over the four grids independently (every
combination of neighbours' masks, also those no bathymetry gives) both step to
the same FP64 state bit for bit, at the edges of the 32 x 8 and 64 x 4 tiles,
with row-compressed and with full static fields."""
import numpy as np
import pytest

from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


def setup(nx, ny, variant, full, seed):
    rng = np.random.default_rng(seed)
    s = configs.basin(nx, ny, 5e3, 5e3, variant=variant, H0=500.0, dt=5.0, Ah=100.0, f0=1e-4, beta=2e-11, drag=1e-6,
                      lateral_mixing=True, quadratic_friction=True, gamma_sq=2e-3, A=6371e3)
    host.add_windstress(s, host.COMP_X, configs.double_gyre_tau(s, 0.1))
    for _ in range(2 if variant == host.FULLY_NONLINEAR else 0):
        host.add_tracer(s, 2.0 + rng.random(s.shape), kappa_h=50.0, gamma_C=1e-6, cons=1e-7)
    for g in s.grids.values():
        g.ocean = (rng.random(s.shape) < 0.8).astype(np.int8)
        g.H = 400.0 + 100.0 * rng.random(s.shape) if full else np.full(s.shape, 500.0)
    if full:
        s.impl_u, s.impl_v, s.impl_eta = (1.0 + 1e-5 * rng.random(s.shape) for _ in range(3))
        s.F_x_const, s.F_y_const, s.F_eta_const = (1e-7 * rng.standard_normal(s.shape) for _ in range(3))
    s.u0, s.v0, s.eta0 = (0.1 * rng.standard_normal(s.shape) for _ in range(3))
    return host.finalize(s)


@pytest.mark.parametrize("nx,ny", [(32, 8), (33, 9), (64, 16), (65, 17), (95, 31), (5, 4)])
@pytest.mark.parametrize("variant", [host.FULLY_NONLINEAR, host.LINEARISED_STATE_OF_REST])
@pytest.mark.parametrize("full", [False, True])
def test_tiles_equal_marching_kernel_on_random_masks(gpu_lib, nx, ny, variant, full):
    s = setup(nx, ny, variant, full, seed=nx * ny + variant)
    names = [("SWM_U", -1), ("SWM_V", -1), ("SWM_ETA", -1), ("G_U", -1), ("G_V", -1), ("G_ETA", -1)]
    names += [(n, k) for k in range(len(s.tracers)) for n in ("CH", "G_CH")]
    out = {}
    for shape in (6, 11, 1, 0, 4):
        with gpu.SwmGpu(s).init_from_setup() as g:
            g.set_kernel_shape(shape)
            g.step(4)
            out[shape] = [g.get(*n) for n in names]
    for shape in (11, 1, 0, 4):
        for n, x, y in zip(names, out[shape], out[6]):
            assert same(x, y), (shape, n)
