"""The stream function's sums at the edges of their kernels: rows of one and of
several 64-cell, 256-cell and 1024-cell groups and of two LDS chunks, columns of
less than one, one and several groups of 64 rows; every value in the oracle's
order of additions, so bit for bit."""
import numpy as np
import pytest

import oracle
from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(3, 3), (64, 63), (65, 64), (66, 65), (257, 127), (258, 128), (321, 129), (1025, 9),
                                   (1026, 200), (2050, 5), (3100, 4)])
def test_psi_at_group_edges(gpu_lib, nx, ny):
    rng = np.random.default_rng(nx + ny)
    s = host.finalize(configs.basin(nx, ny, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=300.0, dt=10.0, f0=1e-4,
                                    beta=2e-11, seed=8, land_fraction=0.05))
    u = rng.standard_normal(s.shape) * s.grids["u"].ocean
    v = rng.standard_normal(s.shape) * s.grids["v"].ocean
    o = oracle.Oracle(s)
    with gpu.SwmGpu(s) as g:
        g.upload_state(u, v, np.zeros(s.shape), itt=0)
        assert same(g.get("PSI"), o.psi(u, v))
    o.close()
