"""Red-black sweeps on register tiles (sor_rows) against one colour per launch
(SWM_GPU_SOR_BLOCK=0): the same chi bit for bit and the same sweep count, at
the edges of its tiles (112 columns; 16, 32 or 48 rows with four sweeps per
launch), over every grid it takes: even extents closed or open in x, odd ones
closed at the seam, islands, one-cell barriers, fewer columns than a
wavefront's; for cadences that do and do not divide the sweeps of a launch,
stopping inside one (the launch is run again up to that sweep) or at the cap."""
import numpy as np
import pytest

from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


def solve(monkeypatch, s, B, chi, blocked, every, tol, sweeps, fp32):
    monkeypatch.setenv("SWM_GPU_SOR_BLOCK", blocked)
    with gpu.SwmGpu(s) as g:
        g.set_sor_check_every(every)
        return g.sor_fixed(B, chi, 1.8, tol, sweeps, fp32_sweeps=fp32)


@pytest.mark.parametrize("nx,ny,walls,land", [
    (112, 16, True, 0.0), (113, 17, True, 0.1), (225, 33, True, 0.1),   # a column / row more than whole tiles
    (3, 3, True, 0.0), (16, 200, False, 0.0),                            # narrower than the halo
    (128, 48, False, 0.1), (226, 31, False, 0.1),                        # periodic in x, odd rows closed
    (900, 700, True, 0.1),                                               # 64-row tiles
    (1790, 1021, True, 0.05),                                            # 48-row tiles
])
@pytest.mark.parametrize("every,fp32", [(1, False), (3, True), (4, False)])
def test_register_tiles_equal_one_colour_per_launch(gpu_lib, monkeypatch, nx, ny, walls, land, every, fp32):
    s = host.finalize(configs.basin(nx, ny, 10e3, 10e3, variant=host.FULLY_NONLINEAR, H0=500.0, dt=10.0,
                                    seed=nx + ny, land_fraction=land, side_walls=walls, A=6371e3))
    rng = np.random.default_rng(nx * ny)
    B = 1e-6 * rng.standard_normal(s.shape)
    chi = 1e3 * rng.standard_normal(s.shape)
    cap = 22 if nx * ny > 1e5 else 50
    for tol in (0.0, None):
        if tol is None:   # passed for the first time about half way: the norm the capped run had there
            half = solve(monkeypatch, s, B, chi, "0", every, 0.0, cap // 2 // every * every, fp32)
            tol = half[2] * (1 + 1e-9)
        want = solve(monkeypatch, s, B, chi, "0", every, tol, cap, fp32)
        got = solve(monkeypatch, s, B, chi, "1", every, tol, cap, fp32)
        assert same(got[0], want[0])
        assert got[1] == want[1] and got[3] == want[3]
        assert got[2] == want[2] or abs(got[2] - want[2]) <= 1e-12 * abs(want[2])
