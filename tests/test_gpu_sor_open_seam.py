"""Red-black sweeps on odd extents that are open across their periodic seam,
where the seam's neighbours have the same colour: the LDS tiles (sor_block),
which only these grids take, and one colour per launch both update the last
column and row after a colour's other cells, as the sequential sweep does, and
so give the oracle's chi bit for bit for every halo and tile height; extents
down to and below the tile's halo, one seam or two (with the corner that both
share), islands, FP32 sweeps, stops inside a launch, and the reference mode."""
import numpy as np
import pytest

import oracle
from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu

# (halo, rows, cadence): 4, 2 and 1 sweeps a launch, and one colour
FORMS = [(-1, 16, 4), (-1, 16, 3), (8, 16, 8), (4, 16, 2), (4, 32, 4), (2, 16, 1), (2, 32, 3), (0, 16, 1)]


def setup(nx, ny, kind):
    """A channel open in x with islands, a torus of ocean, or a torus with one
    land column, open in y only."""
    s = configs.basin(nx, ny, 10e3, 10e3, variant=host.FULLY_NONLINEAR, H0=500.0, dt=10.0, seed=nx + ny,
                      land_fraction=0.1 if kind == "channel" else 0.0, side_walls=False, A=6371e3)
    if kind != "channel":
        for n, g in s.grids.items():
            g.ocean = np.ones(s.shape, np.int8)
            if kind == "wall":
                g.ocean[:, 0] = 0
                g.ocean[:, 1] = n in ("v", "eta")
    return host.finalize(s)


def rhs(o, s, seed):
    rng = np.random.default_rng(seed)
    return o.divergence(rng.standard_normal(s.shape) * s.grids["u"].ocean,
                        rng.standard_normal(s.shape) * s.grids["v"].ocean)


def settings(g, halo, rows, every):
    g.set_sor_tile_rows(rows)
    g.set_sor_check_every(every)
    g.set_sor_halo(halo)


@pytest.mark.parametrize("nx,ny,kind", [
    (301, 40, "channel"), (131, 75, "channel"), (65, 17, "channel"), (11, 16, "channel"), (9, 12, "channel"),
    (5, 8, "channel"), (97, 83, "torus"), (64, 33, "torus"), (33, 48, "torus"), (11, 11, "torus"), (7, 9, "torus"),
    (97, 83, "wall"), (128, 31, "wall")])
def test_sweeps_equal_sequential_sweeps(gpu_lib, nx, ny, kind):
    s = setup(nx, ny, kind)
    assert s.grids["u"].ocean[:, 0].any() == (kind != "wall") and s.grids["v"].ocean[0].any() == (kind != "channel")
    o = oracle.Oracle(s)
    B = rhs(o, s, 3)
    chi0 = 1e3 * np.random.default_rng(5).standard_normal(s.shape)
    want = o.sor_fixed(B, chi0, 1.9, 0.0, 43)
    o.close()
    for form in FORMS:
        with gpu.SwmGpu(s) as g:
            settings(g, *form)
            chi, it, rr, ok = g.sor_fixed(B, chi0, 1.9, 0.0, 43)
        assert it == want[1] == 43 and not ok, form
        assert same(chi, want[0]), form
        assert abs(rr - want[2]) <= 1e-12 * want[2], form


@pytest.mark.parametrize("nx,ny,kind", [(131, 75, "channel"), (33, 35, "torus")])
def test_fp32_sweeps_are_the_same_in_every_form(gpu_lib, nx, ny, kind):
    s = setup(nx, ny, kind)
    o = oracle.Oracle(s)
    B = rhs(o, s, 4)
    o.close()
    out = []
    for form in FORMS:
        with gpu.SwmGpu(s) as g:
            settings(g, *form)
            out.append(g.sor_fixed(B, np.zeros(s.shape), 1.9, 0.0, 37, fp32_sweeps=True))
    assert all(x[1] == 37 and same(x[0], out[-1][0]) for x in out)


@pytest.mark.parametrize("form,stop", [((-1, 16, 4), 40), ((8, 16, 8), 96), ((4, 32, 2), 42), ((2, 16, 1), 39),
                                       ((0, 16, 1), 39)])
def test_stops_at_the_sweep_that_passes(gpu_lib, form, stop):
    """The tolerance is the geometric mean of the oracle's relative residuals at
    the tested sweep before `stop` and at it, and the first one to pass."""
    s = setup(131, 75, "channel")
    o = oracle.Oracle(s)
    B = rhs(o, s, 6)
    every = form[2]
    rr = {k: o.sor_fixed(B, np.zeros(s.shape), 1.7, 0.0, k)[2] for k in range(every, stop + 1, every)}
    tol = float(np.sqrt(rr[stop] * rr[stop - every]))
    assert rr[stop] < tol and all(rr[k] > tol for k in rr if k < stop)
    want = o.sor_fixed(B, np.zeros(s.shape), 1.7, 0.0, stop)
    o.close()
    with gpu.SwmGpu(s) as g:
        settings(g, *form)
        chi, it, res, ok = g.sor_fixed(B, np.zeros(s.shape), 1.7, tol, 5000)
    assert ok and it == stop and same(chi, want[0])
    assert abs(res - rr[stop]) <= 1e-12 * rr[stop]


@pytest.mark.parametrize("halo", [-1, 8, 2, 0])
def test_reference_mode_stops_at_any_sweep_of_a_launch(gpu_lib, halo):
    """With four sweeps a launch its first three keep their chi and sums, and the
    next launch's first block tests the four in order: the oracle's sweep
    count and chi for tolerances that stop at each of them (each the mean of
    the oracle's norms at the sweep and at the one before)."""
    s = setup(65, 40, "channel")
    o = oracle.Oracle(s)
    B = rhs(o, s, 8)
    zero = np.zeros(s.shape)
    first = o.sor(B, zero, epsilon=1e-2, first_guess=True)
    assert first[3] == 0
    with gpu.SwmGpu(s) as g:
        g.set_sor_check_every(4)
        g.set_sor_halo(halo)
        eps = 1e-2
        for _ in range(5):   # each tolerance just below the last stop's norm
            chi, it, an, rc = o.sor(B, zero, epsilon=eps, first_guess=True)
            got = g.sor(B, zero, epsilon=eps, first_guess=True)
            assert rc == 0 and got[3] and got[1] == it, (it, got[1])
            assert same(got[0], chi)
            assert abs(got[2] - an) <= 1e-12 * an
            eps = an * (1 - 1e-6)
    o.close()
