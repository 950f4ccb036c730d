"""The SOR tuner's race without a GPU: every kind of launch enters it once, the
library's own choice among them, so that a tuned context is no slower than an
untuned one whatever cadences are asked for."""
import pytest

from swm_amd import autotune, configs, host


class Clocked:
    """Stands in for SwmGpu: a sweep takes `cost(sweeps per launch)` on its clock."""

    def __init__(self, s, cost):
        self.s, self.precision, self.cost, self.now, self.raced = s, 0, cost, 0.0, []

    def set_sor_halo(self, h):
        self.halo = h

    def set_sor_check_every(self, c):
        self.every = c

    def set_sor_tile_rows(self, r):
        self.rows = r

    def velocity_potential(self, omega, tol, sweeps, **kw):
        k = autotune.sor_sweeps_per_launch(self.s, self.halo, self.every)
        self.raced.append((k, self.every, self.rows, sweeps))
        self.now += sweeps * self.cost(k)


def domain(nx, ny, side_walls):
    return host.finalize(configs.basin(nx, ny, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=500.0, dt=5.0,
                                       side_walls=side_walls))


def tune(monkeypatch, s, cost, **kw):
    m = Clocked(s, cost)
    monkeypatch.setattr(autotune.time, "perf_counter", lambda: m.now)
    return m, autotune.tune_sor(m, sweeps=8, **kw)


@pytest.mark.parametrize("cadences", [(1,), (2,), (3,), (1, 2, 4, 8, 16)])
def test_four_sweeps_a_launch_are_raced_at_every_cadence(monkeypatch, cadences):
    m, res = tune(monkeypatch, domain(64, 48, True), lambda k: 1.0 / (1 + k), cadences=cadences)
    assert res["sweeps_per_launch"] == 4
    assert autotune.sor_sweeps_per_launch(m.s, m.halo, m.every) == 4
    first = [x[:2] for x in m.raced if x[3] == 8][::2]      # each is run twice, once to warm up
    assert len(first) == len(set(first))


@pytest.mark.parametrize("nx,ny,walls,alternate", [(64, 48, False, True), (65, 48, True, True), (65, 48, False, False)])
def test_rows_are_raced_where_they_matter(monkeypatch, nx, ny, walls, alternate):
    s = domain(nx, ny, walls)
    assert autotune.colours_alternate(s) == alternate
    m, _ = tune(monkeypatch, s, lambda k: 1.0, cadences=(4,))
    assert ({x[2] for x in m.raced} == {16}) == alternate
    first = [x[:3] for x in m.raced if x[3] == 8][::2]
    assert len(first) == len(set(first))
