"""Timed workloads of the shallow-water time-stepping path.

Each case is what a program that uses this package has it do between two
points of its own time loop, through the public binding (``swm_amd.gpu``):
some time steps and the register reads of an output step (``step``), the
per-step velocity potential (``potential``, ``elliptic``), one chunk of a
batched ensemble (``batch``), or a run with averaging and diagnostic tasks
(``diag``).  Sizes are those of ``swm_amd/configs.py``, ``bench.py`` and the
tests, or odd ones between them.

``prepare`` does the host initialisation, the hand-over to the device and the
first steps (the multistep scheme's start), ``run`` is one pass of the run
under way.  Time steps advance the state, so a second pass on the same state
continues the run.  FP32 contexts return their fields in single
precision, as such a model writes its output.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from swm_amd import configs, gpu, host

VARIANTS = {"nonlinear": host.FULLY_NONLINEAR, "mean": host.LINEARISED_MEAN_STATE,
            "rest": host.LINEARISED_STATE_OF_REST}
DX = 5e3            # grid spacing of every basin, m
START = 3           # steps behind every run before its first pass


def _step(name, nx, ny, steps, **more):
    return dict(dict(name=name, kind="step", nx=nx, ny=ny, steps=steps, variant="nonlinear", precision="f64",
                     tracers=0, mixing=True, quadratic=False, land=0.05, sphere=False, stream=False), **more)


def listed():
    return [
        # a host model that drives the device one time step at a time and reads
        # the state after each: the smallest call, all latency
        _step("one_step_96x64", 96, 64, 1, tracers=1),
        # the linear non-rotating basin: 200 x 200, output every 200 steps
        _step("linear_200x200", 200, 200, 200, variant="rest", mixing=False, land=0.0),
        # the headline double-gyre basin with its tracer, output every 1000 steps, FP64 and FP32
        _step("gyre_1024x1024_f64", 1024, 1024, 1000, tracers=1),
        _step("gyre_1024x1024_f32", 1024, 1024, 1000, tracers=1, precision="f32"),
        # a basin larger than the last-level cache, without a tracer
        _step("gyre_2304x1800_f64", 2304, 1800, 150),
        # a ragged grid on the sphere: two tracers and quadratic friction (the tracers' undefined
        # values spread from land by a cell a step, so an interior is left after 100)
        _step("ragged_487x333_two_tracers", 487, 333, 100, tracers=2, quadratic=True, sphere=True, land=0.0),
        # perturbations of a mean flow under time-dependent wind (a dataset interpolated every step)
        _step("mean_state_501x383", 501, 383, 300, variant="mean", sphere=True, stream=True),
        # the elliptic workload: a step and the velocity potential of its flow, warm-started, FP64 sweeps
        dict(name="potential_2048x1024_f64", kind="potential", nx=2048, ny=1024, sweeps=5000, every=16, fp32=False,
             land=0.0, sphere=False),
        # the same with FP32 sweeps on an odd basin with islands
        dict(name="potential_1201x800_f32", kind="potential", nx=1201, ny=800, sweeps=5000, every=16, fp32=True,
             land=0.05, sphere=False),
        # the build with the elliptic solver: chi, the non-divergent flow and its
        # streamfunction after a step, by the reference's own iteration
        dict(name="elliptic_build_720x361", kind="elliptic", nx=720, ny=361, land=0.03, sphere=True),
        # one 64-step chunk of an uneven FP32 ensemble, half of it with tracers (no islands there)
        dict(name="ensemble_14_f32", kind="batch", members=14, lo=128, hi=1024, steps=64, precision="f32", pick=3),
        # averaging tasks accumulated over an output interval, then the diagnostics of an output step
        dict(name="diagnostics_1024x768", kind="diag", nx=1024, ny=768, steps=100, land=0.05),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["step", "potential", "elliptic", "batch", "diag"], [6, 2, 1, 2, 1])[0]
    if kind == "step":
        nx, ny = _log(rng, 64, 2048), _log(rng, 64, 1536)
        variant = rng.choice(["nonlinear", "nonlinear", "nonlinear", "rest", "mean"])
        if variant == "mean":
            nx, ny = max(nx, ny), min(nx, ny)
        # up to the work of the largest listed case
        steps = 1 if rng.random() < 0.1 else min(_log(rng, 20, 1000), int(1e9 / (nx * ny)))
        return dict(kind=kind, nx=nx, ny=ny, steps=steps, variant=variant, precision=rng.choice(["f64", "f32"]),
                    tracers=rng.choice([0, 1, 1, 2]) if variant == "nonlinear" else 0,
                    mixing=variant == "nonlinear" or rng.random() < 0.5, quadratic=rng.random() < 0.25,
                    land=rng.choice([0.0, 0.05, 0.1]), sphere=rng.random() < 0.5, stream=rng.random() < 0.2)
    if kind == "potential":
        return dict(kind=kind, nx=_log(rng, 200, 2048), ny=_log(rng, 150, 1024), sweeps=_log(rng, 500, 5000),
                    every=rng.choice([1, 4, 8, 16, 16]), fp32=rng.random() < 0.5, land=rng.choice([0.0, 0.05]),
                    sphere=rng.random() < 0.5)
    if kind == "elliptic":
        return dict(kind=kind, nx=_log(rng, 150, 800), ny=_log(rng, 100, 500), land=rng.choice([0.0, 0.05]),
                    sphere=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind=kind, members=rng.randint(3, 14), lo=64, hi=rng.choice([256, 512, 1024]),
                    steps=rng.choice([16, 64]), precision=rng.choice(["f32", "f32", "f64"]),
                    pick=rng.randint(0, 10 ** 6))
    return dict(kind=kind, nx=_log(rng, 128, 1400), ny=_log(rng, 128, 1000), steps=_log(rng, 20, 100),
                land=rng.choice([0.0, 0.05]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _waves(rng, ny, nx, amp, modes=5, kmax=8):
    """A smooth field: seeded Fourier modes of amplitude amp / sqrt(modes)."""
    x, y = np.arange(nx) / nx, np.arange(ny) / ny
    kx, ky = rng.integers(1, kmax + 1, modes), rng.integers(1, kmax + 1, modes)
    ax = 2 * np.pi * (kx[:, None] * x) + rng.uniform(0, 2 * np.pi, (modes, 1))
    ay = 2 * np.pi * (ky[:, None] * y)
    return amp / math.sqrt(modes) * (np.cos(ay).T @ np.cos(ax) - np.sin(ay).T @ np.sin(ax))


def _setup(seed, nx, ny, variant="nonlinear", tracers=0, mixing=True, quadratic=False, land=0.0, sphere=False,
           stream=False, H0=500.0, Ah=100.0, tau0=0.1):
    """Host initialisation: a wind-driven beta-plane basin in motion."""
    rng = np.random.default_rng([seed, nx, ny])
    dt = configs.stable_dt(H0, 0.8 * DX if sphere else DX)
    psi = None
    if variant == "mean":
        psi = _waves(rng, ny, nx, 0.05 * H0 * DX * 8.0, kmax=3)
    s = configs.basin(nx, ny, DX, DX, variant=VARIANTS[variant], H0=H0, dt=dt, Ah=Ah, lbc=2.0, f0=1e-4, beta=2e-11,
                      drag=1e-6, lateral_mixing=mixing, land_fraction=land, seed=seed % (1 << 31),
                      A=6371e3 if sphere else configs.A_FLAT, quadratic_friction=quadratic, gamma_sq=2e-3, psi_bs=psi)
    wind = configs.double_gyre_tau(s, tau0)
    if stream:      # four records of a wind dataset, an hour apart
        rec = np.stack([wind * (1.0 + 0.3 * math.sin(0.5 * math.pi * k)) for k in range(4)])
        host.add_forcing_stream(s, host.STREAM_WIND, host.COMP_X, rec, 3600.0)
    else:
        host.add_windstress(s, host.COMP_X, wind)
    for _ in range(tracers):
        host.add_tracer(s, 2.0 + _waves(rng, ny, nx, 1.0), kappa_h=50.0)
    s.u0, s.v0 = _waves(rng, ny, nx, 0.1), _waves(rng, ny, nx, 0.1)
    s.eta0 = _waves(rng, ny, nx, 0.2)
    return host.finalize(s)


def _members(case, seed):
    """Setups of a batch: sizes and parameters of the case, fields of the seed."""
    r = np.random.default_rng(case["pick"])
    out = []
    for k in range(case["members"]):
        nx, ny = (int(round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(2))
        out.append(_setup(seed * 64 + k, nx, ny, tracers=k % 2, land=0.05 * (1 - k % 2), H0=float(r.uniform(200.0, 4000.0)),
                          Ah=float(r.uniform(20.0, 500.0)), tau0=float(r.uniform(0.02, 0.2))))
    return out


_SETUP_KEYS = ("nx", "ny", "variant", "tracers", "mixing", "quadratic", "land", "sphere", "stream")


def _case_setup(case, seed):
    return _setup(seed, **{k: case[k] for k in _SETUP_KEYS if k in case}, **({"tracers": 1} if case["kind"] == "diag" else {}))


def prepare(case, seed):
    prec = gpu.FP32 if case.get("precision") == "f32" else gpu.FP64
    if case["kind"] == "batch":
        batch, members = gpu.SwmBatch(), []
        for s in _members(case, seed):
            members.append(gpu.SwmGpu(s, precision=prec).init_from_setup())
            members[-1].step(START)
            batch.attach(members[-1], 1 << 40)
        return dict(case=case, batch=batch, members=members)
    s = _case_setup(case, seed)
    s.elliptic_solver = case["kind"] == "elliptic"
    g = gpu.SwmGpu(s, precision=prec).init_from_setup()
    g.step(START)
    state = dict(case=case, g=g)
    if case["kind"] == "potential":
        g.set_sor_check_every(case["every"])
    if case["kind"] == "diag":
        state["avg"] = [g.avg_add("SWM_U"), g.avg_add("SWM_V"), g.avg_add("SWM_ETA"), g.avg_add("SWM_ETA", square=True)]
    return state


def _fields(g):
    out = {n: g.get("SWM_" + n) for n in ("U", "V", "ETA")}
    for k in range(len(g.s.tracers)):
        out["CH%d" % k] = g.get("CH", k)
    return {n: a.astype(np.float32) for n, a in out.items()} if g.precision == gpu.FP32 else out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        state["batch"].step(case["steps"])
        return [_fields(m) for m in state["members"]]
    g = state["g"]
    if kind == "step":
        g.step(case["steps"])
        return _fields(g)
    if kind == "potential":
        g.step(1)
        sweeps, residual, _ = g.velocity_potential(omega=1.9, rel_tol=1e-10, max_sweeps=case["sweeps"],
                                                   fp32_sweeps=case["fp32"])
        chi = g.get("CHI")
        return dict(chi=chi.astype(np.float32) if case["fp32"] else chi, sweeps=sweeps, residual=residual)
    if kind == "elliptic":
        g.step(1)
        out = {n: g.get(n) for n in ("CHI", "U_ND", "V_ND", "PSI")}
        out["sweeps"] = g.elliptic_stats()[0]
        return out
    g.step(case["steps"])
    out = {"mean%d" % k: g.avg_read(a)[0] for k, a in enumerate(state["avg"])}
    for n in ("PSI", "SWM_RELVORT", "SWM_MU", "SWM_EDENS"):
        out[n] = g.get(n)
    out["sums"] = np.array(g.sums(0))
    return out


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------

def _step_work(cells, steps, size, tracers, extra_fields=0):
    """A step reads u, v, eta and the two newest tendencies of each and writes
    them back with one tendency each, 15 values a cell, 5 more for a tracer,
    and reads the masks; about 250 operations a cell, 70 more a tracer."""
    return (cells * steps * (size * (15 + 5 * tracers + extra_fields) + 1), cells * steps * (250 + 70 * tracers))


def work(case):
    kind = case["kind"]
    if kind == "batch":
        r = np.random.default_rng(case["pick"])
        b = f = 0
        for k in range(case["members"]):
            n = 1
            for _ in range(2):
                n *= int(round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"])))))
            r.uniform(size=3)
            x, y = _step_work(n, case["steps"], 4 if case["precision"] == "f32" else 8, k % 2)
            b, f = b + x, f + y
        return dict(bytes=b, flops=f)
    cells = case["nx"] * case["ny"]
    if kind == "step":
        size = 4 if case["precision"] == "f32" else 8
        b, f = _step_work(cells, case["steps"], size, case["tracers"], 2 if case["stream"] else 0)
        return dict(bytes=b, flops=f)
    b, f = _step_work(cells, case.get("steps", 1), 8, 1 if kind == "diag" else 0)
    if kind == "potential":     # chi read and written once, the divergence's flow once; 13 operations a cell and sweep
        size = 4 if case["fp32"] else 8
        return dict(bytes=b + cells * (2 * size + 17), flops=f + 13 * cells * case["sweeps"])
    if kind == "elliptic":      # some 5000 sweeps: the solver stops at 10 times the larger extent at most
        return dict(bytes=b + cells * (2 * 8 + 17 + 5 * 8), flops=f + 13 * cells * 5000)
    # four averages: read a field, update a buffer, every step; four fields out,
    # of which the streamfunction sums half a row per cell
    return dict(bytes=b + cells * (case["steps"] * 4 * 24 + 8 * 8 + 8 * 8), flops=f + cells * (case["steps"] * 10 + case["nx"] / 2 + 60))


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float64), device=_dev())


def _W(a): return torch.roll(a, 1, 1)      # a(i-1, j)
def _E(a): return torch.roll(a, -1, 1)     # a(i+1, j)
def _S(a): return torch.roll(a, 1, 0)      # a(i, j-1)
def _N(a): return torch.roll(a, -1, 0)     # a(i, j+1)


class _Model:
    """The discrete model of one Setup: Arakawa C grid, energy-type Bernoulli
    function, potential vorticity fluxes, tension/shear mixing, AB3."""

    def __init__(self, s):
        self.s = s
        col = lambda a: _t(a)[:, None]
        g = s.grids
        self.oH, self.ou, self.ov, self.oe = (_t(g[k].ocean) for k in ("H", "u", "v", "eta"))
        self.cH, self.cu, self.cv, self.ce = (col(g[k].cos_lat) for k in ("H", "u", "v", "eta"))
        self.tH, self.tu, self.tv, self.te = (col(g[k].tan_lat) for k in ("H", "u", "v", "eta"))
        self.f = col(g["H"].f)
        self.He, self.Hu, self.Hv = _t(g["eta"].H), _t(g["u"].H), _t(g["v"].H)
        A, dL, dT, Ah = s.A, s.dLambda, s.dTheta, s.Ah
        self.bcH = torch.where(self.oH > 0, 1.0, s.lbc)
        ou, ov, oe, oH = self.ou, self.ov, self.oe, self.oH
        one = lambda a: torch.clamp(a, min=1.0)
        self.wu, self.wv = 1 / one(oe + _W(oe)), 1 / one(oe + _S(oe))
        self.wh = 1 / one(oe + _W(oe) + _S(oe) + _S(_W(oe)))
        self.imp = [_t(a) for a in (s.impl_u, s.impl_v, s.impl_eta)]
        self.F = [_t(a) for a in (s.F_x_const, s.F_y_const, s.F_eta_const)]
        self.tau = [(c, _t(a)) for c, a in s.wind]
        self.streams = [(st, _t(st.records)) for st in s.streams]
        if s.lateral_mixing:
            ot = one(ov + _N(ov))
            self.pll_c = (-(Ah / dL / A / self.ce), Ah / A * (1 / dT + _N(ov) * self.te / ot),
                          Ah / A * (-1 / dT + ov * self.te / ot))
            ot = one(ou + _S(ou))
            self.plt_c = (-(Ah / dL / A / self.cH), -(Ah / A * (1 / dT + ou * self.tH / ot)),
                          -(Ah / A * (-1 / dT + _S(ou) * self.tH / ot)))
            ot = one(oH + _N(oH))
            self.lu = (-(1 / A / self.cu / dL), -(1 / A / dT - 2 * self.tu / A / ot), -(-1 / A / dT - 2 * self.tu / A / ot))
            ot = one(oe + _S(oe))
            self.lv = (-(1 / A / self.cv / dL), -(-1 / A / dT + 2 * self.tv / A / ot), -(1 / A / dT + 2 * self.tv / A / ot))
        if s.quadratic_friction:
            self.gs = _t(s.gamma_sq_u), _t(s.gamma_sq_v)
        if s.variant == host.LINEARISED_MEAN_STATE:
            self.ub, self.vb, self.zb = _t(s.u_bs), _t(s.v_bs), _t(s.zeta_bs)
        if s.tracers:
            nan = lambda d: torch.where(d == 0, math.nan, 1 / one(d))
            cvn = _N(self.cv)
            dE, dW, dN, dS = (nan(oe + x(oe)) for x in (_E, _W, _N, _S))
            ax, ayn, ays = 1 / A / dL / self.ce, cvn / A / dT / self.ce, self.cv / A / dT / self.ce
            self.adv = (-_E(ou) * _E(oe) * dE * ax, ou * _W(oe) * dW * ax, -_N(ov) * _N(oe) * dN * ayn,
                        ov * _S(oe) * dS * ays, -_E(ou) * oe * dE * ax, ou * oe * dW * ax, -_N(ov) * oe * dN * ayn,
                        ov * oe * dS * ays)
            k = 1 / (A * A)
            self.dif = (_E(ou) * k / (dL * dL) / self.cu / self.ce, -ou * k / (dL * dL) / self.cu / self.ce,
                        _N(ov) * k * cvn / (dT * dT) / self.ce, -ov * k * self.cv / (dT * dT) / self.ce)
        # the state after the host's initial conditions: masked fields, no history
        z = torch.zeros_like(oe)
        self.u, self.v, self.eta = ou * _t(s.u0), ov * _t(s.v0), oe * _t(s.eta0)
        self.G = [[z, z] for _ in range(3)]
        D0 = self.D(self.eta)
        self.trc = [dict(CH=D0 * _t(t["C"]), C=_t(t["C"]), G=[z, z], kappa=t["kappa_h"], C0=_t(t["C0"]),
                         gC=_t(t["gamma_C"]), imp=1 + s.dt * _t(t["cons"])) for t in s.tracers]
        self.itt = 0

    def D(self, eta):
        if self.s.variant == host.FULLY_NONLINEAR:
            return torch.where(self.oe > 0, eta + self.He, 1.0)
        return self.He

    def Du(self, D): return self.wu * (self.oe * D + _W(self.oe * D))
    def Dv(self, D): return self.wv * (self.oe * D + _S(self.oe * D))

    def derived(self):
        s, u, v, eta = self.s, self.u, self.v, self.eta
        A, dL, dT = s.A, s.dLambda, s.dTheta
        D = self.D(eta)
        oD = self.oe * D
        r = dict(D=D, Du=self.Du(D), Dv=self.Dv(D), Dh=self.wh * (oD + _W(oD) + _S(oD) + _S(_W(oD))))
        za = torch.where(self.ov + _W(self.ov) > 0, self.bcH / (A * self.cH * dL) * (v - _W(v)), 0.0)
        zb = torch.where(self.ou + _S(self.ou) > 0, self.bcH * (self.cu * u - _S(self.cu * u)) / (A * dT), 0.0)
        r["zeta"] = za - zb / self.cH
        pD = torch.clamp(r["Dh"], min=2.220446049250313e-16)
        if s.variant == host.FULLY_NONLINEAR:
            r["Pot"] = (self.f + r["zeta"]) / pD
            r["Ed"] = self.oe * (((_E(u) ** 2 + u ** 2) / 2 + (_N(v) ** 2 + v ** 2) / 2) / 2 + s.G * eta)
        elif s.variant == host.LINEARISED_MEAN_STATE:
            r["Pot"] = (self.f + self.zb) / pD
            uU, vV = u * self.ub, v * self.vb
            r["Ed"] = self.oe * ((_E(uU) + uU) / 2 + (_N(vV) + vV) / 2 + s.G * eta)
        else:
            r["Pot"] = self.f / pD
            r["Ed"] = self.oe * (s.G * eta)
        r["MU"], r["MV"] = self.ou * r["Du"] * u, self.ov * r["Dv"] * v
        return r

    def forcing(self, r):
        s, ocean = self.s, (self.ou, self.ov, self.oe)
        F = list(self.F)
        for c, tau in self.tau:
            F[c] = F[c] + torch.where(ocean[c] > 0, tau / (s.RHO0 * (r["Du"], r["Dv"])[c]), 0.0)
        for st, rec in self.streams:
            t = self.itt * s.dt / st.rec_dt
            k, n = int(math.floor(t)), rec.shape[0]
            y = rec[k % n] + (t - k) * (rec[(k + 1) % n] - rec[k % n])
            F[st.comp] = F[st.comp] + torch.where(ocean[st.comp] > 0, y / (s.RHO0 * (r["Du"], r["Dv"])[st.comp]), 0.0)
        return F

    def step(self):
        s, u, v = self.s, self.u, self.v
        A, dL, dT, dt = s.A, s.dLambda, s.dTheta, s.dt
        r = self.derived()
        F = self.forcing(r)
        D, Du, Dv, Dh, Pot, Ed, MU, MV = (r[k] for k in ("D", "Du", "Dv", "Dh", "Pot", "Ed", "MU", "MV"))
        ge = -(_E(MU) - MU) / dL - (_N(self.cv * MV) - self.cv * MV) / dT
        gu = (Pot + _N(Pot)) / 2 * (MV + _W(MV) + _N(MV) + _N(_W(MV))) / 4
        gv = -(Pot + _E(Pot)) / 2 * (MU + _E(MU) + _S(MU) + _S(_E(MU))) / 4
        if s.variant == host.LINEARISED_MEAN_STATE:
            # the eastern face interpolates eta at column j+1 of row j
            ny, nx = self.eta.shape
            eu = self.Du(self.eta)
            j = torch.arange(ny, device=eu.device)
            ge = ge - (eu[j, (j + 1) % nx][:, None] * _E(self.ub) - eu * self.ub) / dL
            ev = self.cv * self.Dv(self.eta) * self.vb
            ge = ge - (_N(ev) - ev) / dT
            z = r["zeta"]
            gu = gu + (z + _N(z)) / 2 * (self.vb + _W(self.vb) + _N(self.vb) + _N(_W(self.vb))) / 4
            gv = gv - (z + _E(z)) / 2 * (self.ub + _E(self.ub) + _S(self.ub) + _S(_E(self.ub))) / 4
        gu = gu - (Ed - _W(Ed)) / (A * self.cu * dL)
        gv = gv - (Ed - _S(Ed)) / (A * dT)
        if s.quadratic_friction:
            vi, ui = (v + _W(v) + _N(v) + _N(_W(v))) / 4, (u + _E(u) + _S(u) + _S(_E(u))) / 4
            qu, qv = self.gs[0] * torch.sqrt(u * u + vi * vi) * u, self.gs[1] * torch.sqrt(v * v + ui * ui) * v
            gu, gv = gu - (qu / self.Hu if s.barotropic else qu), gv - (qv / self.Hv if s.barotropic else qv)
        if s.lateral_mixing:
            c = self.pll_c
            pll = self.oe * D * (c[0] * (_E(u) - u) + c[1] * _N(v) + c[2] * v)
            c = self.plt_c
            plt = self.oH * Dh * (c[0] * (v - _W(v)) + c[1] * u + c[2] * _S(u))
            c = self.lu
            gu = gu + (c[0] * (pll - _W(pll)) + c[1] * _N(plt) + c[2] * plt) / Du
            c = self.lv
            gv = gv + (c[0] * (_E(plt) - plt) + c[1] * pll + c[2] * _S(pll)) / Dv
        new = [torch.where(o > 0, g + x, h[1]) for o, g, x, h in
               zip((self.ou, self.ov, self.oe), (gu, gv, ge / (A * self.ce)), F, self.G)]
        self.itt += 1
        chi = s.ab_chi
        ab = [(1.0, 0.0, 0.0), (-0.5 - chi, 1.5 + chi, 0.0), (5 / 12, -16 / 12, 23 / 12)][min(3, self.itt) - 1]
        inc = lambda h, n: dt * (ab[0] * h[0] + (ab[1] * h[1] if self.itt > 1 else 0) + (ab[2] * n if self.itt > 2 else 0))
        out = [(x + inc(h, n)) / i for x, h, n, i in zip((u, v, self.eta), self.G, new, self.imp)]
        if s.variant == host.FULLY_NONLINEAR:
            out[2] = torch.maximum(out[2], s.minD - self.He)
        for t in self.trc:
            CH = t["CH"]
            C = CH / D if t["C"] is None else t["C"]
            ue, vn, k = _E(u), _N(v), t["kappa"]
            a, d = self.adv, self.dif
            g = (_E(CH) * ue * a[0] + _W(CH) * u * a[1] + _N(CH) * vn * a[2] + _S(CH) * v * a[3] + CH * ue * a[4] +
                 CH * u * a[5] + CH * vn * a[6] + CH * v * a[7])
            g = g + torch.where(self.oe > 0, k * (_E(Du) * (_E(C) - C) * d[0] + Du * (C - _W(C)) * d[1] +
                                                  _N(Dv) * (_N(C) - C) * d[2] + Dv * (C - _S(C)) * d[3]), 0.0)
            g = g - t["gC"] * D * (C - t["C0"]) + C * F[2]
            t["CH"], t["C"], t["G"] = (CH + inc(t["G"], g)) / t["imp"], None, [t["G"][1], g]
        self.u, self.v, self.eta = out
        self.G = [[h[1], n] for h, n in zip(self.G, new)]

    def fields(self):
        out = dict(U=self.u, V=self.v, ETA=self.eta)
        out.update({"CH%d" % k: t["CH"] for k, t in enumerate(self.trc)})
        return {k: a.cpu().numpy() for k, a in out.items()}

    def divergence(self):
        s = self.s
        bc = torch.where(self.oe > 0, 1.0, s.lbc)
        za = torch.where(self.ou + _E(self.ou) > 0, bc / (s.A * self.ce * s.dLambda) * (_E(self.u) - self.u), 0.0)
        w = self.cv * self.v
        zb = torch.where(self.ov + _N(self.ov) > 0, bc * (_N(w) - w) / (s.A * s.dTheta), 0.0)
        return za + zb / self.ce

    def relax(self, B, omega, sweeps, stop):
        """Red-black SOR sweeps from chi = 0 of the five-point operator with
        closed coasts; stop(sweep, correction, residual) ends it after a sweep."""
        s = self.s
        x, y = (s.A * self.ce * s.dLambda) ** 2, s.A ** 2 * self.ce * s.dTheta ** 2
        cE, cW, cN, cS = _E(self.ou) / x, self.ou / x, _N(self.ov * self.cv) / y, self.ov * self.cv / y
        c5 = -(cE + cW + cN + cS)
        ny, nx = B.shape
        ij = (torch.arange(nx, device=B.device)[None, :] + torch.arange(ny, device=B.device)[:, None]) % 2
        inv = [torch.where((self.oe > 0) & (ij == c), 1 / c5, 0.0) for c in (0, 1)]
        mine = [torch.where((self.oe > 0) & (ij == c), 1.0, 0.0) for c in (0, 1)]
        chi = torch.zeros_like(B)
        for l in range(1, sweeps + 1):
            parts = []
            for c in (0, 1):
                r = cE * _E(chi) + cW * _W(chi) + cN * _N(chi) + cS * _S(chi) + c5 * chi - B
                d = omega(2 * (l - 1) + c) * r * inv[c]
                chi = chi - d
                parts.append((d, r * mine[c]))
            if stop(l, parts):
                return chi, l
        return chi, sweeps

    def streamfunction(self, u, v):
        s = self.s
        nx = u.shape[1]
        hu, hv = (self.Hu * u, self.Hv * v) if s.barotropic else (u, v)
        hv = torch.cat([(hv * self.ov)[:1], hv[1:]])
        hu = torch.cat([hu[:, :-1], (hu * self.ou)[:, -1:]], 1)
        hv = hv.clone()
        hv[:, -1] = 0
        row = torch.flip(torch.cumsum(torch.flip(hv, [1]), 1), [1]) * s.A * self.cv * s.dLambda
        col = (torch.cumsum(hu, 0) - hu) * s.A * s.dTheta
        psi = torch.zeros_like(u)
        psi[0, :-1] = -row[0, :-1]
        psi[1:, -1] = -col[1:, -1]
        psi[1:, :-1] = (-row[1:, :-1] + psi[1:, -1:] - col[1:, :-1] + psi[:1, :-1]) / 2
        return psi


def _exact_potential(case, m):
    B = m.divergence()
    norm = float(torch.sqrt((B * m.oe).square().sum()))
    last = {}

    def stop(l, parts):
        if l % case["every"] and l != case["sweeps"]:
            return False
        last["r"] = math.sqrt(float(sum(r.square().sum() for _, r in parts))) / norm
        return last["r"] < 1e-10

    chi, n = m.relax(B, lambda h: 1.9, case["sweeps"], stop)
    return dict(chi=chi.cpu().numpy(), sweeps=None, residual=None)


def _exact_elliptic(case, m):
    s = m.s
    rj2 = float(np.float32(9.9999178e-1)) ** 2
    om = [1.0, 1 / (1 - 0.5 * rj2)]
    while len(om) < 4 or om[-1] != om[-2]:
        om.append(1 / (1 - 0.25 * rj2 * om[-1]))
    eps = float(np.float32(1e-4))
    chi, n = m.relax(m.divergence(), lambda h: om[min(h, len(om) - 1)], 10 * max(case["nx"], case["ny"]),
                     lambda l, parts: math.sqrt(float(sum(d.square().sum() for d, _ in parts))) < eps)
    bu, bv = torch.where(m.ou > 0, 1.0, s.lbc), torch.where(m.ov > 0, 1.0, s.lbc)
    und = m.u - torch.where(_W(m.oe) + m.oe > 0, bu / (s.A * m.cu * s.dLambda) * (chi - _W(chi)), 0.0)
    vnd = m.v - torch.where(_S(m.oe) + m.oe > 0, bv * (chi - _S(chi)) / (s.A * s.dTheta), 0.0)
    psi = m.streamfunction(und, vnd)
    return dict(CHI=chi.cpu().numpy(), U_ND=und.cpu().numpy(), V_ND=vnd.cpu().numpy(), PSI=psi.cpu().numpy(), sweeps=None)


def _exact_diag(case, m):
    sums = [0.0] * 4
    for _ in range(case["steps"]):
        m.step()
        sums = [a + b for a, b in zip(sums, (m.u, m.v, m.eta, m.eta ** 2))]
    out = {"mean%d" % k: (a / case["steps"]).cpu().numpy() for k, a in enumerate(sums)}
    r = m.derived()
    out.update(PSI=m.streamfunction(m.u, m.v).cpu().numpy(), SWM_RELVORT=r["zeta"].cpu().numpy(),
               SWM_MU=r["MU"].cpu().numpy(), SWM_EDENS=r["Ed"].cpu().numpy())
    ke = r["D"] * ((m.u ** 2 + _E(m.u) ** 2) / 4 + (m.v ** 2 + _N(m.v) ** 2) / 4)
    en = ke + 0.5 * m.s.G * m.eta ** 2
    out["sums"] = np.array([float((m.oe * m.ce * m.eta).sum()), float((m.oe * m.ce * en).sum()),
                            float(torch.where(m.oe > 0, m.ce * m.trc[0]["CH"], 0.0).sum())])
    return out


def exact(case, seed):
    if case["kind"] == "batch":
        out = []
        for s in _members(case, seed):
            m = _Model(s)
            for _ in range(START + case["steps"]):
                m.step()
            out.append(m.fields())
        return out
    m = _Model(_case_setup(case, seed))
    for _ in range(START):
        m.step()
    if case["kind"] == "diag":
        return _exact_diag(case, m)
    for _ in range(case.get("steps", 1)):
        m.step()
    if case["kind"] == "potential":
        return _exact_potential(case, m)
    if case["kind"] == "elliptic":
        return _exact_elliptic(case, m)
    return m.fields()
