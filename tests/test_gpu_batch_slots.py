"""A batched step writes the members' next step state to the other of two slots,
and the replayed graph holds two steps: any split of a run into even and odd
calls, members that end in the middle of one, and a change of the launch form
between calls leave every member where it gets alone, bit for bit."""
import numpy as np
import pytest

from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu

CALLS = [1, 2, 3, 1, 1, 4, 2]
STEPS = [14, 5, 9, 0]   # of the members; the calls add up to 14


def setup(k):
    rng = np.random.default_rng(k)
    s = host.finalize(configs.basin(33 + 32 * k, 17 + 9 * k, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=300.0, dt=10.0,
                                    f0=1e-4, beta=2e-11, seed=k, land_fraction=0.05))
    return s, [0.1 * rng.standard_normal(s.shape) * s.grids[g].ocean for g in ("u", "v", "eta")]


@pytest.mark.parametrize("precision", [gpu.FP64, gpu.FP32])
@pytest.mark.parametrize("shapes", [[1], [0], [1, 3], [2, 1]])
def test_any_split_of_a_batched_run(gpu_lib, precision, shapes):
    members, want = [], []
    with gpu.SwmBatch() as b:
        for k, n in enumerate(STEPS):
            s, x = setup(k)
            with gpu.SwmGpu(s, precision) as alone:
                alone.upload_state(*x)
                alone.step(n)
                want.append([alone.get(f) for f in ("SWM_U", "SWM_V", "SWM_ETA", "G_U")])
            m = gpu.SwmGpu(s, precision)
            m.upload_state(*x)
            b.attach(m, n)
            members.append(m)
        done = 0
        for q, n in enumerate(CALLS):
            if q == 0 or len(shapes) > 1:
                b.set_shape(shapes[q % len(shapes)])
            active = b.step(n)
            done += n
            assert active == sum(e > done for e in STEPS)
            assert [b.remaining(m) for m in members] == [max(0, e - done) for e in STEPS]
        for m, w, n in zip(members, want, STEPS):
            assert m.itt == n
            for f, x in zip(("SWM_U", "SWM_V", "SWM_ETA", "G_U"), w):
                assert same(m.get(f), x), (n, f)
            b.detach(m)
            m.close()
