"""Fields come to the host in pieces, large ones unpacked by several threads,
and in more than one round where they exceed the 32 MiB staging buffer: every
value arrives as it stands on the device, with the low part added where an FP32
context carries one, and a time average within a rounding of its quotient."""
import numpy as np
import pytest

from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


def bf16(x):
    b = x.astype(np.float32).view(np.uint32)
    return ((b + 0x7FFF + ((b >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("nx,ny", [(3, 3), (511, 255), (513, 257), (801, 703), (4500, 1201)])
@pytest.mark.parametrize("mode", ["f64", "f32", "f32_low"])
def test_every_value_arrives(gpu_lib, nx, ny, mode):
    rng = np.random.default_rng(nx)
    s = host.finalize(configs.basin(nx, ny, 5e3, 5e3, variant=host.LINEARISED_STATE_OF_REST, H0=500.0, dt=5.0))
    x = [rng.standard_normal((ny, nx)) for _ in range(3)]
    with gpu.SwmGpu(s, gpu.FP64 if mode == "f64" else gpu.FP32, low_part=mode == "f32_low") as g:
        g.init_from_setup()
        g.upload_state(*x)
        for name, v in zip(("SWM_U", "SWM_V", "SWM_ETA"), x):
            hi = v if mode == "f64" else v.astype(np.float32).astype(np.float64)
            want = hi + bf16(v - hi) if mode == "f32_low" else hi
            assert np.array_equal(g.get(name), want), name
        if mode == "f64":
            a = g.avg_add("SWM_ETA")
            g.step(1)
            eta = g.get("SWM_ETA")
            mean, _ = g.avg_read(a)
            assert np.all(np.abs(mean - eta) <= 2 * np.finfo(float).eps * np.abs(eta))
