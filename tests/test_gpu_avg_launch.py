"""One launch adds a step's fields to up to eight averaging buffers, two cells
at a time: more buffers than that, odd row lengths and both precisions hold the
same bits as sums formed on the host from the fields read after every step."""
import numpy as np
import pytest

from conftest import same
from swm_amd import configs, gpu, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(3, 3), (65, 33), (514, 7)])
@pytest.mark.parametrize("precision", [gpu.FP64, gpu.FP32])
@pytest.mark.parametrize("count", [1, 8, 9, 17])
def test_buffers_equal_host_sums(gpu_lib, nx, ny, precision, count):
    rng = np.random.default_rng(count)
    s = host.finalize(configs.basin(nx, ny, 5e3, 5e3, variant=host.LINEARISED_STATE_OF_REST, H0=500.0, dt=5.0))
    what = [(("SWM_U", "SWM_V", "SWM_ETA")[k % 3], k % 2 == 1) for k in range(count)]
    want = [np.zeros((ny, nx)) for _ in what]
    with gpu.SwmGpu(s, precision) as g:
        g.init_from_setup()
        g.upload_state(*(0.1 * rng.standard_normal((ny, nx)) for _ in range(3)))
        ids = [g.avg_add(n, square=q) for n, q in what]
        for _ in range(4):
            g.step(1)
            for w, (n, q) in zip(want, what):
                x = g.get(n)
                w += s.dt * (x * x if q else x)
        for k, w in zip(ids, want):
            mean, weight = g.avg_read(k)
            assert weight == 4 * s.dt and same(mean, w / weight), k
