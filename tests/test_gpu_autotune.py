"""The autotuner on rays whose launches do not use the configuration (up to 512 per
CU, non-speculative): it keeps the one that is set, for the large launches that
use it, and reports the time of those rays.  Past the line it chooses among the
shapes.  The hits of the last launch it times are the trace's, bit for bit."""
import numpy as np
import pytest

from conftest import random_rays, random_triangles

pytestmark = pytest.mark.gpu

LINE = 512 * 256


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("n", [1, 4099, LINE, LINE + 1])
def test_autotune(gpu, n, any_hit):
    tr = gpu.CudaTracer(gpu.BVH(random_triangles(500, seed=700)))
    rays = random_rays(n, seed=701)
    d_rays, d_hits = gpu.DeviceBuffer.from_array(rays), gpu.DeviceBuffer(n * 8)
    saved = gpu.get_trace_config()
    try:
        gpu.set_trace_config(**{**saved, "block": 128, "lds_stack": 12, "waves_per_cu": 16})
        before = gpu.get_trace_config()
        best, ms = gpu.autotune(tr, d_rays, n, d_hits, any_hit=any_hit)
        assert ms > 0 and best == gpu.get_trace_config()
        if n <= LINE:
            assert best == before
        got = d_hits.download(gpu.HIT_DTYPE, n)
    finally:
        gpu.set_trace_config(**saved)
    ids, ts = tr.trace(rays, any_hit=any_hit)
    assert np.array_equal(got["id"], ids) and np.array_equal(got["t"].view(np.uint32), ts.view(np.uint32))
