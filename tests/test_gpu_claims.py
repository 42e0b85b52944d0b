"""Every ray of a launch past the line where launches claim their rays in turns
(512 per CU) is traced once, at sizes around the ends of a band's run of claims
and for the smallest, an odd and the largest claim; as one set and as a batched
launch with an empty and a one-ray set.  (id, t) are those of launches below the
line, bit for bit."""
import numpy as np
import pytest

from conftest import random_rays, random_triangles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(gpu):
    v, idx = random_triangles(40, seed=600)
    tr = gpu.CudaTracer(gpu.BVH((v, idx)))
    rays = random_rays(300001, seed=601)
    want = [tr.trace(rays[i:i + 100000]) for i in range(0, len(rays), 100000)]
    return tr, rays, np.concatenate([w[0] for w in want]), np.concatenate([w[1] for w in want])


@pytest.mark.parametrize("chunk", [64, 192, 65536])
@pytest.mark.parametrize("n", [131073, 139263, 139264, 139265, 300001])
def test_every_ray_is_traced(gpu, scene, chunk, n):
    tr, rays, ids, ts = scene
    cfg = gpu.get_trace_config()
    gpu.set_trace_config(**{**cfg, "chunk": chunk})
    try:
        d = gpu.DeviceBuffer.from_array(rays)
        none = np.full(2 * len(rays), 0x55555555, np.uint32)
        one = gpu.DeviceBuffer.from_array(none)
        tr.trace_device(d.ptr, n, one.ptr)
        many = gpu.DeviceBuffer.from_array(none)
        cuts = [0, 1, 1, 1000, n]
        gpu.trace_batch([(tr, d.ptr + 32 * a, b - a, many.ptr + 8 * a, False) for a, b in zip(cuts, cuts[1:])])
        for buf in (one, many):
            h = buf.download(gpu.HIT_DTYPE, len(rays))
            assert np.array_equal(h["id"][:n], ids[:n])
            assert np.array_equal(h["t"][:n].view(np.uint32), ts[:n].view(np.uint32))
            assert (h["id"][n:] == 0x55555555).all()
    finally:
        gpu.set_trace_config(**cfg)
