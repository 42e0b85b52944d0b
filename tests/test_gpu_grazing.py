"""Rays that graze tessellated walls: the rounding of a slab test moves its point
along the ray, the farther the more the ray lies in the wall, so that a leaf's box
can fail though the hit is far from its triangle's edges.  Hit and miss are the
oracle's (whose boxes the wide walk's own equal here: corners on a grid of powers of
two), and (id, t) are the same, bit for bit, in launches of few rays and of many, in
a batched launch and for a kernel's single rays, which all follow one rule."""
import numpy as np
import pytest

from test_gpu_cracks import _room

pytestmark = pytest.mark.gpu

N, FEW = 400000, 100000  # past and below the line where launches give each ray a quad


def _aimed(k, r):
    """From 1e-3 to 1e-1 off a wall to points of it 3e-6 to 3e-4 from a grid line."""
    rows = np.arange(N)
    axis, side = r.integers(0, 3, N), r.choice([-1.0, 1.0], N)
    o, to = r.uniform(-5, 5, (N, 3)), r.uniform(-5, 5, (N, 3))
    o[rows, axis] = side * (5 - 10 ** r.uniform(-3, -1, N))
    to[rows, axis] = side * 5
    line = r.integers(0, k + 1, N) * (10 / k) - 5
    to[rows, (axis + 1) % 3] = line + r.choice([-1.0, 1.0], N) * 10 ** r.uniform(np.log10(3e-6), np.log10(3e-4), N)
    d = to - o
    return o, d / np.linalg.norm(d, axis=1, keepdims=True)


def _unaimed(k, r):
    """Anywhere on a wall, 1e-4 to 1e-1 of the direction across it."""
    rows = np.arange(N)
    axis, side = r.integers(0, 3, N), r.choice([-1.0, 1.0], N)
    across, turn, far = 10 ** r.uniform(-4, -1, N), r.uniform(0, 2 * np.pi, N), r.uniform(0.5, 5, N)
    d = np.empty((N, 3))
    d[rows, axis] = side * across
    d[rows, (axis + 1) % 3] = np.sqrt(1 - across ** 2) * np.cos(turn)
    d[rows, (axis + 2) % 3] = np.sqrt(1 - across ** 2) * np.sin(turn)
    o = r.uniform(-5, 5, (N, 3))
    o[rows, axis] = side * (5 - far * across)
    return o, d


@pytest.mark.parametrize("aim", [_aimed, _unaimed])
@pytest.mark.parametrize("k", [4, 16, 32])
def test_grazing_rays(gpu, orc, k, aim):
    from renderbox2_amd import _lib as L
    b = gpu.BVH(_room(k))
    c = b.export(L.RB_LAYOUT_REF_COMPACT2)
    tr = gpu.CudaTracer(b)
    rays = np.zeros((N, 8), np.float32)
    rays[:, 0:3], rays[:, 4:7] = aim(k, np.random.default_rng(1000 + k))
    rays[:, 3], rays[:, 7] = 1e-3, 3.4e38
    oid, _ = orc.trace_compact2(c[0].reshape(-1, 4), c[1].reshape(-1, 4), c[2], rays)
    assert (oid >= 0).mean() > 0.4

    def same(ids, ts, part=slice(None)):
        bad = int(((ids >= 0) != (oid[part] >= 0)).sum())
        assert bad == 0, f"{bad} rays change hit and miss"
        assert np.array_equal(ids, many[0][part]) and np.array_equal(ts.view(np.uint32), many[1][part].view(np.uint32))

    many = tr.trace(rays)
    same(*many)
    for at in range(0, N, FEW):
        same(*tr.trace(rays[at:at + FEW]), slice(at, at + FEW))
    d_rays, d_hits = gpu.DeviceBuffer.from_array(rays), gpu.DeviceBuffer(N * 8)
    cut = N // 3
    gpu.trace_batch([(tr, d_rays.ptr, cut, d_hits.ptr, False),
                     (tr, d_rays.ptr + 32 * cut, N - cut, d_hits.ptr + 8 * cut, False)])
    h = d_hits.download(gpu.HIT_DTYPE, N)
    same(h["id"], h["t"])
    same(*tr.trace_simple(rays))
