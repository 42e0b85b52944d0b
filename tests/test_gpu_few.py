"""GPU parity of the loops a launch may take: a quad of lanes per ray for
launches of few rays, a lane per ray for the rest and a quad for each of its
waves' last rays.  The same rays traced alone and as the head or the end of a
launch past the line (512 rays per CU) give the same (id, t), bit for bit, which
are the oracle's -- over the wide and the binary records, closest and any hit,
masked, at the edges of a block (16 rays), with leaves of more triangles than a
quad has lanes, ties, NaN and zero rays, and stacks that leave their LDS rows."""
import numpy as np
import pytest

from conftest import random_rays, random_triangles

pytestmark = pytest.mark.gpu

PAST = 512 * 256 + 1


@pytest.fixture(scope="module")
def scene(gpu):
    from renderbox2_amd import _lib as L
    v, idx = random_triangles(1500, seed=500)
    # 23 copies of one triangle (a leaf of many, all ties) and 6 nested ones
    extra = [idx[:1]] * 23 + [idx[7:8]] * 6
    idx = np.concatenate([idx] + extra).astype(idx.dtype)
    b = gpu.BVH((v, idx))
    c = b.export(L.RB_LAYOUT_REF_COMPACT2)
    centre = v[idx[0]].mean(axis=0)
    return gpu.CudaTracer(b), (c[0].reshape(-1, 4), c[1].reshape(-1, 4), c[2]), centre


def _rays(n, centre):
    rays = random_rays(n, seed=501)
    rays[: n // 2, 4:7] = centre - rays[: n // 2, 0:3]  # through the copies
    if n > 8:
        rays[1, 4:7] = 0.0
        rays[2, 0:3] = np.nan
        rays[3, 5] = 0.0
        rays[4, 7] = np.inf
        rays[5, 3] = np.nan
        rays[6, 4:7] = np.inf
    return rays


def _trace(gpu, tr, rays, n, any_hit, mask):
    d_rays, d_hits = gpu.DeviceBuffer.from_array(rays), gpu.DeviceBuffer(n * 8)
    d_mask = gpu.DeviceBuffer.from_array(mask) if mask is not None else None
    tr.trace_device(d_rays.ptr, n, d_hits.ptr, any_hit=any_hit, d_mask=d_mask.ptr if d_mask else None)
    return d_hits.download(gpu.HIT_DTYPE, n)


@pytest.mark.parametrize("wide", [1, 0])
@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("n", [1, 15, 17, 4099])
@pytest.mark.parametrize("lds_stack,block", [(16, 256), (8, 64)])
def test_the_loops_give_the_same_hits(gpu, orc, scene, wide, any_hit, masked, n, lds_stack, block):
    tr, c2, centre = scene
    rays = _rays(n, centre)
    mask = (np.arange(PAST) % 3 != 0).astype(np.uint8) if masked else None
    cfg = gpu.get_trace_config()
    gpu.set_trace_config(**{**cfg, "wide": wide, "lds_stack": lds_stack, "block": block})
    try:
        few = _trace(gpu, tr, rays, n, any_hit, mask)
        rest = np.zeros((PAST - n, 8), np.float32)
        rest[:, 0:3] = 1e6  # rays that miss the root
        rest[:, 4] = rest[:, 7] = 1.0
        head = _trace(gpu, tr, np.concatenate([rays, rest]), PAST, any_hit, mask)[:n]
        if masked:
            mask = np.concatenate([mask[n:], mask[:n]])
        end = _trace(gpu, tr, np.concatenate([rest, rays]), PAST, any_hit, mask)[PAST - n:]
    finally:
        gpu.set_trace_config(**cfg)
    mask = np.arange(PAST) % 3 != 0
    for many in (head, end):
        assert np.array_equal(few["id"], many["id"])
        assert np.array_equal(few["t"].view(np.uint32), many["t"].view(np.uint32))
    ok = np.isfinite(rays[:, :7]).all(axis=1)
    if masked:
        ok &= mask[:n]
    oid, ot = orc.trace_compact2(*c2, np.ascontiguousarray(rays[ok]), any_hit=any_hit)
    assert np.array_equal(few["id"][ok], oid) and np.array_equal(few["t"][ok].view(np.uint32), ot.view(np.uint32))
    if n > 1000 and not masked:
        assert (oid >= 0).sum() > n // 4


@pytest.mark.parametrize("kind", ["pt", "bdpt"])
@pytest.mark.parametrize("lds_stack,block,wide", [(16, 256, 1), (8, 64, 1), (16, 512, 0)])
def test_frames_equal_their_tiles(gpu, kind, lds_stack, block, wide):
    """A frame's bounces, whose launches learn in the kernel that they have few
    rays, against those of its tiles, whose launches are known to have few."""
    s = gpu.scenes.pt_room(spheres_hi=4, spheres_lo=10)
    tr = gpu.CudaTracer(gpu.scenes.build(s), s)
    cam = gpu.scenes.pt_camera(256, 192)
    cfg = gpu.get_trace_config()
    gpu.set_trace_config(**{**cfg, "lds_stack": lds_stack, "block": block, "wide": wide})
    try:
        kw = dict(light_paths=500, light_max_depth=3, connections=1) if kind == "bdpt" else {}
        r = gpu.SamplerRenderer(tr, cam, kind, spp=1, seed=4, max_depth=6, rr_start=1, rr_prob=0.5, **kw)
        frame = r.render()
        assert np.isfinite(frame).all() and frame.max() > 0
        for y in range(0, 192, 48):
            for x in range(0, 256, 128):
                tile = r.render((x, y, 128, 48))
                assert np.array_equal(tile.view(np.uint32), frame[y:y + 48, x:x + 128].view(np.uint32))
    finally:
        gpu.set_trace_config(**cfg)
