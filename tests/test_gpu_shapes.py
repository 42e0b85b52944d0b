"""The step loop in every launch shape that can be selected, in launches past the
line up to which launches ignore the shape (512 rays per CU): closest and any hit,
as one set and in a batched launch, over the wide and the binary records, equal the
oracle, bit for bit, in a shallow tree and in one whose stacks leave their rows; and
frames past the line are those of the default shape.  (In the deep tree rays are aimed
at triangles far smaller than their distances' rounding; closest hits over the wide
records, whose leaf boxes are a little larger than the binary ones, are then those of
single rays, which follow the same rule.)  Thresholds, gates, claims and
waves go through their ranges with the shapes."""
import numpy as np
import pytest

from conftest import random_rays, random_triangles
from test_walk_layout import _nested

pytestmark = pytest.mark.gpu

PAST = 512 * 256 + 1
N = 20000
SHAPES = [(s, b) for s, blocks in ((8, (64, 128, 256, 512, 1024)), (12, (64, 128, 256, 512, 1024)),
                                   (16, (64, 128, 256, 512)), (20, (64, 128, 256)), (24, (64, 128, 256)))
          for b in blocks]


def _config(saved, k, wide):
    s, b = SHAPES[k]
    return {**saved, "lds_stack": s, "block": b, "wide": wide, "fetch_threshold": (0, 24, 52, 64)[k % 4],
            "leaf_gate": (0, 20, 40, 63)[(k + k // 4) % 4], "chunk": (64, 192, 1024)[k % 3],
            "waves_per_cu": (8, 20, 32)[k // 2 % 3]}


@pytest.fixture(scope="module", params=["shallow", "deep"])
def scene(request, gpu, orc):
    from renderbox2_amd import _lib as L
    if request.param == "shallow":
        geometry, rays = random_triangles(3000, seed=800), random_rays(N, seed=801)
    else:  # clusters of ever smaller triangles, and rays at all their sizes
        geometry, rays = _nested(64, 40, 0.25, 2), random_rays(N, seed=802, box=1.0)
        v, idx = geometry
        t = np.random.default_rng(803).integers(0, len(idx), N)
        to = v[idx[t]].mean(axis=1)
        rays[:, 4:7] = to - rays[:, 0:3]
    b = gpu.BVH(geometry)
    c = b.export(L.RB_LAYOUT_REF_COMPACT2)
    c2 = (c[0].reshape(-1, 4), c[1].reshape(-1, 4), c[2])
    if request.param == "deep":  # more entries than a wave's last rays keep when they get a quad each
        assert int(b.export(L.RB_LAYOUT_MI355X_WALK)[2][-1]) > 15 + 48
    want = [orc.trace_compact2(*c2, rays, any_hit=a) for a in (False, True)]
    assert (want[0][0] >= 0).mean() > 0.2
    rest = np.zeros((PAST - N, 8), np.float32)
    rest[:, 0:3], rest[:, 4], rest[:, 7] = 1e6, 1.0, 1.0  # rays that miss the root
    tr = gpu.CudaTracer(b)
    want_wide = [tr.trace_simple(rays) if request.param == "deep" else want[0], want[1]]
    return tr, gpu.DeviceBuffer.from_array(np.concatenate([rays, rest])), (want, want_wide)


@pytest.mark.parametrize("wide", [1, 0])
@pytest.mark.parametrize("k", range(len(SHAPES)))
def test_every_shape_equals_the_oracle(gpu, scene, k, wide):
    tr, d_rays, want = scene
    d_hits = gpu.DeviceBuffer(PAST * 8)
    saved = gpu.get_trace_config()
    gpu.set_trace_config(**_config(saved, k, wide))
    try:
        for any_hit in (False, True):
            got = []
            tr.trace_device(d_rays.ptr, PAST, d_hits.ptr, any_hit=any_hit)
            got.append(d_hits.download(gpu.HIT_DTYPE, PAST))
            cut = N // 3
            gpu.trace_batch([(tr, d_rays.ptr, cut, d_hits.ptr, any_hit),
                             (tr, d_rays.ptr + 32 * cut, PAST - cut, d_hits.ptr + 8 * cut, any_hit)])
            got.append(d_hits.download(gpu.HIT_DTYPE, PAST))
            ids, ts = want[wide][any_hit]
            for h in got:
                assert np.array_equal(h["id"][:N], ids) and (h["id"][N:] == -1).all()
                assert np.array_equal(h["t"][:N].view(np.uint32), ts.view(np.uint32))
    finally:
        gpu.set_trace_config(**saved)


@pytest.fixture(scope="module")
def frames(gpu):
    s = gpu.scenes.pt_room(spheres_hi=4, spheres_lo=10)
    tr = gpu.CudaTracer(gpu.scenes.build(s), s)
    cam = gpu.scenes.pt_camera(256, 256)
    kw = dict(spp=2, seed=6, max_depth=3, rr_start=3, rr_prob=0.5)
    pt = gpu.SamplerRenderer(tr, cam, "pt", **kw)
    bdpt = gpu.SamplerRenderer(tr, cam, "bdpt", **kw, light_paths=2000, light_max_depth=3, connections=1)
    return {r: r.render() for r in (pt, bdpt)}


@pytest.mark.parametrize("wide", [1, 0])
@pytest.mark.parametrize("k", range(len(SHAPES)))
def test_every_shape_renders_the_same_frames(gpu, frames, k, wide):
    saved = gpu.get_trace_config()
    gpu.set_trace_config(**_config(saved, k, wide))
    try:
        for renderer, image in frames.items():
            assert image.max() > 0
            assert np.array_equal(renderer.render().view(np.uint32), image.view(np.uint32))
    finally:
        gpu.set_trace_config(**saved)
