"""The filtered film where its workgroups' tiles (64x4 pixels) and its runs of
staged samples (1024 at a time: whole columns, or parts of one pixel's) end:
the oracle's image, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,spp,radius", [(1, 1, 1, 2.0), (63, 3, 5, 2.0), (65, 5, 20, 1.0), (130, 9, 3, 7.5),
                                            (4, 5, 1024, 1.5), (3, 2, 1030, 1.5)])
def test_film_equals_the_oracle(gpu, orc, w, h, spp, radius):
    from renderbox2_amd import _lib as L
    s = gpu.scenes.pt_room(spheres_hi=2, spheres_lo=4)
    b = gpu.scenes.build(s)
    cam = gpu.scenes.pt_camera(w + 9, h + 4)
    tile, film = (7, 3, w, h), (2, radius, radius, 1.0)
    img = gpu.SamplerRenderer(gpu.CudaTracer(b, s), cam, "raycast", spp=spp, seed=8, shade="normals", filter=film[0],
                              filter_width=(radius, radius), filter_alpha=film[3]).render(tile)
    c = b.export(L.RB_LAYOUT_REF_COMPACT2)
    v, idx, tm, _ = s.geometry()
    k = cam.c
    view = (tuple(k.position), tuple(k.lookat), tuple(k.up), k.hfov_deg, k.width, k.height)
    ref = orc.render_raycast((c[0].reshape(-1, 4), c[1].reshape(-1, 4), c[2]), v, idx, tm, s.materials(), view, tile,
                             spp, 8, gpu.core.SHADES["normals"], film=film)
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
