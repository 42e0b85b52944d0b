"""The work that users of this framework have it do, as cases to measure.

Sizes come from the benchmark's configurations (bench.py) and from the
tests, or are generic ragged ones.  Scenes are the seeded synthetic ones of
renderbox2_amd.scenes, or a triangle soup handed over as arrays.  A program
keeps its scene resident on the GPU, so scenes are kept here by what they
are; rays, seeds and buffers are made anew for every state.  Passes go to the
library's own stream, the default of every entry point.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

import renderbox2_amd as rb
from renderbox2_amd import _lib as L

CACHE = os.path.join(tempfile.gettempdir(), "rb_perf_bvh_%d" % os.getuid())
MESHES = {"spheres": rb.scenes.trace_scaled,  # icospheres and thin quads: open, rays leave the scene
          "rooms": rb.scenes.pt_scaled}       # closed room, mixed materials, four emitters
_resident = {}


def listed():
    return [
        # An application that asks a few thousand visibility or picking
        # queries of a small mesh: one call, latency-bound.
        {"name": "closest_small_soup", "kind": "soup", "tris": 10007, "rays": 4099, "any": False},
        # Primary visibility of one HD frame: coherent rays.
        {"name": "closest_camera_hd", "kind": "trace", "scene": "spheres", "tris": 200000, "rays": 2073600,
         "set": "camera", "any": False},
        # Diffuse bounces of a 2048x1024 view of a million triangles: the
        # framework's headline figure.
        {"name": "closest_diffuse_1m", "kind": "trace", "scene": "spheres", "tris": 1000000, "rays": 2097152,
         "set": "diffuse", "any": False},
        # Any-hit queries with the reported first hit, a ragged count.
        {"name": "any_diffuse_1m", "kind": "trace", "scene": "spheres", "tris": 1000000, "rays": 1000003,
         "set": "diffuse", "any": True},
        # An external integrator that reads whole intersection records
        # (rb_trace_fill), smooth normals, a ragged count.
        {"name": "fill_smooth_room", "kind": "fill", "tris": 78848, "rays": 262147},
        # Many uneven ray batches of several resident scenes in one call.
        {"name": "batch_64_of_4_scenes", "kind": "batch", "batches": 64, "rays_low": 4096, "rays_high": 524288},
        # Ambient-occlusion frame, the first rendering configuration.
        {"name": "ao_512", "kind": "render", "pass": "ao", "scene": "room", "tris": 78848, "width": 512, "height": 512,
         "spp": 1, "depth": 0, "filter": "box", "filter_width": 0.5},
        # The same with antialiasing and the Gaussian film on a ragged frame.
        {"name": "ao_gauss_401x299", "kind": "render", "pass": "ao", "scene": "room", "tris": 78848, "width": 401,
         "height": 299, "spp": 4, "depth": 0, "filter": "gaussian", "filter_width": 2.0},
        # One refresh of a progressive viewer: a small path-traced tile.
        {"name": "pt_tile_128", "kind": "render", "pass": "pt", "scene": "rooms", "tris": 500000, "width": 128,
         "height": 128, "spp": 1, "depth": 8, "filter": "box", "filter_width": 0.5},
        # The path-traced frame configuration, and the largest case.
        {"name": "pt_1024_8spp", "kind": "render", "pass": "pt", "scene": "rooms", "tris": 2000000, "width": 1024,
         "height": 1024, "spp": 8, "depth": 8, "filter": "box", "filter_width": 0.5},
        # The bidirectional frame configuration.
        {"name": "bdpt_512_4spp", "kind": "render", "pass": "bdpt", "scene": "rooms", "tris": 2000000, "width": 512,
         "height": 512, "spp": 4, "depth": 6, "filter": "box", "filter_width": 0.5},
        # A burst of mixed tile requests to the rendering server.
        {"name": "served_24_tiles", "kind": "served", "requests": 24, "tris": 500000, "side_low": 64,
         "side_high": 256},
    ]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["soup", "trace", "trace", "trace", "fill", "batch", "render", "render", "render"])
    if kind == "soup":
        return {"kind": "soup", "tris": _log(rng, 300, 50000), "rays": _log(rng, 100, 30000),
                "any": rng.random() < 0.3}
    if kind == "trace":
        return {"kind": "trace", "scene": rng.choice(["spheres", "rooms"]), "tris": _log(rng, 10000, 1000000),
                "rays": _log(rng, 1000, 4000000), "set": rng.choice(["camera", "diffuse"]),
                "any": rng.random() < 0.3}
    if kind == "fill":
        return {"kind": "fill", "tris": 78848, "rays": _log(rng, 1000, 1000000)}
    if kind == "batch":
        low = _log(rng, 500, 8000)
        return {"kind": "batch", "batches": rng.randint(5, 100), "rays_low": low, "rays_high": low * rng.randint(2, 64)}
    what = rng.choice(["ao", "pt", "bdpt"])
    spp = rng.choice([1, 1, 2, 4, 5])
    side = _log(rng, 48, 640)
    film = rng.choice(["box", "box", "gaussian", "triangle"])
    return {"kind": "render", "pass": what, "scene": "rooms" if what != "ao" else rng.choice(["room", "rooms"]),
            "tris": _log(rng, 20000, 1000000), "width": side + rng.randint(0, 40), "height": side, "spp": spp,
            "depth": 0 if what == "ao" else rng.randint(2, 8), "filter": film,
            "filter_width": 0.5 if film == "box" else rng.choice([1.0, 1.5, 2.0])}


def _scene(mesh, tris=0):
    """The resident scene: built once, or read back from the cache of built
    trees that a renderer keeps beside its scene files."""
    key = (mesh, tris if mesh in MESHES else 0)
    if key not in _resident:
        s = MESHES[mesh](tris) if mesh in MESHES else rb.scenes.ao_room(smooth=mesh == "smooth room")
        os.makedirs(CACHE, exist_ok=True)
        bvh, _ = rb.BVH.build_cached(s, CACHE)
        _resident[key] = rb.CudaTracer(bvh, s)
    return _resident[key]


def _camera(mesh, width, height):
    if mesh == "spheres":
        return rb.scenes.trace_camera(width, height)
    return rb.scenes.ao_camera(width, height) if mesh.endswith("room") else rb.scenes.pt_camera(width, height)


def _rays(n):
    return torch.empty((n, 8), dtype=torch.float32, device="cuda")


def _hits(n):
    """The rb_hit records, as the id and the distance that they hold."""
    h = torch.empty((n, 2), dtype=torch.int32, device="cuda")
    return h, {"id": h[:, 0], "t": h.view(torch.float32)[:, 1]}


def _camera_rays(mesh, n, seed):
    h = max(1, int(math.sqrt(n / 2)))
    cam = _camera(mesh, -(-n // h), h)
    rays = _rays(cam.get_total_pixels())
    cam.generate_rays_device(rays.data_ptr(), seed=seed)
    return rays


def _diffuse_rays(tracer, mesh, n, seed):
    """Rays off the surfaces that a view of as many pixels sees."""
    prim = _camera_rays(mesh, n, seed)
    hits, _ = _hits(len(prim))
    rays = _rays(n)
    tracer.trace_device(prim.data_ptr(), len(prim), hits.data_ptr())
    rb.raygen_diffuse_device(tracer, prim.data_ptr(), hits.data_ptr(), len(prim), n, seed + 1, rays.data_ptr())
    torch.cuda.synchronize()
    return rays


def _soup(case, seed):
    """A triangle soup and rays through it, as numpy arrays."""
    r = np.random.default_rng(seed)
    c = r.uniform(-5, 5, (case["tris"], 1, 3))
    v = (c + r.normal(0, 4.0 / case["tris"] ** (1 / 3), (case["tris"], 3, 3))).astype(np.float32).reshape(-1, 3)
    i = np.arange(len(v), dtype=np.uint32).reshape(-1, 3)
    d = r.normal(size=(case["rays"], 3))
    rays = np.zeros((case["rays"], 8), np.float32)
    rays[:, :3] = r.uniform(-6, 6, (case["rays"], 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 7] = r.uniform(2, 20, case["rays"])
    return v, i, rays


def _params(case, seed):
    w = case["filter_width"]
    p = {"spp": case["spp"], "seed": seed, "filter": case["filter"], "filter_width": (w, w)}
    if case["pass"] == "ao":
        return dict(p, ao_samples=8, ao_radius=1.0)
    p = dict(p, max_depth=case["depth"], rr_start=3, rr_prob=0.5)
    if case["pass"] == "bdpt":
        full = case["width"] * case["height"] >= 1 << 18
        p = dict(p, light_max_depth=6, connections=5, light_paths=0, lvc_capacity=1 << (20 if full else 17))
    return p


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "soup":
        v, i, rays = _soup(case, seed)
        s["tracer"] = rb.CudaTracer(rb.BVH((v, i)))
        s["rays"], s["any"] = torch.from_numpy(rays).cuda(), case["any"]
        s["hits"], s["out"] = _hits(case["rays"])
    elif kind == "trace":
        s["tracer"] = _scene(case["scene"], case["tris"])
        s["rays"] = (_diffuse_rays(s["tracer"], case["scene"], case["rays"], seed) if case["set"] == "diffuse"
                     else _camera_rays(case["scene"], case["rays"], seed)[:case["rays"]])
        s["any"] = case["any"]
        s["hits"], s["out"] = _hits(case["rays"])
    elif kind == "fill":
        n = case["rays"]
        s["tracer"] = _scene("smooth room")
        s["rays"] = _diffuse_rays(s["tracer"], "smooth room", n, seed)
        f = torch.zeros((16, n), dtype=torch.float32, device="cuda")
        u = torch.zeros((2, n), dtype=torch.int32, device="cuda")
        b = torch.zeros((2, n), dtype=torch.uint8, device="cuda")
        s["soa"] = L.rb_isect_soa(*[(ctypes.c_void_p * 3)(*[f[3 * k + c].data_ptr() for c in range(3)]) for k in range(4)],
                                  f[12].data_ptr(), u[0].data_ptr(), u[1].data_ptr(), b[0].data_ptr(), b[1].data_ptr(),
                                  f[14].data_ptr(), f[15].data_ptr())
        s["out"] = {"floats": f, "ids": u, "flags": b}
    elif kind == "batch":
        r = np.random.default_rng(seed)
        scenes = [("spheres", t) for t in (10000, 50000, 200000, 1000000)]
        u = np.random.default_rng(case["batches"]).random(case["batches"])  # the sizes are the case's, not the seed's
        sizes = (case["rays_low"] * (case["rays_high"] / case["rays_low"]) ** u).astype(int)
        pools = []
        for k, (mesh, tris) in enumerate(scenes):
            t, m = _scene(mesh, tris), max(16, int(sizes.max()))
            pools.append((t, _camera_rays(mesh, m, seed + k), _diffuse_rays(t, mesh, m, seed + k)))
        torch.cuda.synchronize()
        s["rays"], s["batches"] = _rays(int(sizes.sum())), []
        s["hits"], s["out"] = _hits(int(sizes.sum()))
        at = 0
        for k, n in enumerate(int(x) for x in sizes):  # the first half camera rays, the rest diffuse ones
            t, a, d = pools[k % len(pools)]
            o1, o2 = (int(x) for x in r.integers(0, len(d) - n + 1, 2))
            s["rays"][at:at + n // 2] = a[o1:o1 + n // 2]
            s["rays"][at + n // 2:at + n] = d[o2:o2 + n - n // 2]
            s["batches"].append((t, s["rays"][at:].data_ptr(), n, s["hits"][at:].data_ptr(), False))
            at += n
    elif kind == "render":
        cam = _camera(case["scene"], case["width"], case["height"])
        s["pass"] = rb.SamplerRenderer(_scene(case["scene"], case["tris"]), cam, case["pass"], **_params(case, seed))
        s["out"] = torch.zeros((case["height"], case["width"], 3), dtype=torch.float32, device="cuda")
    else:
        r = np.random.default_rng(seed)
        cam = rb.scenes.pt_camera(1024, 1024)
        s["server"] = rb.RenderServer(max_inflight=8)
        sid = s["server"].add_scene(_scene("rooms", case["tris"]))
        s["requests"] = []
        sides = np.random.default_rng(case["requests"]).integers(case["side_low"], case["side_high"] + 1,
                                                                 (case["requests"], 2))
        for k in range(case["requests"]):
            what = ("ao", "pt", "ao", "pt", "bdpt")[k % 5]
            w, h = (int(x) for x in sides[k])
            x, y = int(r.integers(0, 1025 - w)), int(r.integers(0, 1025 - h))
            p = _params({"pass": what, "spp": 1 + k % 4, "depth": 6, "filter": "box", "filter_width": 0.5, "width": w,
                         "height": h}, seed + k)
            s["requests"].append((what, sid, cam, (x, y, w, h), p))
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind in ("soup", "trace"):
        s["tracer"].trace_device(s["rays"].data_ptr(), len(s["rays"]), s["hits"].data_ptr(), any_hit=s["any"])
    elif kind == "fill":
        L.check(L.lib().rb_trace_fill(s["tracer"].handle, s["rays"].data_ptr(), len(s["rays"]), L.RB_CLOSEST, None,
                                      None, ctypes.byref(s["soa"]), None))
    elif kind == "batch":
        rb.trace_batch(s["batches"])
    elif kind == "render":
        s["pass"].render_device(s["out"].data_ptr())
    else:
        ids = [s["server"].submit_render(*q[:4], **q[4]) for q in s["requests"]]
        return [s["server"].wait(i)[1] for i in ids]
    return s["out"]


def _per_ray(tris):
    """Floating operations of a ray that meets one box of four children a
    level on its way to one triangle."""
    return math.ceil(math.log(max(tris, 4), 4)) * 4 * 12 + 30


def work(case):
    kind = case["kind"]
    if kind in ("soup", "trace"):
        n = case["rays"]
        return {"bytes": 40 * n + 36 * case["tris"], "flops": n * _per_ray(case["tris"])}
    if kind == "fill":
        n = case["rays"]
        return {"bytes": (32 + 74) * n + 72 * case["tris"], "flops": n * (_per_ray(case["tris"]) + 120)}
    if kind == "batch":
        lo, hi = case["rays_low"], case["rays_high"]
        n = case["batches"] * (hi - lo) / math.log(hi / lo)  # mean of the log-uniform sizes
        return {"bytes": 40 * n + 36 * 1260000, "flops": n * _per_ray(300000)}
    if kind == "render":
        n = case["width"] * case["height"] * case["spp"]
        # nine rays of an AO sample; a path's camera ray and, up to the
        # bounce where roulette starts, a light ray and the next one (with
        # BDPT five connections too)
        rays = 9 if case["pass"] == "ao" else 1 + min(case["depth"] + 1, 4) * (7 if case["pass"] == "bdpt" else 2)
        return {"bytes": 12 * case["width"] * case["height"] + 36 * case["tris"], "flops": n * rays * _per_ray(case["tris"])}
    side = (case["side_low"] + case["side_high"]) / 2
    n = case["requests"] * side * side
    return {"bytes": 12 * n + 36 * case["tris"], "flops": 2.5 * n * 15 * _per_ray(case["tris"])}


def exact(case, seed):
    """Brute force over the soup (Moeller-Trumbore); the other cases have
    too many ray-triangle pairs, or follow random paths."""
    if case["kind"] != "soup" or case["any"] or case["tris"] * case["rays"] > 2e8:
        return None
    v, i, rays = _soup(case, seed)
    t = torch.from_numpy(v[i].astype(np.float64)).cuda()
    a, e1, e2 = t[:, 0], t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    got = []
    for r in torch.from_numpy(rays.astype(np.float64)).cuda().split(max(1, 4000000 // len(t))):
        o, d = r[:, None, :3], r[:, None, 4:7]
        p = torch.cross(d.expand(-1, len(t), -1), e2[None].expand(len(r), -1, -1), dim=2)
        det = (p * e1).sum(2)
        q = torch.cross((o - a), e1[None].expand(len(r), -1, -1), dim=2)
        u, w = ((o - a) * p).sum(2) / det, (d * q).sum(2) / det
        at = (q * e2).sum(2) / det
        far = r[:, 7:8]
        hit = (u >= 0) & (w >= 0) & (u + w <= 1) & (at > r[:, 3:4]) & (at < far)
        got.append(torch.where(hit, at, far).amin(1))
    return {"id": None, "t": torch.cat(got)}
