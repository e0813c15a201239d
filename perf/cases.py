"""The work whose speed is measured: what a renderer built on this package
asks of it, each case through the public entry points of `cudatracer_amd`.

A case is a dict of plain values.  `prepare` makes what a program holds before
the call (a context with an uploaded scene, a camera, rays, a server), `run`
is one pass, `work` the bytes and operations that pass cannot do without, and
`exact` its result in 64 bits where plain torch can compute it.  `listed` are
the fixed cases, `draw` makes another of the same ranges.

Every pass of a frame starts from a cleared accumulator, as a viewer's does
when its camera has moved.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import cudatracer_amd as ct

# triangles, paths' rays (primary, extension and shadow rays per path sample)
# and megabytes of textures of the package's generated scenes
SCENES = {
    "box": (ct.SCENE_C1, 20_494, 7.0, 0.0),
    "atrium": (ct.SCENE_C2, 259_072, 5.3, 0.0),
    "displaced": (ct.SCENE_C3, 7_242_882, 2.2, 0.0),
    "textured": (ct.SCENE_C2_TEXTURED, 259_072, 5.3, 6.0),
}
ACCEL = {"bvh2": ct.ACCEL_BVH2, "bvh4": ct.ACCEL_BVH4}
TRAVERSAL = {"exact": ct.TRAV_EXACT, "fast": ct.TRAV_FAST, "compact": ct.TRAV_COMPACT}
MISS = 1e34
PROBES = 4096  # rays traced into a new mesh
# operations of a ray: about 15 quad node tests (four boxes of 20) and 3
# triangle tests (50); of a shaded hit: about 400
RAY_FLOPS, SHADE_FLOPS = 15 * 80 + 3 * 50, 400


def listed():
    return [
        # an interactive preview of a small scene: one sample, read as floats;
        # the binary tree and the options the scene itself asks for
        dict(name="frame_box_256", kind="frame", scene="box", width=256, height=256, spp=1, depth=4, accel="bvh2",
             traversal="exact", read="accum"),
        # the viewer at its usual size: one sample per frame, shown as bytes
        dict(name="frame_atrium_1080p", kind="frame", scene="atrium", width=1920, height=1080, spp=1, depth=8,
             accel="bvh4", traversal="exact", read="rgba8"),
        # a ragged window with several samples per call on the compact tree
        dict(name="frame_atrium_641x363_compact", kind="frame", scene="atrium", width=641, height=363, spp=4, depth=8,
             accel="bvh4", traversal="compact", read="accum"),
        # a large scan at 4K, deep paths with roulette
        dict(name="frame_displaced_4k", kind="frame", scene="displaced", width=3840, height=2160, spp=1, depth=16,
             accel="bvh4", traversal="exact", read="rgba8"),
        # textures, normal maps and a sky texture; the image read as floats
        dict(name="frame_textured_1080p", kind="frame", scene="textured", width=1920, height=1080, spp=1, depth=8,
             accel="bvh4", traversal="exact", read="image"),
        # a picking or probe query: few rays, already on the GPU
        dict(name="rays_device_1k", kind="rays", triangles=20_001, rays=1_000, query="closest_device", accel="bvh4",
             traversal="exact"),
        # a simulation's rays in GPU memory, enough to fill the chip
        dict(name="rays_device_1m", kind="rays", triangles=524_287, rays=1 << 20, query="closest_device", accel="bvh4",
             traversal="exact"),
        # a baker's queries from host arrays: first hits, then visibility
        dict(name="rays_host_300k", kind="rays", triangles=50_000, rays=300_001, query="both_host", accel="bvh2",
             traversal="exact"),
        # thumbnails: uneven views of one scene in one call
        dict(name="batch_16_views", kind="batch", scene="box", views=16, largest=1024, depth=8),
        # a render service's mix of sizes and sample counts, all waiting at once
        dict(name="serve_8_requests", kind="serve", scene="atrium", requests=8, depth=8),
        # a new mesh in a running program: its trees built on the GPU, then
        # first probes into it
        dict(name="scene_swap_1m", kind="swap", triangles=1_000_003, then="probe"),
        # a smaller one whose trees are read back to be kept with the mesh
        dict(name="tree_export_100k", kind="swap", triangles=100_003, then="export"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "rays", "rays", "rays", "batch", "serve", "swap", "display"])
    if kind == "frame":
        scene = rng.choice(["box", "atrium", "atrium", "textured", "displaced"])
        # from a 64-pixel preview to the scene's own frame size
        most = {"box": 1 << 19, "displaced": 3840 * 2160}.get(scene, 1920 * 1080)
        pixels = _log_int(rng, 64 * 48, most)
        aspect = rng.uniform(0.6, 2.0)
        width = max(8, min(pixels // 8, int(math.sqrt(pixels * aspect))))
        height = max(8, pixels // width)
        spp = rng.choice([s for s in (1, 1, 2, 3, 4, 8) if s * width * height <= most] or [1])
        traversal, accel = rng.choice([("exact", "bvh4")] * 4 + [("compact", "bvh4"), ("exact", "bvh2")])
        return dict(kind=kind, scene=scene, width=width, height=height, spp=spp,
                    depth=rng.randint(2, 16 if scene == "displaced" else 8), accel=accel, traversal=traversal,
                    read=rng.choice(["accum", "image", "rgba8"]))
    if kind == "rays":
        traversal, accel = rng.choice([("exact", "bvh4")] * 4 + [("compact", "bvh4"), ("fast", "bvh4"), ("exact", "bvh2")])
        return dict(kind=kind, triangles=_log_int(rng, 2_000, 524_287), rays=_log_int(rng, 64, 1 << 20),
                    query=rng.choice(["closest_device", "closest_device", "closest_noalloc", "both_host"]),
                    accel=accel, traversal=traversal)
    if kind == "batch":
        return dict(kind=kind, scene="box", views=rng.randint(2, 16), largest=_log_int(rng, 128, 768),
                    depth=rng.randint(2, 8))
    if kind == "serve":
        return dict(kind=kind, scene=rng.choice(["box", "atrium"]), requests=rng.randint(1, 7), depth=rng.randint(3, 8))
    if kind == "swap":
        then = rng.choice(["probe", "probe", "export"])
        return dict(kind=kind, triangles=_log_int(rng, 500, 1_000_003 if then == "probe" else 100_003), then=then)
    pixels = _log_int(rng, 64 * 48, 1920 * 1080)
    width = max(8, int(math.sqrt(pixels * rng.uniform(0.6, 2.0))))
    return dict(kind=kind, width=width, height=max(8, pixels // width), samples=rng.randint(1, 1000),
                read=rng.choice(["image", "rgba8"]))


# ------------------------------------------------------------------ inputs --
_displaced = None  # the 7.24M-triangle host scene takes seconds to generate


def _scene(name, seed):
    global _displaced
    if name != "displaced":
        return ct.HostScene.generate(SCENES[name][0], seed, build=False)
    if _displaced is None:
        _displaced = ct.HostScene.generate(ct.SCENE_C3, 7, build=False)
    return _displaced


def _camera(scene, width, height, seed):
    """The scene's own camera, turned and moved a little by the seed."""
    cam = scene.camera(width, height)
    rng = np.random.default_rng(seed + 101)
    f = np.array(list(cam.forward)) + rng.uniform(-0.08, 0.08, 3)
    p = np.array(list(cam.position))
    p = p + rng.uniform(-0.01, 0.01, 3) * np.linalg.norm(p)
    cam.forward[:] = [float(x) for x in f / np.linalg.norm(f)]
    cam.position[:] = [float(x) for x in p]
    return cam


def _grove(triangles, seed):
    """A mesh of exactly `triangles` triangles: a height field of about nine
    tenths of them, the rest loose leaves above it (world units: cells of 2)."""
    rng = np.random.default_rng(seed)
    g = max(2, int(math.sqrt(0.45 * triangles)))
    cell = 2.0
    x, z = np.meshgrid(np.arange(g + 1) * cell, np.arange(g + 1) * cell, indexing="ij")
    y = np.zeros_like(x)
    for octave in range(4):
        k, a = rng.uniform(0.5, 1.5, 2) * 0.02 * 2.2 ** octave, 12.0 * 0.45 ** octave
        y += a * np.sin(k[0] * x + rng.uniform(0, 6)) * np.cos(k[1] * z + rng.uniform(0, 6))
    y += rng.uniform(-0.3, 0.3, y.shape)
    v = np.stack([x, y, z], -1).reshape(-1, 3)
    i = (np.arange(g)[:, None] * (g + 1) + np.arange(g)[None, :]).reshape(-1)
    ground = np.concatenate([np.stack([i, i + 1, i + g + 1], -1), np.stack([i + 1, i + g + 2, i + g + 1], -1)])
    n = triangles - len(ground)
    centre = rng.uniform(0, g * cell, (n, 1, 3))
    centre[..., 1] = rng.uniform(-5, 25, (n, 1))
    leaf = (centre + rng.normal(size=(n, 3, 3)) * np.exp(rng.uniform(-0.5, 1.0, (n, 1, 1)))).reshape(-1, 3)
    idx = np.concatenate([ground, len(v) + np.arange(3 * n).reshape(-1, 3)]).astype(np.uint32)
    vertices = np.concatenate([v, leaf]).astype(np.float32)
    p = vertices[idx].astype(np.float64)
    cn = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    cn /= np.maximum(np.linalg.norm(cn, axis=1, keepdims=True), 1e-20)
    normals = np.zeros(vertices.shape)
    for k in range(3):
        np.add.at(normals, idx[:, k], cn)
    normals /= np.maximum(np.linalg.norm(normals, axis=1, keepdims=True), 1e-20)
    return dict(vertices=vertices, normals=normals.astype(np.float32), indices=idx,
                center_normals=cn.astype(np.float32), material_idx=np.zeros(triangles, np.uint32),
                light_indices=np.array([triangles - 1], np.uint32), size=g * cell)


def _view(mesh):
    """The mesh as the borrowed arrays an upload takes (they stay alive with it)."""
    m = (ct.Material * 1)()
    m[0].albedo[:] = [0.6, 0.6, 0.6]
    m[0].type, m[0].roughness, m[0].refract_idx = ct.MAT_LAMBERTIAN, 1.0, 1.0
    m[0].diffuse_tex = m[0].normal_tex = m[0].mask_tex = m[0].displace_tex = -1
    mesh["materials"] = m
    v = ct.SceneView()
    f, u = C.POINTER(C.c_float), C.POINTER(C.c_uint32)
    v.n_vertices, v.n_triangles, v.n_lights, v.n_materials = len(mesh["vertices"]), len(mesh["indices"]), 1, 1
    for name, t in (("vertices", f), ("normals", f), ("center_normals", f), ("indices", u), ("material_idx", u),
                    ("light_indices", u)):
        mesh[name] = np.ascontiguousarray(mesh[name])
        setattr(v, name, mesh[name].ctypes.data_as(t))
    v.materials = C.cast(m, C.POINTER(ct.Material))
    v.sky_enabled, v.sky_texture = 1, -1
    return v


def _rays(mesh, n, seed):
    """Origins in and above the leaves; directions mostly downward and flat."""
    rng = np.random.default_rng(seed + 11)
    o = rng.uniform(0, mesh["size"], (n, 3))
    o[:, 1] = rng.uniform(-2, 60, n)
    d = rng.normal(size=(n, 3)) * np.array([1.0, 0.6, 1.0]) - np.array([0.0, 0.5, 0.0])
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return o.astype(np.float32), d.astype(np.float32), rng.uniform(5, 200, n).astype(np.float32)


def _opts(case, scene):
    o = scene.frame_opts()[0]
    o.max_depth, o.spp = case["depth"], case["spp"]
    o.accel, o.traversal = ACCEL[case["accel"]], TRAVERSAL[case["traversal"]]
    return o


def prepare(case, seed):
    ctx = ct.Context(0)
    s = dict(case=case, ctx=ctx)
    kind = case["kind"]
    if kind in ("frame", "batch", "serve"):
        scene = _scene(case["scene"], seed)
        ctx.upload_build(scene)
        if kind == "frame":
            s["opts"] = _opts(case, scene)
            s["cam"] = _camera(scene, case["width"], case["height"], seed)
            ctx.resize(case["width"], case["height"])
        else:
            s["opts"] = scene.frame_opts()[0]
            s["opts"].max_depth = case["depth"]
            # sizes and sample counts are the case's, the cameras the seed's
            sizes, rng = np.random.default_rng(5), np.random.default_rng(seed + 3)
            views = []
            for _ in range(case["views"] if kind == "batch" else case["requests"]):
                if kind == "batch":
                    w = int(round(math.exp(sizes.uniform(math.log(min(128, case["largest"])), math.log(case["largest"])))))
                    h = w if sizes.random() < 0.5 else (w * 3) // 4
                    spp = int(sizes.choice([1, 2, 4, 8, 16]))
                    d = rng.normal(size=3)
                    cam = ct.look_at(42.0 * d / np.linalg.norm(d), rng.uniform(-5, 5, 3), 70.0)
                else:
                    w, h = [(256, 256), (512, 512), (1920, 1080)][int(sizes.choice(3, p=[0.5, 0.35, 0.15]))]
                    spp = int(sizes.choice([1, 4, 16]))
                    cam = _camera(scene, w, h, int(rng.integers(1 << 30)))
                views.append((cam, w, h, spp, 0))
            s["views"] = views
            if kind == "serve":
                s["server"] = ct.Server(ctx)
    elif kind == "rays":
        mesh = _grove(case["triangles"], seed)
        ctx.upload_build(_view(mesh), wide=case["traversal"] == "fast")
        o, d, tmax = _rays(mesh, case["rays"], seed)
        opts = ct.default_opts()
        opts.accel, opts.traversal = ACCEL[case["accel"]], TRAVERSAL[case["traversal"]]
        s.update(opts=opts, origins=o, dirs=d, tmax=tmax)
        if case["query"] != "both_host":
            rows = np.zeros((2, case["rays"], 4), np.float32)
            rows[0, :, :3], rows[1, :, :3] = o, d
            s["rows"] = torch.from_numpy(rows).cuda()
            s["hits"] = torch.empty((case["rays"], 2), dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
    elif kind == "swap":
        n = case["triangles"]
        s["mesh"] = _grove(n, seed)
        s["view"] = _view(s["mesh"])
        if case["then"] == "probe":
            s["origins"], s["dirs"], _ = _rays(s["mesh"], PROBES, seed)
            s["opts"] = ct.default_opts()
        else:  # room for the largest trees of n triangles
            s["trees"] = (np.zeros(32 * 2 * n, np.uint8), np.zeros(128 * n, np.uint8), np.zeros(n, np.uint32))
    else:
        ctx.resize(case["width"], case["height"])
        ctx.write_accum(_accum(case, seed), case["samples"])
    return s


def _accum(case, seed):
    """Sums of a rendered image's range: mostly below 1 per sample, some
    pixels dark, a few much brighter."""
    rng = np.random.default_rng(seed + 29)
    a = rng.gamma(1.5, 0.25, (case["height"], case["width"], 4)) * case["samples"]
    a[rng.random(a.shape[:2]) < 0.05] = 0.0
    a[rng.random(a.shape[:2]) < 0.01] *= 30.0
    a[..., 3] = case["samples"]
    return a.astype(np.float32)


# -------------------------------------------------------------------- pass --
def _read(ctx, how):
    if how == "accum":
        return ctx.read_accum()[0]
    return ctx.read_image() if how == "image" else ctx.read_image_rgba8()


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "frame":
        ctx.reset()
        ctx.trace_frame(s["cam"], s["opts"], stats=False)
        return _read(ctx, case["read"])
    if kind == "batch":
        return ctx.render_batch(s["views"], s["opts"])[0]
    if kind == "serve":
        ids = [s["server"].submit(cam, w, h, spp, s["opts"], fb) for (cam, w, h, spp, fb) in s["views"]]
        return [s["server"].wait(i)[1] for i in ids]
    if kind == "rays":
        if case["query"] == "both_host":
            t, prim = ctx.trace_rays(s["origins"], s["dirs"], s["opts"])
            return {"t": t, "prim": prim,
                    "occluded": ctx.trace_shadow_rays(s["origins"], s["dirs"], s["tmax"], s["opts"])}
        call = ctx.trace_rays_device if case["query"] == "closest_device" else ctx.trace_rays_device_noalloc
        call(s["rows"][0].data_ptr(), s["rows"][1].data_ptr(), case["rays"], s["hits"].data_ptr(), s["opts"])
        return {"t": s["hits"][:, 0], "prim": s["hits"].view(torch.int32)[:, 1]}
    if kind == "swap":
        ctx.upload_build(s["view"])
        if case["then"] == "probe":
            return ctx.trace_rays(s["origins"], s["dirs"], s["opts"])
        n, (bvh, mbvh, prims) = case["triangles"], s["trees"]
        r = ct.lib.ct_scene_read_trees(ctx.handle, bvh.ctypes.data, 2 * n, mbvh.ctypes.data, n, prims.ctypes.data, n)
        if r != ct.CT_OK:
            raise ct.CTError(r, "ct_scene_read_trees")
        return bvh, mbvh, prims
    return _read(ctx, case["read"])


# ------------------------------------------------------------------- bounds --
def _scene_bytes(triangles, megabytes=0.0):
    # triangle records, shading records, a quad node of 64 bytes for every 2.5 triangles
    return triangles * (48 + 112 + 64 / 2.5) + megabytes * 1e6


def work(case):
    kind = case["kind"]
    if kind == "frame":
        _, triangles, rays, mb = SCENES[case["scene"]]
        pixels = case["width"] * case["height"]
        own = {"box": 4, "displaced": 16}.get(case["scene"], 8)
        traced = pixels * case["spp"] * rays * min(1.0, case["depth"] / own)
        return {"bytes": _scene_bytes(triangles, mb) + pixels * (4 if case["read"] == "rgba8" else 16),
                "flops": traced * (RAY_FLOPS + SHADE_FLOPS / 2)}
    if kind in ("batch", "serve"):
        _, triangles, rays, mb = SCENES[case["scene"]]
        sizes, pixels, paths = np.random.default_rng(5), 0, 0
        for _ in range(case["views"] if kind == "batch" else case["requests"]):
            if kind == "batch":
                w = int(round(math.exp(sizes.uniform(math.log(min(128, case["largest"])), math.log(case["largest"])))))
                h = w if sizes.random() < 0.5 else (w * 3) // 4
                spp = int(sizes.choice([1, 2, 4, 8, 16]))
            else:
                w, h = [(256, 256), (512, 512), (1920, 1080)][int(sizes.choice(3, p=[0.5, 0.35, 0.15]))]
                spp = int(sizes.choice([1, 4, 16]))
            pixels, paths = pixels + w * h, paths + w * h * spp
        own = 4 if case["scene"] == "box" else 8
        return {"bytes": _scene_bytes(triangles, mb) + 16.0 * pixels,
                "flops": paths * rays * case["depth"] / own * (RAY_FLOPS + SHADE_FLOPS / 2)}
    if kind == "rays":
        n, calls = case["rays"], 2 if case["query"] == "both_host" else 1
        # a small query cannot touch the whole mesh
        return {"bytes": min(calls * n * 15 * 64.0, case["triangles"] * (48 + 64 / 2.5)) + n * (32.0 + 8 + 9 * (calls - 1)),
                "flops": float(calls * n * RAY_FLOPS)}
    if kind == "swap":
        # the arrays in; the records and both trees out (once more if exported)
        n, again = case["triangles"], 2 if case["then"] == "export" else 1
        return {"bytes": n * (12.0 + 12 + 4 + 0.8 * 24) + n * (48.0 + 128 + again * (32 + 128 / 2.5)),
                "flops": n * 20 * 33.0}
    pixels = case["width"] * case["height"]
    return {"bytes": pixels * (16.0 + (4 if case["read"] == "rgba8" else 16)), "flops": pixels * 3 * 40.0}


# --------------------------------------------------------------- in 64 bits --
def exact(case, seed):
    if case["kind"] == "display":
        if case["read"] != "image":
            return None
        a = _accum(case, seed).astype(np.float64)
        out = np.ones(a.shape)
        out[..., :3] = (a[..., :3] / max(case["samples"], 1)) ** (1.0 / 2.2)
        return out
    if case["kind"] != "rays" or case["rays"] * case["triangles"] > 2e10:
        return None
    # every ray against every triangle
    mesh = _grove(case["triangles"], seed)
    o, d, _ = _rays(mesh, case["rays"], seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.from_numpy(mesh["vertices"][mesh["indices"]].astype(np.float64)).to(dev)
    p0, e1, e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    oo, dd = (torch.from_numpy(a.astype(np.float64)).to(dev) for a in (o, d))
    eps = float(np.float32(1e-3))  # the default triangle epsilon
    best = torch.full((case["rays"],), MISS, dtype=torch.float64, device=dev)
    step = max(1, (1 << 25) // case["triangles"])
    dot = lambda a, b: a[0] * b[0] + a[1] * b[1] + a[2] * b[2]  # noqa: E731
    cross = lambda a, b: (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])  # noqa: E731
    tri = lambda a: [a[None, :, k] for k in range(3)]  # noqa: E731
    q0, f1, f2 = tri(p0), tri(e1), tri(e2)
    for b in range(0, case["rays"], step):
        ro = [oo[b:b + step, None, k] for k in range(3)]
        rd = [dd[b:b + step, None, k] for k in range(3)]
        h = cross(rd, f2)
        a = dot(f1, h)
        w = [ro[k] - q0[k] for k in range(3)]
        u = dot(w, h) / a
        q = cross(w, f1)
        v = dot(rd, q) / a
        t = dot(f2, q) / a
        hit = (a.abs() >= eps) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (t > eps)
        best[b:b + step] = torch.where(hit, t, MISS).amin(1).clamp(max=MISS)
    best = best.cpu()
    return {"t": best, "prim": None, "occluded": None} if case["query"] == "both_host" else {"t": best, "prim": None}
