"""The work that users of this library have it do, as measurable cases.

A case is a dict of plain values; `kind` says which public entry points it goes through:

  frame    Renderer.launch_frame (cx_renderer_frame): the path tracer, ReSTIR PT or Conditional
           ReSTIR, one pass = one frame that continues the renderer's history
  inverse  one view of an inverse-rendering step: material rows from device memory, a residual
           frame, dL/dI, an independent frame and its path-replay adjoint
  batch    cx_batch_frame over views of several scenes and resolutions, then cx_batch_sync
  trace    cx_trace_closest and cx_trace_occluded over ray arrays in device memory
  entries  cx_entries_build and cx_entries_query (or cx_entries_search_static) on device arrays
  tonemap  cx_tonemap of an image in device memory
  bvh      cx_scene_build with the device builder on moved geometry, then a first ray query

Scenes are the repository's own (crisoptix_amd/scenes.py), built once per process as a program
does; cameras, random seeds, rays, entries, images and moved geometry come from the seed.  Work
goes to the null stream, which is torch's default stream.

The library gives the same bits for the same inputs whatever its launch settings: hits, neighbour
sets, reservoir records, radiance and bytes are compared exactly.  Only the adjoint's gradients,
summed in float64 by atomics, have a tolerance.
"""
import ctypes
import math

import numpy as np
import torch

from crisoptix_amd import abi, runtime, scenes

# ------------------------------------------------------------------------------------------
# The cases
# ------------------------------------------------------------------------------------------

MAX_FRAME_COST = 1920 * 1080 * (6 + 8)   # pixels x (rays of the walks + shifted suffixes), about


def listed():
    return [
        # the headline workload: 1080p Conditional ReSTIR, 1.06 M triangles, orbiting camera
        _frame("conditional_1080p", "conditional_restir", 1920, 1080, grid=16),
        # an odd-sized view of a textured scene with two gather prefixes, 16 gathered suffixes and
        # prefix spatial reuse: the options of the renderer's panel away from their defaults
        _frame("conditional_odd_textured", "conditional_restir", 717, 403, grid=10, gather_m=17, gather_n=2,
               prefix_spatial=2, textured=True),
        # a thumbnail: every pass is a handful of wavefronts, launches and gaps are the time
        _frame("conditional_160x90", "conditional_restir", 160, 90, grid=4),
        # the smallest benchmark configuration: ReSTIR PT on the Cornell box, static camera,
        # progressive accumulation
        _frame("restir_pt_256", "restir_pt_cornell", 256, 256, grid=0, accum=True),
        # the reference estimator, 8 vertices, progressive preview at 720p
        _frame("path_tracer_720p", "path_tracer", 1280, 720, grid=16, accum=True),
        # gradient step of the differentiable-rendering configuration: 96 k triangles, 65
        # materials, forward and backward
        {"name": "inverse_512", "kind": "inverse", "mode": "restir_pt_cornell", "width": 512, "height": 512},
        # several viewports of uneven size over three scenes in one enqueue
        {"name": "batch_6_views", "kind": "batch", "views": 6, "spec": 31, "largest": 1.0},
        # baking and picking: ray arrays answered by the traversal entry points
        {"name": "trace_2m", "kind": "trace", "grid": 16, "rays": 2_000_000, "bvh_width": 4},
        {"name": "trace_4k", "kind": "trace", "grid": 0, "rays": 4096, "bvh_width": 4},
        # the prefix-entry search of a 1080p frame through its own entry points
        {"name": "entries_1080p", "kind": "entries", "slots": 1920 * 1080, "queries": 547_060, "k": 8,
         "static": False},
        # display output of a 4K image
        {"name": "tonemap_4k", "kind": "tonemap", "width": 3840, "height": 2160},
        # animated geometry: device build of the 1.06 M-triangle scene and a first query
        {"name": "bvh_1m", "kind": "bvh", "grid": 16, "rays": 65_536, "bvh_width": 4},
    ]


def _frame(name, mode, width, height, grid, gather_m=9, gather_n=1, prefix_spatial=0, accum=False, textured=False,
           bvh_width=4):
    case = {"kind": "frame", "mode": mode, "width": width, "height": height, "grid": grid, "gather_m": gather_m,
            "gather_n": gather_n, "prefix_spatial": prefix_spatial, "accum": accum, "textured": textured,
            "bvh_width": bvh_width}
    return dict(case, name=name) if name else case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: sizes over their logarithm, odd ones among them."""
    kind = rng.choice(["frame"] * 5 + ["inverse", "batch", "trace", "trace", "entries", "entries", "tonemap", "bvh"])
    if kind == "frame":
        mode = rng.choice(["conditional_restir"] * 3 + ["restir_pt_cornell", "path_tracer"])
        cond = mode == "conditional_restir"
        aspect = rng.uniform(0.8, 2.0)
        m, n = (rng.randint(1, 32), rng.choice([1, 1, 2])) if cond else (9, 1)
        pixels = _log(rng, 64 * 48, 1920 * 1080)
        pixels = min(pixels, int(0.9 * MAX_FRAME_COST / (6 + (m - 1) * n)))
        w = max(8, int(math.sqrt(pixels * aspect)))
        return _frame(None, mode, w, max(8, pixels // w), grid=rng.choice([0, 4, 8, 10, 16]), gather_m=m, gather_n=n,
                      prefix_spatial=rng.choice([0, 0, 1, 3]), accum=not cond and rng.random() < 0.5,
                      textured=rng.random() < 0.3, bvh_width=rng.choice([4, 4, 4, 2, 8]))
    if kind == "inverse":
        w = _log(rng, 64, 640)
        return {"kind": "inverse", "mode": rng.choice(["restir_pt_cornell", "path_tracer"]), "width": w,
                "height": max(8, int(w * rng.uniform(0.6, 1.1)))}
    if kind == "batch":
        return {"kind": "batch", "views": rng.randint(2, 6), "spec": rng.randint(100, 10**6),
                "largest": rng.uniform(0.05, 0.6)}
    if kind == "trace":
        return {"kind": "trace", "grid": rng.choice([0, 4, 8, 16]), "rays": _log(rng, 257, 1_900_000),
                "bvh_width": rng.choice([4, 4, 2, 8])}
    if kind == "entries":
        slots = _log(rng, 500, 1_900_000)
        return {"kind": "entries", "slots": slots, "queries": max(1, int(slots * rng.uniform(0.1, 0.4))),
                "k": rng.choice([1, 8, 8, 16, 31]), "static": slots <= 65536 and rng.random() < 0.5}
    if kind == "tonemap":
        w = _log(rng, 64, 3840)
        return {"kind": "tonemap", "width": w, "height": max(1, int(w * rng.uniform(0.4, 0.56)))}
    return {"kind": "bvh", "grid": rng.randint(2, 15), "rays": _log(rng, 1000, 65_536),
            "bvh_width": rng.choice([4, 4, 2, 8])}


# ------------------------------------------------------------------------------------------
# What a program has before the call
# ------------------------------------------------------------------------------------------

_kept = {}


def _keep(key, make):
    """One context and one copy of each scene per process, as a program holds them."""
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _ctx():
    return _keep("ctx", lambda: runtime.Context(0))


def _host_scene(grid, textured=False, batch_seed=False):
    """grid 0: the Cornell box; otherwise grid x grid objects under the tent of lights."""
    def make():
        if grid == 0:
            sc = scenes.cornell_box(1, 8)
        elif batch_seed:
            sc = scenes.object_grid(grid, seed=20 + grid, ground_quads=10 * grid)
        else:
            sc = scenes.object_grid(grid, 2, ground_quads=200 if grid == 16 else 10 * grid)
        return scenes.with_textures(sc) if textured else sc
    return _keep(("host", grid, textured, batch_seed), make)


def _scene(grid, bvh_width=4, textured=False, batch_seed=False):
    return _keep(("scene", grid, bvh_width, textured, batch_seed),
                 lambda: runtime.Scene(_ctx(), _host_scene(grid, textured, batch_seed), width=bvh_width))


def _inverse_scene(width, height):
    """The differentiable-rendering scene, one per size: its material tables change per step."""
    return _keep(("inverse", width, height), lambda: runtime.Scene(_ctx(), _keep("inverse host", scenes.inverse_scene)))


class _View:
    """Device memory of the library as an int32 torch tensor, without a copy; the tensor's storage
    holds this object, and with it the owner of the memory."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<i4", "data": (ptr, False), "version": 2,
                                         "strides": None}

    @staticmethod
    def tensor(owner, ptr, shape):
        return torch.as_tensor(_View(owner, ptr, shape), device="cuda")


def _orbit(scene, width, height, start, count=64):
    cam = scenes.orbit_camera(scene, width, height)
    cam.rotate_around_origin([0, 1, 0], start)
    out = []
    for _ in range(count):
        cam.rotate_around_origin([0, 1, 0], 2 * math.pi / 64)
        out.append(abi.CameraData.from_dict(cam.data()))
    return cam, out


def _camera(case, host, rng):
    """(camera, its data per frame): orbiting, or still for the Cornell box and accumulation."""
    if case["grid"] == 0:
        cam = scenes.cornell_camera(case["width"], case["height"])
        cam.pos = cam.pos + rng.uniform(-0.05, 0.05, 3).astype(np.float32)
        return cam, [abi.CameraData.from_dict(cam.data())]
    cam, cams = _orbit(host, case["width"], case["height"], rng.uniform(0, 2 * math.pi))
    return cam, cams[:1] if case["accum"] else cams


def _frame_params(case, size):
    p = abi.workload_params(case["mode"], case["width"], case["height"], size)
    p.enableAccum = 1 if case["accum"] else 0
    p.gatherM, p.gatherN = case["gather_m"], case["gather_n"]
    if case["prefix_spatial"]:
        p.prefixEnableSpatial, p.prefixSpatialCount = 1, case["prefix_spatial"]
    return p


def _prepare_frame(case, seed):
    rng = np.random.default_rng(seed)
    host = _host_scene(case["grid"], case["textured"])
    gs = _scene(case["grid"], case["bvh_width"], case["textured"])
    cam, cams = _camera(case, host, rng)
    W, H = case["width"], case["height"]
    ren = runtime.Renderer(W, H, _ctx(), cam, gs, params=_frame_params(case, gs.size), seed=seed)
    out = torch.zeros((H, W, 3), dtype=torch.float32, device="cuda")
    v = ren.state()
    st = {"ren": ren, "cams": cams, "moving": len(cams) > 1, "i": 0, "out": out, "optr": runtime.DevicePtr(out.data_ptr())}
    # the reservoirs a frame leaves behind, whole: 9 and 7 words of 16 bytes a pixel
    if case["mode"] != "path_tracer":
        st["prefix"] = [_View.tensor(ren, v.prefixRes[b], (abi.PREFIX_CHUNKS, H * W, 4)) for b in (0, 1)]
    if case["mode"] == "conditional_restir":
        st["suffix"] = [_View.tensor(ren, v.suffixRes[b], (abi.SUFFIX_CHUNKS, H * W, 4)) for b in (0, 1)]
    for _ in range(2):   # a running program has a history to reuse
        _run_frame(st)
    return st


def _run_frame(st):
    ren, i = st["ren"], st["i"]
    st["i"] = i + 1
    ren.launch_frame(st["cams"][i % len(st["cams"])], st["moving"] or i == 0, output=st["optr"])
    res = {"image": st["out"]}
    if "prefix" in st:
        front = (i + 1) & 1   # the buffers swap every frame; the first one writes buffer 1
        res["prefix"] = st["prefix"][front]
        if "suffix" in st:
            res["suffix"] = st["suffix"][front]
    return res


def _prepare_inverse(case, seed):
    rng = np.random.default_rng(seed)
    W, H = case["width"], case["height"]
    gs = _inverse_scene(W, H)
    host = gs.host
    cam, cams = _orbit(host, W, H, rng.uniform(0, 2 * math.pi), 1)
    p = abi.workload_params(case["mode"], W, H, gs.size)
    p.maxPathLen = 4
    ren = runtime.Renderer(W, H, _ctx(), cam, gs, params=p, seed=seed)
    ren.set_device_random(True, seed)
    M = host.materials.shape[0]
    rows = scenes.perturbed_materials(host.materials, seed=seed)
    f64 = dict(dtype=torch.float64, device="cuda")
    f32 = dict(dtype=torch.float32, device="cuda")
    E = host.emitter_color.shape[0]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    st = {"gs": gs, "ren": ren, "cam": cams[0], "M": M, "rows": torch.from_numpy(rows).to("cuda"),
          "target": 0.05 * torch.rand((H, W, 3), generator=gen, **f32), "img": torch.zeros((H, W, 3), **f32),
          "img2": torch.zeros((H, W, 3), **f32), "dl": torch.zeros((H, W, 3), **f32),
          "zero": torch.zeros((), **f32), "scale": 2.0 / (3 * W * H), "gA": torch.zeros((M, 3), **f64),
          "gR": torch.zeros(M, **f64), "gE": torch.zeros((E, 3), **f64)}
    _run_inverse(st)
    return st


def _run_inverse(st):
    """The per-view work of crisoptix_amd.inverse.DeviceStep.step."""
    ren, cam = st["ren"], st["cam"]
    st["gs"].set_materials_device(st["rows"].data_ptr(), st["M"])
    for k in ("gA", "gR", "gE"):
        st[k].zero_()
    ren.reset()
    ren.launch_frame(cam, False, output=runtime.DevicePtr(st["img"].data_ptr()))
    torch.where(st["img"] <= 10.0, (st["img"] - st["target"]) * st["scale"], st["zero"], out=st["dl"])
    ren.reset()
    ren.launch_frame(cam, False, output=runtime.DevicePtr(st["img2"].data_ptr()))
    ren.adjoint(st["dl"].data_ptr(), st["gA"].data_ptr(), st["gR"].data_ptr(), st["gE"].data_ptr())
    return {"image": st["img"], "image2": st["img2"], "dL_dI": st["dl"], "albedo": st["gA"], "roughness": st["gR"],
            "emission": st["gE"]}


BATCH_GRIDS = (4, 10, 24)


def _batch_views(case):
    """Resolutions between 352 x 256 and 1912 x 1072 (`largest` scales the upper end) over the
    three scenes, as crisoptix_amd.batch.view_specs draws them."""
    rng = np.random.default_rng(case["spec"])
    out = []
    for _ in range(case["views"]):
        t = float(rng.random()) * case["largest"]
        w, h = (int(round((320 + 1600 * t) / 8)) * 8, int(round((240 + 840 * t) / 8)) * 8)
        out.append((int(rng.integers(0, len(BATCH_GRIDS))), w, h))
    return out


def _prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    rens, cams, outs = [], [], []
    for i, (s, w, h) in enumerate(_batch_views(case)):
        host, gs = _host_scene(BATCH_GRIDS[s], batch_seed=True), _scene(BATCH_GRIDS[s], batch_seed=True)
        cam, orbit = _orbit(host, w, h, rng.uniform(0, 2 * math.pi), 16)
        p = abi.workload_params("conditional_restir", w, h, gs.size)
        p.maxPathLen = 6
        ren = runtime.Renderer(w, h, _ctx(), cam, gs, params=p, seed=seed * 64 + i)
        ren.set_overlap(False)
        out = torch.zeros((h, w, 3), dtype=torch.float32, device="cuda")
        ren.output = runtime.DevicePtr(out.data_ptr())
        rens.append(ren)
        cams.append(orbit)
        outs.append(out)
    st = {"batch": runtime.Batch(_ctx(), rens), "cams": cams, "outs": outs, "i": 0}
    torch.cuda.synchronize()   # the pool's streams read what the null stream cleared
    _run_batch(st)
    return st


def _run_batch(st):
    i = st["i"]
    st["i"] = i + 1
    st["batch"].frame([c[i % len(c)] for c in st["cams"]], [True] * len(st["cams"]))
    st["batch"].sync()
    return st["outs"]


def _rays(host, n, gen, rng, grid):
    """Half camera rays in scan order, half rays from points in the scene in any direction, as
    picking and baking make them; [n][8] = origin, direction, tmin, tmax."""
    dev = dict(dtype=torch.float32, device="cuda")
    r = torch.empty((n, 8), **dev)
    h = n // 2
    w = max(1, int(math.sqrt(max(1, h))))
    cam = scenes.cornell_camera(w, w) if grid == 0 else _orbit(host, w, w, rng.uniform(0, 2 * math.pi), 1)[0]
    d = {k: torch.from_numpy(np.asarray(v, np.float32)).to("cuda") for k, v in cam.data().items()}
    i = torch.arange(h, device="cuda")
    jit = torch.rand((h, 2), generator=gen, **dev)
    u = ((i % w) + jit[:, 0]) / w * 2 - 1
    v = (torch.div(i, w, rounding_mode="floor") + jit[:, 1]) / w * 2 - 1
    r[:h, 0:3] = d["pos"]
    r[:h, 3:6] = torch.nn.functional.normalize(u[:, None] * d["U"] + v[:, None] * d["V"] + d["W"], dim=1)
    lo, hi = ((-0.9, 0.1, -2.9), (0.9, 1.9, 0.9)) if grid == 0 else \
        ((-1.8 * grid, 0.02, -1.8 * grid), (1.8 * grid, 3.0, 1.8 * grid))
    lo, hi = torch.tensor(lo, **dev), torch.tensor(hi, **dev)
    r[h:, 0:3] = lo + (hi - lo) * torch.rand((n - h, 3), generator=gen, **dev)
    r[h:, 3:6] = torch.nn.functional.normalize(torch.randn((n - h, 3), generator=gen, **dev), dim=1)
    r[:, 6] = 1e-3
    r[:, 7] = 1e16
    return r


def _ray_buffers(n):
    i32, f32 = dict(dtype=torch.int32, device="cuda"), dict(dtype=torch.float32, device="cuda")
    return {"prim": torch.zeros(n, **i32), "t": torch.zeros(n, **f32), "u": torch.zeros(n, **f32),
            "v": torch.zeros(n, **f32), "occluded": torch.zeros(n, **i32)}


def _prepare_trace(case, seed):
    host, gs = _host_scene(case["grid"]), _scene(case["grid"], case["bvh_width"])
    gen, rng = torch.Generator(device="cuda").manual_seed(seed), np.random.default_rng(seed)
    rays = _rays(host, case["rays"], gen, rng, case["grid"])
    # visibility queries between points: the same origins, limited lengths
    short = rays.clone()
    size = 2.0 if case["grid"] == 0 else 4.0 * case["grid"]
    short[:, 7] = size * (0.05 + torch.rand(case["rays"], generator=gen, dtype=torch.float32, device="cuda"))
    return {"gs": gs, "rays": rays, "short": short, "n": case["rays"], **_ray_buffers(case["rays"])}


def _run_trace(st):
    ctx, gs, n = _ctx(), st["gs"], st["n"]
    lib = runtime.lib()
    ctx.check(lib.cx_trace_closest(ctx.h, gs.h, st["rays"].data_ptr(), n, st["prim"].data_ptr(), st["t"].data_ptr(),
                                   st["u"].data_ptr(), st["v"].data_ptr(), None), "cx_trace_closest")
    ctx.check(lib.cx_trace_occluded(ctx.h, gs.h, st["short"].data_ptr(), n, st["occluded"].data_ptr(), None),
              "cx_trace_occluded")
    return {k: st[k] for k in ("prim", "t", "u", "v", "occluded")}


def _prepare_entries(case, seed):
    """Points as last prefix vertices lie: on the ground, on the objects and on the tent's faces
    of the 16 x 16 grid (half-width 36), with the search radius of the frames (1 % of the scene's
    size, scaled by path length / 4.5); a third of the slots are valid."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dev = dict(dtype=torch.float32, device="cuda")
    n, nq = case["slots"], case["queries"]

    def points(m):
        p = torch.empty((m, 3), **dev)
        p[:, 0::2] = (torch.rand((m, 2), generator=gen, **dev) * 2 - 1) * 30.0
        p[:, 1] = 0.0
        which = torch.rand(m, generator=gen, **dev)
        cell = torch.randint(0, 16, (m, 2), generator=gen, device="cuda").float()
        s = 0.3 + 1.2 * ((cell[:, 0] * 16 + cell[:, 1]) * 0.618034 % 1.0)
        c = torch.stack([(cell[:, 0] - 7.5) * 4.0, s, (cell[:, 1] - 7.5) * 4.0], 1)
        d = torch.nn.functional.normalize(torch.randn((m, 3), generator=gen, **dev), dim=1)
        p = torch.where((which < 0.4)[:, None], c + s[:, None] * d, p)
        up = 36.0 * torch.rand(m, generator=gen, **dev)
        a = 2 * math.pi * torch.rand(m, generator=gen, **dev)
        tent = torch.stack([(36.0 - up) * torch.cos(a), up, (36.0 - up) * torch.sin(a)], 1)
        return torch.where((which > 0.8)[:, None], tent, p).contiguous()

    pos, q = points(n), points(nq)
    radius = 1.1 * (20.0 + 50.0 * torch.rand(n, generator=gen, **dev)) / 4.5
    valid = (torch.rand(n, generator=gen, **dev) < 0.355).to(torch.uint8)
    k = case["k"]
    st = {"n": n, "nq": nq, "k": k, "pos": pos, "radius": radius, "valid": valid, "q": q, "static": case["static"],
          "idx": torch.zeros((nq, k), dtype=torch.int32, device="cuda"), "dist": torch.zeros((nq, k), **dev),
          "count": torch.zeros(nq, dtype=torch.int32, device="cuda"),
          "mn": (ctypes.c_float * 3)(-36.0, 0.0, -36.0), "mx": (ctypes.c_float * 3)(36.0, 36.0, 36.0)}
    if not case["static"]:
        st["entries"] = runtime.Entries(_ctx(), n)
    return st


def _run_entries(st):
    ctx, lib = _ctx(), runtime.lib()
    mn, mx = ctypes.addressof(st["mn"]), ctypes.addressof(st["mx"])
    src = (st["pos"].data_ptr(), st["radius"].data_ptr(), st["valid"].data_ptr(), st["n"], mn, mx)
    dst = (st["q"].data_ptr(), st["nq"], st["k"], st["idx"].data_ptr(), st["dist"].data_ptr(), st["count"].data_ptr())
    if st["static"]:
        ctx.check(lib.cx_entries_search_static(ctx.h, *src, *dst, None), "cx_entries_search_static")
    else:
        ctx.check(lib.cx_entries_build(ctx.h, st["entries"].h, *src, None), "cx_entries_build")
        ctx.check(lib.cx_entries_query(ctx.h, st["entries"].h, *dst, None), "cx_entries_query")
    return {"idx": st["idx"], "dist": st["dist"], "count": st["count"]}


def _prepare_tonemap(case, seed):
    """Radiance as frames hold it: lognormal over several stops, unlit pixels, overexposed ones."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["height"], case["width"], 3)
    hdr = torch.exp(1.5 * torch.randn(shape, generator=gen, dtype=torch.float32, device="cuda") - 1.5)
    dark = torch.rand(shape[:2] + (1,), generator=gen, dtype=torch.float32, device="cuda") < 0.1
    hdr = torch.where(dark, torch.zeros_like(hdr), hdr).contiguous()
    return {"hdr": hdr, "ldr": torch.zeros(shape, dtype=torch.uint8, device="cuda"), "n": hdr.numel()}


def _run_tonemap(st):
    ctx = _ctx()
    ctx.check(runtime.lib().cx_tonemap(ctx.h, st["hdr"].data_ptr(), st["ldr"].data_ptr(), st["n"], None), "cx_tonemap")
    return st["ldr"]


def _prepare_bvh(case, seed):
    """The scene's geometry turned about the vertical axis and stretched a little, as host arrays."""
    rng = np.random.default_rng(seed)
    host = _host_scene(case["grid"])
    a, s = rng.uniform(0, 2 * math.pi), rng.uniform(0.95, 1.05, 3)
    c, n = math.cos(a), math.sin(a)
    rot = np.asarray([[c, 0, n], [0, 1, 0], [-n, 0, c]], np.float32)
    pos = np.ascontiguousarray((host.positions @ rot.T) * s.astype(np.float32), np.float32)
    moved = scenes.Scene(**{**host.__dict__, "positions": pos,
                            "normals": np.ascontiguousarray(host.normals @ rot.T, np.float32)})
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rays = _rays(host, case["rays"], gen, rng, case["grid"])
    return {"host": moved, "bvh_width": case["bvh_width"], "rays": rays, "short": rays, "n": case["rays"],
            **_ray_buffers(case["rays"])}


def _run_bvh(st):
    st["gs"] = runtime.Scene(_ctx(), st["host"], width=st["bvh_width"], builder="device")
    return _run_trace(st)


_PREPARE = {"frame": _prepare_frame, "inverse": _prepare_inverse, "batch": _prepare_batch, "trace": _prepare_trace,
            "entries": _prepare_entries, "tonemap": _prepare_tonemap, "bvh": _prepare_bvh}
_RUN = {"frame": _run_frame, "inverse": _run_inverse, "batch": _run_batch, "trace": _run_trace,
        "entries": _run_entries, "tonemap": _run_tonemap, "bvh": _run_bvh}


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, int(seed)), kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)


# ------------------------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is
# ------------------------------------------------------------------------------------------

def _triangles(grid):
    if grid == 0:
        return 2304
    return int(grid * grid * (0.75 * 5120 + 0.25 * 12)) + 2 * (200 if grid == 16 else 10 * grid) ** 2 + 16


def _scene_bytes(t):
    return 28 * t   # positions and normals (half a vertex a triangle), indices, material ids


def _ray_flops(t):
    """One ray down a 4-wide tree to one triangle: box tests of 4 children a level, one triangle."""
    return 4 * 20 * math.ceil(math.log(max(t, 4), 4)) + 60


def work(case):
    kind = case["kind"]
    if kind in ("frame", "inverse"):
        px = case["width"] * case["height"]
        t = 95_760 if kind == "inverse" else _triangles(case["grid"])
        if case["mode"] == "conditional_restir":   # both reservoirs, the pixel's state, the image; rays measured
            per, rays = (9 + 7 + 1) * 16 * 2 + 12, 6.0 + 1.0 * (case["gather_m"] - 1) * case["gather_n"]
        elif case["mode"] == "restir_pt_cornell":
            per, rays = (9 + 1) * 16 * 2 + 12, 8.0
        else:
            per, rays = 12 + (12 if case.get("accum") else 0), 6.0
        if kind == "inverse":   # two frames from a reset history, dL/dI and the replay of the second
            record = 160 if case["mode"] == "restir_pt_cornell" else 0
            return {"bytes": px * (2 * 12 + 2 * record + 48) + _scene_bytes(t), "flops": 3 * rays * px * _ray_flops(t)}
        return {"bytes": px * per + _scene_bytes(t), "flops": rays * px * _ray_flops(t)}
    if kind == "batch":
        views = _batch_views(case)
        px = sum(w * h for _, w, h in views)
        flops = sum(w * h * 13.0 * _ray_flops(_triangles(BATCH_GRIDS[s])) for s, w, h in views)
        return {"bytes": px * ((9 + 7 + 1) * 16 * 2 + 12) +
                sum(_scene_bytes(_triangles(BATCH_GRIDS[s])) for s in {v[0] for v in views}), "flops": flops}
    if kind == "trace":
        t = _triangles(case["grid"])
        return {"bytes": case["rays"] * (48 + 36) + 40 * t, "flops": 2 * case["rays"] * _ray_flops(t)}
    if kind == "entries":
        n, nq, k = case["slots"], case["queries"], case["k"]
        return {"bytes": 17 * n + nq * (12 + 8 * k + 4), "flops": 10.0 * nq * (k + math.log2(n + 2) * 4)}
    if kind == "tonemap":
        return {"bytes": 5 * 3 * case["width"] * case["height"], "flops": 20.0 * 3 * case["width"] * case["height"]}
    t = _triangles(case["grid"])   # geometry in, a tree of two boxes a triangle out, rays
    return {"bytes": _scene_bytes(t) + t * (48 + 64) + case["rays"] * (48 + 36),
            "flops": 60.0 * t * math.log2(t + 2) + 2 * case["rays"] * _ray_flops(t)}


def tolerance(case):
    if case["kind"] == "inverse":
        # float64 sums of about a million 32-bit terms in an order of their own per run: measured
        # 5e-16 apart; other groupings of the 32-bit terms stay below this
        return {"rel": 1e-7, "max": 1e-5}
    return "exact"


def exact(case, seed):
    """Distances and hits in 64 bits where every pair can be tried; frames, gradients and bytes
    follow decisions taken in 32 bits and have no such value."""
    if case["kind"] == "trace" and case["grid"] == 0 and case["rays"] <= 200_000:
        gen, rng = torch.Generator(device="cuda").manual_seed(int(seed)), np.random.default_rng(int(seed))
        host = _host_scene(0)
        r = _rays(host, case["rays"], gen, rng, 0).double()
        tri = torch.from_numpy(host.positions[host.indices.astype(np.int64)]).to("cuda").double()
        best_t = []
        for part in r.split(2048):
            o, d = part[:, None, 0:3], part[:, None, 3:6]
            e1, e2 = tri[None, :, 1] - tri[None, :, 0], tri[None, :, 2] - tri[None, :, 0]
            pv = torch.linalg.cross(d.expand(-1, len(tri), -1), e2.expand(len(part), -1, -1))
            det = (e1 * pv).sum(-1)
            tv = o - tri[None, :, 0]
            u = (tv * pv).sum(-1) / det
            qv = torch.linalg.cross(tv, e1.expand(len(part), -1, -1))
            v = (d * qv).sum(-1) / det
            t = (e2 * qv).sum(-1) / det
            ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 1e-3) & (det != 0)
            t = torch.where(ok, t, torch.inf).min(1).values
            best_t.append(torch.where(torch.isfinite(t), t, 0.0))
        # the boxes stand on the floor: which of two coplanar triangles is hit, and so its u and v,
        # is a matter of 32-bit rounding
        return {"prim": None, "t": torch.cat(best_t), "u": None, "v": None, "occluded": None}
    if case["kind"] == "entries" and case["slots"] * case["queries"] <= 4_000_000_000:
        st = _prepare_entries(dict(case, static=True), int(seed))
        pos, ok = st["pos"].double(), st["valid"].bool()
        r = torch.where(ok, st["radius"].double(), -1.0)
        k = case["k"]
        dist = torch.zeros((st["nq"], k), dtype=torch.float64, device="cuda")
        step = max(1, 200_000_000 // case["slots"])
        for a in range(0, st["nq"], step):
            q = st["q"][a:a + step].double()
            d2 = sum((q[:, None, c] - pos[None, :, c]) ** 2 for c in range(3))
            d = torch.where(d2.sqrt_() <= r[None, :], d2, torch.inf)
            best = d.topk(min(k, case["slots"]), dim=1, largest=False, sorted=True).values
            dist[a:a + step, :best.shape[1]] = torch.where(torch.isfinite(best), best, 0.0)
        return {"idx": None, "dist": dist, "count": None}
    return None
