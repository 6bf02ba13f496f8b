"""The calls that a program built on this framework spends its time in, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" says which entry points it goes through:

  frame   cluster_and_shade of one frame at a time (Batch.PER_FRAME): an interactive renderer's call, where the
          latency of a frame counts. Default configuration, as the benchmark's plain path.
  stages  the four stages called one by one (light BVH, unique clusters, light assignment, shade), as the drop-in
          C++ classes do, with the other options: tight cluster boxes, 30-bit Morton codes, the smooth attenuation, a
          directional light.
  batch   cluster_and_shade of many equal frames in one graph replay: offline and served rendering, the benchmark's
          headline. With "materials" the shade resolves textures; with "sliced" the 32-slice x 6-face keys.
  mixed   the same over frames of different sizes and light counts (640x360 to 3840x2160, 256 to 65536 lights).
  train   one step of an optimiser on light and material parameters: the differentiable shade and its gradients.
  sort    the in-place radix sort of keys, or of keys with values, on some of their bits (32: all; 30 and 15: Morton
          codes); the keys are copied into place first, since a sorted array is not what a program sorts.
  bucket  the counting sort of (key, value) pairs into buckets, with the bucket starts.
  scan    an exclusive prefix sum, in one or several segments.
  reduce  the up-sweep tree of a sum, a minimum or a maximum.

Frames, lights, materials and keys come from the library's own seeded generators (procedural scenes of boxes on a
ground plane, lights of radius 1 to 8 in a 100^3 volume) and from torch's, on the device.
"""
import ctypes
import math

import numpy as np
import torch

import vren_amd
from vren_amd.autograd import ShadeFrame, shade

RESOLUTIONS = [(640, 360), (1280, 720), (1920, 1080), (2560, 1440), (3840, 2160)]
NEAR, FAR = 0.1, 100.0
# frames of the largest batch: what a drawn batch's pixels are held under
MOST_PIXELS = 64 * 1920 * 1080


def listed():
    return [
        # the smallest frame of the mixed workload with its fewest lights: launches and latency are all of it
        {"name": "frame_640x360_256", "kind": "frame", "width": 640, "height": 360, "lights": 256},
        # the ordinary frame
        {"name": "frame_1080p_4096", "kind": "frame", "width": 1920, "height": 1080, "lights": 4096},
        # the largest frame with the most lights of the mixed workload
        {"name": "frame_4k_65536", "kind": "frame", "width": 3840, "height": 2160, "lights": 65536},
        # a ragged screen (neither side a multiple of 32, rows that do not start on 16 bytes) through the stage calls
        {"name": "stages_1366x769_1000", "kind": "stages", "width": 1366, "height": 769, "lights": 1000},
        # the benchmark's batch
        {"name": "batch_64x1080p_4096", "kind": "batch", "frames": 64, "width": 1920, "height": 1080, "lights": 4096,
         "materials": False, "sliced": False},
        # textured materials and the coarser key encoder
        {"name": "batch_16x1080p_materials", "kind": "batch", "frames": 16, "width": 1920, "height": 1080,
         "lights": 4096, "materials": True, "sliced": True},
        # frames of every size in one batch
        {"name": "mixed_32", "kind": "mixed", "frames": 32, "mix": 4444, "ragged": False},
        # one optimiser step on a 1080p frame
        {"name": "train_1080p_4096", "kind": "train", "width": 1920, "height": 1080, "lights": 4096},
        # the sort benchmark
        {"name": "sort_pairs_2p26", "kind": "sort", "n": 1 << 26, "values": True, "bits": 32, "spread": "uniform"},
        # a sort of the size that a frame's own work lists have
        {"name": "sort_pairs_100003", "kind": "sort", "n": 100003, "values": True, "bits": 32, "spread": "uniform"},
        # the reference's 65536 buckets
        {"name": "bucket_2p24", "kind": "bucket", "n": 1 << 24, "buckets": 65536},
        # a prefix sum over a buffer larger than the caches
        {"name": "scan_2p26", "kind": "scan", "n": 1 << 26, "blocks": 1},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _screen(rng, most=3840 * 2160):
    """A screen of 640x360 to 3840x2160: one in three of the common sizes, else any width and height."""
    if rng.random() < 0.34:
        w, h = rng.choice([r for r in RESOLUTIONS if r[0] * r[1] <= most])
    else:
        w = _log_uniform(rng, 640, min(3840, math.sqrt(most * 16 / 9)))
        h = min(max(360, int(w * rng.uniform(0.5, 0.6))), most // w)
    return w, h


def draw(rng):
    kind = rng.choice(["frame", "frame", "stages", "batch", "batch", "mixed", "train", "sort", "sort", "sort", "bucket",
                       "scan", "reduce"])
    if kind in ("frame", "stages"):
        w, h = _screen(rng)
        return {"kind": kind, "width": w, "height": h, "lights": _log_uniform(rng, 256, 65536 if kind == "frame" else 8192)}
    if kind == "train":
        w, h = _screen(rng, 1920 * 1080)
        return {"kind": kind, "width": w, "height": h, "lights": _log_uniform(rng, 256, 4096)}
    if kind == "batch":
        w, h = _screen(rng)
        return {"kind": kind, "frames": _log_uniform(rng, 2, max(2, min(64, MOST_PIXELS // (2 * w * h)))), "width": w,
                "height": h, "lights": _log_uniform(rng, 256, 8192), "materials": rng.random() < 0.25,
                "sliced": rng.random() < 0.25}
    if kind == "mixed":
        return {"kind": kind, "frames": _log_uniform(rng, 4, 24), "mix": rng.randrange(1 << 20), "ragged": rng.random() < 0.5}
    if kind == "sort":
        return {"kind": kind, "n": _log_uniform(rng, 1000, 1 << 26), "values": rng.random() < 0.6,
                "bits": rng.choice([32, 32, 30, 15]), "spread": rng.choice(["uniform", "uniform", "clustered"])}
    if kind == "bucket":
        return {"kind": kind, "n": _log_uniform(rng, 1000, 1 << 25), "buckets": 1 << rng.randint(8, 16)}
    if kind == "scan":
        n = _log_uniform(rng, 1000, 1 << 26)
        return {"kind": kind, "n": n, "blocks": rng.choice([1, 1, max(1, min(64, (1 << 26) // n))])}
    return {"kind": kind, "n": _log_uniform(rng, 1000, 1 << 26), "op": rng.choice(["add", "min", "max"])}


# ---- inputs ------------------------------------------------------------------------------------------------------

_context = None


def _ctx():
    """The program's one context (a context is used from one thread and one stream)."""
    global _context
    if _context is None:
        _context = vren_amd.Context(0)
    return _context


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _i32(*shape):
    return torch.zeros(*shape, dtype=torch.int32, device="cuda")


def _camera(w, h):
    c = vren_amd.Camera()
    c.position[2] = -50.0
    c.fov_y = float(np.float32(math.pi / 2))
    c.aspect_ratio = float(np.float32(w) / np.float32(h))
    c.near_plane, c.far_plane = NEAR, FAR
    return c


def _frame_inputs(seed, w, h, lights, resolved=True):
    """G-buffer, lights and per-pixel materials of one frame."""
    ctx, cam = _ctx(), _camera(w, h)
    f = {"cam": cam, "w": w, "h": h, "L": lights, "depth": _f32(w * h),
         "normals": torch.empty(w * h * 4, dtype=torch.int16, device="cuda"), "pos": _f32(lights, 4), "lig": _f32(lights, 4)}
    ctx.synth_frame(seed, w, h, cam, 64, f["depth"], f["normals"])
    ctx.synth_lights(seed + 7, lights, f["pos"], f["lig"])
    if resolved:
        f["ar"], f["metal"] = _f32(w * h, 4), _f32(w * h)
        ctx.synth_materials(seed, w * h, f["ar"], f["metal"])
    return f


def _descriptor(f, out):
    d = vren_amd.FrameDesc()
    d.width, d.height, d.camera = f["w"], f["h"], f["cam"]
    d.depth, d.normals = f["depth"].data_ptr(), f["normals"].data_ptr()
    if "ar" in f:
        d.albedo_roughness, d.metallic = f["ar"].data_ptr(), f["metal"].data_ptr()
    d.light_positions, d.point_lights, d.light_count = f["pos"].data_ptr(), f["lig"].data_ptr(), f["L"]
    d.output = out.data_ptr()
    return d


def _material_tables(seed):
    """Eight materials over six RGBA8 textures of 1x1 to 256x256 texels, in both filters and every address mode."""
    rng = np.random.default_rng(seed)
    texels, tab = [], (vren_amd.Texture * 6)()
    for k, (w, h) in enumerate([(256, 256), (64, 128), (7, 5), (1, 1), (33, 17), (128, 64)]):
        t = torch.from_numpy(rng.integers(0, 256, (h, w, 4), dtype=np.uint8)).cuda()
        texels.append(t)
        tab[k].texels, tab[k].width, tab[k].height = t.data_ptr(), w, h
        tab[k].filter, tab[k].address_u, tab[k].address_v = k % 2, k % 3, (k + 1) % 3
    mats = (vren_amd.Material * 8)()
    for m in range(8):
        mats[m].base_color_texture_idx, mats[m].metallic_roughness_texture_idx = (2 * m) % 6, (2 * m + 1) % 6
        mats[m].metallic_factor, mats[m].roughness_factor = 0.1 * m, 0.3 + 0.08 * m
        for c in range(4):
            mats[m].base_color_factor[c] = 0.5 + 0.05 * c
    raw = [torch.from_numpy(np.frombuffer(bytes(x), np.uint8).copy()).cuda() for x in (mats, tab)]
    return raw[0], raw[1], texels


def _frame_sizes(case):
    """(width, height, lights) of each frame of a case."""
    if case["kind"] != "mixed":
        return [(case["width"], case["height"], case["lights"])] * case.get("frames", 1)
    rng = np.random.default_rng(case["mix"])
    sizes = []
    for _ in range(case["frames"]):
        w, h = RESOLUTIONS[rng.integers(0, len(RESOLUTIONS))]
        if case["ragged"]:
            w, h = w - int(rng.integers(0, 64)), h - int(rng.integers(0, 36))
        sizes.append((w, h, int(round(float(np.exp(rng.uniform(np.log(256.0), np.log(65536.0))))))))
    return sizes


def _prepare_batch(case, seed):
    state = {"frames": [], "keep": []}
    materials = case.get("materials", False)
    cfg = vren_amd.default_cfg(**({"key_mode": vren_amd.KEYS_SLICED} if case.get("sliced") else {}))
    sizes = _frame_sizes(case)
    out = torch.zeros(sum(w * h for w, h, _ in sizes), 4, dtype=torch.float32, device="cuda")
    tables = _material_tables(seed) if materials else None
    descs, at = [], 0
    for k, (w, h, lights) in enumerate(sizes):
        f = _frame_inputs(64 * seed + k, w, h, lights, resolved=not materials)
        d = _descriptor(f, out[at:at + w * h])
        at += w * h
        if materials:
            gy, gx = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
            f["tc"] = torch.stack([gx.reshape(-1) / w * 3.0 - 1.0, gy.reshape(-1) / h * 2.5 - 0.7], dim=1).float().contiguous()
            f["mi"] = ((gx // 97 + gy // 61 + k) % 8).reshape(-1).to(torch.int16).contiguous()
            ms = vren_amd.MaterialSet()
            ms.texcoords, ms.material_indices = f["tc"].data_ptr(), f["mi"].data_ptr()
            ms.materials, ms.material_count = tables[0].data_ptr(), 8
            ms.textures, ms.texture_count = tables[1].data_ptr(), 6
            d.materials = ctypes.pointer(ms)
            state["keep"].append(ms)
        descs.append(d)
        state["frames"].append(f)
    torch.cuda.synchronize()
    state["keep"].append(tables)
    state["out"] = out
    state["batch"] = vren_amd.Batch(_ctx(), descs, cfg)
    state["mode"] = vren_amd.Batch.PER_FRAME if case["kind"] == "frame" else vren_amd.Batch.GRAPH
    return state


def _stage_buffers(f, key_cap, index_cap):
    lib = _ctx().lib
    L = f["L"]
    return {"key_cap": key_cap, "index_cap": index_cap, "view_pos": _f32(L, 4), "codes": _i32(L, 2),
            "bvh": _i32(lib.vren_calc_bvh_buffer_length(L), 8), "keys": _i32(key_cap), "count": _i32(1),
            "refs": _i32(f["w"] * f["h"]), "counts": _i32(key_cap), "offsets": _i32(key_cap), "indices": _i32(index_cap),
            "total": _i32(1)}


def _light_lists(f, b, cfg):
    """The three stages that give every pixel its light list."""
    ctx = _ctx()
    ctx.construct_point_light_bvh(f["pos"], f["lig"], f["L"], f["cam"], cfg, b["view_pos"], b["codes"], b["bvh"])
    ctx.find_unique_cluster_list(f["w"], f["h"], f["cam"], cfg, f["depth"], f["normals"], b["keys"], b["key_cap"],
                                 b["count"], b["refs"])
    ctx.assign_lights(f["w"], f["h"], f["cam"], cfg, b["keys"], b["count"], b["key_cap"], b["bvh"], f["L"], b["codes"],
                      b["view_pos"], b["counts"], b["offsets"], b["indices"], b["index_cap"], b["total"])


def _stages_cfg():
    return vren_amd.default_cfg(cluster_aabb_mode=vren_amd.CLUSTER_AABB_TIGHT, morton_bits=10,
                                attenuation=vren_amd.ATTEN_SMOOTH)


def _prepare_stages(case, seed):
    f = _frame_inputs(seed, case["width"], case["height"], case["lights"])
    b = _stage_buffers(f, 1 << 17, 1 << 23)
    g = torch.Generator(device="cuda").manual_seed(seed)
    sun = torch.zeros(2, 4, device="cuda")
    sun[0, :3] = torch.nn.functional.normalize(torch.tensor([0.3, -1.0, 0.5], device="cuda") +
                                               0.1 * torch.rand(3, device="cuda", generator=g), dim=0)
    sun[1, :3] = torch.rand(3, device="cuda", generator=g)
    return {"f": f, "b": b, "cfg": _stages_cfg(), "sun": sun,
            "out": torch.zeros(f["w"] * f["h"], 4, dtype=torch.float32, device="cuda")}


def _prepare_train(case, seed):
    f = _frame_inputs(seed, case["width"], case["height"], case["lights"])
    b = _stage_buffers(f, 1 << 18, 1 << 22)
    _light_lists(f, b, vren_amd.default_cfg())
    smooth = vren_amd.default_cfg(attenuation=vren_amd.ATTEN_SMOOTH)
    frame = ShadeFrame(_ctx(), f["w"], f["h"], f["cam"], smooth, f["depth"], f["normals"], f["metal"], b["refs"],
                       b["key_cap"], b["counts"], b["offsets"], b["indices"], b["index_cap"])
    g = torch.Generator(device="cuda").manual_seed(seed)
    target = torch.rand(f["w"] * f["h"], 4, device="cuda", generator=g)
    return {"f": f, "b": b, "frame": frame, "target": target,
            "params": [f[k].clone().requires_grad_(True) for k in ("pos", "lig", "ar")]}


def _keys(n, seed, bits, spread):
    """n random keys below 2^bits: uniform, or clustered around a few centres as the keys of neighbouring pixels are."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if spread == "uniform":
        k = torch.randint(0, 1 << bits, (n,), device="cuda", generator=g, dtype=torch.int64)
    else:
        centre = torch.randint(0, 1 << bits, (32,), device="cuda", generator=g, dtype=torch.int64)
        at = torch.randint(0, 32, (n,), device="cuda", generator=g, dtype=torch.int64)
        k = centre[at] + (torch.randn(n, device="cuda", generator=g) * (1 << (bits // 2))).to(torch.int64)
        k &= (1 << bits) - 1
    return torch.where(k >= 1 << 31, k - (1 << 32), k).to(torch.int32)


def _prepare_sort(case, seed):
    n = case["n"]
    keys = _keys(n, seed, case["bits"], case["spread"])
    s = {"n": n, "bits": case["bits"], "keys_in": keys, "keys": torch.empty_like(keys), "vals": None,
         "scratch": torch.empty(_ctx().radix_sort_scratch_bytes(n, case["values"]), dtype=torch.uint8, device="cuda")}
    if case["values"]:
        s["vals_in"] = torch.arange(n, dtype=torch.int32, device="cuda")
        s["vals"] = torch.empty_like(keys)
    return s


def _prepare_bucket(case, seed):
    n = case["n"]
    pairs = torch.stack([_keys(n, seed, 32, "uniform"), torch.arange(n, dtype=torch.int32, device="cuda")], dim=1)
    return {"n": n, "buckets": case["buckets"], "pairs": pairs.contiguous(), "sorted": torch.empty_like(pairs),
            "starts": _i32(case["buckets"])}


def _prepare_scan(case, seed):
    x = _keys(case["n"] * case["blocks"], seed, 32, "uniform")
    return {"n": case["n"], "blocks": case["blocks"], "x": x, "out": torch.empty_like(x)}


def _prepare_reduce(case, seed):
    n = case["n"]
    ops = {"add": vren_amd.REDUCE_ADD, "min": vren_amd.REDUCE_MIN, "max": vren_amd.REDUCE_MAX}
    return {"n": n, "op": ops[case["op"]], "x": _keys(n, seed, 32, "uniform"), "out": _i32(1 << (n - 1).bit_length())}


_PREPARE = {"frame": _prepare_batch, "batch": _prepare_batch, "mixed": _prepare_batch, "stages": _prepare_stages,
            "train": _prepare_train, "sort": _prepare_sort, "bucket": _prepare_bucket, "scan": _prepare_scan,
            "reduce": _prepare_reduce}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


# ---- one pass ----------------------------------------------------------------------------------------------------


def _run_batch(s):
    s["batch"].run(s["mode"])
    return s["out"]


def _run_stages(s):
    f, b = s["f"], s["b"]
    _light_lists(f, b, s["cfg"])
    _ctx().shade(f["w"], f["h"], f["cam"], s["cfg"], f["depth"], f["normals"], f["ar"], f["metal"], b["refs"],
                 b["key_cap"], b["counts"], b["offsets"], b["indices"], b["index_cap"], f["pos"], f["lig"], f["L"],
                 s["out"], s["sun"], 1)
    return {"image": s["out"], "view_pos": b["view_pos"], "codes": b["codes"], "bvh": b["bvh"], "keys": b["keys"],
            "count": b["count"], "refs": b["refs"], "counts": b["counts"], "offsets": b["offsets"],
            "indices": b["indices"], "total": b["total"]}


def _run_train(s):
    image = shade(*s["params"], s["frame"])
    grads = torch.autograd.grad(image, s["params"], grad_outputs=image.detach() - s["target"])
    return {"image": image.detach(), "pos": grads[0], "lights": grads[1], "albedo_roughness": grads[2]}


def _run_sort(s):
    s["keys"].copy_(s["keys_in"])
    if s["vals"] is not None:
        s["vals"].copy_(s["vals_in"])
    _ctx().radix_sort(s["keys"], s["vals"], s["n"], s["scratch"], 0, s["bits"])
    return [s["keys"]] if s["vals"] is None else [s["keys"], s["vals"]]


def _run_bucket(s):
    _ctx().bucket_sort(s["pairs"], s["n"], s["sorted"], s["starts"], s["buckets"], 0)
    return [s["sorted"], s["starts"]]


def _run_scan(s):
    _ctx().exclusive_scan_u32(s["x"], s["out"], s["n"], s["blocks"])
    return s["out"]


def _run_reduce(s):
    _ctx().reduce_u32(s["x"], s["n"], s["out"], s["op"])
    return s["out"]


_RUN = {"frame": _run_batch, "batch": _run_batch, "mixed": _run_batch, "stages": _run_stages, "train": _run_train,
        "sort": _run_sort, "bucket": _run_bucket, "scan": _run_scan, "reduce": _run_reduce}


def run(state):
    return _RUN[state["kind"]](state)


# ---- what a pass cannot do without -------------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("frame", "batch", "mixed", "stages", "train"):
        nbytes = flops = 0
        for w, h, lights in _frame_sizes(case):
            px = w * h
            # depth 4, normal 8, albedo and roughness 16, metallic 4 (or texcoord 8, material index 2) in, radiance 16 out
            nbytes += px * (38 if case.get("materials") else 48) + 32 * lights
            # the view reconstruction and surface terms of a pixel; about 102 operations for each light that reaches
            # it, 2.6 of 4096 lights on average
            flops += px * (150 + 102 * 2.6 * lights / 4096)
            if kind == "train":
                # also the reference 4 and the loss's target 16 in, the material gradient 16 out; the adjoint's two passes
                # over the pairs
                nbytes += px * 36 + 32 * lights
                flops += px * (150 + 350 * 2.6 * lights / 4096)
        return {"bytes": nbytes, "flops": flops}
    n = case["n"]
    if kind == "sort":
        return {"bytes": n * (16 if case["values"] else 8), "flops": 0}
    if kind == "bucket":
        return {"bytes": n * 16 + 4 * case["buckets"], "flops": 0}
    if kind == "scan":
        return {"bytes": 8 * n * case["blocks"], "flops": 0}
    return {"bytes": 4 * n + 4 * (1 << (n - 1).bit_length()), "flops": 0}


# ---- the radiance in 64 bits -------------------------------------------------------------------------------------


def _world_positions(f):
    """World position of every pixel and whether it is shaded (view depth below far - 0.001), from the camera's float
    matrices: a camera at `position` looking along +z, unrotated."""
    w, h, cam = f["w"], f["h"], f["cam"]
    one, near, far = np.float32(1), np.float32(cam.near_plane), np.float32(cam.far_plane)
    t = np.float32(math.tan(float(np.float32(cam.fov_y) / np.float32(2))))
    p00, p11 = float(one / (t * np.float32(cam.aspect_ratio))), float(one / t)
    p22, p32 = float(far / (far - near)), float(-(far * near) / (far - near))
    z = p32 / (f["depth"].double() - p22)
    p = torch.arange(w * h, device="cuda")
    x = ((p % w).double() / w * 2 - 1) / p00 * z
    y = ((1 - torch.div(p, w, rounding_mode="floor").double() / h) * 2 - 1) / p11 * z
    return torch.stack([x + cam.position[0], y + cam.position[1], z + cam.position[2]], dim=1), z < float(far - np.float32(0.001))


def _reflected(v, n, to_light, f0, albedo, metal, rough):
    """The BRDF times n.l of each row, as the reference's pbr.glsl defines it (PI = 3.14, k = roughness)."""
    pi = float(np.float32(3.14))
    half = torch.nn.functional.normalize(v + to_light, dim=1, eps=1e-300)
    dot = lambda a, b: (a * b).sum(1).clamp(min=0.0)  # noqa: E731
    nh, nv, nl, hv = dot(n, half), dot(n, v), dot(n, to_light), dot(half, v)
    a2 = rough * rough
    ndf = a2 / (pi * (nh * nh * (a2 - 1) + 1) ** 2)
    g = nv / (nv * (1 - rough) + rough) * (nl / (nl * (1 - rough) + rough))
    fresnel = f0 + (1 - f0) * ((1 - hv) ** 5)[:, None]
    diffuse = (1 - fresnel) * (1 - metal)[:, None] * albedo / pi
    return (diffuse + fresnel * (ndf * g / (4 * nv * nl + float(np.float32(0.0001))))[:, None]) * nl[:, None]


def _image(f, points, shaded, pixel, light, pos, lig, ar, sun=None):
    """The frame's radiance from its (pixel, light) pairs, smooth attenuation, in 64 bits (differentiable)."""
    eye = torch.tensor([f["cam"].position[i] for i in range(3)], dtype=torch.float64, device="cuda")
    at = shaded.nonzero()[:, 0]
    slot = torch.full_like(shaded, -1, dtype=torch.int64)
    slot[at] = torch.arange(at.numel(), device="cuda")
    albedo, rough = ar[at, :3], ar[at, 3]
    metal = f["metal"].double()[at]
    f0 = float(np.float32(0.04)) * (1 - metal)[:, None] + albedo * metal[:, None]
    n = f["normals"].view(torch.float16).view(-1, 4)[at, :3].double()
    v = torch.nn.functional.normalize(eye - points[at], dim=1, eps=1e-300)
    row = slot[pixel]
    d = points[pixel] - pos[light, :3]
    dist = d.norm(dim=1)
    fade = (1 - (dist / lig[light, 3]) ** 4).clamp(min=0.0) ** 2
    term = _reflected(v[row], n[row], -d / dist[:, None], f0[row], albedo[row], metal[row], rough[row])
    colour = (float(np.float32(0.03)) * albedo).index_add(0, row, term * lig[light, :3] * fade[:, None])
    if sun is not None:
        colour = colour + _reflected(v, n, (-sun[0, :3]).expand_as(v), f0, albedo, metal, rough) * sun[1, :3]
    rgb = colour ** (1 / float(np.float32(2.2)))
    out = torch.zeros(shaded.numel(), 4, dtype=torch.float64, device="cuda")
    return out.index_copy(0, at, torch.cat([rgb, torch.ones_like(rgb[:, :1])], dim=1))


def _pairs_in_range(points, shaded, pos, lig):
    """Every (pixel, light) pair closer than the light's radius: with tight cluster boxes the lists hold all of them."""
    at = shaded.nonzero()[:, 0]
    p, found = points[at], []
    step = max(1, (1 << 25) // max(1, at.numel()))
    for k in range(0, pos.shape[0], step):
        c, r = pos[k:k + step, :3], lig[k:k + step, 3]
        d2 = sum((p[:, i:i + 1] - c[None, :, i]) ** 2 for i in range(3))
        hit = (d2 < r[None, :] ** 2).nonzero()
        found.append(torch.stack([at[hit[:, 0]], hit[:, 1] + k], dim=1))
    found = torch.cat(found)
    return found[:, 0], found[:, 1]


def _listed_pairs(f, b, shaded):
    """The (pixel, light) pairs of the lists that the call is given."""
    refs = b["refs"].long()
    count = torch.where(shaded, b["counts"].long()[refs], 0)
    pixel = torch.repeat_interleave(torch.arange(refs.numel(), device="cuda"), count)
    first = count.cumsum(0) - count
    entry = torch.arange(pixel.numel(), device="cuda") - first[pixel] + b["offsets"].long()[refs[pixel]]
    return pixel, b["indices"].long()[entry]


def exact(case, seed):
    """run()'s outputs in 64 bits where they are computed numbers. A frame, batch or mixed case has none: its default
    cluster boxes are the reference's, whose lists depend on the order of 32-bit operations, so that the radiance has a
    64-bit value only on given lists, as in train, or on all lights in range, as in stages."""
    if case["kind"] == "stages":
        s = prepare(case, seed)
        f = s["f"]
        points, shaded = _world_positions(f)
        pos, lig = f["pos"].double(), f["lig"].double()
        image = _image(f, points, shaded, *_pairs_in_range(points, shaded, pos, lig), pos, lig, f["ar"].double(),
                       s["sun"].double())
        view = pos.clone()
        view[:, :3] -= torch.tensor([f["cam"].position[i] for i in range(3)], dtype=torch.float64, device="cuda")
        return {"image": image, "view_pos": view, "codes": None, "bvh": None, "keys": None, "count": None, "refs": None,
                "counts": None, "offsets": None, "indices": None, "total": None}
    if case["kind"] == "train":
        s = prepare(case, seed)
        f = s["f"]
        points, shaded = _world_positions(f)
        params = [f[k].double().requires_grad_(True) for k in ("pos", "lig", "ar")]
        image = _image(f, points, shaded, *_listed_pairs(f, s["b"], shaded), *params)
        grads = torch.autograd.grad(image, params, grad_outputs=image.detach() - s["target"].double())
        return {"image": image.detach(), "pos": grads[0], "lights": grads[1], "albedo_roughness": grads[2]}
    return None
