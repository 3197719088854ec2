"""The workloads this library's speed is measured on: views rendered frame
after frame, views batched into fused launches, the denoiser on its own, the
pass-level entry points of a host with its own render graph, and raw ray
queries, from the smallest view a server renders to a 16-view batch.

A case is a dict of plain values; `prepare` makes its inputs on the GPU from a
seed (camera path, noise, rays and which of two scenes), `run` makes one pass
through the public entry points, `exact` gives what a pass returns in 64-bit
torch where that is short to state (ray queries against all triangles, one
a-trous iteration).  Scenes are the benchmark's: boxes and icospheres on a
plane under a sun and a constant sky.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from violet_amd import _abi, _lib, batch, denoiser, gpu, renderer, scene, serve, synth

STORAGE = {"f32": _lib.STORAGE_F32, "f16": _lib.STORAGE_F16}
FLOAT = {"f32": "<f4", "f16": "<f2"}
ORBIT_FRAMES = 60
WARM_FRAMES = 6  # frames rendered before a pass: histories, reservoirs and the radiance cache are filled
DENOISE_FRAMES = 8  # frames of a denoiser sequence; the sequence then starts over after a reset (a camera cut)
SCENES = 2


def listed():
    return [
        # the headline: one 1080p view of the large scene, full precision
        {"name": "frame 1080p", "kind": "frame", "width": 1920, "height": 1080, "triangles": 1_000_000,
         "storage": "f32", "resample": "reference", "lit": False},
        # the 720p frame loop on the smaller scene, with its own resampling constants
        {"name": "frame 720p", "kind": "frame", "width": 1280, "height": 720, "triangles": 200_000,
         "storage": "f32", "resample": "frame_loop", "lit": False},
        # the smallest view a server renders: launches and latency count
        {"name": "frame 256", "kind": "frame", "width": 256, "height": 256, "triangles": 1_000_000,
         "storage": "f16", "resample": "reference", "lit": False},
        # an odd-sized view taken all the way to the lit, anti-aliased image
        {"name": "lit frame odd", "kind": "frame", "width": 803, "height": 451, "triangles": 200_000,
         "storage": "f16", "resample": "reference", "lit": True},
        # 16 uneven views in one batch, each pass one launch over all of them: the largest call
        {"name": "batch 16 views", "kind": "batch", "views": 16, "min_width": 320, "max_width": 1920,
         "min_height": 240, "max_height": 1080, "sizes_seed": 21, "triangles": 1_000_000, "storage": "f16"},
        # what a serving loop issues when a few small requests have queued up
        {"name": "batch 4 small", "kind": "batch", "views": 4, "min_width": 256, "max_width": 640,
         "min_height": 256, "max_height": 360, "sizes_seed": 5, "triangles": 1_000_000, "storage": "f16"},
        # the denoiser alone behind another renderer: a small preview with five iterations ...
        {"name": "denoise 360p", "kind": "denoise", "width": 640, "height": 360, "storage": "f32", "iterations": 5},
        # ... and a large view in half-precision storage
        {"name": "denoise 1440p", "kind": "denoise", "width": 2560, "height": 1440, "storage": "f16",
         "iterations": 3},
        # one wavelet iteration, called by a host that sequences its own denoiser
        {"name": "atrous 1080p", "kind": "atrous", "width": 1920, "height": 1080, "storage": "f32", "step": 2},
        # sampling and spatial reuse pass by pass, as a render graph issues them
        {"name": "passes 1080p", "kind": "passes", "width": 1920, "height": 1080, "triangles": 1_000_000,
         "storage": "f32"},
        # a bulk ray query: bounce rays off the large scene's surfaces, closest hits
        {"name": "rays bounce", "kind": "rays", "rays": 1 << 20, "triangles": 1_000_000, "what": "bounce"},
        # a small one: shadow rays for a ragged handful of points
        {"name": "rays shadow small", "kind": "rays", "rays": 9973, "triangles": 20_000, "what": "shadow"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "denoise", "atrous", "passes", "rays"])
    w, h = _log_int(rng, 200, 2560), _log_int(rng, 150, 1440)
    tris = _log_int(rng, 10_000, 1_000_000)
    storage = rng.choice(["f32", "f16"])
    if kind == "frame":
        return {"kind": kind, "width": w, "height": h, "triangles": tris, "storage": storage,
                "resample": rng.choice(["reference", "frame_loop"]), "lit": rng.random() < 0.4}
    if kind == "batch":
        return {"kind": kind, "views": rng.randint(2, 12), "min_width": 256, "max_width": rng.randint(400, 1600),
                "min_height": 200, "max_height": rng.randint(300, 1000), "sizes_seed": rng.randint(1, 10_000),
                "triangles": tris, "storage": storage}
    if kind == "denoise":
        return {"kind": kind, "width": w, "height": h, "storage": storage, "iterations": rng.randint(2, 5)}
    if kind == "atrous":
        return {"kind": kind, "width": w, "height": h, "storage": storage, "step": 1 << rng.randint(0, 4)}
    if kind == "passes":
        return {"kind": kind, "width": w, "height": h, "triangles": tris, "storage": storage}
    return {"kind": kind, "rays": _log_int(rng, 2_000, 2_000_000), "triangles": tris,
            "what": rng.choice(["camera", "bounce", "shadow"])}


# ---------------------------------------------------------------------------
# what the cases share
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _mesh(triangles, which):
    return scene.make_scene(triangles, seed=13 + which)


@functools.lru_cache(maxsize=4)
def _scene(triangles, which):
    """A program builds a scene once and renders it for as long as it lives."""
    return scene.Scene(_mesh(triangles, which))


def _scene_of(case, seed):
    return _scene(case["triangles"], seed % SCENES)


class _Image:
    """A library-owned device image as torch sees one.  A tensor made from it holds it, and with it the object that
    owns the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


class _Views:
    """Tensors over the images of `owner`, made once per address (they alternate between frames)."""

    def __init__(self, owner):
        self.owner = owner
        self.made = {}

    def __call__(self, ptr, shape, typestr):
        key = (ptr, shape, typestr)
        if key not in self.made:
            self.made[key] = torch.as_tensor(_Image(self.owner, ptr, shape, typestr), device="cuda")
        return self.made[key]


def _orbit(width, height, phase, frame, deg_per_frame, jitter=False):
    a = math.radians(phase + deg_per_frame * frame)
    pos = np.array([30.0 * math.cos(a), 30.0 * math.sin(a), 9.0])
    d = -pos / np.linalg.norm(pos)
    yaw, pitch = math.degrees(math.atan2(d[0], d[1])), math.degrees(math.asin(d[2])) + 8.0
    j = synth.jitter_ndc(frame % 8, width, height) if jitter else (0.0, 0.0)
    return synth.View(synth.Camera(pos, yaw, pitch), width, height, jitter=j)


def _orbit_params(width, height, seed, frames=ORBIT_FRAMES, deg_per_frame=6.0, jitter=False):
    """Frame parameters of a closed orbit; the seed places its start."""
    phase = float(np.random.default_rng(seed).uniform(0.0, 360.0))
    views = [_orbit(width, height, phase, f, deg_per_frame, jitter) for f in range(frames)]
    return [synth.make_frame_params(views[f], views[f - 1]) for f in range(frames)]


def _config(case):
    c = renderer.RestirConfig(storage=STORAGE[case["storage"]])
    if case.get("resample") == "frame_loop":
        c.temporal_m_cap, c.diff_spatial_taps, c.spatial_radius_px = 30, 5, 30.0
    if case.get("lit"):
        c.compose = c.taa = True
    return c


def _outputs(views, case, o, w, h):
    f = FLOAT[case["storage"]]
    out = {"diffuse": views(o.indirect_diffuse, (h, w, 3), f), "specular": views(o.indirect_specular, (h, w, 3), f),
           "depth": views(o.depth, (h, w), "<f4"), "gbuffer": views(o.gbuffer, (4, h, w), "<i4")}
    if o.color:
        out["color"] = views(o.color, (h, w, 3), f)
    return out


# ---------------------------------------------------------------------------
# one view, frame after frame
# ---------------------------------------------------------------------------
def _prepare_frame(case, seed):
    w, h = case["width"], case["height"]
    view = renderer.RestirRenderer(w, h, _config(case))
    s = {"scene": _scene_of(case, seed), "view": view, "frame": 0,
         "params": _orbit_params(w, h, seed, jitter=case["lit"]), "tensors": _Views(view)}
    for _ in range(WARM_FRAMES):
        _run_frame(case, s)
    return s


def _run_frame(case, s):
    k = s["frame"]
    s["frame"] = k + 1
    o = s["view"].add_passes(s["scene"], s["params"][k % ORBIT_FRAMES], k)
    return _outputs(s["tensors"], case, o, case["width"], case["height"])


# ---------------------------------------------------------------------------
# many views in one batch
# ---------------------------------------------------------------------------
def _batch_sizes(case):
    rng = np.random.default_rng(case["sizes_seed"])
    n = case["views"]
    ws = rng.integers(case["min_width"], case["max_width"] + 1, n)
    hs = rng.integers(case["min_height"], case["max_height"] + 1, n)
    return [(int(w), int(h)) for w, h in zip(ws, hs)]


def _prepare_batch(case, seed):
    sizes = _batch_sizes(case)
    views = [renderer.RestirRenderer(w, h, _config(case)) for w, h in sizes]
    s = {"scene": _scene_of(case, seed), "frame": 0, "tensors": _Views(views), "sizes": sizes, "views": views,
         "params": [_orbit_params(w, h, seed * 64 + k) for k, (w, h) in enumerate(sizes)],
         "batch": batch.Batch()}
    for _ in range(WARM_FRAMES):
        _run_batch(case, s)
    return s


def _run_batch(case, s):
    k = s["frame"]
    s["frame"] = k + 1
    out = s["batch"].add_passes(s["scene"], s["views"], [p[k % ORBIT_FRAMES] for p in s["params"]],
                                [k] * len(s["views"]))
    return [_outputs(s["tensors"], case, o, w, h) for o, (w, h) in zip(out, s["sizes"])]


# ---------------------------------------------------------------------------
# the denoiser and one of its iterations
# ---------------------------------------------------------------------------
def _gbuffer(sc, fp, w, h):
    depth = torch.empty((h, w), dtype=torch.float32, device="cuda")
    gb = torch.empty((4, h, w), dtype=torch.int32, device="cuda")
    io = _abi.GBufferIO(w, h, depth.data_ptr(), gb.data_ptr())
    _lib.call("vgi_pass_gbuffer_primary", ctypes.byref(fp), sc.handle, ctypes.byref(io), gpu.stream())
    return depth, gb


def _noisy(depth, generator, lobe, storage):
    """A smooth field over the image times Exp(1) noise, one draw per pixel, zero on the sky."""
    h, w = depth.shape
    y = torch.arange(h, device="cuda", dtype=torch.float32)[:, None] / h
    x = torch.arange(w, device="cuda", dtype=torch.float32)[None, :] / w
    base = 0.6 + 0.35 * torch.sin((7.0 + 2 * lobe) * x + 3.0 * y) * torch.cos(5.0 * y - 2.0 * lobe * x)
    e = torch.empty((h, w), device="cuda").exponential_(generator=generator)
    v = torch.where(depth > 0, base * e, torch.zeros_like(e))
    tint = torch.tensor([[1.0, 0.85, 0.7], [0.7, 0.8, 1.0]][lobe], device="cuda")
    return (v[..., None] * tint).to(torch.float16 if storage == "f16" else torch.float32).contiguous()


def _denoise_scene(seed):
    return _scene(50_000, seed % SCENES)


def _prepare_denoise(case, seed):
    w, h = case["width"], case["height"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    # a slow pan: about two pixels a frame at the image centre
    params = _orbit_params(w, h, seed, DENOISE_FRAMES, 180.0 / w)
    frames = []
    for f, fp in enumerate(params):
        depth, gb = _gbuffer(_denoise_scene(seed), fp, w, h)
        ray_len = torch.where(depth > 0, 1.0, 0.0).to(torch.float16 if case["storage"] == "f16" else torch.float32)
        frames.append((depth, gb, _noisy(depth, g, 0, case["storage"]), _noisy(depth, g, 1, case["storage"]), ray_len))
    den = denoiser.Denoiser(w, h, STORAGE[case["storage"]])
    den.atrous_iterations = case["iterations"]
    s = {"params": params, "frames": frames, "den": den, "frame": 0, "tensors": _Views(den)}
    for _ in range(3):
        _run_denoise(case, s)
    return s


def _run_denoise(case, s):
    k = s["frame"] % DENOISE_FRAMES
    s["frame"] += 1
    depth, gb, diff, spec, ray_len = s["frames"][k]
    if k == 0:
        s["den"].reset()
        prev = (None, None)
    else:
        prev = s["frames"][k - 1][:2]
    o = s["den"].add_passes(s["params"][k], denoiser.Input(depth, gb, prev[0], prev[1], diff, spec, ray_len))
    w, h, f = case["width"], case["height"], FLOAT[case["storage"]]
    v = s["tensors"]
    return {"diffuse": v(o.diffuse, (h, w, 3), f), "specular": v(o.specular, (h, w, 3), f),
            "history_len": v(o.history_len, (h, w), "|u1"), "variance": v(o.variance, (h, w, 2), f)}


def _prepare_atrous(case, seed):
    w, h = case["width"], case["height"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    depth, gb = _gbuffer(_denoise_scene(seed), _orbit_params(w, h, seed, 1)[0], w, h)
    diff, spec = _noisy(depth, g, 0, case["storage"]), _noisy(depth, g, 1, case["storage"])
    var = 0.05 + 0.3 * torch.rand((h, w, 2), device="cuda", generator=g)
    var = torch.where(depth[..., None] > 0, var, torch.zeros_like(var)).to(diff.dtype).contiguous()
    out = [torch.empty_like(diff), torch.empty_like(spec), torch.empty_like(var)]
    io = _lib.DenoiseAtrousIO(w, h, STORAGE[case["storage"]], depth.data_ptr(), gb.data_ptr(), diff.data_ptr(),
                              spec.data_ptr(), var.data_ptr(), *[t.data_ptr() for t in out])
    return {"io": io, "pc": _lib.PCDenoiseAtrous(case["step"]), "in": (depth, gb, diff, spec, var), "out": out}


def _run_atrous(case, s):
    _lib.call("vgi_pass_denoise_atrous", ctypes.byref(s["io"]), ctypes.byref(s["pc"]), gpu.stream())
    return {"diffuse": s["out"][0], "specular": s["out"][1], "variance": s["out"][2]}


def _exact_atrous(case, seed):
    """The edge-stopping 5x5 wavelet iteration of SVGF, taps on the centre row and column left out (as the
    reference leaves them out), in float64."""
    depth, gb, diff, spec, var = (t.double() if t.is_floating_point() else t for t in _prepare_atrous(case, seed)["in"])
    h, w = depth.shape
    step = case["step"]
    enc = gb[1].long() & 0xFFFFFF
    fx, fy = (enc & 0xFFF).double() * (2.0 / 4095.0) - 1.0, (enc >> 12).double() * (2.0 / 4095.0) - 1.0
    fz = 1.0 - fx.abs() - fy.abs()
    t = (-fz).clamp(0.0, 1.0)
    n = torch.stack([fx + torch.where(fx >= 0, -t, t), fy + torch.where(fy >= 0, -t, t), fz], -1)
    n = n / n.norm(dim=-1, keepdim=True)
    fwidth = (gb[2] & 0xFFFF).to(torch.int16).view(torch.float16).double()
    lum = torch.tensor([0.2126, 0.7152, 0.0722], dtype=torch.float64, device="cuda")
    ld, ls = (diff * lum).sum(-1), (spec * lum).sum(-1)
    kd, ks = 1.0 / (4.0 * var[..., 0].sqrt() + 1e-8), 1.0 / (4.0 * var[..., 1].sqrt() + 1e-8)
    kernel = (1.0, 2.0 / 3.0, 1.0 / 6.0)
    dsum, ssum, vsum = diff.clone(), spec.clone(), var.clone()
    wd, ws = torch.ones_like(depth), torch.ones_like(depth)
    for y in (-2, -1, 1, 2):
        for x in (-2, -1, 1, 2):
            ox, oy = x * step, y * step
            # the centre pixels whose tap lies inside the image, and their taps
            c = (slice(max(0, -oy), min(h, h - oy)), slice(max(0, -ox), min(w, w - ox)))
            if c[0].start >= c[0].stop or c[1].start >= c[1].stop:
                continue
            j = (slice(c[0].start + oy, c[0].stop + oy), slice(c[1].start + ox, c[1].stop + ox))
            ez = -(depth[j] - depth[c]).abs() / (fwidth[c] * math.hypot(ox, oy) + 1e-8)
            wn = (n[j] * n[c]).sum(-1).clamp(0.0, 1.0) ** 128
            k = kernel[abs(x)] * kernel[abs(y)]
            a = k * wn * torch.exp(ez - (ld[j] - ld[c]).abs() * kd[c])
            b = k * wn * torch.exp(ez - (ls[j] - ls[c]).abs() * ks[c])
            dsum[c] += diff[j] * a[..., None]
            ssum[c] += spec[j] * b[..., None]
            vsum[c] += torch.stack([a * a * var[j][..., 0], b * b * var[j][..., 1]], -1)
            wd[c] += a
            ws[c] += b
    return {"diffuse": dsum / wd[..., None], "specular": ssum / ws[..., None],
            "variance": vsum / torch.stack([wd, ws], -1) ** 2}


# ---------------------------------------------------------------------------
# pass by pass: sampling and spatial reuse of both lobes
# ---------------------------------------------------------------------------
def _prepare_passes(case, seed):
    w, h = case["width"], case["height"]
    # a rendered view supplies what a host's own passes and history would
    s = _prepare_frame(dict(case, lit=False), seed)
    r, sc = s["view"], s["scene"]
    st = STORAGE[case["storage"]]
    at = lambda name: r.image(name)[0]  # noqa: E731
    rdt = torch.float16 if case["storage"] == "f16" else torch.float32
    new = lambda shape, dt: torch.zeros(shape, dtype=dt, device="cuda")  # noqa: E731
    out = {"diff_hit": new((h, w, 2), torch.int32), "diff_radiance": new((h, w, 3), rdt),
           "spec_hit": new((h, w, 4), torch.float32), "spec_radiance": new((h, w, 3), rdt),
           "diff_reservoir": new((h, w), torch.int32), "diff_reused_hit": new((h, w, 2), torch.int32),
           "diff_reused_radiance": new((h, w, 3), rdt), "diff_lighting": new((h, w, 3), rdt),
           "spec_lighting": new((h, w, 3), rdt), "spec_ray_len": new((h, w), rdt)}
    o = {k: v.data_ptr() for k, v in out.items()}
    queries = new((128 * 1024, 6), torch.int32)
    counter = new((1,), torch.int32)
    tr = _abi.TraceResources()
    tr.scene_tlas = sc.handle
    tr.sky_radiance[:] = [1.0, 1.0, 1.0]
    tr.storage = st
    tr.prev_indirect_diffuse_texture = at("indirect_diffuse_raw")
    tr.prev_depth_texture = at("depth")
    tr.prev_width, tr.prev_height = w, h
    tr.hash_grid_storage_buffer = at("hash_grid_storage")
    tr.rw_hash_grid_query_buffer, tr.rw_hash_grid_query_counter_buffer = queries.data_ptr(), counter.data_ptr()
    rand = int(np.random.default_rng(seed).integers(1, 1 << 31))
    params = s["params"][(s["frame"] - 1) % ORBIT_FRAMES]
    gb, dep = at("gbuffer"), at("depth")
    dg = _abi.DiffSampleGenIO(w, h, st, gb, dep, o["diff_hit"], o["diff_radiance"])
    sg = _abi.SpecSampleGenIO(w, h, st, gb, dep, o["spec_hit"], o["spec_radiance"])
    ds = _abi.DiffSpatialIO(w, h, st, gb, dep, at("ao_filtered"), at("diff_temporal_reservoir"),
                            at("diff_temporal_hit_pos_normal"), at("diff_temporal_hit_radiance"), o["diff_reservoir"],
                            o["diff_reused_hit"], o["diff_reused_radiance"], o["diff_lighting"])
    ss = _abi.SpecSpatialIO(w, h, st, gb, dep, at("spec_reservoir"), at("spec_hit_pos"), at("spec_hit_radiance"),
                            o["spec_lighting"], o["spec_ray_len"])
    gen, fr = _abi.PCSampleGen(rand, 1), _abi.PCFrameRand(rand ^ 0x5BD1E995)
    rp = _abi.ResampleParams(0, 0, 0.0)
    ref = ctypes.byref
    calls = [("vgi_pass_clear_buffer", (counter.data_ptr(), 4, 0)),
             ("vgi_pass_ind_diff_sample_gen", (ref(params), ref(tr), ref(dg), ref(gen))),
             ("vgi_pass_ind_diff_spatial_resample", (ref(params), ref(ds), ref(fr), ref(rp))),
             ("vgi_pass_ind_spec_sample_gen", (ref(params), ref(tr), ref(sg), ref(gen))),
             ("vgi_pass_ind_spec_spatial_resample", (ref(params), ref(ss), ref(fr), ref(rp)))]
    return {"calls": calls, "out": out, "keep": (s, tr, queries, counter)}


def _run_passes(case, s):
    st = gpu.stream()
    for name, args in s["calls"]:
        _lib.call(name, *args, st)
    return s["out"]


# ---------------------------------------------------------------------------
# ray queries
# ---------------------------------------------------------------------------
SUN = (0.3094922, 0.2063282, 0.9284767)


def _rays(case, seed):
    """(n, 8) rays: pinhole camera rays in pixel order, bounces off surface points into the hemisphere above them,
    or shadow rays from surface points towards the sun; surface points in mesh order, as a light baker walks them."""
    m = _mesh(case["triangles"], seed % SCENES)
    n = case["rays"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["what"] == "camera":
        w = max(1, int(math.sqrt(n * 16 / 9)))
        fp = _orbit_params(w, max(1, n // w), seed, 1)[0]
        i = torch.arange(n, device="cuda")
        inv = torch.tensor(list(fp.inv_view_proj), device="cuda", dtype=torch.float64).reshape(4, 4).T
        ndc = torch.stack([((i % w) + 0.5) / w * 2 - 1, ((i // w) + 0.5) / max(1, n // w) * 2 - 1,
                           torch.ones(n, device="cuda"), torch.ones(n, device="cuda")], -1).double()
        e = ndc @ inv.T
        o = torch.tensor(list(fp.view_pos)[:3], device="cuda", dtype=torch.float64).expand(n, 3)
        d = e[:, :3] / e[:, 3:] - o
    else:
        pos = torch.from_numpy(m.positions).cuda().double()
        tri = torch.from_numpy(m.indices.astype(np.int64)).cuda()
        pick = torch.randint(0, len(tri), (n,), device="cuda", generator=g).sort().values
        p0, p1, p2 = (pos[tri[pick, k]] for k in range(3))
        uv = torch.rand((n, 2), device="cuda", generator=g, dtype=torch.float64)
        uv = torch.where(uv.sum(-1, keepdim=True) > 1, 1 - uv, uv)
        nrm = torch.linalg.cross(p1 - p0, p2 - p0)
        nrm = nrm / nrm.norm(dim=-1, keepdim=True).clamp_min(1e-30)
        o = p0 + (p1 - p0) * uv[:, :1] + (p2 - p0) * uv[:, 1:] + nrm * 1e-3
        if case["what"] == "bounce":
            d = torch.randn((n, 3), device="cuda", generator=g, dtype=torch.float64)
            d = d * torch.where((d * nrm).sum(-1, keepdim=True) < 0, -1.0, 1.0)
        else:
            d = torch.tensor(SUN, device="cuda", dtype=torch.float64).expand(n, 3)
    d = d / d.norm(dim=-1, keepdim=True)
    lo, hi = torch.full((n, 1), 0.0005, device="cuda"), torch.full((n, 1), 1000.0, device="cuda")
    return torch.cat([o.float(), lo, d.float(), hi], -1).contiguous()


def _prepare_rays(case, seed):
    rays = _rays(case, seed)
    return {"scene": _scene_of(case, seed), "rays": rays,
            "hits": torch.empty((case["rays"], 4), dtype=torch.int32, device="cuda")}


def _run_rays(case, s):
    any_hit = case["what"] == "shadow"
    s["scene"].trace(s["rays"], case["rays"], any_hit, s["hits"])
    if any_hit:  # only whether something is in the way
        return {"blocked": s["hits"][:, 3] != -1}
    f = s["hits"].view(torch.float32)
    return {"t": f[:, 0], "u": f[:, 1], "v": f[:, 2], "triangle": s["hits"][:, 3]}


def _exact_rays(case, seed):
    """Every ray against every triangle in float64.  The triangle and the place on it have no 64-bit value of their
    own: where triangles meet or coincide (boxes stand on the ground plane) each is right; shadow rays return truth
    values."""
    if case["what"] == "shadow" or case["rays"] * case["triangles"] > 4e9:
        return None
    m = _mesh(case["triangles"], seed % SCENES)
    # what the library is given: single-precision vertices and their single-precision edges
    pos = torch.from_numpy(m.positions).cuda()
    tri = torch.from_numpy(m.indices.astype(np.int64)).cuda()
    v0 = pos[tri[:, 0]]
    e1, e2, v0 = (pos[tri[:, 1]] - v0).double(), (pos[tri[:, 2]] - v0).double(), v0.double()
    r = _rays(case, seed).double()
    n, step = len(r), max(1, 40_000_000 // len(tri))
    nearest = torch.zeros(n, dtype=torch.float64, device="cuda")
    dot = lambda a, b: a[0] * b[0] + a[1] * b[1] + a[2] * b[2]  # noqa: E731
    cross = lambda a, b: (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])  # noqa: E731
    e1c, e2c = e1.T[:, None, :], e2.T[:, None, :]
    for a in range(0, n, step):
        q = r[a:a + step]
        d = q[:, 4:7].T[:, :, None]
        p = cross(d, e2c)
        inv = 1.0 / dot(e1c, p)
        tv = q[:, 0:3].T[:, :, None] - v0.T[:, None, :]
        u = dot(tv, p) * inv
        qv = cross(tv, e1c)
        v = dot(d, qv) * inv
        t = dot(e2c, qv) * inv
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= q[:, 3:4]) & (t < q[:, 7:8])
        nearest[a:a + step] = torch.where(ok, t, q[:, 7:8].expand_as(t)).amin(dim=1)
    return {"t": nearest, "u": None, "v": None, "triangle": None}


# ---------------------------------------------------------------------------
_PREPARE = {"frame": _prepare_frame, "batch": _prepare_batch, "denoise": _prepare_denoise, "atrous": _prepare_atrous,
            "passes": _prepare_passes, "rays": _prepare_rays}
_RUN = {"frame": _run_frame, "batch": _run_batch, "denoise": _run_denoise, "atrous": _run_atrous,
        "passes": _run_passes, "rays": _run_rays}


def prepare(case, seed):
    return {"case": case, "state": _PREPARE[case["kind"]](case, seed)}


def run(state):
    return _RUN[state["case"]["kind"]](state["case"], state["state"])


def exact(case, seed):
    if case["kind"] == "atrous":
        return _exact_atrous(case, seed)
    if case["kind"] == "rays":
        return _exact_rays(case, seed)
    # reservoir selections compare single-precision numbers and feed the frames after them: no 64-bit value
    return None


def work(case):
    """Bytes: every image a pass needs read once and written once (radiance 12 or 6 bytes, pairs 8 or 4).  Operations:
    boxes and triangles of a ray's path through a balanced tree, and the taps' arithmetic."""
    half = case.get("storage") == "f16"
    ray_flops = 40 * 4 * max(1.0, math.log(case.get("triangles", 2), 4)) + 4 * 60
    if case["kind"] == "rays":
        return {"bytes": case["rays"] * 48, "flops": case["rays"] * ray_flops}
    if case["kind"] == "batch":
        px = sum(w * h for w, h in _batch_sizes(case))
    else:
        px = case["width"] * case["height"]
    restir, den, atrous = (414, 94, 46) if half else (524, 244, 76)
    den_flops, atrous_flops, spatial_flops = 2500, 16 * 40, 9 * 200
    if case["kind"] == "atrous":
        return {"bytes": px * atrous, "flops": px * atrous_flops}
    if case["kind"] == "denoise":
        return {"bytes": px * (den + atrous * case["iterations"]),
                "flops": px * (den_flops + atrous_flops * case["iterations"])}
    if case["kind"] == "passes":
        return {"bytes": px * (126 if half else 204), "flops": px * (4 * ray_flops + 2 * spatial_flops)}
    lit = 60 if case.get("lit") else 0
    return {"bytes": px * (restir + den + 3 * atrous + lit),
            "flops": px * (7 * ray_flops + 2 * spatial_flops + den_flops + 3 * atrous_flops)}


def tolerance(case):
    """About four times what the same code with its filter sums in another order showed, and no less than what the
    storage type rounds."""
    if case["kind"] == "rays":
        return "exact"  # smallest t, then lowest triangle, of the single-precision test: the entry point's contract
    half = case["storage"] == "f16"
    if case["kind"] == "passes":
        # the passes are reproducible bit for bit; the denoised history they read (prepare's frames) is not
        return {"rel": 4e-5, "max": 5e-3, "differ": 8e-3} if half else {"rel": 1e-6, "max": 1e-4, "differ": 4e-3}
    if case["kind"] == "atrous":
        return {"rel": 5e-4, "max": 2e-2} if half else {"rel": 2e-5, "max": 1e-3}
    if case["kind"] == "denoise":
        return {"rel": 4e-4, "max": 2e-2, "differ": 1e-5} if half else {"rel": 1e-5, "max": 1e-3, "differ": 1e-5}
    # rounding in the denoiser comes back through the screen-space cache and flips selections
    return {"rel": 1.2e-3, "max": 0.7, "differ": 1e-5}
