"""The voxel-lighting work a program has this framework do, as timed cases.

Each case is one pass through lum_amd.api on a seeded world: a heightmap of
solid blocks under air, a random block palette, random materials and a random
radiance field (lum_amd.synth, the distributions of bench.py).

  probes  radiance update of every probe of one world
  subset  radiance update of a request list (random probes, with or without a stride)
  step    the per-frame update of the renderer: the stored field shift, probe
          selection on the device, the update over the selected probes
  glossy  reflection march over a G-buffer
  diffuse diffuse shading from the field with a shadow map
  frame   models mapped into the world, every probe updated, a glossy frame
  batch   the same chain over many worlds in one launch per pass
  serve   a mixed trace of updates and glossy queries through the server

exact() restates the passes in float64 with plain torch and numpy.
"""
import ctypes
import math

import numpy as np
import torch

from lum_amd import synth
from lum_amd._lib import RADIANCE_BF16, RADIANCE_F16, RADIANCE_F32, check
from lum_amd.api import (Batch, Context, Model, Server, World, camera_default, glossy_request, placement,
                         radiance_params, radiance_request)

FORMATS = {"f32": RADIANCE_F32, "f16": RADIANCE_F16, "bf16": RADIANCE_BF16}
TEXEL_BYTES = {"f32": 16, "f16": 8, "bf16": 8}


def listed():
    return [
        # A small room updated every frame: one short launch, where latency counts.
        {"name": "probes_small", "pass": "probes", "wx": 16, "wy": 16, "wz": 8, "rays": 32, "format": "f32",
         "max_steps": 0},
        # The reference's own world size and ray count.
        {"name": "probes_plain", "pass": "probes", "wx": 48, "wy": 48, "wz": 16, "rays": 64, "format": "f32",
         "max_steps": 64},
        # The largest world of the benchmarks: two million probes, half-precision storage.
        {"name": "probes_large", "pass": "probes", "wx": 256, "wy": 256, "wz": 32, "rays": 128, "format": "f16",
         "max_steps": 96},
        # A served update: a random third of a mid-sized world's probes by request list.
        {"name": "subset_served", "pass": "subset", "wx": 96, "wy": 96, "wz": 32, "rays": 64, "format": "f16",
         "max_steps": 0, "percent": 33, "stride": 1},
        # Odd extents, a ray count that is no power of two, every third entry of the list.
        {"name": "subset_ragged", "pass": "subset", "wx": 53, "wy": 37, "wz": 19, "rays": 192, "format": "bf16",
         "max_steps": 0, "percent": 70, "stride": 3},
        # What the renderer runs each frame: shift, selection, every second selected probe.
        {"name": "step_plain", "pass": "step", "wx": 48, "wy": 48, "wz": 16, "rays": 64, "format": "f32",
         "max_steps": 0, "stride": 2, "special": 96},
        # Full-HD reflections with a normal and a depth of its own for every pixel.
        {"name": "glossy_fullhd", "pass": "glossy", "wx": 48, "wy": 48, "wz": 16, "format": "f32", "max_steps": 128,
         "width": 1920, "height": 1080, "patch": 1},
        # A served reflection query: flat surfaces several pixels wide, part of them too rough to reflect.
        {"name": "glossy_query", "pass": "glossy", "wx": 61, "wy": 45, "wz": 17, "format": "f16", "max_steps": 0,
         "width": 638, "height": 359, "patch": 8},
        # The field's consumer at full HD with a 1024 x 1024 shadow map.
        {"name": "diffuse_fullhd", "pass": "diffuse", "wx": 48, "wy": 48, "wz": 16, "format": "f32", "max_steps": 0,
         "width": 1920, "height": 1080, "patch": 4, "lightmap": 1024},
        # A whole frame with 32 moving models.
        {"name": "frame_models", "pass": "frame", "wx": 48, "wy": 48, "wz": 16, "rays": 64, "format": "f32",
         "max_steps": 64, "models": 32, "model_lo": 16, "model_hi": 64, "width": 1280, "height": 720, "patch": 4},
        # Many worlds stepped together.
        {"name": "batch_worlds", "pass": "batch", "worlds": 24, "wx": 96, "wy": 96, "wz": 32, "format": "f32",
         "max_steps": 64, "models": 4, "model_lo": 16, "model_hi": 32, "width": 640, "height": 360, "patch": 1},
        # A backlog of requests over resident worlds: four fifths updates of 1-100% of the probes, the rest glossy.
        {"name": "serve_backlog", "pass": "serve", "worlds": 24, "wx": 128, "wy": 128, "wz": 32, "format": "f16",
         "max_steps": 0, "requests": 96, "width": 640, "height": 360, "patch": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["probes", "probes", "subset", "subset", "step", "glossy", "glossy", "diffuse", "frame",
                       "batch", "serve"])
    t = rng.random()
    case = {"pass": kind, "format": rng.choice(["f32", "f16", "bf16"]),
            "wx": max(5, int(16 * 8 ** t * rng.uniform(0.8, 1.2))),
            "wy": max(5, int(16 * 8 ** t * rng.uniform(0.8, 1.2))),
            "wz": max(3, int(8 * 4 ** t * rng.uniform(0.8, 1.2))),
            "max_steps": rng.choice([0, 0, 64, 96])}
    if kind in ("probes", "subset", "step", "frame"):
        case["rays"] = rng.choice([32, 64, 64, 128])
    if kind == "subset":
        case["rays"] = rng.choice([32, 64, 128, 192])
        case["percent"] = _log_int(rng, 1, 100)
        case["stride"] = rng.choice([1, 1, 2, 3])
    if kind == "step":
        case["stride"] = rng.choice([1, 2, 3])
        case["special"] = rng.randrange(0, 200)
    if kind in ("glossy", "diffuse", "frame"):
        case["width"] = _log_int(rng, 160, 1920)
        case["height"] = max(64, int(case["width"] * 9 / 16) + rng.randrange(-3, 4))
        case["patch"] = rng.choice([1, 4, 8, 16])
    if kind == "diffuse":
        case["lightmap"] = rng.choice([0, 512, 1024])
    if kind == "frame":
        case["wx"], case["wy"], case["wz"] = (max(a, b) for a, b in
                                              zip((case["wx"], case["wy"], case["wz"]), (20, 20, 10)))
        case["models"] = rng.randrange(1, 33)
        case["model_lo"], case["model_hi"] = 8, rng.choice([24, 40, 64])
    if kind in ("batch", "serve"):
        case["wx"], case["wy"], case["wz"] = rng.choice([(40, 40, 16), (56, 48, 24), (72, 72, 28)])
        case["worlds"] = rng.randrange(3, 17)
        case["width"], case["height"], case["patch"] = 320, 181, rng.choice([1, 8])
    if kind == "batch":
        case["models"], case["model_lo"], case["model_hi"] = rng.randrange(0, 4), 10, 30
    if kind == "serve":
        case["requests"] = rng.randrange(8, 65)
    return case


# ---- inputs ----------------------------------------------------------------

_shared = {}


def _context():
    if "ctx" not in _shared:
        _shared["ctx"] = Context(0)
    return _shared["ctx"]


def _gbuffer(width, height, patch, mats, rng):
    """Flat surfaces of patch x patch pixels.  With patch 1 every pixel has a
    low roughness; with larger patches the materials are drawn from all, so
    the roughness mask leaves some pixels out."""
    pw, ph = -(-width // patch), -(-height // patch)
    mn, dp = synth.make_gbuffer(pw, ph, mats, rng, rough_max=0.3 if patch == 1 else 1.0)
    if patch > 1:
        mn = np.repeat(np.repeat(mn, patch, 0), patch, 1)[:height, :width]
        dp = np.repeat(np.repeat(dp, patch, 0), patch, 1)[:height, :width]
        ramp = np.linspace(0.0, 1e-3, width, dtype=np.float32)
        dp = dp + ramp[None, :]
    return np.ascontiguousarray(mn), np.ascontiguousarray(dp, dtype=np.float32)


class _Inputs:
    """Host inputs of one world, made from the generator alone."""

    def __init__(self, case, size, rng, gbuffer=False):
        self.size = size
        self.blocks = synth.make_world(size, rng, 64)
        self.palette = synth.make_palette(rng, 64)
        self.mats = synth.make_materials(rng)
        self.field = synth.make_field(size, rng)
        self.models, self.quats, self.shifts = [], [], []
        if case.get("models"):
            self.models, self.quats, self.shifts = synth.make_models(
                rng, n=case["models"], lo=case["model_lo"], hi=case["model_hi"], world_size=size)
        self.gbuf = _gbuffer(case["width"], case["height"], case["patch"], self.mats, rng) if gbuffer else None

    @property
    def n(self):
        return self.size[0] * self.size[1] * self.size[2]

    def probe(self, p):
        wx, wy, _ = self.size
        return np.stack([p % wx, p // wx % wy, p // (wx * wy), np.zeros_like(p)], 1).astype(np.int32)


def _size(case):
    return case["wx"], case["wy"], case["wz"]


def _single(case, seed):
    """Inputs of the single-world passes."""
    rng = np.random.default_rng([seed, case["wx"], case["wy"], case["wz"]])
    inp = _Inputs(case, _size(case), rng, gbuffer="width" in case)
    inp.time_seed = int(rng.integers(1 << 20))
    if case["pass"] == "subset":
        count = max(case["stride"], inp.n * case["percent"] // 100)
        inp.requests = inp.probe(rng.permutation(inp.n)[:count])
    if case["pass"] == "step":
        inp.special = inp.probe(rng.permutation(inp.n)[:case["special"]])
        inp.shift = (1, 0, 0) if rng.random() < 0.5 else (0, -1, 0)
    if case.get("lightmap"):
        inp.lightmap = rng.integers(0, 65536, (case["lightmap"], case["lightmap"])).astype(np.uint16)
        proj = np.zeros((4, 4), np.float32)  # column-major: an oblique orthographic light over the world
        ext = 16.0 * max(case["wx"], case["wy"])
        proj[0, 0], proj[1, 1] = 2.0 / ext, 2.0 / ext
        proj[2, 0], proj[2, 1], proj[2, 2] = 0.3 / ext, 0.2 / ext, -1.0 / (16.0 * case["wz"])
        proj[3, 0], proj[3, 1], proj[3, 2] = -1.0, -1.0, 0.0
        inp.proj = proj
    return inp


def _sizes(case):
    """Log-spaced world sizes from 16x16x8 blocks to the case's."""
    hi = _size(case)
    lo = [min(a, b) for a, b in zip((16, 16, 8), hi)]
    n = case["worlds"]
    return [tuple(int(round(a * (b / a) ** ((i + 0.5) / n))) for a, b in zip(lo, hi)) for i in range(n)]


def _many(case, seed):
    """Inputs of the batched and served worlds."""
    rng = np.random.default_rng([seed, case["worlds"], case["wx"]])
    inputs = [_Inputs(case, s, rng, gbuffer=True) for s in _sizes(case)]
    for i, inp in enumerate(inputs):
        inp.rays = (64, 32, 128)[i % 3]
        inp.time_seed = int(rng.integers(1 << 20))
    trace = []
    if case["pass"] == "serve":
        for inp in inputs:
            inp.order = inp.probe(rng.permutation(inp.n))
        for _ in range(case["requests"]):
            i = int(rng.integers(len(inputs)))
            if rng.random() < 0.8:
                count = max(1, int(rng.uniform(0.01, 1.0) * inputs[i].n))
                first = int(rng.integers(inputs[i].n - count + 1))
                trace.append(("radiance", i, first, count, int(rng.choice([32, 64, 128])), int(rng.integers(1 << 20))))
            else:
                trace.append(("glossy", i))
    return inputs, trace


# ---- the framework's side ---------------------------------------------------

class _Owner:
    """Closes a world and its models when the last user is gone.  Every tensor
    over the world's memory refers to it, so the memory outlives them all."""

    def __init__(self):
        self.handles = []

    def keep(self, handle):
        self.handles.append(handle)
        return handle

    def __del__(self):
        for h in reversed(self.handles):
            h.close()


class _DevArray:
    """Memory of a world, for torch.as_tensor (whose tensor keeps this object)."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 3}


class _Scene:
    """One resident world with what its passes take."""

    def __init__(self, ctx, case, inp, palette_slots=0):
        self.owner = _Owner()
        self.world = self.owner.keep(World(ctx, inp.size, static_blocks=64, palette_slots=palette_slots,
                                           radiance_format=FORMATS[case["format"]]))
        self.world.set_blocks(inp.blocks)
        self.world.set_palette(inp.palette)
        self.world.set_materials(inp.mats)
        self.world.write_radiance(inp.field)
        self.world.upload_blocks()
        self.models = [self.owner.keep(Model(ctx, v)) for v in inp.models]
        self.placements = [placement(q, s, m.size) for q, s, m in zip(inp.quats, inp.shifts, self.models)]
        self.format = case["format"]
        self.views = {}
        if inp.gbuf is not None:
            h, w = inp.gbuf[1].shape
            self.matnorm, self.depth = (torch.from_numpy(a).cuda() for a in inp.gbuf)
            self.cam = camera_default(w, h)
            self.out = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")

    def field(self):
        """The current radiance field on the device."""
        ptr, size = ctypes.c_void_p(), ctypes.c_size_t()
        check(self.world.lib.lumx_world_radiance_dev(self.world.handle, ctypes.byref(ptr), ctypes.byref(size)))
        view = self.views.get(ptr.value)
        if view is None:
            wx, wy, wz = self.world.size
            kind = {"f32": "<f4", "f16": "<f2", "bf16": "<i2"}[self.format]
            view = torch.as_tensor(_DevArray(self.owner, ptr.value, (wz, wy, wx, 4), kind), device="cuda")
            if self.format == "bf16":
                view = view.view(torch.bfloat16)
            self.views[ptr.value] = view
        return view


class _Many:
    def __init__(self, case, inputs, trace):
        ctx = _context()
        self.batch = self.server = None
        slots = 0 if case["pass"] == "batch" else 64
        self.scenes = [_Scene(ctx, case, inp, slots) for inp in inputs]
        worlds = [s.world for s in self.scenes]
        if case["pass"] == "batch":
            self.batch = Batch(ctx, worlds)
            self.params = [radiance_params(rays=i.rays, time_seed=i.time_seed, max_steps=case["max_steps"])
                           for i in inputs]
            return
        self.server = Server(ctx, worlds, max_batch=32, streams=4)
        self.lists = [torch.from_numpy(i.order).cuda() for i in inputs]
        self.requests = []
        for t in trace:
            s, wid = self.scenes[t[1]], self.server.ids[t[1]]
            if t[0] == "radiance":
                _, i, first, count, rays, seed = t
                p = radiance_params(rays=rays, time_seed=seed, max_steps=case["max_steps"])
                self.requests.append(radiance_request(wid, p, self.lists[i][first:first + count]))
            else:
                self.requests.append(glossy_request(wid, s.matnorm, s.depth, s.cam, s.out, 128.0, 128))
        self.arrivals = [0.0] * len(self.requests)
        torch.cuda.synchronize()

    def __del__(self):
        for h in (self.batch, self.server):
            if h is not None:
                h.close()


def prepare(case, seed):
    if case["pass"] in ("batch", "serve"):
        return {"case": case, "many": _Many(case, *_many(case, seed))}
    inp = _single(case, seed)
    state = {"case": case, "scene": _Scene(_context(), case, inp)}
    stride = case.get("stride", 1)
    if "rays" in case:
        state["params"] = radiance_params(rays=case["rays"], time_seed=inp.time_seed, size=stride,
                                          shift=inp.time_seed % stride, max_steps=case["max_steps"],
                                          alpha=0.01 if case["pass"] == "step" else 0.1)
    if case["pass"] == "subset":
        state["requests"] = torch.from_numpy(inp.requests).cuda()
    if case["pass"] == "step":
        state["special"] = torch.from_numpy(inp.special).cuda() if len(inp.special) else None
        state["shift"] = inp.shift
    if case.get("lightmap"):
        state["lightmap"] = torch.from_numpy(inp.lightmap.view(np.int16)).cuda()
        state["proj"] = inp.proj.reshape(16)
    return state


def run(state):
    case = state["case"]
    kind = case["pass"]
    if kind in ("batch", "serve"):
        many = state["many"]
        if kind == "serve":
            many.server.run_trace(many.requests, many.arrivals)
        else:
            sc = many.scenes
            many.batch.map_models([s.models for s in sc], [s.placements for s in sc])
            many.batch.radiance(many.params)
            many.batch.glossy([s.matnorm for s in sc], [s.depth for s in sc], [s.cam for s in sc],
                              [s.out for s in sc], 128.0, case["max_steps"])
        return {"fields": [s.field() for s in many.scenes], "glossy": [s.out for s in many.scenes]}
    s = state["scene"]
    if kind == "probes":
        s.world.radiance_update(None, state["params"])
        return {"field": s.field()}
    if kind == "subset":
        s.world.radiance_update(state["requests"], state["params"])
        return {"field": s.field()}
    if kind == "step":
        s.world.shift_radiance(state["shift"])
        requests, count = s.world.select_probes_device(state["special"])
        s.world.radiance_update_counted(requests, count, state["params"])
        return {"field": s.field(), "count": count}
    if kind == "glossy":
        return {"out": s.world.glossy(s.matnorm, s.depth, s.cam, 128.0, case["max_steps"], out=s.out)}
    if kind == "diffuse":
        return {"out": s.world.diffuse(s.matnorm, s.depth, s.cam, lightmap=state.get("lightmap"),
                                       lightmap_proj=state.get("proj"), out=s.out)}
    s.world.map_models_device(s.models, s.placements)
    s.world.radiance_update(None, state["params"])
    s.world.glossy(s.matnorm, s.depth, s.cam, 128.0, case["max_steps"], out=s.out)
    return {"field": s.field(), "out": s.out}


# ---- what a pass cannot do without ------------------------------------------
# Bytes: each input read once, each output written once.  Flops: a ray's
# origin and direction, one march sample, one refined hit and one trilinear
# tap come to about 200 single operations; a glossy pixel adds its surface tap.

RAY_FLOPS, PIXEL_FLOPS, DIFFUSE_FLOPS, VOXEL_FLOPS = 200, 300, 200, 24


def _world_bytes(n, fmt):
    return n * (2 + 2 * TEXEL_BYTES[fmt]) + 64 * 4096 + 6144


def work(case):
    kind, fmt = case["pass"], case["format"]
    if kind in ("batch", "serve"):
        n = sum(x * y * z for x, y, z in _sizes(case)) / case["worlds"]
        pixels = case["width"] * case["height"]
        if kind == "batch":
            k = case["models"] * ((case["model_lo"] + case["model_hi"]) / 2) ** 3
            return {"bytes": case["worlds"] * (_world_bytes(n, fmt) + 24 * pixels + 2 * k),
                    "flops": case["worlds"] * (n * 75 * RAY_FLOPS + pixels * PIXEL_FLOPS + k * VOXEL_FLOPS)}
        updates, queries = 0.8 * case["requests"], 0.2 * case["requests"]
        return {"bytes": updates * 0.5 * n * (16 + 2 * TEXEL_BYTES[fmt]) + queries * 24 * pixels,
                "flops": updates * 0.5 * n * 75 * RAY_FLOPS + queries * pixels * PIXEL_FLOPS}
    n = case["wx"] * case["wy"] * case["wz"]
    pixels = case.get("width", 0) * case.get("height", 0)
    if kind == "probes":
        return {"bytes": _world_bytes(n, fmt), "flops": n * case["rays"] * RAY_FLOPS}
    if kind == "subset":
        m = n * case["percent"] // 100 // case["stride"]
        return {"bytes": n * 2 + m * (16 + 2 * TEXEL_BYTES[fmt]) + 64 * 4096, "flops": m * case["rays"] * RAY_FLOPS}
    if kind == "step":
        m = 0.6 * n / case["stride"]
        return {"bytes": _world_bytes(n, fmt) + m * (16 + 2 * TEXEL_BYTES[fmt]),
                "flops": m * case["rays"] * RAY_FLOPS}
    if kind == "glossy":
        return {"bytes": _world_bytes(n, fmt) - n * TEXEL_BYTES[fmt] + 24 * pixels, "flops": pixels * PIXEL_FLOPS}
    if kind == "diffuse":
        return {"bytes": n * TEXEL_BYTES[fmt] + 24 * pixels + 2 * case["lightmap"] ** 2,
                "flops": pixels * DIFFUSE_FLOPS}
    k = case["models"] * ((case["model_lo"] + case["model_hi"]) / 2) ** 3
    return {"bytes": _world_bytes(n, fmt) + 24 * pixels + 2 * k,
            "flops": n * case["rays"] * RAY_FLOPS + pixels * PIXEL_FLOPS + k * VOXEL_FLOPS}


# ---- float64 restatement ------------------------------------------------------

F64 = torch.float64
CHUNK = 1 << 23  # rays or pixels at a time


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Exact:
    """A world in float64: blocks, palette, materials, field."""

    def __init__(self, inp):
        d = _dev()
        self.size = inp.size
        self.wh = torch.tensor(inp.size, device=d)
        self.blocks = torch.from_numpy(inp.blocks.astype(np.int64)).to(d).reshape(-1)
        self.palette = torch.from_numpy(inp.palette).to(d).reshape(-1)
        self.mats = torch.from_numpy(inp.mats).to(d, F64)
        self.field = torch.from_numpy(inp.field).to(d, F64).reshape(-1, 4)

    def linear(self, b):
        wx, wy, _ = self.size
        return b[:, 0] + wx * (b[:, 1] + wy * b[:, 2])

    def voxel(self, i):
        """Block id and voxel at integer positions (block coordinates truncate, outside reads 0)."""
        b = torch.div(i, 16, rounding_mode="trunc")
        inside = ((b >= 0) & (b < self.wh)).all(1)
        blk = torch.where(inside, self.blocks[torch.where(inside, self.linear(b), 0)], 0)
        v = i & 15
        return blk, self.palette[blk * 4096 + v[:, 0] + 16 * v[:, 1] + 256 * v[:, 2]]

    def sample(self, bp):
        """Trilinear filter with wrapped addressing at texel coordinates."""
        f = torch.floor(bp)
        t = bp - f
        i = f.long()
        lo, hi = i % self.wh, (i + 1) % self.wh
        acc = torch.zeros((len(bp), 3), dtype=F64, device=bp.device)
        for c in range(8):
            pick = torch.tensor([bool(c >> a & 1) for a in range(3)], device=bp.device)
            wgt = torch.where(pick, t, 1.0 - t).prod(1, keepdim=True)
            acc += wgt * self.field[self.linear(torch.where(pick, hi, lo)), :3]
        return acc

    def march(self, o, d, max_dist, max_steps):
        """hit, voxel, fraction, normal of each ray."""
        n, dev = len(o), o.device
        hit = torch.zeros(n, dtype=torch.bool, device=dev)
        frac = torch.zeros(n, dtype=F64, device=dev)
        live = torch.arange(n, device=dev)
        lo, ld, lf, it = o, d, torch.zeros(n, dtype=F64, device=dev), 0
        ext = self.wh.to(F64) * 16.0
        while len(live):
            it += 1
            lf = lf + 0.5
            pos = lo + ld * lf[:, None]
            i = pos.long()
            blk, vox = self.voxel(i)
            edge = (torch.div(i, 16, rounding_mode="trunc") * 16).to(F64) + torch.where(ld > 0, 16.0, 0.0)
            skip = ((edge - pos) / ld).amin(1).clamp(min=0.01)
            lf = torch.where(blk == 0, lf + skip, lf)
            h = vox != 0
            out = (pos < 0).any(1) | (pos >= ext).any(1) | (lf >= max_dist)
            if max_steps and it >= max_steps:
                out[:] = True
            hit[live[h]] = True
            frac[live[h]] = lf[h]
            keep = ~(h | out)
            live, lo, ld, lf = live[keep], lo[keep], ld[keep], lf[keep]
        voxel = torch.zeros(n, dtype=torch.long, device=dev)
        normal = torch.zeros((n, 3), dtype=F64, device=dev)
        k = torch.nonzero(hit)[:, 0]
        ok, dk = o[k], d[k]
        p = ok + dk * (frac[k] - 1.5)[:, None]
        step = torch.where(dk > 0, 1, -1)
        fl = torch.floor(p)
        c1 = (fl - p) / dk
        tmax, tdelta = torch.maximum(c1, c1 + 1.0 / dk), 1.0 / dk.abs()
        v = p.long()
        st = torch.zeros_like(dk)
        cv = self.voxel(v)[1]
        for _ in range(5):
            go = cv == 0
            x, y, z = tmax.unbind(1)
            now = torch.stack([(x <= y) & (x <= z), (x >= y) & (y <= z), (z <= x) & (z <= y)], 1) & go[:, None]
            st = torch.where(go[:, None], now.to(F64), st)
            v = v + step * now
            tmax = torch.where(now, tmax + tdelta, tmax)
            cv = torch.where(go, self.voxel(v)[1], cv)
        voxel[k] = cv.long()
        normal[k] = -(step.to(F64) * st)
        frac[k] = ((tmax - tdelta) * st).sum(1)
        return hit, voxel, frac, normal

    def update(self, probes, keys, rays, time_seed, alpha, max_steps):
        """New texels of probes (linear index), rays keyed by keys."""
        dev = self.field.device
        fib = _fibonacci(rays, dev)
        wx, wy, _ = self.size
        new = torch.ones((len(probes), 4), dtype=F64, device=dev)
        light_dir = _unit(torch.tensor([0.5, 0.5, -0.9], dtype=F64, device=dev))
        sun = torch.tensor([0.9, 0.9, 0.6], dtype=F64, device=dev) * 3.0
        sky = torch.tensor([0.53, 0.81, 0.92], dtype=F64, device=dev) * 0.1
        per = max(1, CHUNK // rays)
        lane = torch.arange(rays, device=dev)
        for a in range(0, len(probes), per):
            p = probes[a:a + per]
            g = (keys[a:a + per, None] * rays + lane).reshape(-1)
            base = torch.stack([p % wx, p // wx % wy, p // (wx * wy)], 1).to(F64) * 16.0 + 8.0
            d = _unit((fib[None] + 0.1 * (_hash(g + time_seed, time_seed) - 0.5).view(len(p), rays, 3) * 2.0))
            o = base[:, None] + d * 6.0 + (_hash(g + time_seed + 1, time_seed) - 0.5).view(len(p), rays, 3) * 2.0
            d = torch.where((lane % 2 == 1)[None, :, None], -d, d)
            o, d = o.reshape(-1, 3), d.reshape(-1, 3)
            hit, vox, frac, normal = self.march(o, d, 128.0, max_steps)
            gl = -(d @ light_dir)
            light = sky + torch.where(gl > 0.95, gl, 0.0)[:, None] * sun
            k = torch.nonzero(hit)[:, 0]
            m = self.mats[vox[k]]
            bounce = self.sample((o[k] + frac[k, None] * d[k] + normal[k] * 16.0) / 16.0)
            light[k] = m[:, :3] * (bounce + m[:, 4:5])
            mean = light.view(len(p), rays, 3).mean(1)
            old = self.field[p, :3].clamp(0.0, 1.0)
            new[a:a + per, :3] = torch.nan_to_num(old * (1.0 - alpha) + mean * alpha, nan=0.0)
        return new

    def view(self):
        wx, wy, wz = self.size
        return self.field.view(wz, wy, wx, 4).cpu()

    def map(self, inp):
        """Models into the world: boxes of blocks get palette slots of their own, then the voxels."""
        dev = self.field.device
        wx, wy, wz = self.size
        blocks = inp.blocks.astype(np.int64).copy()
        source, placed = [], []
        for vox, q, shift in zip(inp.models, inp.quats, inp.shifts):
            rot = synth.quat_matrix(q)
            ext = np.array(vox.shape[::-1], float) - 1.0
            corner = np.array([[x, y, z] for x in (0, ext[0]) for y in (0, ext[1]) for z in (0, ext[2])])
            c = corner @ rot.T + np.array(shift)
            lo, hi = c.min(0), c.max(0)
            bl = np.clip(((lo.astype(int) - 1) / 16).astype(int), 0, np.array(self.size) - 1)
            bh = np.clip(((hi.astype(int) + 1) / 16).astype(int), 0, np.array(self.size) - 1)
            box = blocks[bl[2]:bh[2] + 1, bl[1]:bh[1] + 1, bl[0]:bh[0] + 1]
            fresh = box < 64
            source += list(box[fresh])
            box[fresh] = 64 + len(source) - fresh.sum() + np.arange(fresh.sum())
            placed.append((vox, rot, np.array(shift), np.floor(lo).astype(int), np.ceil(hi).astype(int)))
        static = self.palette[:64 * 4096].view(64, 4096)
        self.blocks = torch.from_numpy(blocks).to(dev).reshape(-1)
        slots = static[torch.tensor(np.array(source, np.int64), device=dev)] if source else static[:0]
        self.palette = torch.cat([static, slots]).reshape(-1)
        for vox, rot, shift, lo, hi in placed:
            count = (hi - lo + 3) // 4 * 4
            axes = [torch.arange(int(c), device=dev) + int(a) for c, a in zip(count, lo)]
            z, y, x = torch.meshgrid(axes[2], axes[1], axes[0], indexing="ij")
            w = torch.stack([x, y, z], -1).reshape(-1, 3)
            inv = torch.from_numpy(np.linalg.inv(rot)).to(dev, F64)
            m = ((w.to(F64) + 0.5 - torch.from_numpy(shift).to(dev, F64)) @ inv.T).long()
            b = torch.div(w, 16, rounding_mode="trunc")
            dims = torch.tensor(vox.shape[::-1], device=dev)
            ok = ((m >= 0) & (m < dims)).all(1) & ((b >= 0) & (b < self.wh)).all(1)
            m, w, b = m[ok], w[ok], b[ok]
            val = torch.from_numpy(vox).to(dev)[m[:, 2], m[:, 1], m[:, 0]]
            slot = self.blocks[self.linear(b)]
            put = (val != 0) & (slot >= 64)
            v = w[put] & 15
            self.palette[slot[put] * 4096 + v[:, 0] + 16 * v[:, 1] + 256 * v[:, 2]] = val[put]

    def pixels(self, inp):
        """Material row, normal and origin of every pixel, and the camera direction."""
        dev = self.field.device
        mn, dp = (torch.from_numpy(a).to(dev) for a in inp.gbuf)
        h, w = dp.shape
        cam = camera_default(w, h)
        vec = {k: torch.tensor(list(getattr(cam, k)), dtype=F64, device=dev)
               for k in ("campos", "camdir", "horiz_scaled", "verti_scaled", "light_dir")}
        cx = (torch.arange(w, device=dev).to(F64) + 0.5) / w * 2.0 - 1.0
        cy = (torch.arange(h, device=dev).to(F64) + 0.5) / h * 2.0 - 1.0
        origin = (vec["campos"] + vec["horiz_scaled"] * cx[None, :, None] + vec["verti_scaled"] * cy[:, None, None]
                  + vec["camdir"] * (dp.to(F64) * 1000.0)[..., None]).reshape(-1, 3)
        normal = mn[..., 1:].reshape(-1, 3).to(F64) / 255.0 * 2.0 - 1.0
        return self.mats[mn[..., 0].reshape(-1).long()], normal, origin, vec, (h, w)

    def glossy(self, inp, max_steps):
        mat, normal, origin, vec, (h, w) = self.pixels(inp)
        out = torch.zeros((h * w, 4), dtype=F64, device=mat.device)
        sun = torch.tensor([0.9, 0.9, 0.6], dtype=F64, device=mat.device) * 0.5
        sky = torch.tensor([0.53, 0.81, 0.92], dtype=F64, device=mat.device) * 0.1
        keep = torch.nonzero(mat[:, 5] <= 0.5)[:, 0]
        for a in range(0, len(keep), CHUNK):
            p = keep[a:a + CHUNK]
            m, nrm, o = mat[p], normal[p], origin[p]
            r = m[:, :3].clone()
            light = r * (m[:, 4:5] + self.sample((o + nrm * 16.0) / 16.0))
            d = vec["camdir"] - 2.0 * (nrm @ vec["camdir"])[:, None] * nrm
            hit, vox, frac, hn = self.march(o, d, 128.0, max_steps)
            s = -(d @ vec["light_dir"])
            add = sky * r + torch.where(s > 0.9, s - 0.9, 0.0)[:, None] * 10.0 * sun * r
            k = torch.nonzero(hit)[:, 0]
            hm = self.mats[vox[k]]
            add[k] = r[k] * hm[:, :3] * (hm[:, 4:5] + self.sample((o[k] + frac[k, None] * d[k] + hn[k] * 16.0) / 16.0))
            out[p, :3] = (light + add) / 8.0
            out[p, 3] = 1.0 - m[:, 5]
        return out.view(h, w, 4).cpu()

    def diffuse(self, inp):
        mat, normal, origin, vec, (h, w) = self.pixels(inp)
        light = 2.0 * self.sample((origin + normal * 6.0) / 16.0 - 0.5) + mat[:, 4:5]
        if hasattr(inp, "lightmap"):
            lm = torch.from_numpy(inp.lightmap.astype(np.int64)).to(mat.device)
            size = lm.shape[0]
            side = torch.where((normal @ vec["light_dir"] > 0.0)[:, None], -0.9, 0.9)
            q = origin + normal * side
            proj = torch.from_numpy(inp.proj).to(mat.device, F64)
            c = q @ proj[:3, :3] + proj[3, :3]
            uv, ref = (c[:, :2] + 1.0) / 2.0, (1.0 + c[:, 2]).clamp(0.0, 1.0)
            lit = torch.zeros(len(q), dtype=F64, device=mat.device)
            for tap in ((-1, 0), (0, 0), (1, 0), (0, -1), (0, 1)):
                t = uv + torch.tensor(tap, dtype=F64, device=mat.device) / 1024.0
                i = torch.floor(t * size).long() % (2 * size)
                i = torch.where(i >= size, 2 * size - 1 - i, i)
                lit += (ref < lm[i[:, 1], i[:, 0]].to(F64) / 65535.0).to(F64)
            light = light + (lit / 5.0 * 0.15)[:, None]
        out = torch.ones((h * w, 4), dtype=F64, device=mat.device)
        out[:, :3] = light * mat[:, :3] / 8.0
        return out.view(h, w, 4).cpu()


def _unit(v):
    return v / v.square().sum(-1, keepdim=True).sqrt()


def _fibonacci(rays, dev):
    """The reference's directions from its single-precision angle."""
    i = np.arange(rays, dtype=np.float32)
    phi = np.float32(np.sqrt(np.float32(5.0)) * np.float32(0.5) + np.float32(0.5))
    a = i * (phi - np.float32(1.0))
    ang = np.float32(2.0) * np.float32(math.pi) * (a - np.floor(a))
    ct = np.float32(1.0) - (np.float32(2.0) * i + np.float32(1.0)) * (np.float32(1.0) / np.float32(rays))
    st = np.sqrt(np.clip(1.0 - ct.astype(np.float64) ** 2, 0.0, 1.0))
    c, s = np.cos(ang.astype(np.float64)), np.sin(ang.astype(np.float64))
    return torch.from_numpy(np.stack([c * st, s * st, ct.astype(np.float64)], 1)).to(dev)


def _hash(x, t):
    """Three uniform numbers in [0, 1) per key (32-bit integer hash)."""
    mask, mul = 0xffffffff, 1103515245
    x = x & mask
    y, z = torch.full_like(x, t & mask), torch.full_like(x, t & mask)
    for _ in range(3):
        x, y, z = (((x >> 8) ^ y) * mul) & mask, (((y >> 8) ^ z) * mul) & mask, (((z >> 8) ^ x) * mul) & mask
    return torch.stack([x, y, z], 1).to(F64) / 4294967296.0


def _selected(inp):
    """Probes with a solid block among their 27 clamped neighbours, then the specials not among them."""
    solid = np.pad(inp.blocks > 0, 1, mode="edge")
    wz, wy, wx = inp.blocks.shape
    near = np.zeros(inp.blocks.shape, bool)
    for dz in range(3):
        for dy in range(3):
            for dx in range(3):
                near |= solid[dz:dz + wz, dy:dy + wy, dx:dx + wx]
    flat = near.reshape(-1)
    special = inp.special[:, 0] + wx * (inp.special[:, 1] + wy * inp.special[:, 2]).astype(np.int64)
    return np.concatenate([np.nonzero(flat)[0], special[~flat[special]]])


def exact(case, seed):
    kind = case["pass"]
    if kind in ("batch", "serve"):
        inputs, trace = _many(case, seed)
        worlds = [_Exact(i) for i in inputs]
        h, w = inputs[0].gbuf[1].shape
        glossy = [torch.zeros((h, w, 4), dtype=F64) for _ in inputs]
        if kind == "batch":
            for k, (ew, inp) in enumerate(zip(worlds, inputs)):
                ew.map(inp)
                every = torch.arange(inp.n, device=_dev())
                ew.field = ew.update(every, every, inp.rays, inp.time_seed, 0.1, case["max_steps"])
                glossy[k] = ew.glossy(inp, case["max_steps"])
        for t in trace:
            ew, inp = worlds[t[1]], inputs[t[1]]
            if t[0] == "radiance":
                _, _, first, count, rays, time_seed = t
                rows = torch.from_numpy(inp.order[first:first + count].astype(np.int64)).to(_dev())
                p = ew.linear(rows)
                ew.field[p] = ew.update(p, torch.arange(count, device=_dev()), rays, time_seed, 0.1,
                                        case["max_steps"])
            else:
                glossy[t[1]] = ew.glossy(inp, 128)
        return {"fields": [ew.view() for ew in worlds], "glossy": glossy}
    inp = _single(case, seed)
    ew = _Exact(inp)
    if kind == "glossy":
        return {"out": ew.glossy(inp, case["max_steps"])}
    if kind == "diffuse":
        return {"out": ew.diffuse(inp)}
    every = torch.arange(inp.n, device=_dev())
    if kind in ("probes", "frame"):
        if kind == "frame":
            ew.map(inp)
        ew.field = ew.update(every, every, case["rays"], inp.time_seed, 0.1, case["max_steps"])
        return {"field": ew.view()} if kind == "probes" else {"field": ew.view(),
                                                              "out": ew.glossy(inp, case["max_steps"])}
    stride = case["stride"]
    if kind == "subset":
        listed_probes = ew.linear(torch.from_numpy(inp.requests.astype(np.int64)).to(_dev()))
        alpha = 0.1
    else:
        wx, wy, wz = inp.size
        old = ew.field.view(wz, wy, wx, 4)
        moved = old.clone()
        dst, src = [slice(None)] * 3, [slice(None)] * 3
        for axis, s in zip((2, 1, 0), inp.shift):
            size = old.shape[axis]
            dst[axis], src[axis] = slice(max(-s, 0), size - max(s, 0)), slice(max(s, 0), size - max(-s, 0))
        moved[tuple(dst)] = old[tuple(src)]
        ew.field = moved.reshape(-1, 4)
        listed_probes = torch.from_numpy(_selected(inp)).to(_dev())
        alpha = 0.01
    count = len(listed_probes)
    p = listed_probes[inp.time_seed % stride::stride][:count // stride]
    ew.field[p] = ew.update(p, torch.arange(len(p), device=_dev()), case["rays"], inp.time_seed, alpha,
                            case["max_steps"])
    if kind == "subset":
        return {"field": ew.view()}
    return {"field": ew.view(), "count": torch.tensor([count])}
