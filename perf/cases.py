"""Measured cases: what programs built on this library have it do.

Twelve listed cases through the public Python binding (`solhip`, the C ABI's
ctypes face), from a pick of a few hundred rays to a 1080p path-traced frame
of an animated 10,000-instance scene; `draw` gives more of the same ranges.
Rendered images start a new accumulation in every pass (accum_start_frame =
frame), so a pass's image depends on the state's inputs alone.

Kinds (field "kind" of a case):
  query     solhip_trace_rays on rays and hits resident on the GPU
  ao_glsl   the example-4 program (ao.rgen / rchit / rmiss) on the Cornell box
  pt_glsl   the example-5 program (pathtrace.*) on the Cornell box
  ao        plain ambient occlusion, one primary and n_ao rays per hit
  pt        the wavefront path tracer; rebuild = 1: every BLAS and the TLAS
            rebuilt before the frame (an animated scene)
  load      a static mesh: fast-trace BLAS build, TLAS build, first rays,
            all released again
  rebuild   BLASes and TLAS of a moving scene rebuilt, then rays against it
  server    a burst of jobs on the render server
  mlp       the radiance-cache network: a query batch, then training steps
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "sol-rs_amd", "python"))

import solhip  # noqa: E402
from solhip import scenes  # noqa: E402
from solhip.records import HIT, RAY  # noqa: E402


def listed():
    return [
        # object picking / line-of-sight checks of an interactive tool: a few rays, latency only
        {"name": "pick", "kind": "query", "scene": "cornell", "size": 0, "fast": 0, "n": 257, "any": 0},
        # a lightmap or visibility bake: incoherent rays in one large call
        {"name": "bake", "kind": "query", "scene": "terrain", "size": 512, "fast": 1, "n": 1500007, "any": 0},
        # example 4 at its own window size
        {"name": "ao_example", "kind": "ao_glsl", "W": 900, "H": 600},
        # example 5 at its own window size, 8 samples and 32 bounces
        {"name": "pathtrace_example", "kind": "pt_glsl", "W": 1280, "H": 720, "spp": 8, "depth": 32, "sky": 0},
        # the benchmark's frame: 2.1M triangles, 1080p, 8 AO rays per hit
        {"name": "ao_1080p", "kind": "ao", "scene": "terrain", "size": 1024, "fast": 1, "W": 1920, "H": 1080,
         "n_ao": 8, "any": 0},
        # a small preview with sizes that are no multiple of a tile, first-hit occlusion, a quick build
        {"name": "ao_preview", "kind": "ao", "scene": "terrain", "size": 181, "fast": 0, "W": 357, "H": 243,
         "n_ao": 16, "any": 1},
        # path tracing a closed room with direct light sampling, replayed as a graph
        {"name": "pt_room", "kind": "pt", "scene": "cornell", "size": 0, "fast": 1, "W": 512, "H": 512, "spp": 16,
         "depth": 4, "nee": 1, "rr": 0, "sky": 0, "streams": 1, "graph": 1, "rebuild": 0},
        # one frame of an animated scene: 10,000 instances of 5 BLASes, all rebuilt, 1080p
        {"name": "pt_animated", "kind": "pt", "scene": "instances", "size": 10000, "fast": 0, "W": 1920, "H": 1080,
         "spp": 16, "depth": 8, "nee": 1, "rr": 3, "sky": 2, "streams": 1, "graph": 0, "rebuild": 1},
        # loading a 2.1M-triangle mesh for static use
        {"name": "load_mesh", "kind": "load", "scene": "terrain", "size": 1024, "n": 500},
        # physics or animation of a few hundred bodies: latency of the rebuilds
        {"name": "rebuild_bodies", "kind": "rebuild", "scene": "instances", "size": 500, "n": 60001},
        # a server's burst of mixed jobs
        {"name": "serve_burst", "kind": "server", "jobs": 8, "edge": 320, "spp": 24, "depth": 6, "streams": 0},
        # the radiance cache of a frame: queries of its pixels, 4 training steps
        {"name": "cache_network", "kind": "mlp", "n": 1000003, "rows": 65536, "steps": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "query", "ao_glsl", "pt_glsl", "ao", "pt", "load", "rebuild", "server", "mlp"])
    if kind == "query":
        scene = rng.choice(["cornell", "terrain", "instances"])
        size = {"cornell": 0, "terrain": _log(rng, 16, 512), "instances": _log(rng, 20, 2000)}[scene]
        return {"kind": kind, "scene": scene, "size": size, "fast": rng.randint(0, 1), "n": _log(rng, 1, 3000000),
                "any": rng.randint(0, 1)}
    if kind == "ao_glsl":
        return {"kind": kind, "W": _log(rng, 100, 1280), "H": _log(rng, 100, 720)}
    if kind == "pt_glsl":
        return {"kind": kind, "W": _log(rng, 100, 1280), "H": _log(rng, 100, 720), "spp": rng.randint(1, 8),
                "depth": rng.choice([4, 8, 32]), "sky": rng.randint(0, 1)}
    if kind == "ao":
        return {"kind": kind, "scene": "terrain", "size": _log(rng, 16, 1024), "fast": rng.randint(0, 1),
                "W": _log(rng, 60, 1920), "H": _log(rng, 60, 1080), "n_ao": rng.choice([1, 4, 8, 16]),
                "any": rng.randint(0, 1)}
    if kind == "pt":
        scene = rng.choice(["cornell", "terrain", "instances"])
        size = {"cornell": 0, "terrain": _log(rng, 16, 512), "instances": _log(rng, 20, 2000)}[scene]
        return {"kind": kind, "scene": scene, "size": size, "fast": rng.randint(0, 1), "W": _log(rng, 100, 1280),
                "H": _log(rng, 100, 720), "spp": _log(rng, 1, 16), "depth": rng.randint(2, 8),
                "nee": rng.randint(0, 1), "rr": rng.choice([0, 3]), "sky": rng.choice([0, 1, 2]),
                "streams": rng.randint(0, 1), "graph": rng.randint(0, 1), "rebuild": rng.randint(0, 1)}
    if kind == "load":
        return {"kind": kind, "scene": "terrain", "size": _log(rng, 16, 1024), "n": _log(rng, 1, 500)}
    if kind == "rebuild":
        return {"kind": kind, "scene": "instances", "size": _log(rng, 2, 3000), "n": _log(rng, 1000, 200000)}
    if kind == "server":
        return {"kind": kind, "jobs": rng.randint(1, 8), "edge": _log(rng, 64, 320), "spp": _log(rng, 1, 24),
                "depth": rng.randint(4, 8), "streams": rng.randint(0, 1)}
    return {"kind": "mlp", "n": _log(rng, 100, 1000003), "rows": _log(rng, 100, 65536), "steps": rng.randint(1, 4)}


# ---- inputs -------------------------------------------------------------------

_context = []


def _ctx():
    """the program's one context"""
    if not _context:
        _context.append(solhip.Context(0))
    return _context[0]


class _Mem:
    """a device buffer of the library seen as a torch tensor; the tensor keeps
    this object, and with it the buffer, alive"""

    def __init__(self, count, dtype):
        dt = np.dtype(dtype)
        self.buf = _ctx().buffer(max(16, count * dt.itemsize))
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": dt.str, "data": (self.buf.addr, False),
                                         "version": 2, "strides": None}

    def __del__(self):
        self.buf.destroy()

    def tensor(self):
        return torch.as_tensor(self, device="cuda:0")


class _Scene:
    """a GpuScene with an end"""

    def __init__(self, sd, fast):
        self.sd = sd
        self.gs = solhip.GpuScene(_ctx(), sd, build_flags=solhip.BUILD_PREFER_FAST_TRACE if fast else 0)

    def __del__(self):
        c = _ctx()
        c.sync()
        c.tlas_destroy(self.gs.tlas)
        for b in self.gs.blas:
            c.blas_destroy(b)
        for b in self.gs.bufs:
            b.destroy()


class _Program:
    def __init__(self, kind, spec):
        self.h = _ctx().program(kind, spec)

    def __del__(self):
        _ctx().program_destroy(self.h)


def _scene_data(kind, size, seed):
    if kind == "cornell":
        return scenes.cornell_box()
    if kind == "terrain":
        return scenes.heightfield(size, seed=1 + seed)
    # the 10,000-instance scene holds the full 1M-triangle tube; smaller scenes a coarser one
    tube = (500, 1000) if size >= 4000 else (60, 120)
    return scenes.instanced(size, seed=2 + seed, tube=tube, spread=50.0 * (size / 10000.0) ** (1.0 / 3.0))


def _rays(sd, scene, n, rng):
    """camera-like rays into the room; from above a terrain, or from anywhere
    among the instances, into all directions"""
    r = np.zeros(n, RAY)
    if scene == "cornell":
        o = np.tile(np.array([0.0, 0.0, 3.4]), (n, 1))
        d = rng.uniform(-1.0, 1.0, size=(n, 3)) - o
    else:
        if scene == "terrain":
            o = rng.uniform(-1.0, 1.0, size=(n, 3))
            o[:, 1] = rng.uniform(0.15, 0.6, size=n)
        else:
            o = rng.uniform(-0.5, 0.5, size=(n, 3)) * sd.extent
        d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r["o"], r["d"], r["tmin"], r["tmax"] = o, d, 1e-4, 10000.0
    return r


class _Query:
    """rays and hit records on the GPU, the hits also as tensors"""

    def __init__(self, sd, scene, n, flags, rng):
        self.n, self.flags = n, flags
        self.rays = _Mem(n * RAY.itemsize, np.uint8)
        self.rays.buf.upload(_rays(sd, scene, n, rng))
        self.hits = _Mem(n * (HIT.itemsize // 4), np.float32)
        t = self.hits.tensor().view(n, HIT.itemsize // 4)
        if flags & solhip.TRACE_TERMINATE_ON_FIRST_HIT:
            # which of a ray's hits a first-hit query reports is left open; whether it hit is not
            # (the geometry index: 0, or ~0 on a miss)
            self.out = {"hit": t.view(torch.int32)[:, 5]}
        else:
            self.out = {"tuv": t[:, :3], "ids": t.view(torch.int32)[:, 3:]}

    def trace(self, tlas):
        _ctx().trace_rays_dev(tlas, self.rays.buf, self.hits.buf, self.n, self.flags)


class _Image:
    def __init__(self, W, H, rgba8=False):
        self.W, self.H = W, H
        self.acc = _Mem(W * H * 4, np.float32)
        self.acc.buf.fill(0)
        self.out = {"image": self.acc.tensor().view(H, W, 4)}
        self.rgba8 = _Mem(W * H, np.int32) if rgba8 else None
        if rgba8:
            self.out["rgba8"] = self.rgba8.tensor()
        self.desc = solhip.Images(self.acc.buf.h, self.rgba8.buf.h if rgba8 else 0, 0, 0, 0, 0)


class _Owned:
    """a server or network with an end"""

    def __init__(self, obj):
        self.obj = obj

    def __del__(self):
        self.obj.close()


class _State:
    pass


def _moved(sd, rng):
    """the scene's instances turned and shifted a little (the next frame of an animation)"""
    xf = []
    for m in scenes.instance_xforms(sd):
        m = m.copy()
        m[:3, 3] += rng.uniform(-0.5, 0.5, size=3)
        xf.append(m)
    return scenes.with_transforms(sd, xf)


def _mlp_inputs(n, rng):
    """feature rows as the cache makes them: sin / cos octaves of a position,
    directions, albedo, roughness, metallic, 1, zeros (BF16)"""
    x = np.zeros((n, 64), np.float32)
    p = rng.random(size=(n, 3), dtype=np.float32)
    for a in range(3):
        for o in range(6):
            x[:, 12 * a + 2 * o] = np.sin(p[:, a] * np.float32(math.pi * 2 ** o))
            x[:, 12 * a + 2 * o + 1] = np.cos(p[:, a] * np.float32(math.pi * 2 ** o))
    x[:, 36:42] = rng.random(size=(n, 6), dtype=np.float32) * 2.0 - 1.0
    x[:, 42:46] = rng.random(size=(n, 4), dtype=np.float32)
    x[:, 47] = 1.0
    return torch.from_numpy(x).to(torch.bfloat16), p


def _mlp_targets(p, rng):
    t = np.zeros((len(p), 4), np.float32)
    t[:, 0] = 0.5 + 0.4 * np.sin(6.0 * p[:, 0]) * np.cos(5.0 * p[:, 1])
    t[:, 1] = 0.5 + 0.3 * p[:, 1] * p[:, 2]
    t[:, 2] = 0.6 + 0.2 * np.tanh(p[:, 0] - p[:, 2])
    t[:, :3] *= rng.random(size=(len(p), 3), dtype=np.float32) + 0.5
    return t


def _mlp_data(c, seed):
    rng = np.random.default_rng(1000 + seed)
    xq, _ = _mlp_inputs(c["n"], rng)
    xt, pt = _mlp_inputs(c["rows"], rng)
    return xq, xt, _mlp_targets(pt, rng)


def _jobs(c, seed):
    """(scene index, W, H, samples) of a burst: sizes and sample counts around the case's"""
    sizes, rng = np.random.default_rng(7), np.random.default_rng(7000 + seed)
    out = []
    for k in range(c["jobs"]):
        w, h = (int(max(16, c["edge"] * f)) for f in sizes.uniform(0.5, 1.0, size=2))
        out.append((k % 2, w, h, int(max(1, c["spp"] * rng.uniform(0.25, 1.0)))))
    return out


def prepare(case, seed):
    c = dict(case)
    kind = c["kind"]
    rng = np.random.default_rng(seed)
    s = _State()
    s.c = c
    frame = seed % 100000
    if kind == "query":
        sd = _scene_data(c["scene"], c["size"], seed % 5)
        s.scene = _Scene(sd, c["fast"])
        s.q = _Query(sd, c["scene"], c["n"], solhip.TRACE_TERMINATE_ON_FIRST_HIT if c["any"] else 0, rng)
    elif kind in ("ao_glsl", "pt_glsl", "ao", "pt"):
        sd = _scene_data(c.get("scene", "cornell"), c.get("size", 0), seed % 5)
        s.scene = _Scene(sd, c.get("fast", 1))
        s.img = _Image(c["W"], c["H"], kind in ("pt_glsl", "pt"))
        s.frame, s.uniforms = frame, sd.uniforms(c["W"], c["H"], frame)
        code = {"ao_glsl": solhip.PROG_AO_GLSL, "pt_glsl": solhip.PROG_PATHTRACE_GLSL, "ao": solhip.PROG_AO,
                "pt": solhip.PROG_PATHTRACE}[kind]
        spec = solhip.spec_default(code)
        if kind == "ao_glsl":
            s.blue = _Mem(256 * 256 * 4, np.uint8)
            s.blue.buf.upload(scenes.blue_noise_synthetic(256, seed=7 + seed))
            s.img.desc.blue_noise, s.img.desc.blue_w, s.img.desc.blue_h = s.blue.buf.h, 256, 256
        elif kind == "pt_glsl":
            spec.spp_per_frame, spec.max_depth, spec.enable_sky = c["spp"], c["depth"], c["sky"]
        elif kind == "ao":
            spec.n_ao, spec.ao_tmin, spec.ao_tmax = c["n_ao"], 1e-4 * sd.extent, 0.1 * sd.extent
            spec.ao_any_hit = c["any"]
        else:
            spec.spp_per_frame, spec.max_depth, spec.enable_sky = c["spp"], c["depth"], c["sky"]
            spec.nee, spec.rr_start, spec.sample_streams, spec.wf_graph = c["nee"], c["rr"], c["streams"], c["graph"]
        s.prog = _Program(code, spec)
        if c.get("rebuild"):
            s.descs = _moved(sd, rng).instance_descs if c["scene"] == "instances" else sd.instance_descs
    elif kind == "load":
        sd = _scene_data(c["scene"], c["size"], seed % 5)
        b = sd.blas[0]
        s.sd, s.blas = sd, b
        s.vb, s.ib = _Mem(b.vertices.nbytes, np.uint8), _Mem(b.indices.nbytes, np.uint8)
        s.vb.buf.upload(b.vertices)
        s.ib.buf.upload(b.indices)
        s.q = _Query(sd, c["scene"], c["n"], 0, rng)
    elif kind == "rebuild":
        sd = _scene_data(c["scene"], c["size"], seed % 5)
        s.scene = _Scene(sd, 0)
        s.descs = _moved(sd, rng).instance_descs
        s.q = _Query(sd, c["scene"], c["n"], 0, rng)
    elif kind == "server":
        s.scenes = [_Scene(_scene_data("cornell", 0, 0), 1), _Scene(_scene_data("terrain", 256, seed % 5), 1)]
        s.jobs = [(sc, s.scenes[sc].sd.uniforms(w, h, frame + k), spp, _Image(w, h))
                  for k, (sc, w, h, spp) in enumerate(_jobs(c, seed))]
        s.owned = _Owned(solhip.Server(_ctx(), 1 << 30, 16))
        s.server = s.owned.obj
        s.ids = [s.server.scene(x.gs) for x in s.scenes]
        s.frame = frame
    else:
        xq, xt, t = _mlp_data(c, seed)
        s.owned = _Owned(solhip.Mlp(_ctx(), seed=1 + seed % 1000))
        s.net = s.owned.obj
        s.xq, s.xt = _Mem(xq.numel() * 2, np.uint8), _Mem(xt.numel() * 2, np.uint8)
        s.xq.buf.upload(xq.view(torch.int16).numpy())
        s.xt.buf.upload(xt.view(torch.int16).numpy())
        s.t = _Mem(t.size, np.float32)
        s.t.buf.upload(t)
        s.y = _Mem(c["n"] * 4, np.float32)
        s.out = s.y.tensor().view(c["n"], 4)[:, :3]
    return s


# ---- one pass -------------------------------------------------------------------

def _rebuild(gs, descs):
    for k in range(len(gs.blas)):
        gs.rebuild_blas(k)
    gs.update_instances(descs)


def run(s):
    c, ctx, kind = s.c, _ctx(), s.c["kind"]
    if kind == "query":
        s.q.trace(s.scene.gs.tlas)
        return s.q.out
    if kind in ("ao_glsl", "pt_glsl", "ao", "pt"):
        gs = s.scene.gs
        if c.get("rebuild"):
            _rebuild(gs, s.descs)
        ctx.trace(s.prog.h, gs.tlas, gs.tables, s.uniforms, s.frame, s.img.desc, s.img.W, s.img.H)
        return s.img.out
    if kind == "load":
        blas = ctx.blas_build(s.vb.buf, 64, len(s.blas.vertices), s.ib.buf, len(s.blas.indices),
                              flags=solhip.BUILD_PREFER_FAST_TRACE)
        descs = s.sd.instance_descs.copy()
        descs["blas"] = blas
        tlas = ctx.tlas_build(descs)
        s.q.trace(tlas)
        ctx.tlas_destroy(tlas)
        ctx.blas_destroy(blas)
        return s.q.out
    if kind == "rebuild":
        _rebuild(s.scene.gs, s.descs)
        s.q.trace(s.scene.gs.tlas)
        return s.q.out
    if kind == "server":
        spec = solhip.spec_default(solhip.PROG_PATHTRACE)
        spec.max_depth, spec.enable_sky, spec.nee, spec.rr_start = c["depth"], 2, 1, 3
        spec.sample_streams = c["streams"]
        for k, (sc, uniforms, spp, img) in enumerate(s.jobs):
            spec.spp_per_frame = spp
            s.server.submit(s.ids[sc], img.W, img.H, spec, uniforms, img.acc.buf, accum_start=s.frame + k)
        s.server.run()
        return [img.out["image"] for _, _, _, img in s.jobs]
    s.net.forward(s.xq.buf, c["n"], s.y.buf)
    # the gradient of the training batch, then the training steps
    grad, loss = s.net.gradient(s.xt.buf, s.t.buf, c["rows"])
    s.net.train(s.xt.buf, s.t.buf, c["rows"], c["steps"])
    return {"y": s.out, "grad": grad, "loss": loss}


# ---- what a pass cannot do without ------------------------------------------------

def _triangles(c):
    if c.get("scene") == "terrain":
        return 2 * c["size"] ** 2
    if c.get("scene") == "instances":
        return 20 + 1280 + 20480 + 12 + (1000000 if c["size"] >= 4000 else 14400)
    return 36


def work(case):
    """Bytes: inputs read once and outputs written once (rays 32 B, hits 24 B,
    triangles 36 B of positions, instances 64 B, pixels).  Flops: only the
    network has a count that does not depend on the method."""
    c, kind = case, case["kind"]
    tri = _triangles(c) * 36
    inst = 64 * c["size"] if c.get("scene") == "instances" else 0
    if kind == "query":
        return {"bytes": c["n"] * 56 + tri + inst, "flops": 0}
    if kind in ("load", "rebuild"):
        return {"bytes": c["n"] * 56 + tri + inst, "flops": 0}
    if kind == "server":
        return {"bytes": c["jobs"] * 0.5625 * c["edge"] ** 2 * 16 + 36 * 2 * 256 ** 2, "flops": 0}
    if kind == "mlp":
        macs = 4 * 64 * 64 + 64 * 3
        train = c["rows"] * (1 + c["steps"])
        return {"bytes": c["n"] * (128 + 12) + train * (128 + 12), "flops": 2.0 * macs * (c["n"] + 3 * train)}
    px = c["W"] * c["H"]
    return {"bytes": px * (16 if kind in ("ao", "ao_glsl") else 20) + tri + inst, "flops": 0}


# ---- the same in 64 bits ------------------------------------------------------------

def _closest(sd, rays):
    """closest hits by brute force in float64: (t, u, v), misses (-1, 0, 0)"""
    dev = "cuda:0" if torch.cuda.is_available() else "cpu"
    o = torch.from_numpy(rays["o"].astype(np.float64)).to(dev)
    d = torch.from_numpy(rays["d"].astype(np.float64)).to(dev)
    best = torch.full((len(rays),), float("inf"), dtype=torch.float64, device=dev)
    bu, bv = torch.zeros_like(best), torch.zeros_like(best)
    tmin, tmax = float(rays["tmin"][0]), float(rays["tmax"][0])
    for k, m in enumerate(scenes.instance_xforms(sd)):
        b = sd.blas[int(sd.instance_descs[k]["blas"])]
        p = b.vertices["pos"][:, :3].astype(np.float64) @ m[:3, :3].T + m[:3, 3]
        tri = torch.from_numpy(p[b.indices.reshape(-1, 3)]).to(dev)
        step = max(1, (1 << 24) // len(rays))
        for i in range(0, len(tri), step):
            v0, e1, e2 = tri[i:i + step, 0], tri[i:i + step, 1], tri[i:i + step, 2]
            e1, e2 = e1 - v0, e2 - v0
            n = torch.linalg.cross(e1, e2)
            det = -(d @ n.T)
            ao = o[:, None, :] - v0[None]
            dao = torch.linalg.cross(ao, d[:, None, :].expand_as(ao))
            t = (ao * n).sum(-1) / det
            u, v = (dao * e2).sum(-1) / det, -(dao * e1).sum(-1) / det
            hit = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= tmin) & (t <= tmax)
            t = torch.where(hit, t, torch.full_like(t, float("inf")))
            tt, j = t.min(dim=1)
            at = torch.arange(len(rays), device=dev)
            new = tt < best
            best = torch.where(new, tt, best)
            bu, bv = torch.where(new, u[at, j], bu), torch.where(new, v[at, j], bv)
    miss = torch.isinf(best)
    zero = torch.zeros_like(best)
    return torch.stack([torch.where(miss, zero - 1.0, best), torch.where(miss, zero, bu),
                        torch.where(miss, zero, bv)], dim=1).cpu()


def exact(case, seed):
    """Closest hits by brute force where rays times triangles stay within
    about a billion; the network in float64.  Images have no such value: they
    are means over rays whose directions come from a 32-bit generator, each
    decided by comparisons."""
    c, kind = dict(case), case["kind"]
    if kind in ("query", "load") and not c.get("any") and c["scene"] != "instances":
        if c["n"] * _triangles(c) > 1.1e9:
            return None
        sd = _scene_data(c["scene"], c["size"], seed % 5)
        rays = _rays(sd, c["scene"], c["n"], np.random.default_rng(seed))
        return {"tuv": _closest(sd, rays), "ids": None}
    if kind != "mlp":
        return None
    dev = "cuda:0" if torch.cuda.is_available() else "cpu"
    net = solhip.Mlp(_ctx(), seed=1 + seed % 1000)   # the initial weights of the same seed
    w = net.params()
    net.close()
    W = [torch.from_numpy(w[4096 * i:4096 * (i + 1)].reshape(64, 64).astype(np.float64)).to(dev) for i in range(4)]
    W.append(torch.from_numpy(w[16384:].reshape(64, 16).astype(np.float64)).to(dev))
    for x in W:
        x.requires_grad_(True)

    def net64(x):
        h = x.to(dev).to(torch.float64)
        for i in range(4):
            h = torch.relu(h @ W[i])
        return (h @ W[4])[:, :3]

    xq, xt, t = _mlp_data(c, seed)
    with torch.no_grad():
        y = net64(xq)
    p, tt = net64(xt), torch.from_numpy(t[:, :3].astype(np.float64)).to(dev)
    loss = (((p - tt) ** 2) / (p.detach() ** 2 + 0.01)).sum() / c["rows"]
    loss.backward()
    grad = torch.cat([x.grad.reshape(-1) for x in W])
    return {"y": y.cpu(), "grad": grad.cpu(), "loss": float(loss.detach())}
