"""Wavefront path tracer: small queues finished path by path (k_pt_finish)
against the bounce-by-bounce passes (which SOLHIP_PROFILE_TIME keeps) and the
oracle: the same image, bit for bit, and the same number of extension and shadow
rays; also frames that start in passes and end in the finishing kernel."""
import numpy as np
import pytest

import solhip
from solhip import scenes
from solhip.api import PROFILE_TIME

pytestmark = pytest.mark.gpu

SCENES = {"cornell": scenes.cornell_box, "instances": scenes.random_instances,
          "terrain": lambda: scenes.heightfield(48)}


def _spec(spp, depth, nee, rr, sky, streams, graph=0):
    s = solhip.spec_default(solhip.PROG_PATHTRACE)
    s.spp_per_frame, s.max_depth, s.nee, s.rr_start, s.enable_sky = spp, depth, nee, rr, sky
    s.sample_streams, s.wf_graph = streams, graph
    return s


def _run(ctx, gs, sd, spec, W, H, frames, profile=0):
    prog = ctx.program(solhip.PROG_PATHTRACE, spec)
    acc = ctx.upload(np.zeros((H, W, 4), np.float32))
    img = solhip.Images(acc.h, 0, 0, 0, 0, 0)
    for k in ("pt_extend", "pt_shadow"):
        ctx.kernel_stats(k, reset=True)
    ctx.profile(profile)
    for f in range(frames):
        ctx.trace(prog, gs.tlas, gs.tables, sd.uniforms(W, H, 3 + f), 3, img, W, H)
    ctx.sync()
    ctx.profile(0)
    rays = [ctx.kernel_stats(k, reset=True).counters for k in ("pt_extend", "pt_shadow")]
    assert all(r.overflow == 0 for r in rays)
    out = acc.download(np.float32).reshape(H, W, 4)
    ctx.program_destroy(prog)
    return out, [r.rays for r in rays]


def _oracle(oracle, sd, s, W, H, frames):
    ref = np.zeros((H, W, 4), np.float32)
    cfg = oracle.PTConfig(s.enable_sky, s.spp_per_frame, s.max_depth, s.rr_start, s.nee, s.sample_streams)
    sc = oracle.Scene(sd)
    n = sum(sc.render_pathtrace(sd.uniforms(W, H, 3 + f), cfg, 3, ref, None, W, H) for f in range(frames))
    return ref, n


@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("spp,depth,nee,rr,sky,streams", [
    (1, 0, 1, 0, 1, 0), (3, 4, 1, 0, 0, 0), (3, 8, 1, 2, 2, 1), (2, 6, 0, 3, 1, 1), (4, 33, 1, 3, 0, 0)])
def test_finish_equals_passes_and_oracle(ctx, oracle, name, spp, depth, nee, rr, sky, streams):
    sd = SCENES[name]()
    gs = solhip.GpuScene(ctx, sd)
    W, H = 61, 47
    s = _spec(spp, depth, nee, rr, sky, streams)
    print(name, spp, depth, nee, rr, sky, streams, flush=True)
    a, na = _run(ctx, gs, sd, s, W, H, 2)
    b, nb = _run(ctx, gs, sd, s, W, H, 2, PROFILE_TIME)
    ref, n = _oracle(oracle, sd, s, W, H, 2)
    assert np.array_equal(a.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(b.view(np.uint32), ref.view(np.uint32))
    assert na == nb and sum(na) == n


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("name,W,H,spp,streams", [
    ("cornell", 901, 603, 1, 0), ("cornell", 901, 603, 4, 1), ("terrain", 901, 603, 2, 1), ("instances", 1601, 1101, 1, 0)])
def test_passes_then_finish(ctx, oracle, name, W, H, spp, streams, graph):
    """more paths than the finishing kernel takes at once: the first bounces
    run as passes"""
    sd = SCENES[name]()
    gs = solhip.GpuScene(ctx, sd)
    s = _spec(spp, 6, 1, 3, 2, streams, graph)
    print(name, W, H, spp, streams, graph, flush=True)
    a, na = _run(ctx, gs, sd, s, W, H, 2)
    ref, n = _oracle(oracle, sd, s, W, H, 2)
    assert np.array_equal(a.view(np.uint32), ref.view(np.uint32))
    assert sum(na) == n
