"""The two kernels of SOLHIP_PROG_PATHTRACE_GLSL (lanes in lockstep, and the
per-lane state machine with refill) against the oracle: bit-identical
accumulation and the same ray count on both sides of every boundary of the choice
(depth 8 and 16, a second sample, twice the resident lanes), on images smaller
than a tile, ragged ones, and one where every lane takes several pixels."""
import numpy as np
import pytest

import solhip
from solhip import scenes

pytestmark = pytest.mark.gpu

SCENES = {"cornell": scenes.cornell_box, "instances": scenes.random_instances,
          "terrain": lambda: scenes.heightfield(32)}


@pytest.mark.parametrize("name,W,H,spp,depth,sky", [
    ("cornell", 1, 1, 2, 32, 0), ("cornell", 7, 9, 2, 16, 1), ("cornell", 65, 33, 1, 16, 0),
    ("cornell", 65, 33, 2, 15, 0), ("instances", 61, 35, 3, 20, 1), ("terrain", 130, 71, 2, 17, 1),
    ("cornell", 1027, 611, 1, 8, 1), ("cornell", 1027, 611, 1, 7, 1), ("terrain", 1024, 640, 1, 16, 1)])
def test_pathtrace_glsl_kernels(ctx, oracle, name, W, H, spp, depth, sky):
    sd = SCENES[name]()
    gs = solhip.GpuScene(ctx, sd)
    spec = solhip.spec_default(solhip.PROG_PATHTRACE_GLSL)
    spec.spp_per_frame, spec.max_depth, spec.enable_sky = spp, depth, sky
    prog = ctx.program(solhip.PROG_PATHTRACE_GLSL, spec)
    acc = ctx.upload(np.zeros((H, W, 4), np.float32))
    img = solhip.Images(acc.h, 0, 0, 0, 0, 0)
    sc = oracle.Scene(sd)
    ref = np.zeros((H, W, 4), np.float32)
    for frame in (5, 6):
        u = sd.uniforms(W, H, frame)
        print(name, W, H, spp, depth, frame, flush=True)
        ctx.stats(reset=True)
        ctx.trace(prog, gs.tlas, gs.tables, u, 5, img, W, H)
        st = ctx.stats(reset=True)
        nrays = sc.render_pathtrace_glsl(u, oracle.PTParams(sky, spp, depth), 5, ref, None, W, H)
        g = acc.download(np.float32).reshape(H, W, 4)
        assert np.array_equal(g.view(np.uint32), ref.view(np.uint32))
        assert st.rays == nrays and st.overflow == 0
