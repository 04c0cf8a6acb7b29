"""The two kernels of the GLSL programs on every traversal form (trees of a few levels,
identity transforms, one instance, general), on both sides of the choice between
them (half the resident lanes, twice them, a second sample): accumulation equal to the
oracle's, bit for bit."""
import numpy as np
import pytest

import solhip
from solhip import scenes

pytestmark = pytest.mark.gpu


def _tiles():
    """a terrain in four BLASes at the identity transform, deeper than the few levels' form takes"""
    h = scenes.heightfield(32)
    idx = h.blas[0].indices.reshape(32, 32, 6)
    bl = [scenes.Blas(h.blas[0].vertices, np.ascontiguousarray(idx[i:i + 16, j:j + 16].reshape(-1)))
          for i in (0, 16) for j in (0, 16)]
    return scenes.assemble("tiles", bl, [0, 1, 2, 3], [np.eye(4)] * 4, [0] * 4, [scenes.material((0.8, 0.8, 0.8))],
                           h.camera, 2.0)


SCENES = {"cornell": scenes.cornell_box, "instances": scenes.random_instances, "tiles": _tiles,
          "terrain": lambda: scenes.heightfield(32)}
SIZES = [(5, 3), (361, 363), (363, 363)]   # 131,072 pixels: half the lanes of 256 CUs


@pytest.mark.parametrize("W,H", SIZES)
@pytest.mark.parametrize("name", sorted(SCENES))
def test_ao_glsl_forms(ctx, oracle, name, W, H):
    sd = SCENES[name]()
    gs = solhip.GpuScene(ctx, sd)
    blue = scenes.blue_noise_synthetic()
    prog = ctx.program(solhip.PROG_AO_GLSL)
    acc, bn = ctx.upload(np.zeros((H, W, 4), np.float32)), ctx.upload(blue)
    img = solhip.Images(acc.h, 0, bn.h, blue.shape[1], blue.shape[0], 0)
    ref = np.zeros((H, W, 4), np.float32)
    u = sd.uniforms(W, H, 2)
    print("ao glsl", name, W, H, flush=True)
    ctx.stats(reset=True)
    ctx.trace(prog, gs.tlas, gs.tables, u, 2, img, W, H)
    assert ctx.stats(reset=True).overflow == 0
    oracle.Scene(sd).render_ao_glsl(u, 2, ref, blue, W, H)
    assert np.array_equal(acc.download(np.float32).view(np.uint32), ref.view(np.uint32).reshape(-1))


@pytest.mark.parametrize("W,H,spp,depth", [(5, 3, 2, 3), (361, 363, 2, 4), (363, 363, 2, 4), (725, 725, 1, 3)])
@pytest.mark.parametrize("name", ["instances", "tiles", "terrain"])
def test_pathtrace_glsl_forms(ctx, oracle, name, W, H, spp, depth):
    sd = SCENES[name]()
    gs = solhip.GpuScene(ctx, sd)
    spec = solhip.spec_default(solhip.PROG_PATHTRACE_GLSL)
    spec.spp_per_frame, spec.max_depth, spec.enable_sky = spp, depth, 1
    prog = ctx.program(solhip.PROG_PATHTRACE_GLSL, spec)
    acc = ctx.upload(np.zeros((H, W, 4), np.float32))
    ref = np.zeros((H, W, 4), np.float32)
    u = sd.uniforms(W, H, 4)
    print("pt glsl", name, W, H, spp, depth, flush=True)
    ctx.stats(reset=True)
    ctx.trace(prog, gs.tlas, gs.tables, u, 4, solhip.Images(acc.h, 0, 0, 0, 0, 0), W, H)
    st = ctx.stats(reset=True)
    rays = oracle.Scene(sd).render_pathtrace_glsl(u, oracle.PTParams(1, spp, depth), 4, ref, None, W, H)
    assert np.array_equal(acc.download(np.float32).view(np.uint32), ref.view(np.uint32).reshape(-1))
    assert st.rays == rays and st.overflow == 0
