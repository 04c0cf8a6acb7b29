"""Programs on trees of every depth at which a block's traversal stacks come to
exactly 64 KiB of LDS or pass it (stack entries per lane: the levels of the scene
and two more), and the levels beside them: images equal the oracle's, bit for
bit, and no stack overflows.

Levels come from a BLAS over clusters of triangles, each an eighth of the size and of the
distance of the one before (the binned-SAH build splits off one a level), and from instances
in ever smaller halves of space (the Morton order's bits one by one)."""
import numpy as np
import pytest

import solhip
from solhip import scenes

pytestmark = pytest.mark.gpu


def _clusters(n, first=0, tris=24):
    """n clusters of triangles at scales 8^first, 8^(first - 1), ..."""
    rng = np.random.default_rng(1)
    v = [(rng.uniform(0.5, 1.0, size=(tris, 1, 3)) + rng.uniform(-0.3, 0.3, size=(tris, 3, 3))) * 8.0 ** (first - k)
         for k in range(n)]
    return scenes.soup_blas(np.concatenate(v).reshape(-1, 3).astype(np.float32))


def _scene(blas, xforms):
    cam = scenes.Camera((1.4, 1.2, 1.6), (0.4, 0.4, 0.4))
    n = len(xforms)
    return scenes.assemble("deep", [blas], [0] * n, xforms, [0] * n, [scenes.material((0.8, 0.7, 0.6))], cam, 2.0)


def _levels(ctx, gs):
    """SceneView::stack_depth"""
    return ctx.tlas_info(gs.tlas).depth + max(ctx.blas_info(b).depth for b in gs.blas) + 1


def _halves(each, size=2.0 ** 63):
    """the identity, then `each` shifts into half of a cube, a quarter, an eighth, ..."""
    rng, xf = np.random.default_rng(3), [np.eye(4)]
    for k in range(10):
        for axis in range(3):
            lo, hi = np.zeros(3), np.full(3, size)
            lo[axis], hi[:axis] = size / 2, size / 2
            for _ in range(each):
                xf.append(np.eye(4))
                xf[-1][:3, 3] = rng.uniform(lo, hi)
        size /= 2
    return xf


def _image(ctx, sd, gs, prog, u, W, H, blue=None):
    acc = ctx.upload(np.zeros((H, W, 4), np.float32))
    bn = ctx.upload(blue) if blue is not None else None
    img = solhip.Images(acc.h, 0, bn.h, blue.shape[1], blue.shape[0], 0) if bn else solhip.Images(acc.h, 0, 0, 0, 0, 0)
    ctx.stats(reset=True)
    ctx.trace(prog, gs.tlas, gs.tables, u, 0, img, W, H)
    st = ctx.stats(reset=True)
    assert st.overflow == 0
    return acc.download(np.float32).view(np.uint32)


@pytest.mark.parametrize("clusters,levels", [(10, 13), (11, 14), (12, 15), (25, 28), (26, 30), (27, 31)])
def test_state_machine(ctx, oracle, clusters, levels):
    """blocks of 512 lanes up to 14 levels, of 256 up to 30, then of 128"""
    sd = _scene(_clusters(clusters), [np.eye(4)])
    gs = solhip.GpuScene(ctx, sd, build_flags=solhip.BUILD_PREFER_FAST_TRACE)
    assert _levels(ctx, gs) == levels
    W, H = 363, 365   # more than half of the resident lanes, several samples: k_pixels
    u = sd.uniforms(W, H, 0)
    sc = oracle.Scene(sd)
    blue = scenes.blue_noise_synthetic()
    print("deep ao glsl", levels, flush=True)
    got = _image(ctx, sd, gs, ctx.program(solhip.PROG_AO_GLSL), u, W, H, blue)
    ref = np.zeros((H, W, 4), np.float32)
    sc.render_ao_glsl(u, 0, ref, blue, W, H)
    assert np.array_equal(got, ref.view(np.uint32).reshape(-1))
    print("deep pathtrace glsl", levels, flush=True)
    spec = solhip.spec_default(solhip.PROG_PATHTRACE_GLSL)
    spec.spp_per_frame, spec.max_depth, spec.enable_sky = 2, 4, 1
    got = _image(ctx, sd, gs, ctx.program(solhip.PROG_PATHTRACE_GLSL, spec), u, W, H)
    ref = np.zeros((H, W, 4), np.float32)
    sc.render_pathtrace_glsl(u, oracle.PTParams(1, 2, 4), 0, ref, None, W, H)
    assert np.array_equal(got, ref.view(np.uint32).reshape(-1))


@pytest.mark.parametrize("any_hit", [0, 1])
@pytest.mark.parametrize("clusters,tris,each,levels", [(46, 24, 64, 61), (50, 24, 24, 62), (50, 24, 64, 63), (58, 32, 64, 64)])
def test_ao(ctx, oracle, clusters, tris, each, levels, any_hit):
    """primary rays in blocks of two waves up to the deepest scene that is accepted"""
    sd = _scene(_clusters(clusters, 20, tris), _halves(each))
    gs = solhip.GpuScene(ctx, sd, build_flags=solhip.BUILD_PREFER_FAST_TRACE)
    assert _levels(ctx, gs) == levels
    spec = solhip.spec_default(solhip.PROG_AO)
    spec.n_ao, spec.ao_tmin, spec.ao_tmax, spec.ao_any_hit = 4, 2e-4, 0.5, any_hit
    W, H = 45, 27
    u = sd.uniforms(W, H, 0)
    print("deep ao", levels, any_hit, flush=True)
    got = _image(ctx, sd, gs, ctx.program(solhip.PROG_AO, spec), u, W, H)
    ref = np.zeros((H, W, 4), np.float32)
    oracle.Scene(sd).render_ao(u, oracle.AOParams(4, 2e-4, 0.5, any_hit), 0, ref, W, H)
    assert 0.0 < ref[..., 0].mean() < 1.0   # some rays hit
    assert np.array_equal(got, ref.view(np.uint32).reshape(-1))
