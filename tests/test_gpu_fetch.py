"""Work distribution of the persistent traversal kernels (fetch.h): AO queues at
the sizes where its split changes -- below one wave, around one wave, around the
4096 rays from which 64 partitions are used, and more rays than the GPU's lanes.
Every ray's hit record and the image equal the oracle's: a ray not claimed, or
claimed twice, shows in the records or in the ray count."""
import numpy as np
import pytest

import solhip
from solhip import scenes
from solhip.records import HIT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,n_ao", [(1, 1, 1), (9, 7, 1), (8, 8, 1), (13, 5, 1), (64, 63, 1), (65, 63, 1), (64, 64, 1),
                                      (241, 17, 1), (1, 257, 16), (313, 270, 8)])
def test_every_ray_is_traced_once(ctx, oracle, W, H, n_ao):
    sd = scenes.cornell_box()
    gs = solhip.GpuScene(ctx, sd)
    spec = solhip.spec_default(solhip.PROG_AO)
    spec.n_ao = n_ao
    prog = ctx.program(solhip.PROG_AO, spec)
    acc = ctx.upload(np.zeros((H, W, 4), np.float32))
    n = W * H * (1 + n_ao)
    hits = ctx.upload(np.full(n * HIT.itemsize, 0xA5, np.uint8))
    img = solhip.Images(acc.h, 0, 0, 0, 0, hits.h)
    sc = oracle.Scene(sd)
    ref = np.zeros((H, W, 4), np.float32)
    print("ao", W, H, n_ao, flush=True)
    for frame in range(2):
        u = sd.uniforms(W, H, frame)
        ctx.stats(reset=True)
        ctx.trace(prog, gs.tlas, gs.tables, u, 0, img, W, H)
        rays, ph, ah = sc.render_ao(u, oracle.AOParams(n_ao, spec.ao_tmin, spec.ao_tmax, 0), 0, ref, W, H, want_hits=True)
        assert hits.download(HIT).tobytes() == np.concatenate([ph, ah]).tobytes()
        assert np.array_equal(acc.download(np.float32).view(np.uint32).reshape(-1), ref.view(np.uint32).reshape(-1))
        assert ctx.stats().rays == rays
    ctx.program_destroy(prog)
