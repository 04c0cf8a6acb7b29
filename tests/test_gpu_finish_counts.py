"""Fetch counts of a path-traced frame by kernel (SOLHIP_PROFILE_COUNT): a queue
that is finished path by path counts the same nodes, triangles and instances for
extension and for shadow rays as the bounce-by-bounce passes (which
SOLHIP_PROFILE_TIME keeps)."""
import numpy as np
import pytest

import solhip
from solhip import scenes
from solhip.api import PROFILE_COUNT, PROFILE_TIME

pytestmark = pytest.mark.gpu

SCENES = {"cornell": scenes.cornell_box, "instances": scenes.random_instances, "terrain": lambda: scenes.heightfield(48)}


def _counts(ctx, sd, gs, spec, W, H, profile):
    prog = ctx.program(solhip.PROG_PATHTRACE, spec)
    acc = ctx.upload(np.zeros((H, W, 4), np.float32))
    for k in ("pt_extend", "pt_shadow"):
        ctx.kernel_stats(k, reset=True)
    ctx.profile(profile)
    ctx.trace(prog, gs.tlas, gs.tables, sd.uniforms(W, H, 5), 5, solhip.Images(acc.h, 0, 0, 0, 0, 0), W, H)
    ctx.sync()
    ctx.profile(0)
    ctx.program_destroy(prog)
    c = [ctx.kernel_stats(k, reset=True).counters for k in ("pt_extend", "pt_shadow")]
    return [(x.rays, x.node_fetches, x.tri_fetches, x.inst_fetches, x.overflow) for x in c]


@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("nee", [0, 1])
def test_counts_by_kernel(ctx, name, nee):
    sd = SCENES[name]()
    gs = solhip.GpuScene(ctx, sd)
    s = solhip.spec_default(solhip.PROG_PATHTRACE)
    s.spp_per_frame, s.max_depth, s.nee, s.rr_start, s.enable_sky = 2, 5, nee, 3, 2
    print("counts", name, nee, flush=True)
    passes = _counts(ctx, sd, gs, s, 61, 47, PROFILE_COUNT | PROFILE_TIME)
    assert _counts(ctx, sd, gs, s, 61, 47, PROFILE_COUNT) == passes
