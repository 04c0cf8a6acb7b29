"""solhip_trace_rays at sizes around its launch forms (one ray per wave up to
full waves; the persistent grid and its deal of rays to waves) against the host
replay: every hit bit-identical and every ray traced once."""
import numpy as np
import pytest

import raygen
import solhip
from cpu_harness import build as harness_build
from cpu_harness import harness
from solhip import scenes

pytestmark = pytest.mark.gpu

SCENES = {"cornell": scenes.cornell_box, "terrain": lambda: scenes.heightfield(48),
          "instances": lambda: scenes.random_instances(40)}


@pytest.fixture(scope="module")
def scene_pairs(ctx):
    import os
    if not os.path.exists(harness.LIB):
        harness_build.build()
    out = {}
    for name, f in SCENES.items():
        sd = f()
        out[name] = (sd, solhip.GpuScene(ctx, sd), harness.HostScene(sd, 0))
    return out


@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("n", [1, 63, 1025, 2047, 65537, 327680, 327681, 400003])
def test_query_sizes(ctx, scene_pairs, name, n):
    sd, gs, host = scene_pairs[name]
    rays = raygen.random_rays(n, (0, 0, 0), 2.0 if name != "instances" else 6.0, seed=n)
    ctx.stats(reset=True)
    g = ctx.trace_rays(gs.tlas, rays)
    st = ctx.stats(reset=True)
    h, _ = host.trace(rays)
    assert g.tobytes() == h.tobytes()
    assert st.rays == n and st.overflow == 0
    a = ctx.trace_rays(gs.tlas, rays, solhip.TRACE_TERMINATE_ON_FIRST_HIT)
    assert np.array_equal(a["inst"] == 0xFFFFFFFF, h["inst"] == 0xFFFFFFFF)
