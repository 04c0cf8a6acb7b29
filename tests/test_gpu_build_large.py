"""The binned-SAH builder's rules for large nodes against the host replay, where
even soups do not take it: nodes of more than one workgroup's primitives far below the
levels that are launched blind and below the level at which ranges are halved, and
a root of so many primitives that its chunks are larger than usual.  The same
tree gives the same node count, depth, hits and fetches per ray."""
import numpy as np
import pytest

import raygen
import solhip
from cpu_harness import build as harness_build
from cpu_harness import harness
from solhip import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _built():
    import os
    if not os.path.exists(harness.LIB):
        harness_build.build()


def _clusters():
    """60 stacks of 1100 equal triangles, each an eighth as large and as far out as the one before:
    the build splits off one a level, down to level 48 with thousands of triangles left"""
    one = np.array([[0.6, 0.6, 0.6], [0.9, 0.6, 0.75], [0.6, 0.9, 0.9]])
    return np.concatenate([np.tile(one * 8.0 ** (14 - k), (1100, 1)) for k in range(60)])


def _soup():
    """2.2M small triangles: more than 512 chunks of 4096"""
    rng = np.random.default_rng(5)
    n = 2200000
    return (rng.uniform(-1.0, 1.0, size=(n, 1, 3)) + rng.uniform(-0.005, 0.005, size=(n, 3, 3))).reshape(-1, 3)


@pytest.mark.parametrize("name,points", [("clusters", _clusters), ("soup", _soup)])
def test_tree_equals_the_replay(ctx, name, points):
    b = scenes.soup_blas(points().astype(np.float32))
    cam = scenes.Camera((0.0, 0.0, 4.0), (0.0, 0.0, 0.0))
    sd = scenes.assemble("large", [b], [0], [np.eye(4)], [0], [scenes.material((1, 1, 1))], cam, 2.0)
    print("build", name, len(b.indices) // 3, flush=True)
    gs = solhip.GpuScene(ctx, sd, build_flags=solhip.BUILD_PREFER_FAST_TRACE)
    print("replay", name, flush=True)
    host = harness.HostScene(sd, solhip.BUILD_PREFER_FAST_TRACE)
    info = ctx.blas_info(gs.blas[0])
    assert (info.nodes, info.depth) == host.info(0)
    rays = np.concatenate([raygen.random_rays(400, (0, 0, 0), 1.5, seed=3), raygen.aimed_rays(sd, 400, seed=4)])
    ctx.stats(reset=True)
    g = ctx.trace_rays(gs.tlas, rays, solhip.TRACE_COUNT)
    st = ctx.stats(reset=True)
    h, counts = host.trace(rays)
    assert g.tobytes() == h.tobytes()
    assert (st.node_fetches, st.tri_fetches, st.inst_fetches, st.overflow) == tuple(int(c) for c in counts)
