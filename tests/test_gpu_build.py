"""The GPU builders against the host replay of their rules (bvh_logic.h): the
same tree gives the same node count, depth, hits and node / triangle /
instance fetches per ray, at primitive counts around the builders' own edges
(16-lane nodes, one-workgroup subtrees, chunks of large nodes, several levels
of each), on even, clustered and degenerate geometry."""
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


def _soup(n, kind):
    rng = np.random.default_rng(n)
    if kind == "even":
        c = rng.uniform(-1.0, 1.0, size=(n, 1, 3))
    elif kind == "clustered":
        # most of the triangles in a corner, a few far away: lopsided splits
        c = np.where(rng.random((n, 1, 1)) < 0.02, rng.uniform(-1.0, 1.0, size=(n, 1, 3)),
                     0.9 + rng.normal(scale=0.01, size=(n, 1, 3)))
    else:
        # duplicates: whole groups of triangles share one box (no usable split)
        c = rng.integers(-2, 3, size=(n, 1, 3)) * 0.4
    shape = rng.uniform(-0.1, 0.1, size=(1 if kind == "duplicates" else n, 3, 3))
    b = scenes.soup_blas((c + shape).reshape(-1, 3))
    cam = scenes.Camera((0.0, 0.0, 4.0), (0.0, 0.0, 0.0))
    return scenes.assemble("soup", [b], [0], [np.eye(4)], [0], [scenes.material((1, 1, 1))], cam, 2.0)


@pytest.mark.parametrize("build", [0, solhip.BUILD_PREFER_FAST_TRACE], ids=["morton", "sah"])
@pytest.mark.parametrize("kind", ["even", "clustered", "duplicates"])
@pytest.mark.parametrize("n", [1, 2, 3, 9, 16, 17, 33, 255, 1024, 1025, 2051, 4097, 9001, 20000])
def test_tree_equals_the_replay(ctx, n, kind, build):
    sd = _soup(n, kind)
    print("build", n, kind, build, flush=True)
    gs = solhip.GpuScene(ctx, sd, build_flags=build)
    host = harness.HostScene(sd, build)
    info = ctx.blas_info(gs.blas[0])
    assert (info.nodes, info.depth) == host.info(0)
    rays = np.concatenate([raygen.random_rays(700, (0, 0, 0), 1.5, seed=n), raygen.aimed_rays(sd, 300, seed=n)])
    ctx.stats(reset=True)
    g = ctx.trace_rays(gs.tlas, rays, solhip.TRACE_COUNT)
    st = ctx.stats(reset=True)
    h, counts = host.trace(rays)
    assert g.tobytes() == h.tobytes()
    assert (st.node_fetches, st.tri_fetches, st.inst_fetches, st.overflow) == tuple(int(c) for c in counts)


@pytest.mark.parametrize("n", [2, 9, 64, 500, 1025])
def test_instance_tree_equals_the_replay(ctx, n):
    sd = scenes.random_instances(n, seed=n)
    gs = solhip.GpuScene(ctx, sd)
    host = harness.HostScene(sd, 0)
    info = ctx.tlas_info(gs.tlas)
    assert (info.nodes, info.depth) == host.info(0xFFFFFFFF)
    rays = raygen.random_rays(1000, (0, 0, 0), 5.0, seed=n)
    ctx.stats(reset=True)
    g = ctx.trace_rays(gs.tlas, rays, solhip.TRACE_COUNT)
    st = ctx.stats(reset=True)
    h, counts = host.trace(rays)
    assert g.tobytes() == h.tobytes()
    assert (st.node_fetches, st.tri_fetches, st.inst_fetches, st.overflow) == tuple(int(c) for c in counts)
