"""Morton builds around the sizes up to which one workgroup makes the binary tree,
walks the refit's frontier and scans the radix sort's counts:
the same node count, depth, hits and fetches as the host replay, for triangles
and for instances."""
import numpy as np
import pytest

import raygen
import solhip
from cpu_harness import harness
from solhip import scenes
from test_gpu_build import _built, _soup  # noqa: F401

pytestmark = pytest.mark.gpu


def _same(ctx, sd, handle, info, extent):
    host = harness.HostScene(sd, 0)
    assert (info.nodes, info.depth) == host.info(handle)
    rays = np.concatenate([raygen.random_rays(600, (0, 0, 0), extent, seed=3), raygen.aimed_rays(sd, 200, seed=4)])
    return host.trace(rays), rays


@pytest.mark.parametrize("kind", ["even", "duplicates"])
@pytest.mark.parametrize("n", [1, 2, 31, 1023, 1024, 1025, 2047, 2048, 2049])
def test_triangles(ctx, n, kind):
    sd = _soup(n, kind)
    print("small build", n, kind, flush=True)
    gs = solhip.GpuScene(ctx, sd)
    for k in range(2):   # again into the same structure
        if k:
            gs.rebuild_blas(0)
            gs.update_instances(sd.instance_descs)
        (h, counts), rays = _same(ctx, sd, 0, ctx.blas_info(gs.blas[0]), 1.5)
        ctx.stats(reset=True)
        g = ctx.trace_rays(gs.tlas, rays, solhip.TRACE_COUNT)
        st = ctx.stats(reset=True)
        assert g.tobytes() == h.tobytes()
        assert (st.node_fetches, st.tri_fetches, st.inst_fetches, st.overflow) == tuple(int(c) for c in counts)


@pytest.mark.parametrize("n", [1024, 2047, 2048, 2049])
def test_instances(ctx, n):
    sd = scenes.random_instances(n, seed=n)
    gs = solhip.GpuScene(ctx, sd)
    (h, counts), rays = _same(ctx, sd, 0xFFFFFFFF, ctx.tlas_info(gs.tlas), 5.0)
    ctx.stats(reset=True)
    g = ctx.trace_rays(gs.tlas, rays, solhip.TRACE_COUNT)
    st = ctx.stats(reset=True)
    assert g.tobytes() == h.tobytes()
    assert (st.node_fetches, st.tri_fetches, st.inst_fetches, st.overflow) == tuple(int(c) for c in counts)


@pytest.mark.parametrize("kind", ["even", "duplicates"])
@pytest.mark.parametrize("n", [8192, 8193, 32768, 32769, 131072, 131073])
def test_frontier_and_scan(ctx, n, kind):
    sd = _soup(n, kind)
    print("build", n, kind, flush=True)
    gs = solhip.GpuScene(ctx, sd)
    (h, counts), rays = _same(ctx, sd, 0, ctx.blas_info(gs.blas[0]), 1.5)
    ctx.stats(reset=True)
    g = ctx.trace_rays(gs.tlas, rays[:64], solhip.TRACE_COUNT)
    assert ctx.stats(reset=True).overflow == 0
    assert g.tobytes() == h[:64].tobytes()
