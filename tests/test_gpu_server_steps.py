"""What max_steps of solhip_server_run buys: a step traces, shades, answers the
shadow rays of what it shaded and retires what ended in it, so a job of one
sample per pixel whose longest path has max_depth + 1 segments is done after as many
steps, in one call or in several.  Images equal the oracle's bit for bit."""
import numpy as np
import pytest

import solhip
from solhip import scenes

pytestmark = pytest.mark.gpu

W, H = 72, 56


def _jobs(ctx, srv, sid, sd, n, depth, spp, streams):
    out = []
    for k in range(n):
        s = solhip.spec_default(solhip.PROG_PATHTRACE)
        s.spp_per_frame, s.max_depth, s.nee, s.enable_sky, s.sample_streams = spp, depth, 1, 0, streams
        s.wf_samples_per_pass = spp if streams else 0
        acc = ctx.upload(np.zeros((H, W, 4), np.float32))
        out.append((srv.submit(sid, W, H, s, sd.uniforms(W, H, k), acc), s, k, acc))
    return out


def _check(oracle, srv, sd, jobs):
    for jid, s, k, acc in jobs:
        assert srv.job(jid).state == solhip.JOB_DONE
        cfg = oracle.PTConfig(s.enable_sky, s.spp_per_frame, s.max_depth, s.rr_start, s.nee, s.sample_streams)
        ref = np.zeros((H, W, 4), np.float32)
        oracle.Scene(sd).render_pathtrace(sd.uniforms(W, H, k), cfg, 0, ref, None, W, H)
        assert np.array_equal(acc.download(np.float32).view(np.uint32), ref.view(np.uint32).reshape(-1))


@pytest.mark.parametrize("depth", [0, 1, 4, 9])
@pytest.mark.parametrize("n,spp,streams", [(1, 1, 0), (3, 1, 0), (2, 3, 1)])
def test_steps_until_done(ctx, oracle, depth, n, spp, streams):
    """all samples of a pixel side by side (or one): as many steps as the longest path has segments"""
    sd = scenes.cornell_box()
    gs = solhip.GpuScene(ctx, sd)
    srv = solhip.Server(ctx, 16 << 20, 8)
    sid = srv.scene(gs)
    print("server steps", depth, n, spp, streams, flush=True)
    jobs = _jobs(ctx, srv, sid, sd, n, depth, spp, streams)
    assert srv.run(depth + 1) == 0
    _check(oracle, srv, sd, jobs)
    jobs = _jobs(ctx, srv, sid, sd, n, depth, spp, streams)
    for _ in range(depth):
        assert srv.run(1) == n
    assert srv.run(1) == 0
    _check(oracle, srv, sd, jobs)
    srv.close()


@pytest.mark.parametrize("steps", [1, 2, 3, 7])
def test_samples_in_sequence_by_pieces(ctx, oracle, steps):
    """new samples start in the step after the last one's end, however the steps are
    divided among calls"""
    sd = scenes.cornell_box()
    gs = solhip.GpuScene(ctx, sd)
    srv = solhip.Server(ctx, 16 << 20, 8)
    jobs = _jobs(ctx, srv, srv.scene(gs), sd, 2, 3, 5, 0)
    print("server pieces", steps, flush=True)
    for k in range(21):
        if srv.run(steps) == 0:
            break
    assert (k + 1) * steps <= 20 + steps - 1   # 5 samples of at most 4 segments
    _check(oracle, srv, sd, jobs)
    srv.close()
