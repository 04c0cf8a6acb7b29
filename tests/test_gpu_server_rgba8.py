"""The render server's 8-bit output: every pixel of every job, with samples in
sequence and side by side, one step of 255 at most from the oracle's (the GPU's
powf against the host's), as for solhip_trace's."""
import numpy as np
import pytest

import solhip
from solhip import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 1 << 30])
@pytest.mark.parametrize("streams", [0, 1])
def test_rgba8(ctx, oracle, streams, steps):
    sd = scenes.cornell_box()
    gs = solhip.GpuScene(ctx, sd)
    srv = solhip.Server(ctx, 16 << 20, 3)
    sid = srv.scene(gs)
    jobs = []
    for k, (W, H) in enumerate([(1, 1), (33, 31), (8, 8), (101, 67), (64, 9)]):
        s = solhip.spec_default(solhip.PROG_PATHTRACE)
        s.spp_per_frame, s.max_depth, s.nee, s.sample_streams, s.wf_samples_per_pass = 4, 3, 1, streams, 2 * streams
        acc, out = ctx.upload(np.zeros((H, W, 4), np.float32)), ctx.upload(np.full((H, W, 4), 77, np.uint8))
        jobs.append((srv.submit(sid, W, H, s, sd.uniforms(W, H, k), acc, out), W, H, s, k, acc, out))
    print("server rgba8", streams, steps, flush=True)
    for _ in range(300):
        if srv.run(steps) == 0:
            break
    for jid, W, H, s, k, acc, out in jobs:
        assert srv.job(jid).state == solhip.JOB_DONE
        ref, ref8 = np.zeros((H, W, 4), np.float32), np.zeros((H, W, 4), np.uint8)
        cfg = oracle.PTConfig(0, 4, 3, 0, 1, streams)
        oracle.Scene(sd).render_pathtrace(sd.uniforms(W, H, k), cfg, 0, ref, ref8, W, H)
        assert np.array_equal(acc.download(np.float32).view(np.uint32), ref.view(np.uint32).reshape(-1))
        got = out.download(np.uint8, W * H * 4).reshape(H, W, 4)
        assert np.abs(got.astype(int) - ref8.astype(int)).max() <= 1
        assert (got[..., 3] == 255).all()
    srv.close()
