"""The render server's traversal forms and its step-ahead host: jobs over scenes of one
form, of two (one instance and several, all at the identity transform; or general), at
image sizes around a wave and a block of the shade kernel, with job indices
used again, and run in pieces.  Images equal the oracle's bit for bit; the
rays counted equal its rays."""
import numpy as np
import pytest

import solhip
from solhip import scenes

pytestmark = pytest.mark.gpu

SCENES = {"cornell": scenes.cornell_box, "terrain": lambda: scenes.heightfield(40), "instances": scenes.random_instances}
SIZES = [(1, 1), (9, 7), (8, 8), (65, 1), (64, 48), (33, 31), (101, 97)]


@pytest.mark.parametrize("names,max_jobs,steps", [
    (["terrain"], 16, 1 << 30), (["cornell"], 2, 1 << 30), (["cornell", "terrain"], 3, 1), (["terrain", "cornell"], 1, 3),
    (["instances", "terrain"], 2, 2), (["instances", "cornell", "terrain"], 16, 5)])
def test_forms_and_pieces(ctx, oracle, names, max_jobs, steps):
    sds = [SCENES[n]() for n in names]
    gss = [solhip.GpuScene(ctx, sd) for sd in sds]
    srv = solhip.Server(ctx, 16 << 20, max_jobs)
    ids = [srv.scene(g) for g in gss]
    print("server", names, max_jobs, steps, flush=True)
    for k in ("srv_extend", "srv_shadow"):
        ctx.kernel_stats(k, reset=True)
    jobs = []
    for k, (W, H) in enumerate(SIZES):
        i = k % len(names)
        s = solhip.spec_default(solhip.PROG_PATHTRACE)
        s.spp_per_frame, s.max_depth, s.nee, s.rr_start, s.enable_sky = 1 + k, (0, 4, 8)[k % 3], k % 2, (0, 2)[k % 2], 2
        s.sample_streams, s.wf_samples_per_pass = k // 3 % 2, (0, 2)[k % 2]
        acc, out = ctx.upload(np.zeros((H, W, 4), np.float32)), ctx.upload(np.zeros((H, W, 4), np.uint8))
        jobs.append((srv.submit(ids[i], W, H, s, sds[i].uniforms(W, H, k), acc, out), i, W, H, s, k, acc, out))
    for _ in range(3000):
        if srv.run(steps) == 0:
            break
    rays = 0
    for jid, i, W, H, s, k, acc, out in jobs:
        assert srv.job(jid).state == solhip.JOB_DONE
        cfg = oracle.PTConfig(s.enable_sky, s.spp_per_frame, s.max_depth, s.rr_start, s.nee, s.sample_streams)
        ref, ref8 = np.zeros((H, W, 4), np.float32), np.zeros((H, W, 4), np.uint8)
        rays += oracle.Scene(sds[i]).render_pathtrace(sds[i].uniforms(W, H, k), cfg, 0, ref, ref8, W, H)
        assert np.array_equal(acc.download(np.float32).view(np.uint32), ref.view(np.uint32).reshape(-1)), (names, k)
    stats = [ctx.kernel_stats(k, reset=True).counters for k in ("srv_extend", "srv_shadow")]
    assert sum(c.rays for c in stats) == rays and all(c.overflow == 0 for c in stats)
    srv.close()
