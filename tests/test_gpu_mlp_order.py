"""The order of the weight gradients' sums, which training carries into all later
weights: FP32 sums over chunks of 1024 rows, in row order within a chunk (32
rows per matrix instruction, one accumulator) and chunk after chunk.  Both are
pinned by equality, bit for bit:

- chunks: with 2^k chunks the loss's 1/n is a power of two, so 2^k times the
  gradient of all rows is the running sum, made by numpy, of the chunks' own gradients;
- within a chunk: a row of zeros adds nothing to any weight's gradient (the network
  has no biases), so blocks of 32 rows give the same gradient wherever they
  stand in the chunk, as long as their order is the same."""
import numpy as np
import pytest

import solhip
from test_gpu_mlp import _inputs

pytestmark = pytest.mark.gpu

CHUNK = 1024


def _targets(ctx, n):
    t = np.zeros((n, 4), np.float32)
    t[:, :3] = np.random.default_rng(n).uniform(0.0, 2.0, size=(n, 3))
    return t, ctx.upload(t)


def _running_sum(parts):
    s = np.zeros_like(parts[0])
    for p in parts:
        s = s + p
    return s


@pytest.mark.parametrize("chunks", [2, 8, 64, 256])
def test_chunks_are_summed_in_order(ctx, chunks):
    n = chunks * CHUNK
    m = solhip.Mlp(ctx, seed=3)
    x, xbuf = _inputs(ctx, n, chunks)
    t, tbuf = _targets(ctx, n)
    print("mlp chunks", chunks, flush=True)
    g, _ = m.gradient(xbuf, tbuf, n)
    words = xbuf.download(np.int16).reshape(n, 64)
    parts = []
    for c in range(chunks):
        rows = slice(c * CHUNK, (c + 1) * CHUNK)
        xb, tb = ctx.upload(words[rows]), ctx.upload(t[rows])
        parts.append(m.gradient(xb, tb, CHUNK)[0])
        xb.destroy()
        tb.destroy()
    assert np.array_equal(g * np.float32(chunks), _running_sum(parts))
    m.close()


@pytest.mark.parametrize("n,chunk", [(1024, 0), (1000, 0), (2500, 1), (2500, 2)])
def test_blocks_of_a_chunk_are_summed_in_order(ctx, n, chunk):
    m = solhip.Mlp(ctx, seed=5)
    x, full = _inputs(ctx, 96, n)
    words = full.download(np.int16).reshape(96, 64)
    t, _ = _targets(ctx, n)
    xbuf, tbuf = ctx.buffer(n * 128), ctx.buffer(n * 16)
    last = min(32, (n - chunk * CHUNK) // 32) - 1   # the chunk's last whole block

    def gradient(places):
        w, tt = np.zeros((n, 64), np.int16), np.ones((n, 4), np.float32)
        for k, p in enumerate(places):
            at = chunk * CHUNK + 32 * p
            w[at:at + 32], tt[at:at + 32] = words[32 * k:32 * k + 32], t[32 * k:32 * k + 32]
        xbuf.upload(w)
        tbuf.upload(tt)
        return m.gradient(xbuf, tbuf, n)[0]

    print("mlp blocks", n, chunk, flush=True)
    g = gradient((0, 1, 2))
    assert np.abs(g).max() > 0
    for places in ((0, 1, last), (1, 2, 3), (0, last // 2, last), (2, 5, 9), (last - 2, last - 1, last)):
        assert np.array_equal(g, gradient(places)), places
    m.close()
