"""The radiance-cache network's kernels at the edges of their bands (16 rows),
tiles (64 rows) and grids (a workgroup's second tile from 16,385 rows on), against
a plain PyTorch fp32 reference with the kernels' BF16 roundings of inputs,
weights and hidden activations.  Outputs within 2e-2 of their scale, the gradient
of every layer within 3 % in norm and 0.999 in direction (BF16 gradients: 2^-9
per rounding, a few roundings in a chain), the loss within 2 %."""
import numpy as np
import pytest
import torch

import solhip
from test_gpu_mlp import P, _inputs, bf16_round, pack_grad, ref_forward, unpack

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [15, 16, 17, 32, 33, 127, 129, 16384, 65537, 131073])
def test_forward_bands(ctx, n):
    m = solhip.Mlp(ctx, seed=4)
    x, xbuf = _inputs(ctx, n, n)
    ybuf = ctx.buffer(n * 16)
    ybuf.fill(0x7F800001)
    print("mlp forward", n, flush=True)
    m.forward(xbuf, n, ybuf)
    out = ybuf.download(np.float32).reshape(n, 4)
    ref = ref_forward(x, m.params()).numpy()
    assert np.abs(out[:, :3] - ref).max() <= 2e-2 * np.abs(ref).max()
    assert (out.view(np.uint32)[:, 3] == 0x7F800001).all()   # the fourth component is not written
    m.close()


@pytest.mark.parametrize("n", [63, 64, 65, 200, 16384, 16385, 40001])
def test_gradient_tiles(ctx, n):
    m = solhip.Mlp(ctx, seed=6)
    x, xbuf = _inputs(ctx, n, n)
    t = np.zeros((n, 4), np.float32)
    t[:, :3] = np.random.default_rng(n).uniform(0.0, 2.0, size=(n, 3))
    tbuf = ctx.upload(t)
    print("mlp gradient", n, flush=True)
    g, loss = m.gradient(xbuf, tbuf, n)
    Ws = [bf16_round(W.numpy()).requires_grad_(True) for W in unpack(m.params())]
    h = bf16_round(x)
    for l in range(4):
        h = torch.relu(h @ Ws[l])
        h = h + (h.detach().to(torch.bfloat16).to(torch.float32) - h).detach()   # rounded, gradient passed on
    p = h @ Ws[4]
    ref_loss = (((p - torch.from_numpy(t[:, :3])) ** 2) / (p.detach() ** 2 + 0.01)).sum() / n
    ref_loss.backward()
    ref = pack_grad([W.grad.numpy() for W in Ws])
    assert abs(loss - ref_loss.item()) <= 2e-2 * ref_loss.item()
    for l in range(5):
        sl = slice(l * 4096, (l + 1) * 4096) if l < 4 else slice(16384, P)
        a, b = g[sl].astype(np.float64), ref[sl].astype(np.float64)
        assert a @ b / (np.linalg.norm(a) * np.linalg.norm(b)) > 0.999, l
        assert abs(np.linalg.norm(a) / np.linalg.norm(b) - 1.0) < 0.03, l
    assert (g[16384:].reshape(64, 16)[:, 3:] == 0).all()
    m.close()
