"""The 64-channel mixed-precision training step against the FP64 oracle with
the same operand rounding, at the edges of its tiles: images whose last layer
is one pixel, odd batches and class counts, positions that fill no tile, one
convolution only, and enough positions for several splits.

Bar: as for the general mixed-precision step (tests/test_gpu_cnn.py), whose
arithmetic it shares: FP32 sums in another order, and operands at a BF16
rounding boundary one step apart (2^-8 of one operand among hundreds): 5e-3
relative L2 per gradient segment, losses 1e-3.
"""
import os
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
import cnn_oracle as CO  # noqa: E402

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no HIP device", allow_module_level=True)

from frealign_amd import api, proposal  # noqa: E402


@pytest.mark.parametrize("shape,B", [((2, 64, 1, 1), 1), ((16, 64, 1, 3), 5), ((8, 64, 3, 33), 17),
                                     ((48, 64, 4, 100), 3), ((32, 64, 2, 31), 65),
                                     ((20, 64, 2, 64), 33)])
def test_step_vs_oracle(shape, B):
    S, C, L, K = shape
    rng = np.random.default_rng(S * 1000 + K)
    ctx = api.Context(0)
    net = proposal.Network(ctx, shape, seed=3, device="cuda")
    img = rng.standard_normal((B, S, S)).astype(np.float32)
    lab = rng.integers(0, K, B).astype(np.int32)
    loss = ctx.cnn_gradients(shape, net.wq, torch.from_numpy(img).cuda(),
                             torch.from_numpy(lab).cuda(), net.grad, bf16=True)
    rl, rg = CO.loss_grad(net.wq.cpu().numpy(), shape, img, lab, bf16_ops=True)
    # one class: the loss and every gradient are zero
    rel = lambda a, b: np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-6)  # noqa: E731
    assert rel(loss.cpu().numpy(), rl) < 1e-3
    g = net.grad.cpu().numpy()
    offs, fw, fb, F, n = CO.layout(*shape)
    assert n == g.size
    for a, b in [w for w, _, _ in offs] + [b for _, b, _ in offs] + [fw, fb]:
        assert rel(g[a:b], rg[a:b]) < 5e-3, (shape, a, b)
    # the same bits again (fixed orders throughout)
    first = net.grad.clone()
    ctx.cnn_gradients(shape, net.wq, torch.from_numpy(img).cuda(), torch.from_numpy(lab).cuda(),
                      net.grad, bf16=True)
    assert torch.equal(first, net.grad)
    ctx.close()
