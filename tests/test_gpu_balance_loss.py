"""The sequence balance loss and its gradient at the edges of the kernels' token chunks and lane groups.

A wave takes 64 / W tokens at a time, W = 8, 16, 32 or 64 lanes by the expert count; a sequence is cut
into chunks of at least 16 tokens.  Bars: the loss is a sum of positive fp32 terms in another order than
the oracle's (relative error below its number of dependent additions times 2^-24, far under 1e-5 here);
the gradient's as for the existing check.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe_grad_oracle as G
from oracle import moe_oracle as O
from research_amd import ops
from test_gpu_parity import dev, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,seq,experts,top_k", [
    (1, 1, 1, 1),        # one token, one expert
    (2, 15, 8, 2),       # less than a chunk, eight lanes per token
    (3, 17, 9, 3),       # two chunks, the second of one token; sixteen lanes
    (1, 257, 32, 4),     # thirty-two lanes, a ragged last chunk
    (5, 100, 33, 2),     # a whole wave per token, lanes without an expert
    (2, 1025, 65, 8),    # two experts per lane, one of them absent
    (1, 2048, 256, 16),  # the largest expert count and top-k
    (300, 40, 12, 2),    # more sequences than workgroups wanted: one chunk each
])
def test_balance_loss_and_gradient_at_the_edges(gpu, batch, seq, experts, top_k):
    rng = np.random.default_rng(batch * 1000 + seq)
    scores = (1.0 / (1.0 + np.exp(-rng.standard_normal((batch, seq, experts))))).astype(np.float32)
    scores[0, 0] = 0.0  # a row whose sum is clamped
    ids = rng.random((batch, seq, experts)).argsort(axis=-1)[..., :top_k].astype(np.int32)
    sd, idd = dev(scores, gpu), dev(ids, gpu)
    loss = ops.sequence_balance_loss(idd, sd, top_k=top_k)
    assert float(loss) == pytest.approx(float(O.sequence_balance_loss(ids, scores, top_k)), rel=1e-5)
    assert torch.equal(loss, ops.sequence_balance_loss(idd, sd, top_k=top_k))
    want = G.sequence_balance_loss_backward(ids, scores, top_k, d_loss=1.0)
    got = host(ops.sequence_balance_loss_backward(idd, sd, top_k=top_k))
    whole = np.ones((batch, seq), bool)
    whole[0, 0] = False  # of the clamped row only the sign and size are checked: its scale is 1e20
    scale = float(np.max(np.abs(want[whole]), initial=1e-30))
    np.testing.assert_allclose(got[whole] / scale, want[whole] / scale, rtol=1e-4, atol=2e-6)
    np.testing.assert_allclose(got[0, 0], want[0, 0], rtol=1e-5)
