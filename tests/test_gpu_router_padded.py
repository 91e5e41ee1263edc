"""The matrix-core router where experts or columns do not fill its tiles: expert counts that are multiples of 8 but not
16, 32, 64, 128 or 256, and rows that end inside a chunk (both read as zeros beyond their ends).  The bar is that of
the other projection kernels: one ulp of bf16 on the logits, then bit-exact decisions, and the same bits in every batch.
On top of it the logits are one chain of fused multiply-adds in k order, rounded once, whichever kernel takes the call.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import test_gpu_parity as P
from research_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,hidden,experts,top_k", [
    (1, 8, 8, 1),        # one piece of one row
    (3, 56, 16, 2),      # full columns, a row that ends inside the first chunk
    (17, 128, 8, 8),     # one whole chunk of the sliced kernel, every expert chosen
    (65, 72, 24, 3),     # a second chunk of one piece
    (40, 1024, 8, 2),    # eight slices
    (300, 1152, 40, 4),  # slices of two chunks, the last of one; middle-sized
    (33, 1000, 96, 4),
    (257, 264, 200, 8),
    (20, 384, 248, 16),
])
def test_padded_projection_against_the_oracle(gpu, tokens, hidden, experts, top_k):
    rng = np.random.default_rng(tokens * 31 + hidden)
    x = rng.standard_normal((tokens, hidden)).astype(np.float32)
    w = (rng.standard_normal((hidden, experts)) * 0.02).astype(np.float32)
    bias = (rng.standard_normal(experts) * 0.05).astype(np.float32)
    P.check_router_end_to_end(gpu, x, w, bias, top_k, 1.0, "bf16")


@pytest.mark.parametrize("hidden,experts,top_k", [(1024, 8, 2), (1920, 24, 3), (1000, 96, 4), (1152, 200, 4), (136, 64, 2)])
@pytest.mark.parametrize("score_func", ["sigmoid", "softmax"])
def test_padded_rows_do_not_depend_on_the_batch(gpu, hidden, experts, top_k, score_func):
    """Stand-alone calls and layer calls of every size against one call of all rows; rows beyond an end hold NaN."""
    generator = torch.Generator(device=gpu).manual_seed(hidden + experts)

    def normal(*shape, std=1.0):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    tokens, inter = 2600, 64
    room = torch.full((tokens + 1, hidden), float("nan"), dtype=torch.bfloat16, device=gpu)
    room[:tokens] = normal(tokens, hidden)
    x, w, bias = room[:tokens], normal(hidden, experts, std=0.02), torch.randn(experts, generator=generator, device=gpu) * 0.05
    experts_w = (normal(experts, hidden, inter, std=0.05), normal(experts, hidden, inter, std=0.05),
                 normal(experts, inter, hidden, std=0.05))
    full = ops.router(x, w, bias, top_k, 1.0, score_func=score_func)
    for rows in (1, 5, 16, 64, 65, 200, 256, 257, 1000, 2561):
        part = room[tokens - rows:tokens]  # the last rows: what follows them is not theirs
        alone = ops.router(part, w, bias, top_k, 1.0, score_func=score_func)
        layer = ops.moe_forward(part, w, bias, *experts_w, top_k, 1.0, score_func=score_func)
        for name in ("scores", "expert_ids", "weights"):
            want = getattr(full, name)[tokens - rows:]
            assert torch.equal(getattr(alone, name), want), f"{rows} rows: {name}"
            assert torch.equal(getattr(layer, name), want), f"{rows} rows in a layer call: {name}"
        assert torch.equal(layer.expert_counts, alone.expert_counts) and torch.equal(layer.importance, alone.importance)


@pytest.mark.parametrize("tokens,hidden,experts,top_k", [
    (4096, 1024, 8, 2),    # one column block, half of it experts
    (64, 1024, 8, 2),      # small batches: the sums of a workgroup's 64 experts, then the finishing one
    (250, 1152, 200, 4),   # ... of four column blocks
    (2931, 1000, 24, 3),   # rows that end inside a chunk
    (500, 136, 64, 8),     # ... of eight columns past the first one, experts that fill their blocks
    (700, 712, 96, 4),     # two blocks to a wave
    (600, 520, 160, 3),    # three
    (300, 1384, 248, 16),  # four
])
def test_padded_logits_are_one_chain_in_k_order(gpu, tokens, hidden, experts, top_k):
    """Products of two bf16 values are exact in fp32, so that a rounded sum of each is a fused multiply-add.  Operands two
    bytes off a 16-byte boundary, which the staged kernel takes, have the same bits."""
    rng = np.random.default_rng(tokens + hidden)
    x = P.O.bf16_round(rng.standard_normal((tokens, hidden)).astype(np.float32))
    w = P.O.bf16_round((rng.standard_normal((hidden, experts)) * 0.02).astype(np.float32))
    chain = np.zeros((tokens, experts), np.float32)
    for k in range(hidden):
        chain += x[:, k, None] * w[None, k]
    dx, dw = P.dev(x, gpu, "bf16"), P.dev(w, gpu, "bf16")
    got = ops.router(dx, dw, None, top_k, 1.0, return_logits=True)
    differ = int((P.host(got.logits) != P.O.bf16_round(chain)).sum())
    assert differ == 0, f"{differ} of {chain.size} logits differ"

    def shifted(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view_as(t)

    staged = ops.router(shifted(dx), shifted(dw), None, top_k, 1.0, return_logits=True)
    for name in ("logits", "scores", "expert_ids", "weights", "expert_counts", "importance"):
        assert torch.equal(getattr(got, name), getattr(staged, name)), name
