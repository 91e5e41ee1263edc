"""Widths that are multiples of 8 but end inside a k step of the matrix-core kernels.

The cases take every kernel through a ragged last step: 64-row tiles (few rows per group), the two-stage
256-row kernels (short reductions), the streaming gate/up kernel (at least eight 32-deep steps), and the
data gradients.  Bars are those of the existing checks against the oracle.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import test_gpu_grad as G
import test_gpu_parity as P
from research_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter", [
    (40, 8, 4, 2, 8),        # a single 8-wide chunk in each direction
    (60, 72, 5, 2, 40),      # 64-row tiles, one whole step and one chunk
    (500, 200, 2, 2, 136),   # 256-row tiles, seven gate/up steps: the two-stage kernel
    (400, 264, 2, 1, 520),   # the streaming kernel with nine steps, the last of one chunk
    (300, 504, 2, 2, 328),   # ... the last of three chunks; the down product ends one chunk into a step
])
def test_experts_and_gradients_at_ragged_widths(gpu, tokens, hidden, experts, top_k, inter):
    P.test_grouped_swiglu_matches_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")
    G.test_expert_gradients_match_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")


@pytest.mark.parametrize("tokens,hidden,inter", [(30, 72, 40), (600, 264, 136)])
def test_a_row_does_not_read_the_row_behind_it(gpu, tokens, hidden, inter):
    """What follows a row's last element in memory is the next row: with infinities there, the row before
    must come out as without them."""
    gen = torch.Generator(device=gpu).manual_seed(3)
    draw = lambda *shape: (torch.randn(*shape, device=gpu, generator=gen) * 0.2).to(torch.bfloat16)
    x, w_router = draw(tokens, hidden), draw(hidden, 2)
    gate, up, down = draw(2, hidden, inter), draw(2, hidden, inter), draw(2, inter, hidden)
    clean = ops.moe_forward(x, w_router, None, gate, up, down, 1, 1.0).y
    bad = torch.arange(1, tokens, 2, device=gpu)
    x[bad, :8] = float("inf")
    got = ops.moe_forward(x, w_router, None, gate, up, down, 1, 1.0).y
    good = torch.arange(0, tokens, 2, device=gpu)
    assert torch.equal(got[good], clean[good])
