"""Widths that are multiples of 8 but end inside a k step of the matrix-core kernels.

The cases take every kernel through a ragged last step and name the ones they are about: gate/up, down, and the two
data gradients; a rule that sends a case elsewhere fails it.  Bars are those of the existing checks against the oracle.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import test_gpu_grad as G
import test_gpu_parity as P
from kernel_choice import forward_kernels, gradient_kernels
from research_amd import ops

pytestmark = pytest.mark.gpu


SHAPES = [
    # tokens, hidden, experts, top_k, inter, gate/up and down, data gradients
    (40, 8, 4, 2, 8, "stream_16x64 stream_16x64", "half half"),      # a single 8-wide chunk in each direction
    (60, 72, 5, 2, 40, "stream_16x64 stream_16x64", "half half"),    # one whole step and one chunk
    (500, 200, 2, 2, 136, "stream_16x64 stream_16x64", "half half"),
    (400, 264, 2, 1, 520, "stream_16x64 stream_16x64", "half half_deep"),
    (300, 504, 2, 2, 328, "stream_16x64 stream_32x64", "half_deep half_deep"),
    (250, 72, 64, 8, 136, "rows64_tail stream_32x64", "half half"),  # three 32-deep steps, the last of one chunk
    (350, 264, 40, 4, 136, "stream_16x128 rows64", "half half"),     # ... five of them
    (900, 1000, 2, 2, 328, "half_tail half", "half_deep half_deep"),
    (4500, 72, 2, 1, 200, "rows256_short_tail half_deep", "half half_deep"),
    # 256-row tiles throughout: several whole steps, then one of a single chunk; a second segment behind it
    (16500, 136, 3, 2, 200, "rows256_short_tail rows256_tail", "rows256_tail rows256_tail"),
    (12000, 264, 3, 2, 264, "rows256_tail rows256_tail", "rows256_tail rows256_tail"),
    # ... five chunks, several tiles per workgroup, groups of a few hundred rows: the module call of perf/cases.py
    (2931, 1000, 24, 3, 2664, "rows256_tail rows256_tail", "rows256_tail rows256_tail"),
]


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter,forward,gradients", SHAPES)
def test_experts_and_gradients_at_ragged_widths(gpu, tokens, hidden, experts, top_k, inter, forward, gradients):
    assert " ".join(forward_kernels(tokens * top_k, hidden, inter, experts)) == forward
    assert " ".join(gradient_kernels(tokens * top_k, hidden, inter, experts)) == gradients
    P.test_grouped_swiglu_matches_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")
    G.test_expert_gradients_match_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")


LAST_ROWS = [
    # tokens, hidden, inter, experts, kernels
    (30, 72, 40, 2, "stream_16x64 stream_16x64"),
    (600, 264, 136, 2, "stream_16x64 stream_16x64"),
    (2000, 72, 136, 64, "rows64_tail stream_32x64"),
    (2000, 136, 72, 64, "stream_32x64 rows64"),
    (1300, 72, 136, 24, "stream_16x128 stream_16x64"),
    (4500, 264, 72, 2, "half_tail rows256_tail"),
    (4500, 72, 264, 2, "rows256_short_tail half"),
    (9000, 264, 264, 40, "rows256_tail half_deep"),
]


@pytest.mark.parametrize("tokens,hidden,inter,experts,kernels", LAST_ROWS)
def test_a_row_does_not_read_the_row_behind_it(gpu, tokens, hidden, inter, experts, kernels):
    """What follows a row's last element in memory is the next row: with infinities there, the row before
    must come out as without them."""
    gen = torch.Generator(device=gpu).manual_seed(3)
    draw = lambda *shape: (torch.randn(*shape, device=gpu, generator=gen) * 0.2).to(torch.bfloat16)
    x, w_router = draw(tokens, hidden), draw(hidden, experts)
    gate, up, down = draw(experts, hidden, inter), draw(experts, hidden, inter), draw(experts, inter, hidden)
    assert " ".join(forward_kernels(tokens, hidden, inter, experts)) == kernels
    clean = ops.moe_forward(x, w_router, None, gate, up, down, 1, 1.0).y
    bad = torch.arange(1, tokens, 2, device=gpu)
    x[bad, :8] = float("inf")
    got = ops.moe_forward(x, w_router, None, gate, up, down, 1, 1.0).y
    good = torch.arange(0, tokens, 2, device=gpu)
    assert torch.equal(got[good], clean[good])
