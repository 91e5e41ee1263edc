"""Every kernel the bf16 expert products are dealt to, at the edges of its tiles, against the oracle.

Which one takes a product depends on the rows, the groups and the columns (grouped_gemm.hip): streaming tiles of
16 or 32 rows where the launch has at most a tile per CU, or a few per CU and groups of a few rows; 64-row LDS tiles
for groups of up to 52 rows; 128-row tiles where 256-row ones would leave CUs idle; 256-row tiles.  The shapes below
take each of them with ragged rows, columns and reductions, and name the kernels of gate/up and down and those of the
two data gradients; a rule that sends a case elsewhere fails it.  The bar is that of the other expert checks.
"""

from __future__ import annotations

import pytest
import torch

import test_gpu_grad as G
import test_gpu_parity as P
from kernel_choice import forward_kernels, gradient_kernels
from research_amd import ops

pytestmark = pytest.mark.gpu


GROUPED = [
    (1, 8, 1, 1, 8, "stream_16x64 stream_16x64", "half half"),                # one row, one 8-wide chunk
    (3, 136, 4, 2, 72, "stream_16x64 stream_16x64", "half half"),             # a reduction that ends one chunk into a block
    (17, 264, 2, 1, 200, "stream_16x64 stream_16x64", "half half_deep"),      # a second 16-row tile with one row
    (40, 96, 48, 1, 704, "stream_16x128 stream_16x64", "half half_deep"),     # more than 256 tiles of 64 columns
    (30, 1024, 64, 8, 1408, "rows64 stream_16x128", "half half"),             # groups of four rows, more tiles than CUs
    (128, 72, 8, 2, 2056, "rows64_tail stream_16x64", "half half_deep"),      # the last column tile eight wide
    (512, 2056, 8, 2, 40, "stream_16x64 rows256_tail", "half_deep half"),     # a reduction of one ragged step
    (350, 264, 40, 4, 136, "stream_16x128 rows64", "half half"),
    (700, 296, 4, 2, 520, "half_tail stream_32x64", "half half_deep"),        # ten 32-deep steps, the last of one chunk
    (2600, 328, 8, 2, 264, "half_tail half", "half half_deep"),
    (512, 72, 64, 8, 1416, "rows256_short_tail half", "half half_deep"),      # a gradient with several tiles per workgroup
    (500, 512, 64, 8, 704, "rows256 half", "half half_deep"),                 # ragged ends of 64 groups
    (1100, 320, 4, 2, 1032, "half half", "half half_deep"),
    (16500, 256, 3, 2, 192, "rows256 rows256", "rows256 rows256"),
    (9000, 64, 8, 2, 1024, "rows256_short half", "half half_deep"),           # two 64-deep steps
]


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter,forward,gradients", GROUPED)
def test_grouped_products_on_every_kernel(gpu, tokens, hidden, experts, top_k, inter, forward, gradients):
    assert " ".join(forward_kernels(tokens * top_k, hidden, inter, experts)) == forward
    assert " ".join(gradient_kernels(tokens * top_k, hidden, inter, experts)) == gradients
    P.test_grouped_swiglu_matches_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")
    G.test_expert_gradients_match_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")
    x, gate, up, down, ids, _ = P.random_problem(5, tokens, hidden, experts, top_k, inter, 0.05)
    xd, gd, ud, dd = (P.dev(a, gpu, "bf16") for a in (x, gate, up, down))
    d = ops.dispatch(P.dev(ids, gpu), experts, xd)
    if hidden % 64 == 0 and inter % 64 == 0:  # fetched through the permutation: the same sums
        assert torch.equal(ops.grouped_swiglu_gather(xd, d.source_order, top_k, gd, ud, dd, d.group_sizes, d.offsets),
                           ops.grouped_swiglu(d.packed_x, gd, ud, dd, d.group_sizes, d.offsets))


DENSE = [
    (1, 2048, 2816, "stream_16x64 stream_16x64", "half_deep half_deep"),
    (16, 136, 264, "stream_16x64 stream_16x64", "half half_deep"),
    (65, 200, 1000, "stream_16x64 stream_16x64", "half half_deep"),
    (130, 264, 2816, "stream_32x64 stream_16x64", "half half_deep"),
    (300, 328, 2056, "half_tail stream_16x64", "half half_deep"),
    (1100, 520, 1352, "half_tail half", "half_deep half_deep"),
    (4300, 264, 1032, "rows256_tail half", "half half_deep"),
    (5000, 1024, 1032, "rows256 half_deep", "half half"),
]


@pytest.mark.parametrize("tokens,hidden,inter,forward,gradients", DENSE)
def test_shared_products_on_every_kernel(gpu, tokens, hidden, inter, forward, gradients):
    assert " ".join(forward_kernels(tokens, hidden, inter)) == forward
    assert " ".join(gradient_kernels(tokens, hidden, inter)) == gradients
    P.test_shared_swiglu_matches_oracle(gpu, tokens, hidden, inter, "bf16")
    G.test_shared_gradients_match_oracle(gpu, tokens, hidden, inter, "bf16")
