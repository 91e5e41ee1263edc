"""Every kernel the bf16 expert products are dealt to, at the edges of its tiles, against the oracle.

Which one takes a product depends on the rows, the groups and the columns (grouped_gemm.hip): streaming tiles of
16, 32 or 64 rows by 64 or 128 columns where the launch has at most a tile per CU or groups of a row or four,
64-row LDS tiles for groups of up to 48 rows, 128-row tiles where 256-row ones would leave CUs idle.  The shapes
below take each of them with ragged rows, columns and reductions.  The bar is that of the other expert checks.
"""

from __future__ import annotations

import pytest
import torch

import test_gpu_grad as G
import test_gpu_parity as P
from research_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter", [
    (1, 8, 1, 1, 8),             # one row, one 8-wide chunk
    (3, 136, 4, 2, 72),          # 64-column tiles, a reduction that ends one chunk into a block
    (17, 264, 2, 1, 200),        # a second 16-row tile with one row; three blocks of 64 over two waves
    (40, 96, 48, 1, 704),        # 128-column tiles: more than 256 of 64 columns
    (30, 1024, 64, 8, 1408),     # groups of four rows, more tiles than CUs
    (128, 72, 8, 2, 2056),       # 32-row, 128-column tiles, the last column tile eight wide
    (512, 2056, 8, 2, 40),       # down: 64-row, 128-column tiles
    (350, 264, 40, 4, 136),      # 64-row LDS tiles
    (700, 296, 4, 2, 520),       # 128-row tiles with gathered rows, ten 32-deep steps and one chunk
    (2600, 328, 8, 2, 264),      # 128-row tiles of the down product, several per workgroup
    (512, 72, 64, 8, 1416),      # 128-row tiles of a data gradient, several per workgroup, a ragged second k step
])
def test_grouped_products_on_every_kernel(gpu, tokens, hidden, experts, top_k, inter):
    P.test_grouped_swiglu_matches_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")
    G.test_expert_gradients_match_oracle(gpu, tokens, hidden, experts, top_k, inter, "bf16")
    x, gate, up, down, ids, _ = P.random_problem(5, tokens, hidden, experts, top_k, inter, 0.05)
    xd, gd, ud, dd = (P.dev(a, gpu, "bf16") for a in (x, gate, up, down))
    d = ops.dispatch(P.dev(ids, gpu), experts, xd)
    if hidden % 64 == 0 and inter % 64 == 0:  # fetched through the permutation: the same sums
        assert torch.equal(ops.grouped_swiglu_gather(xd, d.source_order, top_k, gd, ud, dd, d.group_sizes, d.offsets),
                           ops.grouped_swiglu(d.packed_x, gd, ud, dd, d.group_sizes, d.offsets))


@pytest.mark.parametrize("tokens,hidden,inter", [
    (1, 2048, 2816), (16, 136, 264), (65, 200, 1000),  # 16-row tiles of 64 columns
    (130, 264, 2816),                                  # 32-row tiles of 64 columns
    (300, 328, 2056),                                  # 32-row tiles of 128 columns; down: 16- and 32-row tiles
    (1100, 520, 1352),                                 # 128-row tiles, one per CU
    (4300, 264, 1032),                                 # 256-row gate/up; down: 128-row tiles
])
def test_shared_products_on_every_kernel(gpu, tokens, hidden, inter):
    P.test_shared_swiglu_matches_oracle(gpu, tokens, hidden, inter, "bf16")
    G.test_shared_gradients_match_oracle(gpu, tokens, hidden, inter, "bf16")
