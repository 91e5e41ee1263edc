"""The single-precision matrix-core products at the edges of their tiles (64 and 128 rows and columns, k steps
of 32, chunks of 4), against the oracle.

Bars: the forward's f32_tol.  Gradients: max|g - ref| / max|ref| <= 2^-23 * sqrt(n) * 8 for sums of n terms --
each of two summation orders is off by about sqrt(n) roundings of 2^-24 of the terms' size, and a factor of
eight covers the largest of the elements and the chain of three products.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import test_gpu_grad as G
import test_gpu_parity as P
from kernel_choice import MI355X_CUS, f32_backward_kernel
from oracle import moe_grad_oracle as GO
from oracle import moe_oracle as O
from research_amd import grad
from test_gpu_parity import dev, host, random_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter", [
    (1, 4, 1, 1, 4),          # one row, one chunk
    (65, 36, 3, 2, 68),       # a second 32-deep step of one chunk, tiles with one row
    (400, 128, 2, 2, 192),    # whole tiles with gathered rows
    (600, 260, 3, 1, 132),    # columns and steps that end one chunk in
    (2500, 64, 4, 2, 256),    # enough tiles for 128-row gate/up tiles: 168 of them against 324 in two rounds of 256
    (2500, 644, 4, 2, 652),   # ... and 128 x 128 down products and data gradients (252 against 891 tiles), ragged ends
    (1200, 508, 8, 2, 1020),  # ... and weight gradients, single (256 against 1024) and dual
])
def test_f32_experts_at_tile_edges(gpu, tokens, hidden, experts, top_k, inter):
    P.test_grouped_swiglu_matches_oracle(gpu, tokens, hidden, experts, top_k, inter, "f32")
    x, gate, up, down, ids, w = random_problem(7 + tokens, tokens, hidden, experts, top_k, inter, 0.1)
    dy = np.random.default_rng(tokens).standard_normal((tokens, hidden)).astype(np.float32)
    want = GO.experts_backward(x, ids, w, gate, up, down, dy)
    got, _ = G.expert_grads(gpu, x, ids, w, gate, up, down, dy, "f32")
    bar = 2.0 ** -23 * 8 * np.sqrt(max(hidden, inter, tokens * top_k))
    for name in ("dx", "d_weights", "d_gate", "d_up", "d_down"):
        assert P.report(f"f32 {name}", host(getattr(got, name)), getattr(want, name).astype(np.float32)) <= bar, name


@pytest.mark.parametrize("tokens,hidden,inter", [(130, 68, 36), (1000, 128, 64), (4100, 256, 4)])
def test_f32_shared_experts_with_split_reductions(gpu, tokens, hidden, inter):
    """One group: the weight gradients are cut into runs of rows whose partial sums are added in order."""
    rng = np.random.default_rng(tokens)
    x, dy = (rng.standard_normal((tokens, hidden)).astype(np.float32) for _ in range(2))
    mats = [(rng.standard_normal(s) * 0.1).astype(np.float32) for s in ((hidden, inter), (hidden, inter), (inter, hidden))]
    md = [dev(m, gpu) for m in mats]
    y, res = grad.shared_swiglu_train(dev(x, gpu), *md)
    np.testing.assert_allclose(host(y), O.shared_swiglu(x, *mats, "f32"), **P.f32_tol(O.shared_swiglu(x, *mats, "f32")))
    got = grad.shared_backward(dev(x, gpu), dev(dy, gpu), *md, res)
    again = grad.shared_backward(dev(x, gpu), dev(dy, gpu), *md, res)
    leaves = [torch.from_numpy(a.astype(np.float64)).requires_grad_() for a in (x, *mats)]
    h = torch.nn.functional.silu(leaves[0] @ leaves[1]) * (leaves[0] @ leaves[2])
    want = torch.autograd.grad(h @ leaves[3], leaves, torch.from_numpy(dy.astype(np.float64)))
    bar = 2.0 ** -23 * 8 * np.sqrt(max(hidden, inter, tokens))
    for g, a, ref in zip(got, again, want):
        assert torch.equal(g, a)
        assert P.report("f32 shared", host(g), ref.numpy().astype(np.float32)) <= bar


# tokens, hidden, experts, d_ff, how the products of the backward pass run, and (tokens, experts) of a larger call whose
# first groups are these and whose products have launches of their own
BACKWARD_SHAPES = [
    (3, 4, 5, 4, "joint", (4099, 250)),         # one chunk, groups of at most three rows, two of them empty
    (300, 260, 5, 132, "joint", (1200, 64)),    # columns one chunk past a tile; a group without rows between groups with some
    (700, 132, 16, 68, "joint", (1700, 250)),   # short reductions, most tiles partly filled
    (2048, 512, 8, 1024, "joint", (3048, 10)),
    (8192, 512, 8, 1024, "separate", (9192, 10)),  # rounds of the launches of their own are nearly full
]


@pytest.mark.parametrize("tokens,hidden,experts,inter,launches,larger", BACKWARD_SHAPES)
def test_f32_backward_products_in_one_launch(gpu, tokens, hidden, experts, inter, launches, larger):
    """dXp and the three weight gradients with uneven groups and empty ones, against float64.  The same groups among the
    first of a larger call, whose products run in launches of their own, have the same bits."""
    if torch.cuda.get_device_properties(gpu).multi_processor_count == MI355X_CUS:
        assert f32_backward_kernel(tokens, hidden, inter, experts) == launches
        assert f32_backward_kernel(larger[0], hidden, inter, larger[1]) == "separate"
    rng = np.random.default_rng(tokens + hidden)
    share = np.where(np.arange(experts) % 4 == 1, 0.0, 1.0 + np.arange(experts) ** 2)
    first = rng.choice(experts, tokens, p=share / share.sum())
    ids = first.astype(np.int32)[:, None]
    x, dy = (rng.standard_normal((tokens, hidden)).astype(np.float32) for _ in range(2))
    w = rng.uniform(0.5, 1.0, (tokens, 1)).astype(np.float32)
    gate, up = ((rng.standard_normal((experts, hidden, inter)) * 0.1).astype(np.float32) for _ in range(2))
    down = (rng.standard_normal((experts, inter, hidden)) * 0.1).astype(np.float32)
    got, _ = G.expert_grads(gpu, x, ids, w, gate, up, down, dy, "f32")

    def extended(a, n, scale):
        return np.concatenate([a, (rng.standard_normal((n - len(a), *a.shape[1:])) * scale).astype(np.float32)])

    more = rng.integers(experts, larger[1], (larger[0] - tokens, 1)).astype(np.int32)
    alone, _ = G.expert_grads(gpu, extended(x, larger[0], 1.0), np.concatenate([ids, more]), extended(w, larger[0], 1.0),
                              *(extended(m, larger[1], 0.1) for m in (gate, up, down)), extended(dy, larger[0], 1.0), "f32")
    leaves = [torch.from_numpy(a.astype(np.float64)).requires_grad_() for a in (x, gate, up, down)]
    y = torch.zeros(tokens, hidden, dtype=torch.float64)
    for e in range(experts):
        rows = torch.from_numpy(np.flatnonzero(first == e))
        h = torch.nn.functional.silu(leaves[0][rows] @ leaves[1][e]) * (leaves[0][rows] @ leaves[2][e])
        y = y.index_put((rows,), (h @ leaves[3][e]) * torch.from_numpy(w[rows].astype(np.float64)))
    want = torch.autograd.grad(y, leaves, torch.from_numpy(dy.astype(np.float64)))
    bar = 2.0 ** -23 * 8 * np.sqrt(max(hidden, inter, tokens))
    for name, ref in zip(("dx", "d_gate", "d_up", "d_down"), want):
        assert torch.equal(getattr(got, name), getattr(alone, name)[:len(ref)]), name
        assert P.report(f"f32 {name}", host(getattr(got, name)), ref.numpy().astype(np.float32)) <= bar, name
