"""Layer calls of some hundred tokens, whose shared products run beside the router's finishing launch and the dispatch:
every output equals that of the operators called one by one, bit for bit, also on replays of a captured call."""

from __future__ import annotations

import pytest
import torch

from research_amd import grad, graph, ops
from test_gpu_layer_paths import test_decode_path_equals_the_stand_alone_operators as check_layer

pytestmark = pytest.mark.gpu

SHAPES = [
    # tokens, hidden, experts, top_k, d_ff, shared width
    (387, 2048, 64, 8, 1408, 2816),  # 128 x 64 and 64 x 64 tiles, the first beside 25 router workgroups
    (257, 1024, 64, 8, 704, 2048),   # the router's smallest launch of its own per 16 tokens, 64 x 64 tiles
    (129, 1024, 128, 8, 768, 2816),  # the small batch's finish in blocks
    (512, 2048, 64, 8, 704, 1032),   # the most assignments; a ragged reduction and a part-filled column tile
    (513, 2048, 64, 8, 704, 1032),   # a dispatch in two launches: only the first product beside the router
    (300, 1152, 24, 8, 512, 1024),   # a router of one launch: the dispatch takes the first product
    (300, 1024, 64, 8, 704, 8192),   # more tiles than CUs: nothing beside
]
RAGGED = (300, 1000, 64, 8, 704, 1024)  # a ragged gate/up reduction: nothing beside


@pytest.mark.parametrize("tokens,hidden,experts,top_k,d_ff,shared_width", SHAPES)
def test_layer_equals_the_stand_alone_operators(gpu, tokens, hidden, experts, top_k, d_ff, shared_width):
    check_layer(gpu, tokens, hidden, experts, top_k, d_ff, shared_width)


def operands(gpu, tokens, hidden, experts, d_ff, shared_width):
    generator = torch.Generator(device=gpu).manual_seed(tokens)

    def normal(*shape, std=0.05):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    weights = (normal(hidden, experts), torch.zeros(experts, device=gpu), normal(experts, hidden, d_ff),
               normal(experts, hidden, d_ff), normal(experts, d_ff, hidden))
    shared = normal(hidden, shared_width), normal(hidden, shared_width), normal(shared_width, hidden)
    return lambda: normal(tokens, hidden, std=1.0), weights, shared


@pytest.mark.parametrize("shape", [SHAPES[1], RAGGED])
def test_training_forward_keeps_the_products(gpu, shape):
    tokens, hidden, experts, top_k, d_ff, shared_width = shape
    draw, weights, shared = operands(gpu, tokens, hidden, experts, d_ff, shared_width)
    x = draw()
    trained, kept = grad.moe_forward_train(x, *weights, top_k, 1.0, shared=shared)
    shared_y, alone = grad.shared_swiglu_train(x, *shared)
    plan = ops.dispatch(trained.expert_ids, experts, x)
    packed_y = ops.grouped_swiglu(plan.packed_x, *weights[2:], plan.group_sizes, plan.offsets)
    assert torch.equal(trained.y, ops.combine(packed_y, plan.inverse, trained.weights, shared_y))
    assert torch.equal(kept.shared.gate_pre, alone.gate_pre) and torch.equal(kept.shared.up_pre, alone.up_pre)


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[5]])
def test_replays_equal_eager_calls(gpu, shape):
    tokens, hidden, experts, top_k, d_ff, shared_width = shape
    draw, weights, shared = operands(gpu, tokens, hidden, experts, d_ff, shared_width)
    captured = graph.GraphedLayer(draw(), *weights, top_k, 1.0, shared=shared)
    for _ in range(4):
        x = draw()
        want = ops.moe_forward(x, *weights, top_k, 1.0, shared=shared)
        got = captured.replay(x)
        for name in ("y", "expert_ids", "weights", "expert_counts", "importance"):
            assert torch.equal(getattr(got, name), getattr(want, name)), name
