"""Layer calls of some hundred tokens, whose shared products run beside the router's finishing launch and the dispatch:
every output equals that of the operators called one by one, bit for bit, also on replays of a captured call.

The last two entries of a shape say beside which launch and in which tiles, on a device of 256 compute units;
tests/test_kernel_choice.py holds them to the rules.
"""

from __future__ import annotations

import pytest
import torch

from kernel_choice import MI355X_CUS, shared_beside
from research_amd import grad, graph, ops
from test_gpu_layer_paths import test_decode_path_equals_the_stand_alone_operators as check_layer

pytestmark = pytest.mark.gpu

SHAPES = [
    # tokens, hidden, experts, top_k, d_ff, shared width, where gate/up and down run and in which tiles
    (387, 2048, 64, 8, 1408, 2816, "router 128x64", "dispatch 64x64"),   # 25 router workgroups in front of the tiles
    (257, 1024, 64, 8, 704, 2048, "router 64x64", ""),                   # (down in the launch of the routed product)
    (234, 640, 32, 2, 128, 2544, "router 64x64", ""),                    # a small batch that finishes in blocks
    (256, 640, 24, 4, 256, 3288, "router 64x64", ""),                    # ... behind the chained router
    (677, 1024, 16, 4, 128, 832, "router 64x64", "dispatch 64x64"),
    (1128, 1024, 16, 2, 128, 496, "router 64x64", "dispatch 128x64"),    # ragged reductions, part-filled column tiles
    (1607, 1024, 16, 2, 128, 680, "router 128x64", "dispatch 128x64"),
    (512, 1152, 16, 8, 64, 1032, "router 64x64", "dispatch 64x64"),      # the most assignments
    (513, 1152, 16, 8, 64, 1032, "router 64x64", ""),                    # a dispatch in two launches
    (541, 640, 24, 2, 128, 1264, "dispatch 64x64", ""),                  # routers of one launch, chained ...
    (421, 640, 16, 1, 128, 2448, "dispatch 128x64", ""),                 # ... and not
    (300, 1152, 24, 8, 512, 1024, "", ""),                               # joint gate/up
    (300, 1024, 64, 8, 704, 8192, "", ""),                               # more tiles than CUs
]
RAGGED = (300, 1000, 64, 8, 704, 1024, "", "")  # a ragged gate/up reduction


@pytest.mark.parametrize("tokens,hidden,experts,top_k,d_ff,shared_width,gate_up,down", SHAPES)
def test_layer_equals_the_stand_alone_operators(gpu, tokens, hidden, experts, top_k, d_ff, shared_width, gate_up, down):
    if torch.cuda.get_device_properties(gpu).multi_processor_count == MI355X_CUS:
        assert shared_beside(tokens, top_k, hidden, d_ff, shared_width, experts, cus=0) == [gate_up, down]
    check_layer(gpu, tokens, hidden, experts, top_k, d_ff, shared_width)


def operands(gpu, tokens, hidden, experts, d_ff, shared_width):
    generator = torch.Generator(device=gpu).manual_seed(tokens)

    def normal(*shape, std=0.05):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    weights = (normal(hidden, experts), torch.zeros(experts, device=gpu), normal(experts, hidden, d_ff),
               normal(experts, hidden, d_ff), normal(experts, d_ff, hidden))
    shared = normal(hidden, shared_width), normal(hidden, shared_width), normal(shared_width, hidden)
    return lambda: normal(tokens, hidden, std=1.0), weights, shared


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[6], SHAPES[9], RAGGED])
def test_training_forward_keeps_the_products(gpu, shape):
    tokens, hidden, experts, top_k, d_ff, shared_width = shape[:6]
    draw, weights, shared = operands(gpu, tokens, hidden, experts, d_ff, shared_width)
    x = draw()
    trained, kept = grad.moe_forward_train(x, *weights, top_k, 1.0, shared=shared)
    shared_y, alone = grad.shared_swiglu_train(x, *shared)
    plan = ops.dispatch(trained.expert_ids, experts, x)
    packed_y = ops.grouped_swiglu(plan.packed_x, *weights[2:], plan.group_sizes, plan.offsets)
    assert torch.equal(trained.y, ops.combine(packed_y, plan.inverse, trained.weights, shared_y))
    assert torch.equal(kept.shared.gate_pre, alone.gate_pre) and torch.equal(kept.shared.up_pre, alone.up_pre)


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[4], SHAPES[9]])
def test_replays_equal_eager_calls(gpu, shape):
    tokens, hidden, experts, top_k, d_ff, shared_width = shape[:6]
    draw, weights, shared = operands(gpu, tokens, hidden, experts, d_ff, shared_width)
    captured = graph.GraphedLayer(draw(), *weights, top_k, 1.0, shared=shared)
    for _ in range(4):
        x = draw()
        want = ops.moe_forward(x, *weights, top_k, 1.0, shared=shared)
        got = captured.replay(x)
        for name in ("y", "expert_ids", "weights", "expert_counts", "importance"):
            assert torch.equal(getattr(got, name), getattr(want, name)), name
