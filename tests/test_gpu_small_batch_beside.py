"""Small batches in four launches: router and shared gate/up, routed gate/up and shared down, routed down, combine.

At up to 64 tokens whose shared products run in streaming tiles, the shared gate/up tiles share the router's launch (or
the decode launch) and the shared down tiles the routed gate/up launch (or the decode path's down launch).  Every output
equals that of the operators called one by one, bit for bit, also on replays of a captured call.
"""

from __future__ import annotations

import pytest
import torch

from kernel_choice import MI355X_CUS, forward_kernels
from research_amd import _ffi, grad, graph, ops
from test_gpu_layer_paths import test_decode_path_equals_the_stand_alone_operators as check_layer

pytestmark = pytest.mark.gpu

SHAPES = [
    # tokens, hidden, experts, top_k, d_ff, shared width, the routed kernel beside the shared down tiles
    (1, 1024, 8, 2, 512, 264, "stream_16x64"),      # experts that do not fill the router's tiles
    (10, 512, 64, 8, 1408, 512, "stream_16x128"),
    (64, 1024, 8, 2, 2048, 2048, "stream_32x64"),   # four token blocks
    (64, 384, 24, 8, 2048, 64, "rows64"),           # one shared column tile
    (24, 512, 128, 8, 768, 1408, "rows64"),
    (15, 1024, 64, 8, 704, 2816, "stream_16x128"),  # the last batch before the decode launch, and the decode launch,
    (16, 1024, 64, 8, 704, 2816, "decode"),         # whose down kernels are streaming tiles
    (64, 2048, 64, 8, 64, 1000, "decode"),          # and 64-row ones
    (20, 128, 16, 2, 64, 72, "decode"),
]


@pytest.mark.parametrize("tokens,hidden,experts,top_k,d_ff,shared_width,kernel", SHAPES)
def test_layer_equals_the_stand_alone_operators(gpu, tokens, hidden, experts, top_k, d_ff, shared_width, kernel):
    assert forward_kernels(tokens, hidden, shared_width, cus=MI355X_CUS) == ("stream_16x64", "stream_16x64")
    decode = ops._lib().jtmoe_moe_forward_takes_decode_path(tokens, hidden, experts, top_k, d_ff, _ffi.JTMOE_BF16) == 1
    assert decode == (kernel == "decode")
    if not decode:
        assert forward_kernels(tokens * top_k, hidden, d_ff, experts, MI355X_CUS)[0] == kernel
    check_layer(gpu, tokens, hidden, experts, top_k, d_ff, shared_width)


@pytest.mark.parametrize("tokens,hidden,experts,top_k,d_ff,shared_width,kernel", [
    (2, 256, 32, 2, 64, 136, "stream_16x64"),
    (64, 1024, 8, 2, 2048, 2048, "stream_32x64"),
    (64, 384, 24, 8, 2048, 64, "rows64"),
    (24, 512, 16, 2, 396, 264, "general"),  # takes no tiles along: the shared down product in a launch of its own
])
def test_training_forward_keeps_every_product(gpu, tokens, hidden, experts, top_k, d_ff, shared_width, kernel):
    """The training forward, whose routed gate/up beside the shared down tiles keeps its two products, and the inference
    call, against the operators one by one."""
    assert forward_kernels(tokens, hidden, shared_width, cus=MI355X_CUS) == ("stream_16x64", "stream_16x64")
    assert forward_kernels(tokens * top_k, hidden, d_ff, experts, MI355X_CUS)[0] == kernel
    generator = torch.Generator(device=gpu).manual_seed(tokens + d_ff)

    def normal(*shape, std=0.05):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    x, weights = normal(tokens, hidden, std=1.0), (normal(hidden, experts), torch.zeros(experts, device=gpu),
                                                   normal(experts, hidden, d_ff), normal(experts, hidden, d_ff),
                                                   normal(experts, d_ff, hidden))
    shared = normal(hidden, shared_width), normal(hidden, shared_width), normal(shared_width, hidden)
    trained, kept = grad.moe_forward_train(x, *weights, top_k, 1.0, shared=shared)
    plan = ops.dispatch(trained.expert_ids, experts, x)
    packed_y, _, routed = grad.grouped_swiglu_train(plan.packed_x, None, top_k, *weights[2:], plan.group_sizes, plan.offsets)
    shared_y, dense = grad.shared_swiglu_train(x, *shared)
    want = ops.combine(packed_y, plan.inverse, trained.weights, shared_y)
    assert torch.equal(trained.y, want)
    assert torch.equal(ops.moe_forward(x, *weights, top_k, 1.0, shared=shared).y, want)
    for got, alone in ((kept.routed, routed), (kept.shared, dense)):
        assert torch.equal(got.gate_pre, alone.gate_pre) and torch.equal(got.up_pre, alone.up_pre)


@pytest.mark.parametrize("tokens,hidden,experts,top_k,d_ff,shared_width", [(1, 1024, 8, 2, 512, 264), (9, 512, 64, 8, 704, 1408),
                                                                           (40, 512, 64, 8, 704, 1408)])
def test_replays_equal_eager_calls(gpu, tokens, hidden, experts, top_k, d_ff, shared_width):
    """Four replays on four inputs, with eager calls through the same kind of workspace in between."""
    generator = torch.Generator(device=gpu).manual_seed(tokens)

    def normal(*shape, std=0.05):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    weights = (normal(hidden, experts), torch.zeros(experts, device=gpu), normal(experts, hidden, d_ff),
               normal(experts, hidden, d_ff), normal(experts, d_ff, hidden))
    shared = normal(hidden, shared_width), normal(hidden, shared_width), normal(shared_width, hidden)
    captured = graph.GraphedLayer(normal(tokens, hidden, std=1.0), *weights, top_k, 1.0, shared=shared)
    for _ in range(4):
        x = normal(tokens, hidden, std=1.0)
        want = ops.moe_forward(x, *weights, top_k, 1.0, shared=shared)
        got = captured.replay(x)
        torch.cuda.synchronize()
        for name in ("y", "expert_ids", "weights", "scores", "expert_counts", "importance"):
            assert torch.equal(getattr(got, name), getattr(want, name)), name
