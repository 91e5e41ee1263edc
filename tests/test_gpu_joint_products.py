"""Routed and shared experts in the same launches: every output equals that of launches of their own, bit for bit.

The last four entries of a shape name the kernels of the joint launches on a device of 256 compute units (gate/up, down,
the gradients dZ and dX); tests/test_kernel_choice.py holds them to the rules.
"""

from __future__ import annotations

import pytest
import torch

from kernel_choice import MI355X_CUS, joint_kernels
from research_amd import grad, ops

pytestmark = pytest.mark.gpu

# tokens, hidden, experts, top-k, d_ff, shared d_ff: shared reductions shorter and longer than the routed ones, ragged
# widths, less than a tile of shared rows, more shared tiles than routed ones, products that stay apart
SHAPES = [
    (387, 1024, 64, 8, 1408, 2816, "separate separate separate separate"),
    (387, 1024, 8, 2, 512, 512, "separate half half_deep half_deep"),
    (500, 520, 4, 2, 512, 1352, "half_tail half half_deep half_deep"),
    (700, 1024, 8, 2, 2048, 2048, "rows256 half separate half_deep"),
    (500, 512, 4, 2, 512, 4096, "half half half_deep half_deep"),
    (900, 712, 4, 2, 1032, 520, "half_tail half half_deep half_deep"),
    (2048, 2048, 64, 8, 1408, 2816, "rows256 separate separate separate"),
    (4096, 1024, 8, 2, 2048, 2048, "separate rows256 rows256 rows256"),
    (2931, 1000, 24, 3, 2664, 2664, "separate rows256_tail separate rows256_tail"),
    (6000, 1384, 96, 2, 904, 904, "separate rows256_tail rows256_tail rows256_tail"),
    (3000, 1024, 5, 1, 768, 3072, "rows256 separate rows256 separate"),
    (2048, 1000, 8, 2, 2056, 2056, "rows256_tail rows256_tail rows256_tail rows256_tail"),
    (2600, 328, 12, 2, 1800, 4104, "rows256_tail half separate half_deep"),
    # the shortest reductions that half tiles take, eight 32-deep steps, and the longest that they do not
    (1000, 232, 8, 2, 512, 512, "half_tail half separate half_deep"),
    (1000, 224, 8, 2, 512, 512, "separate half separate half_deep"),
    (1000, 512, 8, 2, 232, 256, "half half half_deep half_deep"),
    (1000, 512, 8, 2, 224, 232, "half separate half_deep half_deep"),
]


@pytest.mark.parametrize("tokens,hidden,experts,top_k,inter,shared,kernels", SHAPES)
def test_joint_launches_have_the_bits_of_separate_ones(gpu, tokens, hidden, experts, top_k, inter, shared, kernels):
    if torch.cuda.get_device_properties(gpu).multi_processor_count == MI355X_CUS:
        assert " ".join(joint_kernels(tokens, top_k, hidden, inter, shared, experts)) == kernels
    generator = torch.Generator(device=gpu).manual_seed(tokens + hidden)

    def normal(*shape, std=0.05):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    x, dy = normal(tokens, hidden, std=1.0), normal(tokens, hidden, std=1.0)
    weights = (normal(hidden, experts), torch.zeros(experts, device=gpu), normal(experts, hidden, inter),
               normal(experts, hidden, inter), normal(experts, inter, hidden))
    extra = normal(hidden, shared), normal(hidden, shared), normal(shared, hidden)
    layer = ops.moe_forward(x, *weights, top_k, 1.0, shared=extra)
    plan = ops.dispatch(layer.expert_ids, experts, x)
    packed_y, _, routed = grad.grouped_swiglu_train(plan.packed_x, None, top_k, *weights[2:], plan.group_sizes, plan.offsets)
    shared_y, dense = grad.shared_swiglu_train(x, *extra)
    want = ops.combine(packed_y, plan.inverse, layer.weights, shared_y)
    assert torch.equal(layer.y, want), f"{int((layer.y != want).sum())} values differ"

    trained, kept = grad.moe_forward_train(x, *weights, top_k, 1.0, shared=extra)
    assert torch.equal(trained.y, want)
    for got, separate in ((kept.routed, routed), (kept.shared, dense)):
        assert torch.equal(got.gate_pre, separate.gate_pre) and torch.equal(got.up_pre, separate.up_pre)

    got = grad.moe_backward(x, dy, None, weights[0], *weights[2:], extra, trained, kept)
    dx_shared, *d_shared = grad.shared_backward(x, dy, *extra, kept.shared)
    alone = grad.experts_backward(x, dy, plan, trained.weights, *weights[2:], kept.routed)
    dx_router, d_w_router = grad.router_backward(x, weights[0], trained.scores, trained.expert_ids, alone.d_weights)
    for name, a, b in (("router", got.d_w_router, d_w_router), ("gate", got.d_gate, alone.d_gate),
                       ("up", got.d_up, alone.d_up), ("down", got.d_down, alone.d_down),
                       *zip(("shared gate", "shared up", "shared down"), got.d_shared, d_shared)):
        assert torch.equal(a, b), f"gradient of {name}: {int((a != b).sum())} values differ"
    alone = grad.experts_backward(x, dy, plan, trained.weights, *weights[2:], kept.routed, dx_extra=dx_shared + dx_router)
    assert torch.equal(got.dx, alone.dx)
