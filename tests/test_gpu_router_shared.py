"""The shared experts beside a small batch's router: the bits of the operators called one by one.

At up to 64 tokens whose shared products run in 16-row, 64-column streaming tiles, the layer's two router launches
take the shared gate/up and down tiles along.  The shapes stand at the edges of that rule and just beyond it.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kernel_choice import forward_kernels
from research_amd import _ffi, grad, ops
from test_gpu_layer_paths import test_decode_path_equals_the_stand_alone_operators as check_layer
from test_gpu_parity import dev

pytestmark = pytest.mark.gpu


SHAPES = [
    # tokens, hidden, experts, top_k, d_ff, shared width, whether the router takes the shared experts along
    (1, 2048, 64, 8, 1408, 2816, True),   # the benchmark's model
    (1, 128, 16, 1, 64, 8, True),         # one slice, one 8-wide column tile, a reduction of one chunk
    (3, 384, 16, 1, 64, 200, True),       # three slices, a ragged last column tile
    (15, 256, 64, 8, 64, 1000, True),     # the last row of a 16-row tile missing
    (17, 2176, 256, 1, 64, 72, True),     # two token blocks, the second of one token; 256 experts
    (64, 1024, 128, 2, 64, 2816, True),   # the largest batch
    (65, 1024, 128, 1, 64, 2816, False),  # a token more: launches of their own
    (64, 128, 128, 1, 64, 8200, False),   # more tiles than CUs: launches of their own
]


@pytest.mark.parametrize("tokens,hidden,experts,top_k,d_ff,shared_width,beside", SHAPES)
def test_layer_equals_the_stand_alone_operators(gpu, tokens, hidden, experts, top_k, d_ff, shared_width, beside):
    assert beside == (tokens <= 64 and forward_kernels(tokens, hidden, shared_width) == ("stream_16x64", "stream_16x64"))
    check_layer(gpu, tokens, hidden, experts, top_k, d_ff, shared_width)


@pytest.mark.parametrize("tokens", [2, 33])
def test_training_forward_keeps_the_shared_products(gpu, tokens):
    hidden, experts, top_k, d_ff, shared_width = 256, 32, 2, 64, 136
    rng = np.random.default_rng(tokens)

    def normal(scale, *shape):
        return dev((rng.standard_normal(shape) * scale).astype(np.float32), gpu, "bf16")

    x, w_router = normal(1.0, tokens, hidden), normal(0.1, hidden, experts)
    gate, up, down = normal(0.05, experts, hidden, d_ff), normal(0.05, experts, hidden, d_ff), normal(0.05, experts, d_ff, hidden)
    shared = normal(0.05, hidden, shared_width), normal(0.05, hidden, shared_width), normal(0.05, shared_width, hidden)
    _, kept = grad.moe_forward_train(x, w_router, None, gate, up, down, top_k, 1.0, shared=shared)
    _, alone = grad.shared_swiglu_train(x, *shared)
    assert torch.equal(kept.shared.gate_pre, alone.gate_pre)
    assert torch.equal(kept.shared.up_pre, alone.up_pre)


@pytest.mark.parametrize("tokens", [1, 20])
def test_a_timed_call_times_the_shared_experts_as_such(gpu, tokens):
    generator = torch.Generator(device=gpu).manual_seed(tokens)

    def normal(*shape):
        return (torch.randn(shape, generator=generator, device=gpu) * 0.05).to(torch.bfloat16)

    args = (normal(tokens, 512), normal(512, 64), None, normal(64, 512, 64), normal(64, 512, 64), normal(64, 64, 512), 4, 1.0)
    shared = normal(512, 1024), normal(512, 1024), normal(1024, 512)
    stage_ms = []
    timed = ops.moe_forward(*args, shared=shared, stage_ms=stage_ms)
    assert torch.equal(timed.y, ops.moe_forward(*args, shared=shared).y)
    stages = dict(zip(_ffi.STAGE_NAMES, stage_ms))
    assert stages["shared_gate_up"] > 0.0 and stages["shared_down"] > 0.0, stages
