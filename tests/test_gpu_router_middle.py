"""The router of middle-sized layer calls (slices of the k range in workgroups of their own) and the dispatch behind
it: the bits of the stand-alone entry points, at the edges of the rules that choose the launches."""

from __future__ import annotations

import pytest

from test_gpu_layer_paths import test_layer_routing_outputs_equal_the_stand_alone_entry_points as check_routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,hidden,experts,top_k", [
    (257, 2048, 64, 8),   # the smallest batch; one row in the last block of 16
    (2560, 2176, 64, 2),  # the largest; 17 chunks of 128: slices of three, the last of two
    (2561, 2048, 64, 2),  # a token more: 64-token workgroups
    (1000, 2048, 128, 8),
    (600, 2048, 128, 1),
    (257, 1024, 16, 2),   # the narrowest rows: eight slices of one chunk
    (700, 1152, 32, 4),   # nine chunks: slices of two, the last of one
    (2560, 1024, 256, 8), # the most experts
    (700, 896, 256, 2),   # narrower: 64-token workgroups
    (512, 128, 16, 8),    # 4096 assignments: one workgroup
    (513, 128, 16, 8),    # 4104: histogram and rank passes
])
def test_routing_outputs_equal_the_stand_alone_entry_points(gpu, tokens, hidden, experts, top_k):
    # (d_ff as wide as the partial sums need: they live where the activations go later)
    check_routing(gpu, tokens, hidden, experts, top_k, 64 if top_k * 64 >= 16 * experts else 16 * experts // top_k, "bf16")
