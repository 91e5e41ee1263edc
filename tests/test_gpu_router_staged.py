"""The projection of everything the matrix-core router does not take, at the edges of its chunks.

A chunk is 128 (bf16) or 64 (fp32) k rows of 16 tokens; a thread owns ceil(16 E / 256) logits.  The cases
sit either side of those limits and of the 16-byte rows that the vector loads need.  The bar is that of
the other projection kernels (one ulp of the compute dtype on the logits, then bit-exact decisions).
"""

from __future__ import annotations

import numpy as np
import pytest

import test_gpu_parity as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,hidden,experts,top_k,dtype", [
    (1, 1, 1, 1, "bf16"),          # a single logit of a single term
    (16, 128, 17, 2, "bf16"),      # one whole chunk, two logits per thread
    (17, 136, 15, 3, "bf16"),      # a ragged second chunk and token block
    (33, 1000, 24, 3, "bf16"),     # several chunks, the last of 104 rows
    (15, 129, 33, 4, "bf16"),      # rows that are no whole vectors
    (40, 264, 96, 4, "bf16"),      # eight logits per thread
    (20, 72, 255, 8, "bf16"),      # sixteen logits per thread
    (31, 64, 8, 2, "f32"),         # one whole fp32 chunk
    (65, 68, 16, 2, "f32"),        # a second chunk of one vector
    (18, 127, 65, 5, "f32"),       # no whole vectors
    (50, 200, 256, 16, "f32"),     # the largest expert count and top-k
])
def test_projection_at_the_edges_of_its_chunks(gpu, tokens, hidden, experts, top_k, dtype):
    rng = np.random.default_rng(tokens * 31 + hidden)
    x = rng.standard_normal((tokens, hidden)).astype(np.float32)
    w = (rng.standard_normal((hidden, experts)) * 0.02).astype(np.float32)
    bias = (rng.standard_normal(experts) * 0.05).astype(np.float32)
    P.check_router_end_to_end(gpu, x, w, bias, top_k, 1.0, dtype)
