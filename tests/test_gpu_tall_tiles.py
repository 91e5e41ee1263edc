"""256-row tiles of up to 320 rows, and part-filled ones beside them: every row has the bits of its group alone.

The group sizes stand on either side of what tiles take beyond 256 rows (64 each, from a group's first tile on) and of
the row blocks that a part-filled tile leaves out; taller tiles spare a round in each of the products named, which
tests/test_kernel_choice.py holds to the rules.
"""

from __future__ import annotations

import pytest
import torch

from research_amd import grad, ops

pytestmark = pytest.mark.gpu

SIZES = (257, 320, 577, 1100, 0, 1279, 1025, 1, 300, 65, 2303, 33)


WIDTHS = [
    # ..., the products (gate/up, down, dZ, dX) that take them
    (256, 4096, (0, 2)),  # the fewest whole steps
    (264, 4104, (0, 2)),  # ... whose last step holds one chunk
    (4096, 256, (1, 3)),
    (4104, 264, (1, 3)),
]


@pytest.mark.parametrize("hidden,inter", [widths[:2] for widths in WIDTHS])
def test_rows_have_the_bits_of_their_group_alone(gpu, hidden, inter):
    generator = torch.Generator(device=gpu).manual_seed(hidden)

    def normal(*shape, std=0.05):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    experts, tokens = len(SIZES), sum(SIZES)
    x, dy = normal(tokens, hidden, std=1.0), normal(tokens, hidden, std=1.0)
    weights = normal(experts, hidden, inter), normal(experts, hidden, inter), normal(experts, inter, hidden)
    ids = torch.repeat_interleave(torch.arange(experts, device=gpu), torch.tensor(SIZES, device=gpu)).to(torch.int32)
    ids = ids[torch.randperm(tokens, generator=torch.Generator().manual_seed(1)).to(gpu)].view(tokens, 1).contiguous()

    def run(x, dy, ids, weights):
        plan = ops.dispatch(ids, weights[0].shape[0], x)
        y, _, kept = grad.grouped_swiglu_train(x, plan.source_order, 1, *weights, plan.group_sizes, plan.offsets)
        route = torch.ones((x.shape[0], 1), dtype=x.dtype, device=gpu)
        return y, grad.experts_backward(x, dy, plan, route, *weights, kept).dx

    packed_y, dx = run(x, dy, ids, weights)
    at = 0
    for e, size in enumerate(SIZES):
        if size == 0:
            continue
        rows = torch.nonzero(ids.view(-1) == e).view(-1)
        alone_y, alone_dx = run(x[rows], dy[rows], torch.zeros((size, 1), dtype=torch.int32, device=gpu),
                                [m[e:e + 1].contiguous() for m in weights])
        assert torch.equal(packed_y[at:at + size], alone_y), f"group of {size} rows"
        assert torch.equal(dx[rows], alone_dx), f"dx of a group of {size} rows"
        at += size
