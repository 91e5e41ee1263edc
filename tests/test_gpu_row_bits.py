"""A row of the expert products has the same bits whichever kernel takes it.

The reference's invariant is prefill + decode == full forward (tests/jaxtitan/test_infer.py:270-301).  Which kernel
takes a product depends on the size of the call, so all of them add up a result in one order: 16 k values per
instruction, chained in k order, one rounding at the end.  The sizes below stand on either side of the rules that
choose: streaming tiles of 16 and 32 rows, 64-row LDS tiles, half tiles, 256-row tiles, the decode launch, shared
experts beside the router.  Equal means equal: no tolerance.
"""

from __future__ import annotations

import pytest
import torch

from research_amd import grad, ops

pytestmark = pytest.mark.gpu

WIDTHS = [(1024, 704), (512, 2816), (2048, 192), (1000, 264), (264, 1352), (72, 2056)]
DENSE_ROWS = (1, 3, 16, 17, 64, 65, 130, 260, 520, 1030, 2600)
EXPERTS = (5, 64)
GROUP_ROWS, MOST_ROWS = (1, 2, 3, 9, 20, 40, 70), 6000


def drawer(gpu, seed):
    generator = torch.Generator(device=gpu).manual_seed(seed)

    def normal(*shape, std=1.0):
        return (torch.randn(shape, generator=generator, device=gpu) * std).to(torch.bfloat16)

    return normal


@pytest.mark.parametrize("hidden,inter", WIDTHS)
def test_shared_rows_do_not_depend_on_the_call(gpu, hidden, inter):
    normal = drawer(gpu, hidden)
    x = normal(DENSE_ROWS[-1], hidden)
    matrices = normal(hidden, inter, std=0.05), normal(hidden, inter, std=0.05), normal(inter, hidden, std=0.05)
    whole = ops.shared_swiglu(x, *matrices)
    for rows in DENSE_ROWS[:-1]:
        part = ops.shared_swiglu(x[:rows].contiguous(), *matrices)
        assert torch.equal(part, whole[:rows]), f"{rows} rows: {int((part != whole[:rows]).sum())} values differ"


@pytest.mark.parametrize("hidden,inter", WIDTHS)
@pytest.mark.parametrize("experts", EXPERTS)
def test_routed_rows_do_not_depend_on_the_call(gpu, hidden, inter, experts):
    """Rows of every group: the first few of each alone against all of them."""
    normal = drawer(gpu, hidden + experts)
    per_group = MOST_ROWS // experts
    x = normal(experts * per_group, hidden)
    matrices = (normal(experts, hidden, inter, std=0.05), normal(experts, hidden, inter, std=0.05),
                normal(experts, inter, hidden, std=0.05))

    def run(rows):
        sizes = torch.full((experts,), rows, dtype=torch.int32, device=gpu)
        offsets = (torch.cumsum(sizes, 0) - sizes).to(torch.int32)
        part = x.view(experts, per_group, hidden)[:, :rows].reshape(-1, hidden).contiguous()
        return ops.grouped_swiglu(part, *matrices, sizes, offsets).view(experts, rows, hidden)

    whole = run(per_group)
    for rows in GROUP_ROWS:
        part = run(rows)
        assert torch.equal(part, whole[:, :rows]), f"{rows} rows: {int((part != whole[:, :rows]).sum())} values differ"


@pytest.mark.parametrize("hidden,inter,experts,top_k,shared", [
    (512, 704, 64, 8, 1408),  # streaming tiles and shared experts beside the router at the small sizes
    (1024, 192, 16, 2, 0),    # the decode launch from 16 tokens on
    (2048, 64, 128, 2, 128),  # the sliced router in between
])
def test_layer_rows_do_not_depend_on_the_call(gpu, hidden, inter, experts, top_k, shared):
    normal = drawer(gpu, experts)
    x, bias = normal(2700, hidden), torch.zeros(experts, device=gpu)
    weights = (normal(hidden, experts, std=0.05), bias, normal(experts, hidden, inter, std=0.05),
               normal(experts, hidden, inter, std=0.05), normal(experts, inter, hidden, std=0.05))
    extra = (normal(hidden, shared, std=0.05), normal(hidden, shared, std=0.05), normal(shared, hidden, std=0.05)) if shared else None
    whole = ops.moe_forward(x, *weights, top_k, 1.0, shared=extra)
    for rows in (1, 2, 7, 16, 33, 64, 65, 200, 257, 700, 1300):
        part = ops.moe_forward(x[:rows].contiguous(), *weights, top_k, 1.0, shared=extra)
        assert torch.equal(part.expert_ids, whole.expert_ids[:rows])
        assert torch.equal(part.y, whole.y[:rows]), f"{rows} rows: {int((part.y != whole.y[:rows]).sum())} values differ"


def off_by_one_element(t):
    """The same values at an address that is no multiple of 16: only the general kernel takes such an operand."""
    room = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    moved = room[1:].view(t.shape)
    moved.copy_(t)
    return moved


@pytest.mark.parametrize("tokens,experts,top_k,hidden,inter", [
    (2, 3, 1, 200, 72), (40, 2, 1, 264, 1352), (30, 64, 8, 1000, 264), (350, 40, 4, 264, 1352), (900, 2, 2, 1000, 328),
    (2931, 24, 3, 264, 1352), (2600, 8, 2, 104, 520), (700, 3, 1, 72, 136),
])
def test_ragged_widths_have_the_bits_of_the_general_kernel(gpu, tokens, experts, top_k, hidden, inter):
    """Routed and shared products, and the two products that a training forward keeps."""
    normal = drawer(gpu, tokens)
    x = normal(tokens, hidden)
    matrices = (normal(experts, hidden, inter, std=0.05), normal(experts, hidden, inter, std=0.05),
                normal(experts, inter, hidden, std=0.05))
    ids = torch.rand(tokens, experts, device=gpu).topk(top_k, dim=1).indices.to(torch.int32)
    plan = ops.dispatch(ids, experts, x)
    general = [off_by_one_element(m) for m in matrices]
    groups = plan.group_sizes, plan.offsets
    assert torch.equal(ops.grouped_swiglu(plan.packed_x, *matrices, *groups), ops.grouped_swiglu(plan.packed_x, *general, *groups))
    one = [m[0].contiguous() for m in matrices]
    want, kept_by_general = grad.shared_swiglu_train(x, *(off_by_one_element(m) for m in one))
    got, kept = grad.shared_swiglu_train(x, *one)
    assert torch.equal(got, want)
    assert torch.equal(kept.gate_pre, kept_by_general.gate_pre) and torch.equal(kept.up_pre, kept_by_general.up_pre)
