"""Norm and combine with a wave per 512 columns of a row: bits of a wave per row.  Rows of two waves to eight, with
ends inside a wave, and batches on either side of the line between the two forms of either."""

from __future__ import annotations

import pytest
import torch

from research_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [520, 1024, 2048, 3080, 4096])
def test_norm(gpu, hidden):
    generator = torch.Generator(device=gpu).manual_seed(hidden)
    x = torch.randn(67, hidden, generator=generator, device=gpu).to(torch.bfloat16)
    scale = torch.randn(hidden + 1, generator=generator, device=gpu)
    # a scale that starts between two 16-byte boundaries takes the kernel of a wave per row
    assert torch.equal(ops.rmsnorm(x, scale[1:].clone(), 1e-6), ops.rmsnorm(x, scale[1:], 1e-6))


@pytest.mark.parametrize("hidden", [520, 1032, 3080, 4096])
def test_norm_of_the_most_rows(gpu, hidden):
    """As many rows as a workgroup each takes, and one more: the bits of any of them alone."""
    generator = torch.Generator(device=gpu).manual_seed(hidden)
    most = 8192 // ((hidden + 511) // 512)
    x = torch.randn(most + 1, hidden, generator=generator, device=gpu).to(torch.bfloat16)
    scale = torch.randn(hidden, generator=generator, device=gpu)
    over = ops.rmsnorm(x, scale, 1e-6)
    assert torch.equal(ops.rmsnorm(x[:most].contiguous(), scale, 1e-6), over[:most])
    assert torch.equal(ops.rmsnorm(x[most - 5:].contiguous(), scale, 1e-6), over[most - 5:])


@pytest.mark.parametrize("top_k", [1, 2, 8])
@pytest.mark.parametrize("hidden", [520, 1024, 2048, 3080, 4096])
def test_combine(gpu, hidden, top_k):
    """Some rows of a batch past the line, and the same rows alone."""
    generator = torch.Generator(device=gpu).manual_seed(hidden + top_k)
    waves = (hidden + 511) // 512
    tokens, few = (16384 if waves > 2 else 8192) // waves + 1, 61
    packed = torch.randn(tokens * top_k, hidden, generator=generator, device=gpu).to(torch.bfloat16)
    weights = torch.rand(tokens, top_k, generator=generator, device=gpu).to(torch.bfloat16)
    residual, shared = (torch.randn(tokens, hidden, generator=generator, device=gpu).to(torch.bfloat16) for _ in range(2))
    scale = torch.randn(hidden, generator=generator, device=gpu)
    order = torch.randperm(tokens * top_k, generator=generator, device=gpu).to(torch.int32)
    inverse = order[: few * top_k]
    alone = torch.arange(few * top_k, device=gpu, dtype=torch.int32)
    rows = packed[inverse.long()].contiguous()
    assert torch.equal(ops.combine(packed, order, weights, shared)[:few], ops.combine(rows, alone, weights[:few], shared[:few]))
    want = ops.combine_norm_residual(packed, order, weights, residual, scale, 1e-6, shared)
    got = ops.combine_norm_residual(rows, alone, weights[:few], residual[:few], scale, 1e-6, shared[:few])
    assert torch.equal(want[:few], got)
