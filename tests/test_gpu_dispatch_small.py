"""The dispatch plan of one workgroup, whose waves own runs of consecutive assignments: sizes around a wave, a run of
one load and of several, and the largest; fewer experts than lanes and more; ids outside the experts are dropped."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from research_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts", [1, 3, 64, 129, 256])
@pytest.mark.parametrize("tokens,top_k", [(1, 1), (63, 1), (65, 1), (341, 3), (1025, 1), (387, 8), (1024, 4), (4097, 1), (8191, 1), (1024, 8)])
def test_plan(gpu, tokens, top_k, experts):
    ids = np.random.default_rng(tokens + experts).integers(0, experts, (tokens, top_k)).astype(np.int32)
    want = O.dispatch(ids, experts)
    got = ops.dispatch(torch.from_numpy(ids).to(gpu), experts)
    for name in ("group_sizes", "offsets", "source_order", "inverse"):
        np.testing.assert_array_equal(getattr(got, name).cpu().numpy(), getattr(want, name), err_msg=name)


def test_ids_outside_the_experts_have_no_row(gpu):
    ids = np.random.default_rng(5).integers(-2, 9, (700, 3)).astype(np.int32)
    got = ops.dispatch(torch.from_numpy(ids).to(gpu), 7)
    flat = ids.reshape(-1)
    valid = np.flatnonzero((flat >= 0) & (flat < 7))
    order = valid[np.argsort(flat[valid], kind="stable")]
    np.testing.assert_array_equal(got.group_sizes.cpu().numpy(), np.bincount(flat[valid], minlength=7))
    np.testing.assert_array_equal(got.source_order.cpu().numpy()[: order.size], order)
    inverse = np.full(flat.size, -1)
    inverse[order] = np.arange(order.size)
    np.testing.assert_array_equal(got.inverse.cpu().numpy(), inverse)
