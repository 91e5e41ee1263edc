"""The sequence balance loss where a workgroup takes a whole sequence: many or short ones, either side of the rule.

The bars are those of test_gpu_balance_loss.py.
"""

from __future__ import annotations

import pytest

from research_amd import _ffi
from test_gpu_balance_loss import test_balance_loss_and_gradient_at_the_edges as check


@pytest.mark.gpu
@pytest.mark.parametrize("batch,seq,experts,top_k", [
    (255, 16, 256, 8),   # short sequences: whole, though two chunks could be had
    (255, 33, 7, 2),     # the same with eight tokens at a time: in chunks
    (256, 64, 256, 8),   # one workgroup per CU: whole whatever the length
    (257, 3, 12, 2),
    (64, 64, 256, 8),
    (70000, 1, 4, 2),    # more sequences than a grid's second dimension holds
    (3000, 5, 40, 3),
])
def test_balance_loss_of_many_sequences(gpu, batch, seq, experts, top_k):
    check(gpu, batch, seq, experts, top_k)


def test_workspace_is_one_number_per_sequence_once_they_fill_the_chip():
    lib = _ffi.load_library()
    for batch in (256, 300, 16384, 1 << 20):
        assert lib.jtmoe_balance_workspace_bytes(batch, 256) == (4 * batch + 255) // 256 * 256
