"""A branch whose sum is left to the next norm: it is added once, and what it sums is let go then."""
import gc
import weakref

import pytest
import torch

from ullm_amd.parts.base import SummedBranch


def _branch():
    rows = torch.ones(2, 3)
    return SummedBranch(lambda: rows + 0, lambda residual, *rest: residual + rows, torch.bfloat16, 0.5), weakref.ref(rows)


def test_what_is_summed_is_let_go_once_it_is_added():
    b, rows = _branch()
    y = b.added_and_squashed(torch.zeros(2, 3), None, None, None, torch.bfloat16)
    gc.collect()
    assert rows() is None and y.sum() == 6


def test_what_is_summed_is_let_go_once_the_sum_is_made():
    b, rows = _branch()
    assert b.added_and_squashed(torch.zeros(2, 3), None, None, None, torch.float32) is None and rows() is not None
    total = b.branch
    gc.collect()
    assert rows() is None and b.joined() is total
    assert b.added_and_squashed(torch.zeros(2, 3), None, None, None, torch.bfloat16) is None


def test_it_is_added_once():
    b, _ = _branch()
    b.added_and_squashed(torch.zeros(2, 3), None, None, None, torch.bfloat16)
    with pytest.raises(RuntimeError, match="twice"):
        b.added_and_squashed(torch.zeros(2, 3), None, None, None, torch.bfloat16)
    with pytest.raises(RuntimeError, match="twice"):
        b.branch
    with pytest.raises(RuntimeError, match="twice"):
        b.joined()
