"""A branch whose sum is left to the next norm: it is added once, what it sums is let go then, and who hands such a branch on."""
import gc
import weakref
from types import SimpleNamespace

import pytest
import torch

from ullm_amd.parts import NormedBranch
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


@pytest.mark.parametrize("takes,offers", [(True, True), (True, False), (False, True)])
def test_the_sum_is_left_to_norms_that_take_it(takes, offers):
    from ullm_amd.parts.block import ParallelBlock
    x, mixed = torch.zeros(2, 3), torch.ones(2, 3)
    norm = SimpleNamespace(takes_sums=takes, add_norm=lambda *a, **k: x)
    ffn = SimpleNamespace(forward_onto=lambda h, ctx, base: base + 1)
    if offers:
        ffn.branch_onto = lambda h, ctx, base, mult: SummedBranch(lambda: base + 1, None, torch.bfloat16, mult)
    block = ParallelBlock(norm, SimpleNamespace(forward=lambda h, ctx, cache: mixed), ffn, 0.25)
    _, b = block.forward(x, None, SimpleNamespace(dtype=torch.bfloat16, whole_branch=False), None)
    assert isinstance(b, SummedBranch) == (takes and offers) and isinstance(b, NormedBranch)
    assert b.mult == 0.25 and torch.equal(b.joined(), mixed + 1)


def test_a_subclass_that_sums_otherwise_is_asked():
    from ullm_amd.parts.moe import RoutedExperts

    class Doubled(RoutedExperts):
        def __init__(self):
            pass

        def forward_onto(self, x, ctx, base, bias=None):
            return 2 * base
    b = Doubled().branch_onto(None, None, torch.ones(2, 3), 0.5)
    assert not isinstance(b, SummedBranch) and b.mult == 0.5 and b.joined().sum() == 12
