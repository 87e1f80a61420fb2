"""The grouping of (token, expert) pairs: pair counts on both sides of what a block's threads keep in registers
(16 each of 1024 threads), expert counts on both sides of one wave's running sum, experts without weights among them."""
import pytest
import torch

from ullm_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,top,experts,outputs,tile_rows", [
    (1, 1, 1, 1, 16), (1, 4, 3, 7, 16), (255, 4, 32, 32, 32), (4096, 4, 64, 65, 128), (4097, 4, 65, 65, 64), (8193, 4, 130, 144, 256)])
def test_every_pair_has_a_slot_of_its_expert(tokens, top, experts, outputs, tile_rows):
    gen = torch.Generator().manual_seed(tokens)
    ids = torch.rand(tokens, outputs, generator=gen).topk(top, -1).indices.int()
    slot, token, tiles, offsets = (t.cpu() for t in ops.moe_sort(ids.cuda(), experts, tile_rows))
    flat = ids.view(-1).long()
    counts = torch.bincount(flat, minlength=outputs)[:experts]
    ends = torch.cumsum(counts, 0)
    assert offsets.tolist() == [0] + ends.tolist()
    inside = flat < experts
    assert (slot[~inside] == -1).all()
    taken = slot[inside].long()
    assert torch.equal(taken.sort().values, torch.arange(int(ends[-1])))
    assert (taken >= (ends - counts)[flat[inside]]).all() and (taken < ends[flat[inside]]).all()
    assert torch.equal(token[taken].long(), inside.nonzero().view(-1) // top)
    expect = [(e, int(ends[e] - counts[e]) + i, min(tile_rows, int(counts[e]) - i))
              for e in range(experts) for i in range(0, int(counts[e]), tile_rows)]
    assert int(tiles[-1, 0]) == len(expect)
    assert [tuple(t) for t in tiles[:len(expect)].tolist()] == expect and (tiles[len(expect):-1, 2] == 0).all()
