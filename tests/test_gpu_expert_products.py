"""The experts' products over large tiles: rows on both sides of a wave's 64 and a tile's edge, one to five stages of K,
columns past the last block's, a gathered and a plain row order, against 64-bit results."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from ullm_amd.kernels import ops
    return ops


@pytest.mark.parametrize("tile_rows", [128, 256])
@pytest.mark.parametrize("K,n_out", [(64, 130), (128, 256), (192, 64), (256, 388), (320, 260)])
@pytest.mark.parametrize("limit", [0.0, 1.5])
def test_experts_with_rows_at_every_edge(ops, tile_rows, K, n_out, limit):
    g = torch.Generator().manual_seed(K + n_out + tile_rows)
    counts = [1, 63, 64, 65, 0, 127, 128, 129, 255, 256, 257, 16]
    experts, T = len(counts), sum(counts)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=g)].int()[:, None].contiguous().to(DEV)
    wide = torch.randn(T, K + 8, generator=g).bfloat16().to(DEV)
    x = wide[:, :K]                                                   # rows further apart than they are long
    w_gu = (torch.randn(experts, 2 * n_out, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    w = (torch.randn(experts, n_out, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    slot, token, tiles, offsets = ops.moe_sort(ids, experts, tile_rows)
    gated = ops.moe_rows(x, token, w_gu, tiles, tile_rows, T, gated=True, limit=limit, alpha=1.3)
    by_slot = x[token.long()].contiguous()
    plain = ops.moe_rows(by_slot, None, w, tiles, tile_rows, T, gated=False)
    at = offsets.cpu().tolist()
    for e, n in enumerate(counts):
        rows = slice(at[e], at[e] + n)
        assert at[e + 1] - at[e] == n
        h = by_slot[rows].double()
        size = h.abs() @ w[e].double().abs().T
        assert ((plain[rows].double() - h @ w[e].double().T).abs() <= (K + 1) * 2.0 ** -24 * size).all()    # K 32-bit sums
        gu = h @ w_gu[e].double().T
        a, u = gu[:, :n_out], gu[:, n_out:]
        if limit:
            a, u = a.clamp(max=limit), u.clamp(-limit, limit)
            want = a * torch.sigmoid(1.3 * a) * (u + 1)
        else:
            want = a * torch.sigmoid(a) * u
        # the result's rounding to bfloat16, and of the 32-bit sums what the unit makes of it (its slopes are below 3 + |u|)
        off = (K + 8) * 2.0 ** -24 * (h.abs() @ w_gu[e].double().abs().T).amax(-1, keepdim=True) * (4 + u.abs() + a.abs())
        assert ((gated[rows].double() - want).abs() <= 2.0 ** -8 * want.abs() + off).all()
    # a row's result does not depend on the rows beside it: 128 and 256 rows a tile add up the same way
    other = 384 - tile_rows
    slot2, token2, tiles2, _ = ops.moe_sort(ids, experts, other)
    again = ops.moe_rows(x[token2.long()].contiguous(), None, w, tiles2, other, T, gated=False)
    assert torch.equal(again[slot2.long()], plain[slot.long()])


@pytest.mark.parametrize("tile_rows", [16, 32])
@pytest.mark.parametrize("K,n_out", [(256, 40), (320, 16), (448, 129), (704, 34), (1024, 4), (200, 48)])
@pytest.mark.parametrize("limit", [0.0, 1.5])
def test_few_rows_an_expert(ops, tile_rows, K, n_out, limit):
    """Each wave's share of K one to several stages long, rows on both sides of a tile's edge, columns past the last block's."""
    g = torch.Generator().manual_seed(K + n_out + tile_rows)
    counts = [1, 0, 15, 16, 17, 31, 32, 33]
    experts, T = len(counts), sum(counts)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=g)].int()[:, None].contiguous().to(DEV)
    x = torch.randn(T, K + 8, generator=g).bfloat16().to(DEV)[:, :K]
    w_gu = (torch.randn(experts, 2 * n_out, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    w = (torch.randn(experts, n_out, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    slot, token, tiles, offsets = ops.moe_sort(ids, experts, tile_rows)
    gated = ops.moe_rows(x, token, w_gu, tiles, tile_rows, T, gated=True, limit=limit, alpha=1.3)
    by_slot = x[token.long()].contiguous()
    plain = ops.moe_rows(by_slot, None, w, tiles, tile_rows, T, gated=False)
    at = offsets.cpu().tolist()
    for e, n in enumerate(counts):
        rows = slice(at[e], at[e] + n)
        h = by_slot[rows].double()
        size = h.abs() @ w[e].double().abs().T
        assert ((plain[rows].double() - h @ w[e].double().T).abs() <= (K + 1) * 2.0 ** -24 * size).all()    # K 32-bit sums
        gu = h @ w_gu[e].double().T
        a, u = gu[:, :n_out], gu[:, n_out:]
        if limit:
            a, u = a.clamp(max=limit), u.clamp(-limit, limit)
            want = a * torch.sigmoid(1.3 * a) * (u + 1)
        else:
            want = a * torch.sigmoid(a) * u
        off = (K + 8) * 2.0 ** -24 * (h.abs() @ w_gu[e].double().abs().T).max() * (4 + u.abs() + a.abs()) if n else 0.0
        assert ((gated[rows].double() - want).abs() <= 2.0 ** -8 * want.abs() + off).all()


@pytest.mark.parametrize("K,n_out,experts", [(64, 1040, 24), (192, 1096, 24), (128, 520, 300)])
def test_tiles_of_every_height_in_more_than_a_round(ops, K, n_out, experts):
    """Lists of more blocks than a round, the last of them begun, whose long tiles go before the others, and one of more tiles than
    that order takes: the same sums as in tiles of 128, whose blocks go by the list."""
    g = torch.Generator().manual_seed(K + n_out)
    cycle = [300, 1, 64, 65, 0, 128, 129, 256, 257, 520, 20, 192]
    counts = [cycle[e % len(cycle)] if experts < 256 else 3 + e % 5 for e in range(experts)]
    T = sum(counts)
    if experts < 256:
        blocks = -(-n_out // 128)
        used, short = sum(-(-n // 256) for n in counts) * blocks, sum(0 < n % 256 <= 128 for n in counts) * blocks
        assert used > 256 and 0 < used % 256 <= 204 and 0 < short <= 160
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=g)].int()[:, None].contiguous().to(DEV)
    x = torch.randn(T, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(experts, 2 * n_out, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    results = []
    for tile_rows in (128, 256):
        slot, token, tiles, _ = ops.moe_sort(ids, experts, tile_rows)
        at = slot.long()
        results.append((ops.moe_rows(x, token, w, tiles, tile_rows, T, gated=True)[at],
                        ops.moe_rows(x[token.long()].contiguous(), None, w, tiles, tile_rows, T, gated=False)[at]))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
