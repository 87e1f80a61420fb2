"""The 32-bit product and the tiled 32-bit attention at the edges of their tiles, against 64-bit results."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from ullm_amd.kernels import ops
    return ops


# rows on both sides of every tile's edge; K below, at and past a chunk, a stage and two, and no multiple of four
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 65, 33), (16, 64, 64), (17, 31, 100), (33, 130, 128), (64, 1024, 257),
                                   (129, 1000, 72), (640, 2600, 96), (1300, 1281, 68)])
@pytest.mark.parametrize("a_dtype,w_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                             (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_products_at_tile_edges(ops, M, N, K, a_dtype, w_dtype):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + N * 3 + K)
    wide = torch.randn(M, K + 3, generator=g, device=DEV).to(a_dtype)
    w = torch.randn(N, K, generator=g, device=DEV).to(w_dtype)
    bias = torch.randn(N, generator=g, device=DEV)
    a = wide[:, :K]
    want = a.double() @ w.double().T + bias.double()
    got = ops.gemm_simple(a, w, bias, out_dtype=torch.float32)
    # K products rounded into two chains and the bias: at most K + 2 roundings of the largest sum of absolute products
    bound = (K + 2) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs())
    assert ((got.double() - want).abs() <= bound).all()
    # a row's result depends on the row alone, whatever tile it lies in and however its operands are aligned
    for rows in (slice(0, 1), slice(M // 2, M // 2 + 17), slice(0, 40)):
        assert torch.equal(ops.gemm_simple(a[rows].contiguous(), w, bias, out_dtype=torch.float32), got[rows])


def _batch(g, lens, starts, nq, nkv, hd, page, dtype):
    """Queries of every request's new tokens, pools with its keys and values under shuffled pages, and the step's arrays."""
    B, keys = len(lens), [s + n for s, n in zip(starts, lens)]
    need = [-(-k // page) for k in keys]
    order = torch.randperm(sum(need) + 2, generator=g).tolist()
    table = torch.full((B, max(need)), -1, dtype=torch.int32)
    k_pool = torch.randn(sum(need) + 2, nkv, page, hd, generator=g).to(dtype)
    v_pool = torch.randn(sum(need) + 2, nkv, hd, page, generator=g).to(dtype)
    for b in range(B):
        for i in range(need[b]):
            table[b, i] = order.pop()
    entry = torch.tensor([b for b, n in enumerate(lens) for _ in range(n)], dtype=torch.int32)
    pos = torch.tensor([s + i for s, n in zip(starts, lens) for i in range(n)], dtype=torch.int32)
    q = torch.randn(len(entry), nq * hd, generator=g).to(dtype)
    return [t.to(DEV) for t in (q, k_pool, v_pool, pos, entry, table)]


def _reference(q, k_pool, v_pool, pos, entry, table, nq, nkv, hd, page, scale, window, bias, sink):
    out = torch.empty(q.shape[0], nq, hd, dtype=torch.float64, device=DEV)
    for t in range(q.shape[0]):
        p, row = int(pos[t]), table[int(entry[t])]
        j = torch.arange(p + 1, device=DEV)
        lo = p - window + 1 if window > 0 else p // -window * -window if window < 0 else 0
        j = j[j >= lo]
        pages = row[j // page].long()
        for h in range(nq):
            kv = h // (nq // nkv)
            k, v = k_pool[pages, kv, j % page].double(), v_pool[pages, kv, :, j % page].double()
            s = k @ q[t, h * hd:(h + 1) * hd].double() * scale
            if bias is not None:
                s = s + bias[h, (p - j).clamp(max=bias.shape[1] - 1)].double()
            top = s.max() if sink is None else torch.maximum(s.max(), sink[h].double())
            e = torch.exp(s - top)
            out[t, h] = e @ v / (e.sum() + (0 if sink is None else torch.exp(sink[h].double() - top)))
    return out.view(q.shape[0], nq * hd)


# heads a kv head has that divide 16, do not, and exceed it; pages of 4, 16 and 20 tokens; contexts at the edges of 64 keys
@pytest.mark.parametrize("nq,nkv,hd,page,window,extras,lens,starts", [
    (2, 1, 16, 4, 0, False, [1, 1, 1], [0, 63, 64]),
    (4, 2, 128, 16, 0, False, [70, 3, 1], [0, 62, 130]),
    (5, 1, 48, 20, 33, True, [9, 20, 1], [0, 55, 127]),
    (20, 1, 32, 16, -48, True, [50, 2], [0, 95]),
    (6, 2, 256, 16, 0, True, [1, 33], [191, 0]),
    (3, 3, 96, 16, 17, False, [64, 65], [64, 0]),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_tiles(ops, nq, nkv, hd, page, window, extras, lens, starts, dtype):
    g = torch.Generator().manual_seed(hd + nq)
    q, k_pool, v_pool, pos, entry, table = _batch(g, lens, starts, nq, nkv, hd, page, dtype)
    bias = torch.randn(nq, 40, generator=g).to(DEV) if extras else None
    sink = torch.randn(nq, generator=g).to(DEV) if extras else None
    scale = hd ** -0.5

    def run(rows=slice(None)):
        return ops.paged_attention_generic(q[rows].contiguous(), k_pool, v_pool, pos[rows].contiguous(), entry[rows].contiguous(),
                                           table, page, nq, nkv, hd, scale, window, bias=bias, sink=sink)
    got = run()
    want = _reference(q, k_pool, v_pool, pos, entry, table, nq, nkv, hd, page, scale, window, bias, sink)
    step = 2e-5 if dtype == torch.float32 else 2.0 ** -8          # 32-bit sums; one rounding of the result to bfloat16
    assert (got.double() - want).abs().max() <= step * float(want.abs().max())
    # a token's result has the same bits alone, in a step of single tokens and beside others
    for t in {0, len(pos) // 2, len(pos) - 1}:
        assert torch.equal(run(slice(t, t + 1)), got[t:t + 1])
    for cut in (1, len(pos) // 3):
        assert torch.equal(torch.cat((run(slice(0, cut)), run(slice(cut, None)))), got)


def test_values_that_are_not_finite_reach_only_rows_that_see_them(ops):
    """A value of infinity at position 40: rows before it, and rows of another request in the same tile, are as without it."""
    g = torch.Generator().manual_seed(5)
    nq, nkv, hd, page = 4, 2, 64, 16
    q, k_pool, v_pool, pos, entry, table = _batch(g, [60, 9], [0, 0], nq, nkv, hd, page, torch.float32)

    def run():
        return ops.paged_attention_generic(q, k_pool, v_pool, pos, entry, table, page, nq, nkv, hd, 0.125, 0)
    clean = run()
    v_pool[int(table[0, 40 // page]), :, 3, 40 % page] = math.inf
    k_pool[int(table[0, 45 // page]), :, 45 % page, 3] = math.nan
    got = run()
    seen = (entry == 0) & (pos >= 40)
    # the tile that holds a value of infinity is added in another order: 32-bit rounding
    assert (got[~seen] - clean[~seen]).abs().max() <= 2e-5 * float(clean.abs().max())
    assert torch.isinf(got.view(-1, nq, hd)[(entry == 0) & (pos >= 40) & (pos < 45)][:, :, 3]).all()
    assert torch.isnan(got[(entry == 0) & (pos >= 45)]).all()
