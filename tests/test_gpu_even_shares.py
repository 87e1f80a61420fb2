"""Decode attention whose blocks share out all tokens' keys evenly: against softmax in 64 bits, with contexts of a key, of whole tiles and of thousands,
as many tokens as it takes, windows, heads' extras, fewer tiles than blocks; and which launches go that way."""
import pytest
import torch

from gpu_util import DEV, paged_cache, table_tensor, tol
from test_gpu_two_head_prompts import _attention
from ullm_amd.kernels.ops import DECODE_EVEN, decode_cuts, decode_split

# keys of every token, heads, kv heads, window, blocks a kv head
CASES = [([1], 2, 1, 0, 2), ([1, 1, 1], 2, 1, 0, 64), ([31, 32, 33, 2, 1, 700], 4, 2, 0, 7), ([2500, 1, 64, 65, 900], 4, 1, 0, 40),
         ([37 * i % 211 + 1 for i in range(64)], 6, 3, 0, 65), ([37 * i % 411 + 1 for i in range(64)], 2, 2, 0, 200), ([90, 600, 301, 33], 6, 3, 50, 16),
         ([200, 65, 64, 129], 8, 8, -64, 9), ([1500, 40, 333], 32, 1, 0, 30), ([4000, 17], 18, 1, 0, 100)]


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("lens,nq,nkv,window,blocks", CASES)
def test_every_share(lens, nq, nkv, window, blocks, hd):
    from ullm_amd.kernels import ops
    g = torch.Generator().manual_seed(nq + window + hd)
    P, dtype, scale, B = 16, torch.bfloat16, hd ** -0.5, len(lens)
    ks, vs = ([torch.randn(n, nkv, hd, generator=g).to(dtype).float() for n in lens] for _ in range(2))
    k_pool, v_pool, tables = paged_cache(ks, vs, P, dtype, DEV)
    bt = table_tensor(tables, DEV)
    q = torch.randn(B, nq * hd, generator=g).to(dtype)
    positions, entry = torch.tensor(lens, dtype=torch.int32, device=DEV) - 1, torch.arange(B, dtype=torch.int32, device=DEV)
    order = torch.tensor(sorted(range(B), key=lambda i: -lens[i]), dtype=torch.int32, device=DEV)
    want = torch.cat([_attention(row.view(1, nq, hd), k, v, window, scale) for row, k, v in zip(q, ks, vs)])
    for listed in (None, order):
        out = torch.full((B, nq * hd), float("nan"), dtype=dtype, device=DEV)
        ops.attention_decode_mfma(q.to(DEV), out, k_pool, v_pool, listed, B, positions, entry, bt, P, nq, nkv, hd, scale, window, max(lens),
                                  splits=blocks, waves=DECODE_EVEN)
        assert (out.float().cpu() - want.float()).abs().max() <= tol(dtype, want)
    # the step's norm, rotation and cache write in it: the bits in the cache of equal cuts, and of the output up to the shares' order of adding
    raw = torch.randn(B, (nq + 2 * nkv) * hd, generator=g).to(DEV, dtype)
    got = []
    for splits, waves in ((blocks, DECODE_EVEN), (1, 1)):
        k_one, v_one, out = k_pool.clone(), v_pool.clone(), torch.full((B, nq * hd), float("nan"), dtype=dtype, device=DEV)
        ops.attention_decode_fused(raw, out, None, None, 1e-5, None, 0, 0, k_one, v_one, order, B, positions, entry, bt, P, nq, nkv, hd, scale, window,
                                   max(lens), write_kv=True, splits=splits, waves=waves, entry_is_token=True)
        got.append((k_one, v_one, out.float().cpu()))
    assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(got[0][:2], got[1][:2]))
    assert (got[0][2] - got[1][2]).abs().max() <= tol(dtype, got[1][2])
    # heads' extras: a sink and a gate
    sink, gate = torch.randn(nq, generator=g).to(DEV), torch.randn(B, nq, generator=g).to(DEV, dtype)
    got = []
    for splits, waves in ((blocks, DECODE_EVEN), (1, 1)):
        out = torch.full((B, nq * hd), float("nan"), dtype=dtype, device=DEV)
        ops.attention_decode_mfma(q.to(DEV), out, k_pool, v_pool, order, B, positions, entry, bt, P, nq, nkv, hd, scale, window, max(lens), splits=splits,
                                  waves=waves, gate=gate, sink_log2=sink)
        got.append(out.float().cpu())
    assert (got[0] - got[1]).abs().max() <= tol(dtype, got[1])


@pytest.mark.gpu
def test_shapes_it_does_not_take_are_refused():
    from ullm_amd.kernels import ops
    hd, nq, P = 128, 2, 16
    pool = torch.zeros(1, 1, P, hd, dtype=torch.bfloat16, device=DEV)
    for B, blocks in ((65, 100), (4, 4), (1, 1)):
        q = torch.zeros(B, nq * hd, dtype=torch.bfloat16, device=DEV)
        zeros = torch.zeros(B, dtype=torch.int32, device=DEV)
        with pytest.raises(ops.KernelError):
            ops.attention_decode_mfma(q, torch.empty_like(q), pool, pool.view(1, 1, hd, P), None, B, zeros, zeros, zeros.view(B, 1), P, nq, 1, hd, 1.0, 0, 1,
                                      splits=blocks, waves=DECODE_EVEN)


def test_which_launches_go_that_way():
    """Only single waves a block, that are a wave a SIMD together, with long ways; everything else is cut as it was."""
    even = set()
    for nkv, groups in ((1, 1), (2, 1), (4, 1), (8, 1), (16, 2), (40, 1), (128, 1)):
        for items in (1, 2, 3, 4, 8, 15, 17, 28, 31, 32, 64, 65, 200, 300):
            for max_kv in (1, 500, 4096, 8160, 8161, 8192, 16384, 40000, 131072):
                for hd, window, units in ((128, 0, 256), (64, 0, 256), (256, 0, 256), (128, 200, 256), (128, -9000, 256), (128, 0, 128)):
                    args = (items, nkv, groups, max_kv, hd, window, units)
                    waves, n = decode_cuts(*args)
                    if waves != DECODE_EVEN:
                        assert (waves, n) == decode_split(*args)
                        continue
                    even.add(args)
                    assert decode_split(*args)[0] == 1 and items < n and 4 <= items <= 64 and n * nkv * groups <= 4 * units
                    assert hd <= 128 and max_kv > 8160 and abs(window) != 200
    assert (15, 8, 1, 8192, 128, 0, 256) in even and (15, 8, 1, 8160, 128, 0, 256) not in even
    assert (8, 8, 1, 16384, 128, 0, 256) in even and (8, 8, 1, 8192, 128, 0, 256) not in even
