"""Decoded tokens beside prompt portions in one attention launch: every way against softmax in 64 bits, at teams without a token, tiles at their
edges, windows, chunks and contexts of every remainder; and which steps go that way."""
import ctypes

import pytest
import torch

from gpu_util import DEV, paged_cache, table_tensor, tol
from test_gpu_two_head_prompts import _attention


# (new tokens, keys before them) of every request, heads, kv heads, window: pairs of tokens and kv heads that leave teams without one, kv heads that
# are no multiple of the dies, groups of one to sixteen heads, contexts below, at and past a tile for each of four waves
CASES = [([(1, 0), (33, 5), (1, 40), (1, 31)], 2, 1, 0), ([(1, 127), (70, 0), (1, 128), (1, 129), (31, 100), (1, 700)], 4, 2, 0),
         ([(1, 300), (130, 400), (1, 49), (1, 50)], 6, 3, 50), ([(1, 200), (65, 63), (1, 64)], 8, 8, -64), ([(1, 15), (97, 60), (1, 500)], 10, 2, 0),
         ([(1, 90), (40, 333), (1, 17)], 16, 1, 0), ([(1, 37 * i) for i in range(20)] + [(600, 17)], 16, 8, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("entries,nq,nkv,window", CASES)
def test_every_way_of_the_launch(entries, nq, nkv, window):
    from ullm_amd.kernels import ops
    from ullm_amd.parts import StepShape
    from ullm_amd.parts.attention import plan_attention_step
    g = torch.Generator().manual_seed(nq + window)
    hd, P, dtype, scale = 128, 16, torch.bfloat16, 128 ** -0.5
    ks, vs = ([torch.randn(n + s, nkv, hd, generator=g).to(dtype).float() for n, s in entries] for _ in range(2))
    k_pool, v_pool, tables = paged_cache(ks, vs, P, dtype, DEV)
    bt = table_tensor(tables, DEV)
    plan = plan_attention_step(StepShape(tuple(n for n, _ in entries), tuple(s for _, s in entries)))
    f, arrays = plan.facts, {k: torch.tensor(v, device=DEV) for k, v in plan.arrays.items()}
    assert f["decode_keys"] == sum(s + 1 for n, s in entries if n == 1)
    T = sum(n for n, _ in entries)
    q = torch.randn(T, nq * hd, generator=g).to(dtype)
    positions = torch.cat([torch.arange(s, s + n) for n, s in entries]).int().to(DEV)
    entry = torch.cat([torch.full((n,), b) for b, (n, _) in enumerate(entries)]).int().to(DEV)
    want = torch.cat([_attention(part.view(-1, nq, hd), k, v, window, scale)
                      for part, k, v in zip(q.split([n for n, _ in entries]), ks, vs)])
    for way in ((3, 4, 5) if nq // nkv <= 2 else (1, 2)):
        out = torch.full((T, nq * hd), float("nan"), dtype=dtype, device=DEV)
        assert ops.attention_mixed_mfma(
            q.to(DEV), out, k_pool, v_pool, arrays["decode_tokens"], f["num_decode"], arrays["tiles"], f["num_tiles"], positions, entry, bt, P, nq,
            nkv, hd, scale, window, f["decode_keys"], f["max_decode_kv"], wide_tiles=arrays["wide_tiles"], n_wide=f["num_wide"], way=way)
        assert (out.float().cpu() - want.float()).abs().max() <= tol(dtype, want), way
    with pytest.raises(ops.KernelError):
        ops.attention_mixed_mfma(q.to(DEV), out, k_pool, v_pool, arrays["decode_tokens"], f["num_decode"], arrays["tiles"], f["num_tiles"], positions,
                                 entry, bt, P, nq, nkv, hd, scale, window, f["decode_keys"], f["max_decode_kv"], way=6)


# keys of the decoded tokens, and where their blocks then stand among the prompt's: few with a long walk before them, many behind the first round, few
# short ones behind all
ORDERS = {"first": [3000, 2500], "between": [600, 520, 590] * 20, "last": [60, 31, 1, 47]}


@pytest.mark.gpu
@pytest.mark.parametrize("order", ORDERS)
@pytest.mark.parametrize("nq", [16, 64])
def test_every_order_of_the_blocks(nq, order):
    """More prompt blocks than the chip holds: the bits of the prompt's own launch, and softmax in 64 bits for the decoded tokens."""
    from ullm_amd.kernels import build, ops
    from ullm_amd.parts import StepShape
    from ullm_amd.parts.attention import plan_attention_step
    g = torch.Generator(DEV).manual_seed(nq)
    nkv, hd, P, dtype, scale = 16, 128, 16, torch.bfloat16, 128 ** -0.5
    entries = [(1, n - 1) for n in ORDERS[order]] + [(2133, 0)]
    pages = [-(-(n + s) // P) for n, s in entries]
    k_pool = torch.randn(sum(pages), nkv, P, hd, generator=g, device=DEV).to(dtype)
    v_pool = torch.randn(sum(pages), nkv, hd, P, generator=g, device=DEV).to(dtype)
    ids = torch.randperm(sum(pages), generator=g, device=DEV).int().split(pages)
    bt = table_tensor([i.tolist() for i in ids], DEV)
    plan = plan_attention_step(StepShape(tuple(n for n, _ in entries), tuple(s for _, s in entries)))
    f, arrays = plan.facts, {k: torch.tensor(v, device=DEV) for k, v in plan.arrays.items()}
    T = sum(n for n, _ in entries)
    q = torch.randn(T, nq * hd, generator=g, device=DEV).to(dtype)
    positions = torch.cat([torch.arange(s, s + n) for n, s in entries]).int().to(DEV)
    entry = torch.cat([torch.full((n,), b) for b, (n, _) in enumerate(entries)]).int().to(DEV)
    figures = dict(keys_total=f["tile_keys_total"], keys_max=f["tile_keys_max"], wide_tiles=arrays["wide_tiles"], n_wide=f["num_wide"],
                   wide_keys_total=f["wide_keys_total"], wide_keys_max=f["wide_keys_max"])
    want = []
    for b, n in enumerate(ORDERS[order]):
        k = k_pool[ids[b].long()].transpose(1, 2).reshape(-1, nkv, hd)[:n]
        v = v_pool[ids[b].long()].permute(0, 3, 1, 2).reshape(-1, nkv, hd)[:n]
        want.append(_attention(q[b:b + 1].view(1, nq, hd).cpu(), k.cpu(), v.cpu(), 0, scale))
    want, decoded = torch.cat(want), len(ORDERS[order])
    long, i = ctypes.c_longlong, ctypes.c_int
    lead = build.load("attention_mfma").ullm_attention_mixed_lead
    lead.restype = long
    for way in ((3, 4, 5) if nq // nkv <= 2 else (1, 2)):
        wide = way in (4, 5)
        blocks = (f["num_wide"] if wide else f["num_tiles"]) * nkv * -(-nq // nkv // 4)
        keys = f["wide_keys_total" if wide else "tile_keys_total"] * nkv * -(-nq // nkv // 4)
        slots = ops.compute_units(DEV) * (2 if way in (1, 4) else 1)
        assert blocks > slots
        before = lead(i(way), long(blocks), long(keys), long(decoded * nkv), long(f["decode_keys"]), i(f["max_decode_kv"]), i(nkv),
                      i(ops.compute_units(DEV)))
        assert before == {"first": 0, "between": slots, "last": blocks}[order], way
        out, alone = (torch.full((T, nq * hd), float("nan"), dtype=dtype, device=DEV) for _ in range(2))
        assert ops.attention_mixed_mfma(
            q, out, k_pool, v_pool, arrays["decode_tokens"], f["num_decode"], arrays["tiles"], f["num_tiles"], positions, entry, bt, P, nq, nkv, hd, scale,
            0, f["decode_keys"], f["max_decode_kv"], way=way, **figures)
        ops.attention_prefill_mfma(q, alone, k_pool, v_pool, arrays["tiles"], f["num_tiles"], positions, entry, bt, P, nq, nkv, hd, scale, 0, halves=way,
                                   **figures)
        assert torch.equal(out[decoded:], alone[decoded:]) and not torch.isnan(out).any(), way
        assert (out[:decoded].float().cpu() - want.float()).abs().max() <= tol(dtype, want), way


def test_orders_on_other_chips():
    """CPU: what the chip holds at once is its units'; blocks between two of the prompt's are a multiple of the eight dies."""
    from ullm_amd.kernels import build
    long, i = ctypes.c_longlong, ctypes.c_int
    f = build.load("attention_mfma").ullm_attention_mixed_lead
    f.restype = long
    for way, per_unit in ((1, 2), (2, 1), (3, 1), (4, 2), (5, 1)):
        for units in (256, 250, 64):
            slots = units * per_unit
            lead = lambda blocks, pairs, keys, longest: f(i(way), long(blocks), long(1000 * blocks), long(pairs), long(keys), i(longest), i(8), i(units))  # noqa: E731
            assert lead(slots, 8, 9000, 9000) == slots and lead(slots - 3, 800, 90000, 900) == slots - 3
            assert lead(slots + 1, 8, 9000, 9000) == 0 and lead(slots + 5, 8, 40, 40) == slots + 5
            assert lead(slots + 1, 2 * slots, 10 ** 6, 900) == slots // 8 * 8


# requests and keys of the longest (the others down to 0.58 of it), the portion and the keys before it, heads, kv heads: us of two launches (0) and of the ways
MEASURED = [(4, 640, 700, 2100, 16, {0: 52.1, 3: 39.5, 5: 57.8, 4: 85.7}), (40, 640, 300, 600, 16, {0: 43.5, 3: 26.8, 5: 26.8, 4: 37.0}),
            (100, 640, 300, 600, 16, {0: 66.8, 3: 44.2, 5: 45.0, 4: 41.7}), (100, 640, 700, 0, 16, {0: 64.0, 3: 54.0, 5: 45.2, 4: 43.0}),
            (100, 640, 700, 2100, 16, {0: 88.6, 3: 65.5, 5: 60.3, 4: 93.0}), (100, 300, 1500, 3000, 16, {0: 123.7, 3: 98.2, 5: 88.8, 4: 136.5}),
            (30, 2000, 300, 600, 16, {0: 62.1, 3: 66.0, 5: 66.7, 4: 41.5}), (8, 4000, 300, 600, 16, {0: 47.2, 3: 115.5, 5: 115.1, 4: 63.0}),
            (100, 640, 700, 2100, 32, {0: 108.8, 1: 94.2, 2: 80.1}), (100, 640, 1900, 0, 32, {0: 102.6, 1: 77.9, 2: 100.2}),
            (100, 64, 300, 600, 32, {0: 36.2, 1: 33.8, 2: 27.0}), (8, 4000, 700, 0, 32, {0: 50.4, 1: 64.6, 2: 117.0}),
            # what a walk waits for: another team's on its unit, the prompt's blocks, which take every slot, and its own beginning
            (40, 2881, 35, 0, 16, {0: 74.2, 3: 96.3, 4: 86.7, 5: 96.8}), (37, 3175, 216, 25, 16, {0: 82.8, 3: 104.1, 4: 91.5, 5: 103.8}),
            (1, 1906, 488, 3319, 40, {0: 89.4, 2: 126.7}), (2, 743, 43, 0, 16, {0: 16.0, 3: 27.0, 4: 17.7, 5: 27.4})]


@pytest.mark.parametrize("case", range(len(MEASURED)))
def test_near_the_best_of_those_measured(case):
    """CPU: the way of a step."""
    from ullm_amd.kernels import build
    from ullm_amd.parts import StepShape
    from ullm_amd.parts.attention import plan_attention_step
    b, c, portion, behind, nq, times = MEASURED[case]
    starts = [max(16, int(c * (1 - 0.45 * ((7 * i) % 16) / 16))) for i in range(b)]
    f = plan_attention_step(StepShape((1,) * b + (portion,), tuple(starts) + (behind,))).facts
    i, long = ctypes.c_int, ctypes.c_longlong
    way = build.load("attention_mfma").ullm_attention_mixed_way(
        i(f["num_decode"]), long(f["decode_keys"]), i(f["max_decode_kv"]), i(f["num_tiles"]), long(f["tile_keys_total"]), i(f["tile_keys_max"]),
        i(f["num_wide"]), long(f["wide_keys_total"]), i(f["wide_keys_max"]), i(nq), i(8), i(0), i(256))
    assert times[way] <= 1.07 * min(times.values())
