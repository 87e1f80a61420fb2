"""Prompt attention of groups of at most two heads of size 128 in every way its launch knows: tiles that end inside a block's second half,
requests without one, contexts before the tokens, windows, chunks and the extras; against softmax in 64 bits."""
import pytest
import torch

from gpu_util import DEV, paged_cache, table_tensor, tol

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from ullm_amd.kernels import ops
    return ops


def _attention(q, k, v, window, scale, bias=None, sink=None):
    """64-bit: queries at the end of the keys; q [n, heads, 128], k and v [S, kv heads, 128]."""
    n, heads, S = q.shape[0], q.shape[1], k.shape[0]
    at, key = torch.arange(S - n, S)[:, None], torch.arange(S)[None, :]
    seen = (key <= at) & ((key > at - window) if window > 0 else (key >= at - at % -window) if window < 0 else key >= 0)
    out = []
    for h in range(heads):
        kv = h // (heads // k.shape[1])
        s = (q[:, h].double() @ k[:, kv].double().T) * scale
        if bias is not None:
            s = s + bias[h].double()[(at - key).clamp(0, bias.shape[1] - 1)]
        s = s.masked_fill(~seen, float("-inf"))
        top = s.amax(-1, keepdim=True)
        e = torch.exp(s - top)
        total = e.sum(-1, keepdim=True) + (torch.exp(sink[h].double() - top) if sink is not None else 0)
        out.append(e / total @ v[:, kv].double())
    return torch.stack(out, 1).reshape(n, -1)


# (new tokens, keys before them) of every request, heads, kv heads, window
CASES = [([(70, 0), (33, 5), (1, 40), (64, 0), (31, 100)], 4, 2, 0), ([(130, 400), (2, 3)], 2, 2, 0), ([(97, 60), (40, 333)], 4, 2, 50),
         ([(200, 90)], 6, 3, -64), ([(900, 17), (350, 1)], 16, 8, 0)]


@pytest.mark.parametrize("extras", [False, True])
@pytest.mark.parametrize("entries,nq,nkv,window", CASES)
def test_every_way_of_the_launch(ops, entries, nq, nkv, window, extras):
    from ullm_amd.parts import StepShape
    from ullm_amd.parts.attention import plan_attention_step
    g = torch.Generator().manual_seed(nq + window)
    hd, P, dtype, scale = 128, 16, torch.bfloat16, 128 ** -0.5
    sizes = [n + before for n, before in entries]
    ks, vs = ([torch.randn(S, nkv, hd, generator=g).to(dtype).float() for S in sizes] for _ in range(2))
    k_pool, v_pool, tables = paged_cache(ks, vs, P, dtype, DEV)
    bt = table_tensor(tables, DEV)
    plan = plan_attention_step(StepShape(tuple(n for n, _ in entries), tuple(s for _, s in entries)))
    f, arrays = plan.facts, {k: torch.tensor(v, device=DEV) for k, v in plan.arrays.items()}
    T = sum(n for n, _ in entries)
    q = torch.randn(T, nq * hd, generator=g).to(dtype)
    positions = torch.cat([torch.arange(s, s + n) for n, s in entries]).int().to(DEV)
    entry = torch.cat([torch.full((n,), b) for b, (n, _) in enumerate(entries)]).int().to(DEV)
    bias, gate, sink = (torch.randn(nq, 37, generator=g), torch.randn(T, nq, generator=g).to(dtype), torch.randn(nq, generator=g)) if extras else (None,) * 3
    log2e = 1.4426950408889634
    more = dict(bias_log2=(bias * log2e).to(DEV), gate=gate.to(DEV), sink_log2=(sink * log2e).to(DEV)) if extras else {}
    at, want, of_tiles = 0, [], []
    for (n, _), k, v in zip(entries, ks, vs):
        want.append(_attention(q[at:at + n].view(n, nq, hd), k, v, window, scale, bias, sink))
        of_tiles += [n > 1] * n
        at += n
    want = torch.cat(want)
    if extras:
        want = (want.view(T, nq, hd) * torch.sigmoid(gate.double())[:, :, None]).view(T, -1)
    rows = torch.tensor(of_tiles)                                # one-token entries go another way
    for way in (0, 1, 2, 3, 4, 5):
        out = torch.full((T, nq * hd), float("nan"), dtype=dtype, device=DEV)
        ops.attention_prefill_mfma(q.to(DEV), out, k_pool, v_pool, arrays["tiles"], f["num_tiles"], positions, entry, bt, P, nq, nkv, hd, scale,
                                   window, halves=way, keys_total=f["tile_keys_total"], keys_max=f["tile_keys_max"],
                                   wide_tiles=arrays["wide_tiles"], n_wide=f["num_wide"], wide_keys_total=f["wide_keys_total"],
                                   wide_keys_max=f["wide_keys_max"], **more)
        got = out.float().cpu()[rows]
        assert (got - want[rows].float()).abs().max() <= tol(dtype, want[rows]), way
        assert torch.isnan(out.float().cpu()[~rows]).all()


@pytest.mark.parametrize("window,gated", [(0, False), (0, True), (16700, False)])
def test_more_keys_than_the_page_ids_in_shared_memory(ops, window, gated):
    """Every part of the keys has the page ids of 128 tiles (4096 keys) at hand and refills them on the way: with 17 001 keys all of the
    ways do, the quarters with their two tiles in turn from the 129th of their 132 or 133 steps on.  Every query looks at one key beside
    a part's first or a refill's (its score there is about 128 / 2, elsewhere 60 / 2 at most)."""
    S, n, nq, nkv, hd, P, scale = 17001, 94, 2, 1, 128, 16, 0.5
    g = torch.Generator().manual_seed(7 + window)
    k, v = (torch.randn(S, nkv, hd, generator=g).bfloat16().float() for _ in range(2))
    begin = max(0, S - n - window + 1) // 32 * 32 if window else 0           # of the first tile's keys
    seams = set()
    for parts in (1, 2, 4):
        share = -(-(-(-(S - begin) // 32)) // parts) * 32
        for first in range(begin, S, share):
            seams |= {first + at + by for at in range(0, share, 4096) for by in (-1, 0, 31, 32)}
    seams = sorted(t for t in seams if (S - window if window else 0) <= t <= S - n)       # those that every query sees
    assert 40 < len(seams) <= n * nq // 3
    at = torch.tensor((seams * 5)[:n * nq])                                  # each by queries of three waves at least
    q = k[at, 0].view(n, nq, hd).bfloat16()
    k_pool, v_pool, tables = paged_cache([k], [v], P, torch.bfloat16, DEV)
    tiles, wide = (torch.tensor([x for f in range(0, n, size) for x in (f, min(size, n - f))], dtype=torch.int32, device=DEV)
                   for size in (ops.PREFILL_TILE, 2 * ops.PREFILL_TILE))
    want = _attention(q, k, v, window, scale)
    gate = torch.randn(n, nq, generator=g).bfloat16()
    if gated:
        want = (want.view(n, nq, hd) * torch.sigmoid(gate.double())[:, :, None]).view(n, -1)
    for way in (0, 1, 2, 3, 4, 5):
        out = torch.full((n, nq * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.attention_prefill_mfma(q.view(n, -1).to(DEV), out, k_pool, v_pool, tiles, len(tiles) // 2, torch.arange(S - n, S).int().to(DEV),
                                   torch.zeros(n, dtype=torch.int32, device=DEV), table_tensor(tables, DEV), P, nq, nkv, hd, scale, window, halves=way,
                                   wide_tiles=wide, n_wide=len(wide) // 2, gate=gate.to(DEV) if gated else None)
        assert (out.float().cpu() - want.float()).abs().max() <= tol(torch.bfloat16, want), way


def test_ways_that_other_groups_do_not_have(ops):
    """Wide tiles and quarters are for groups of at most two heads of size 128."""
    nq, nkv, hd, P = 8, 2, 128, 16
    k_pool = torch.zeros(4, nkv, P, hd, dtype=torch.bfloat16, device=DEV)
    v_pool = torch.zeros(4, nkv, hd, P, dtype=torch.bfloat16, device=DEV)
    q = torch.zeros(20, nq * hd, dtype=torch.bfloat16, device=DEV)
    tiles = torch.tensor([0, 20], dtype=torch.int32, device=DEV)
    ints = torch.zeros(20, dtype=torch.int32, device=DEV)
    for way in (3, 4, 5):
        with pytest.raises(ops.KernelError):
            ops.attention_prefill_mfma(q, torch.empty_like(q), k_pool, v_pool, tiles, 1, ints, ints, torch.zeros(1, 4, dtype=torch.int32, device=DEV), P,
                                       nq, nkv, hd, 1.0, 0, halves=way, wide_tiles=tiles, n_wide=1)
