"""How prompt attention adds up the parts of a tile's keys, to the bit: the sums and the outputs so far times their factor in one rounding, with the
other part's product rounded ahead of it, in every launch that cuts the keys, alone and beside decoded tokens."""
import pytest
import torch

from gpu_util import DEV, paged_cache, table_tensor

pytestmark = pytest.mark.gpu

HD, NKV, NEW, REQUESTS = 128, 8, 64, 2
LOG2E = 1.4426950408889634
HIDDEN = -400.0                                            # a key with it weighs exactly 0


def _merged(parts, weights, swapped=False):
    """acc = acc * fa + its * fb over the parts, 32-bit; `swapped`: the product that is rounded by itself is the first."""
    acc = parts[0]
    for its, (fa, fb) in zip(parts[1:], weights):
        a, fa, b, fb = acc.double(), fa.double(), its.double(), fb.double()
        # (a product of two 32-bit values is exact in 64 bits)
        acc = (a * fa).float().double() + b * fb if swapped else a * fa + (b * fb).float().double()
        acc = acc.float()
    return acc


def _weights(reference):
    """The two factors of every merge; reference: [parts, ...], the exponent of every live key of a part."""
    m, weights = reference[0], []
    for its in reference[1:]:
        top = torch.maximum(m, its)
        weights.append((torch.exp2(m - top), torch.exp2(its - top)))
        m = top
    return weights


def _total(weights, swapped=False):
    """A column's keys lie in four lanes, 24 live ones of a part in each."""
    return 4 * _merged([torch.full_like(weights[0][0], 24.0)] * (len(weights) + 1), weights, swapped)


def _outputs(values, weights, total):
    """values: [parts, ..., n], every live key's value."""
    acc = _merged([96 * v for v in values], [(a[..., None], b[..., None]) for a, b in weights])
    return (acc * (1 / total)[..., None]).to(torch.bfloat16)


def _telling(parts, g):
    """Scores [REQUESTS * NKV, parts] whose sum's reciprocal has other bits in the other order of rounding, values [parts, REQUESTS * NKV, HD] that show
    them in bfloat16 (as many different ones as were found), and the outputs in both orders."""
    score = (0.3 * torch.randn(4096, parts, generator=g)).to(torch.bfloat16).float().to(DEV)
    weights = _weights(score.T * LOG2E)
    score = score[1 / _total(weights) != 1 / _total(weights, True)]
    weights = _weights(score.T * LOG2E)
    totals, kept, values = (_total(weights), _total(weights, True)), [], []
    draws = torch.Generator(DEV).manual_seed(parts)
    for i in range(len(score)):
        v = torch.randn(parts, 1 << 22, generator=draws, device=DEV).to(torch.bfloat16).float()
        at = [(a[i], b[i]) for a, b in weights]
        shown = (_outputs(v, at, totals[0][i]) != _outputs(v, at, totals[1][i])).nonzero()[:, 0]
        if len(shown) == 0:
            continue
        kept.append(i)
        values.append(v[:, shown.repeat(HD)[:HD]])
        if len(kept) == REQUESTS * NKV:
            break
    values, weights = torch.stack(values, 1), [(a[kept], b[kept]) for a, b in weights]
    return score[kept], values, [_outputs(values, weights, t[kept]) for t in totals]


@pytest.mark.parametrize("group,way,parts", [(2, 3, 4), (2, 5, 2), (2, 2, 2), (4, 2, 2)])
@pytest.mark.parametrize("kind", ["alone", "extras", "mixed"])
def test_bits_of_the_merge(group, way, parts, kind):
    """Parts of five 32-key tiles, three of keys of one score and two that count nothing (the last two of all are the queries' own)."""
    if kind == "mixed" and group == 2 and way == 2:
        pytest.skip("groups of two heads go another way beside decoded tokens")
    from ullm_amd.kernels import ops
    from ullm_amd.parts import StepShape
    from ullm_amd.parts.attention import plan_attention_step
    g = torch.Generator().manual_seed(7)
    nq, dtype, S, P = group * NKV, torch.bfloat16, 160 * parts, 16
    score, value, (want, other) = _telling(parts, g)
    assert (want != other).all()
    score, value = score.cpu().view(REQUESTS, NKV, parts), value.cpu().view(parts, REQUESTS, NKV, HD)
    ks, vs = [], []
    for b in range(REQUESTS):
        k, v = torch.zeros(S, NKV, HD), torch.zeros(S, NKV, HD)
        k[..., 0] = HIDDEN
        for p in range(parts):
            live = slice(160 * p, 160 * p + 96)
            k[live, :, 0], v[live] = score[b, :, p], value[p, b]
        ks.append(k)
        vs.append(v)
    entries = [(NEW, S - NEW)] * REQUESTS
    if kind == "mixed":
        entries.append((1, 40))
        ks.append(torch.randn(41, NKV, HD, generator=g))
        vs.append(torch.randn(41, NKV, HD, generator=g))
    k_pool, v_pool, tables = paged_cache(ks, vs, P, dtype, DEV)
    plan = plan_attention_step(StepShape(tuple(n for n, _ in entries), tuple(s for _, s in entries)))
    f, arrays = plan.facts, {k: torch.tensor(v, device=DEV) for k, v in plan.arrays.items()}
    T, rows = sum(n for n, _ in entries), NEW * REQUESTS
    q = torch.zeros(T, nq, HD)
    q[:, :, 0] = 1.0
    positions = torch.cat([torch.arange(s, s + n) for n, s in entries]).int().to(DEV)
    entry = torch.cat([torch.full((n,), b) for b, (n, _) in enumerate(entries)]).int().to(DEV)
    out = torch.full((T, nq * HD), float("nan"), dtype=dtype, device=DEV)
    args = (positions, entry, table_tensor(tables, DEV), P, nq, NKV, HD, 1.0, 0)
    qs = q.view(T, -1).to(dtype).to(DEV)
    wide = dict(wide_tiles=arrays["wide_tiles"], n_wide=f["num_wide"])
    if kind == "mixed":
        assert ops.attention_mixed_mfma(qs, out, k_pool, v_pool, arrays["decode_tokens"], f["num_decode"], arrays["tiles"], f["num_tiles"], *args,
                                        f["decode_keys"], f["max_decode_kv"], way=way, **wide)
    else:
        more = dict(bias_log2=torch.zeros(nq, 1, device=DEV)) if kind == "extras" else {}
        ops.attention_prefill_mfma(qs, out, k_pool, v_pool, arrays["tiles"], f["num_tiles"], *args, halves=way, **wide, **more)
    # a score is the product of two bfloat16 values, exact, times log2(e), rounded once
    got = out[:rows].view(REQUESTS, NEW, NKV, group, HD)
    assert torch.equal(got, want.view(REQUESTS, 1, NKV, 1, HD).expand_as(got))
