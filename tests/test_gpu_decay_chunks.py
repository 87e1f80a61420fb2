"""The decaying recurrence in chunks and segments: against a 64-bit walk token by token, at portions on both sides of a chunk's and
a segment's edge beside single tokens, with states found and left in rows of their own."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _walk(q, k, v, d, S, bonus):
    out = torch.empty(q.shape[0], *v.shape[1:], dtype=torch.float64)
    for t in range(q.shape[0]):
        kv = k[t][:, :, None] * v[t][:, None, :]
        if bonus is None:
            S = d[t][:, :, None] * S + kv
            out[t] = (S * q[t][:, :, None]).sum(1)
        else:
            out[t] = ((S + bonus[:, :, None] * kv) * q[t][:, :, None]).sum(1)
            S = d[t][:, :, None] * S + kv
    return out, S


def _case(kind, heads, N, P, lens, seed):
    g = torch.Generator().manual_seed(seed)
    T = sum(lens)
    wide = torch.randn(T, heads * (2 * N + P) + 5, generator=g) * 0.7
    z = torch.randn(T, heads * N, generator=g) * 2.0
    per_head = 1.0 - torch.rand(heads, generator=g) * 0.2
    bonus = torch.randn(heads, N, generator=g) if kind == "exp_exp_bonus" else None
    state = torch.randn(len(lens) + 2, 7 + heads * N * P, generator=g)
    slots = torch.randperm(len(lens) + 2, generator=g)[:len(lens)].int()
    return wide, z, per_head, bonus, state, slots


def _run(ops, kind, heads, N, P, lens, wide, z, per_head, bonus, state, slots, write_state=True):
    from ullm_amd.parts.decay import chunk_plan
    plan = chunk_plan(lens)
    plan.arrays = {n: torch.from_numpy(a).to(DEV) for n, a in plan.arrays.items()}
    x, st = wide.to(DEV), state.to(DEV)
    q, k, v = x[:, :heads * N], x[:, heads * N:2 * heads * N], x[:, 2 * heads * N:heads * (2 * N + P)]
    code = {"per_head": ops.DECAY_PER_HEAD, "sigmoid_root": ops.DECAY_SIGMOID_ROOT, "exp_exp_bonus": ops.DECAY_EXP_EXP}[kind]
    o = ops.decay_chunks(q, k, v, (per_head if kind == "per_head" else z).to(DEV), code, st, 7, slots.to(DEV), len(lens), heads, N, P,
                         plan, tau=3.0, bonus=None if bonus is None else bonus.to(DEV), silu_inputs=kind == "per_head",
                         q_scale=0.5, write_state=write_state)
    return o.cpu(), st.cpu(), plan.facts


@pytest.mark.parametrize("heads,N,P", [(1, 16, 16), (3, 48, 32), (2, 64, 144), (2, 128, 128)])
@pytest.mark.parametrize("kind", ["per_head", "sigmoid_root", "exp_exp_bonus"])
@pytest.mark.parametrize("lens", [[128], [129, 1, 15], [16, 300, 17, 1, 400], [143, 2500]])
def test_against_a_walk_token_by_token(heads, N, P, kind, lens):
    from ullm_amd.kernels import ops
    if sum(lens) > 2000 and heads * N > 64:
        pytest.skip("the long portion once per kind")
    assert ops.decay_chunks_supports(N, P)
    wide, z, per_head, bonus, state, slots = _case(kind, heads, N, P, lens, N + len(lens))
    got, left, facts = _run(ops, kind, heads, N, P, lens, wide, z, per_head, bonus, state, slots)
    assert facts["several"] == any(n > 128 for n in lens)
    q, k, v = (wide[:, a:b].double().view(len(wide), heads, -1) for a, b in
               ((0, heads * N), (heads * N, 2 * heads * N), (2 * heads * N, heads * (2 * N + P))))
    if kind == "per_head":
        q, k, v = (t * torch.sigmoid(t) for t in (q, k, v))
        d = per_head.double()[None, :, None].expand_as(q)
    else:
        zd = z.double().view(len(wide), heads, N)
        d = torch.sigmoid(zd).pow(1 / 3.0) if kind == "sigmoid_root" else torch.exp(-torch.exp(zd))
    t0 = 0
    touched = torch.zeros(len(state), dtype=torch.bool)
    for b, n in enumerate(lens):
        rows, slot = slice(t0, t0 + n), int(slots[b])
        S = state[slot, 7:].double().view(heads, N, P)
        want, S = _walk(q[rows] * 0.5, k[rows], v[rows], d[rows], S, None if bonus is None else bonus.double())
        # 32-bit: the sums behind an output or a state are some hundred terms of about the largest one's size
        assert (got[rows].double().view(n, heads, P) - want).abs().max() <= 2e-5 * want.abs().max()
        assert (left[slot, 7:].double().view(heads, N, P) - S).abs().max() <= 2e-5 * S.abs().max()
        assert torch.equal(left[slot, :7], state[slot, :7])
        touched[slot] = True
        t0 += n
    assert torch.equal(left[~touched], state[~touched])
    # without leave to write the state, only the outputs
    again, kept, _ = _run(ops, kind, heads, N, P, lens, wide, z, per_head, bonus, state, slots, write_state=False)
    assert torch.equal(again, got) and torch.equal(kept, state)


def test_a_value_that_is_not_finite_reaches_no_earlier_token_and_no_other_request():
    from ullm_amd.kernels import ops
    heads, N, P, lens = 2, 32, 16, [200, 140]
    case = _case("sigmoid_root", heads, N, P, lens, 3)
    clean, _, _ = _run(ops, "sigmoid_root", heads, N, P, lens, *case)
    case[0][70, 2 * heads * N + 3] = math.inf                          # token 70's value 3 of head 0
    got, left, _ = _run(ops, "sigmoid_root", heads, N, P, lens, *case)
    assert (got[:70] - clean[:70]).abs().max() <= 2e-5 * clean.abs().max() and torch.equal(got[200:], clean[200:])
    assert not torch.isfinite(got[70:200, 3]).any() and not torch.isfinite(left[int(case[5][0]), 7:].view(heads, N, P)[0, :, 3]).any()
    other = [c for c in range(heads * P) if c != 3]
    assert torch.equal(got[:, other][:64], clean[:, other][:64])
    assert (got[70:200][:, other] - clean[70:200][:, other]).abs().max() <= 2e-5 * clean.abs().max()
