"""Norm, rotation and cache write of the heads over many tokens (several heads a thread, values in runs of eight): the bits of the same
tokens in short portions, which take a head a thread and write their values one by one."""
import pytest
import torch

from gpu_util import DEV, table_tensor

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from ullm_amd.kernels import ops
    return ops


# heads, kv heads, head size, page size, rotated dims, pairing, q gain, k gain
@pytest.mark.parametrize("nq,nkv,hd,P,rot,style,q_norm,k_norm", [
    (4, 2, 128, 16, 128, 1, True, True), (16, 8, 128, 16, 128, 1, True, False), (40, 8, 128, 16, 64, 1, True, True),
    (60, 4, 128, 8, 128, 2, False, True), (24, 4, 64, 16, 64, 1, True, True), (8, 8, 256, 32, 256, 1, False, False),
    (64, 8, 128, 16, 128, 1, True, True)])                                # two blocks a token, three heads a thread in both
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens", [[127, 1], [128], [511], [300, 1, 7, 204], [9, 3, 700], [1024]])
def test_long_batches_write_what_short_ones_do(ops, nq, nkv, hd, P, rot, style, q_norm, k_norm, dtype, lens):
    g = torch.Generator().manual_seed(nq + len(lens))
    T = sum(lens)
    starts = [(5 * b) % 11 for b in range(len(lens))]                   # runs of eight begin and end inside the requests
    positions = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lens)]).int().to(DEV)
    entry = torch.cat([torch.full((n,), b) for b, n in enumerate(lens)]).int().to(DEV)
    need = [-(-(s + n) // P) for s, n in zip(starts, lens)]
    ids = torch.randperm(sum(need) + 2, generator=g).tolist()
    tables = [ids[sum(need[:b]):sum(need[:b + 1])] for b in range(len(lens))]
    bt = table_tensor(tables, DEV)
    bt[-1, 0] = -1                                                      # a page given back: its tokens are written nowhere
    qkv = torch.randn(T, (nq + 2 * nkv) * hd, generator=g).to(DEV, dtype)
    gain = lambda on: (torch.rand(hd, generator=g) + 0.5).to(DEV) if on else None      # noqa: E731
    qg, kg = gain(q_norm), gain(k_norm)
    table = torch.randn(max(lens) + 20, rot, generator=g).to(DEV)
    got = []
    for portion, write in ((T, True), (100, True), (T, False), (100, False)):
        k_pool, v_pool = torch.zeros(len(ids), nkv, P, hd, dtype=dtype, device=DEV), torch.zeros(len(ids), nkv, hd, P, dtype=dtype, device=DEV)
        q = torch.zeros(T, nq * hd, dtype=dtype, device=DEV)
        for at in range(0, T, portion):
            end = min(T, at + portion)
            ops.qk_norm_rope_write(qkv[at:end], q[at:end], qg, kg, 1e-6, table, rot, style, positions[at:end], entry[at:end], bt, k_pool, v_pool, P,
                                   nq, nkv, hd, write_kv=write)
        got.append((q, k_pool, v_pool))
    for a, b in ((0, 1), (2, 3)):
        assert all(torch.equal(x, y) for x, y in zip(got[a], got[b]))
    assert torch.equal(got[0][0], got[2][0]) and not got[2][1].any() and not got[2][2].any()
    written = sum(lens) - min(max(P - starts[-1], 0), lens[-1])         # all but those of the page given back
    assert int((got[0][1].float().abs().sum(-1) > 0).sum()) == written * nkv and bool((got[0][0] != 0).any())
    assert int((got[0][2].float().abs().sum(2) > 0).sum()) == written * nkv
