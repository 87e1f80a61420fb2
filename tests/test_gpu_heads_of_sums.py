"""Heads' norm, rotation and cache write straight from a product's stacks of sums: the bits of adding the stacks up first."""
import ctypes

import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu
PAGE = 16


def _call(name, *args):
    from ullm_amd.kernels import build, ops
    out = [ctypes.c_void_p(a.data_ptr()) if isinstance(a, torch.Tensor) else ctypes.c_float(a) if isinstance(a, float)
           else ctypes.c_void_p(0) if a is None else ctypes.c_int(a) for a in args]
    return getattr(build.load("elementwise"), name)(*out, ops._stream())


def _both_ways(slices, T, nq, nkv, hd, bias, gains, rot):
    """(status, [q, keys, values] from the sums, the same from the rows that ``sum_stacks`` leaves)."""
    from ullm_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(T + hd + slices)
    width, need = (nq + 2 * nkv) * hd, -(-(T + 9) // PAGE)
    sums = torch.randn(slices, T, width, device=DEV, generator=g)
    b = torch.randn(width, device=DEV, generator=g) if bias else None
    # two requests: the first from position 5 on, the second, of the last third of the tokens, from 0
    cut = T - T // 3
    positions = torch.cat([torch.arange(cut) + 5, torch.arange(T - cut)]).int().to(DEV)
    entry = (torch.arange(T) >= cut).int().to(DEV)
    table = torch.randperm(2 * need, generator=torch.Generator().manual_seed(T)).view(2, need).int().to(DEV)
    table[0, 0] = -1                                         # an entry without a page: nothing is written
    qg, kg = (torch.rand(hd, device=DEV, generator=g) + 0.5 for _ in range(2)) if gains else (None, None)
    cs = torch.randn(T + 16, rot, device=DEV, generator=g) if rot else None
    style = 1 if rot else 0

    def fresh():
        return [torch.zeros(T, nq * hd, dtype=torch.bfloat16, device=DEV), torch.zeros(2 * need, nkv, PAGE, hd, dtype=torch.bfloat16, device=DEV),
                torch.zeros(2 * need, nkv, hd, PAGE, dtype=torch.bfloat16, device=DEV)]
    got, want = fresh(), fresh()
    rc = _call("ullm_qk_norm_rope_write_sums", sums, slices, b, width, got[0], nq * hd, qg, kg, 1e-6, cs, T + 16 if rot else 0, rot, style,
               positions, entry, table, need, got[1], got[2], PAGE, T, nq, nkv, hd, 1)
    ops.qk_norm_rope_write(ops.sum_stacks(sums, b, torch.bfloat16), want[0], qg, kg, 1e-6, cs, rot, style, positions, entry, table,
                           want[1], want[2], PAGE, nq, nkv, hd, True)
    return rc, got, want


# one token; both sides of where values go in runs and where threads take several heads of finished rows
@pytest.mark.parametrize("T", [1, 65, 127, 128, 131, 511, 515])
@pytest.mark.parametrize("slices,nq,nkv,hd,bias,gains,rot", [
    (2, 32, 8, 128, False, True, 128), (4, 40, 8, 128, True, True, 128), (2, 6, 2, 64, True, False, 32), (4, 3, 1, 256, False, True, 0),
    (4, 8, 8, 32, False, False, 32)])
def test_heads_from_sums(T, slices, nq, nkv, hd, bias, gains, rot):
    rc, got, want = _both_ways(slices, T, nq, nkv, hd, bias, gains, rot)
    assert rc == 0
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("slices,hd", [(1, 128), (3, 128), (2, 24), (4, 48)])
def test_what_is_left_to_two_launches(slices, hd):
    rc, got, _ = _both_ways(slices, 20, 4, 2, hd, False, True, 0)
    torch.cuda.synchronize()
    assert rc == -3 and not any(t.any() for t in got)
