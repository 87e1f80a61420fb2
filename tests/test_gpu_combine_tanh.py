"""The experts' sum added to the stream and squashed in one kernel: the bits of the two kernels one after the other."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


# one token and many; columns in one block, on both sides of two, and that no thread takes four of
@pytest.mark.parametrize("T,H", [(1, 2048), (48, 1024), (300, 1028), (7, 33), (130, 2050)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("base_dtype,shared,identity,mult", [(None, False, 0, 1.0), (torch.float32, True, 2, 0.3), ("rows", False, 1, 1.0)])
def test_sum_stream_and_squashing(T, H, dtype, base_dtype, shared, identity, mult):
    from ullm_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(T + H)
    experts, top = 6, 3

    def normal(*shape, of=torch.float32):
        return torch.randn(*shape, device=DEV, generator=g).to(of)
    x, y = normal(T, H, of=dtype), normal(T * top, H)
    ids = torch.rand(T, experts + identity, device=DEV, generator=g).argsort(-1)[:, :top].int().contiguous()
    slots = torch.randperm(T * top, device=DEV, generator=g).int()
    weights = torch.rand(T, top, device=DEV, generator=g)
    base = None if base_dtype is None else normal(T, H, of=dtype if base_dtype == "rows" else base_dtype)
    more = normal(T, H, of=dtype) if shared else None
    alpha, gain, shift, stream = normal(()), normal(H), normal(H), normal(T, H)
    want_stream = stream.clone()
    total = ops.moe_combine(y, x, ids, weights, slots, experts, base=base, shared=more)
    want = ops.add_tanh(total, want_stream, alpha, gain, shift, dtype, mult=mult)
    got = ops.moe_combine_tanh(y, x, ids, weights, slots, experts, stream, alpha, gain, shift, mult, base=base, shared=more)
    assert got.dtype == dtype and torch.equal(got, want) and torch.equal(stream, want_stream)


def test_a_sum_that_is_asked_for_runs_once():
    from ullm_amd.parts.base import NormedBranch, SummedBranch
    made = []

    def total():
        made.append(torch.ones(2, 3))
        return made[-1]
    b = SummedBranch(total, lambda *args: args, torch.bfloat16, 0.5)
    assert isinstance(b, NormedBranch) and b.post is None and b.second is None
    assert b.added_and_squashed(1, 2, 3, 4, torch.float32) is None and not made
    assert b.joined() is b.branch is made[0] and len(made) == 1
    assert b.added_and_squashed(1, 2, 3, 4, torch.bfloat16) is None
