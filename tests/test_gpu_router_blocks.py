"""The router kernel's block shapes: a token's choice and weights have the same bits in all of them, and are those of 64 bits."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


# rows that fit four, two and one to a block, as 32-bit values or as they come; outputs on both sides of a round of waves and of
# what several tokens a block take; rows that no 16-byte load takes
@pytest.mark.parametrize("H,R,top", [(512, 16, 2), (1024, 33, 4), (2048, 32, 4), (2052, 7, 1), (4096, 64, 6), (5120, 24, 2), (9000, 30, 3), (640, 300, 5),
                                     (1030, 256, 8), (65, 5, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("corrected", [False, True])
def test_a_token_is_routed_alike_in_every_block(H, R, top, dtype, corrected):
    from ullm_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(H + R)
    x = torch.randn(4100, H, device=DEV, generator=g).to(dtype)
    w = torch.randn(R, H, device=DEV, generator=g) * 0.2
    c = torch.randn(R, device=DEV, generator=g) * 0.1 if corrected else None
    # the one token a block of sixteen waves, in rows of a wider tensor that begin off a 16-byte address
    wide = torch.empty(300, H + 3, dtype=dtype, device=DEV)
    wide[:, 1:H + 1] = x[:300]
    ids, weights = ops.moe_router(wide[:, 1:H + 1], w, c, top)
    for T in (1, 299, 301, 512, 513, 1023, 1027, 4100):
        i, p = ops.moe_router(x[:T].contiguous(), w, c, top)
        n = min(T, 300)
        assert torch.equal(i[:n], ids[:n]) and torch.equal(p[:n], weights[:n]), T
        again, again_p = ops.moe_router(x[T - 1:T].contiguous(), w, c, top)
        assert torch.equal(i[-1], again[0]) and torch.equal(p[-1], again_p[0]), T
    s = torch.softmax(x[:300].double() @ w.double().T, -1)
    choice, order = (s + (c.double() if corrected else 0)).sort(-1, descending=True)
    # a choice is clear where no neighbour among the first is nearer than 32-bit sums of H products are off
    clear = (choice[:, :top] - choice[:, 1:top + 1] > 1e-5).all(-1) if R > top else torch.zeros(300, dtype=torch.bool, device=DEV)
    assert torch.equal(ids[clear].long(), order[clear, :top])
    picked = s.gather(1, ids.long())
    # a sum of H products has H roundings of its terms at most: far below 1e-4 of a logit here, and so of a weight
    assert ((weights.double() - picked / picked.sum(-1, keepdim=True)).abs() <= 1e-4).all()
