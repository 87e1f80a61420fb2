"""Every tile of the 32-bit product, at its edges and those of its stages, against a plain loop of fused multiply-adds over K."""
import ctypes
import ctypes.util
import random

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

fmaf = ctypes.CDLL(ctypes.util.find_library("m")).fmaf
fmaf.restype, fmaf.argtypes = ctypes.c_float, [ctypes.c_float] * 3


# tiles of 32 x 32, 32 x 64, 64 x 32 in stages of 64 and of 32, 64 x 64, 16 x 64; K of one stage, of two and of three, with and
# without a last one that is not whole, and of rows that no 16-byte load takes
@pytest.mark.parametrize("M,N", [(33, 1000), (150, 6100), (450, 1030), (192, 2720), (380, 4100), (1000, 4097), (13, 9000)])
@pytest.mark.parametrize("K", [20, 64, 101, 128, 192, 196])
@pytest.mark.parametrize("a_dtype", [torch.float32, torch.bfloat16])
def test_a_tile_has_the_bits_of_a_loop_over_k(M, N, K, a_dtype):
    from ullm_amd.kernels import ops
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g).to(a_dtype), torch.randn(N, K, generator=g)
    a[M // 2, K - 1] = w[N // 3, 0] = float("inf")          # past a row's end lie the next row's values: none may be read as this one's
    got = ops.gemm_simple(a.to(DEV), w.to(DEV), None, out_dtype=torch.float32)
    finite = torch.isfinite(got)
    assert not finite[M // 2].any() and not finite[:, N // 3].any()
    assert int(finite.sum()) == (M - 1) * (N - 1)
    got, af = got.cpu(), a.float()
    rng = random.Random(K)
    for m, n in [(rng.randrange(M), rng.randrange(N)) for _ in range(40)] + [(M - 1, N - 1), (0, N - 1), (M - 1, 0)]:
        if m == M // 2 or n == N // 3:
            continue
        total = 0.0
        for x, y in zip(af[m].tolist(), w[n].tolist()):
            total = fmaf(x, y, total)
        assert float(got[m, n]) == total, (m, n)
