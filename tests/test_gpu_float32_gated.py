"""The gated 32-bit product: the bits of the product and the activation kernel behind it."""
import pytest
import torch

from gpu_util import DEV

pytestmark = pytest.mark.gpu


# rows and columns on both sides of a tile's edge, in tiles of 32 and of 64 rows; K of whole stages, of whole pieces and of neither
@pytest.mark.parametrize("M,I", [(1, 16), (17, 33), (33, 100), (64, 31), (130, 3072), (500, 1024), (1000, 2050)])
@pytest.mark.parametrize("K", [5, 64, 100, 192, 1024])
def test_gated_product(M, I, K):
    from ullm_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(M + I + K)
    x, w = torch.randn(M, K + 4, device=DEV, generator=g)[:, :K], torch.randn(2 * I, K, device=DEV, generator=g) * 0.3
    w[I // 2] *= 100.0                                        # units that saturate on both sides
    assert torch.equal(ops.gemm_simple_silu(x, w), ops.silu_mul(ops.gemm_simple(x, w)))
