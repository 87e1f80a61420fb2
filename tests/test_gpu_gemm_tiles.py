"""The large bfloat16 product at the edges of its tiles: rows and columns past the last tile's, one stage of K to many,
with and without a bias, the gated unit and its clamped form, against 64-bit results; and its rule of use."""
import pytest
import torch

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from ullm_amd.kernels import ops
    return ops


def _operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K + 8, generator=g, device=DEV).bfloat16()[:, :K]            # rows further apart than they are long
    return x, (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16(), torch.randn(N, generator=g, device=DEV)


@pytest.mark.gpu
@pytest.mark.parametrize("groups", [2, 4])
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (63, 256, 128), (129, 264, 192), (256, 120, 256), (257, 520, 320), (700, 1032, 1024),
                                   (2300, 264, 448)])
def test_products_at_tile_edges(ops, M, N, K, groups):
    x, w, bias = _operands(M, N, K, M + N)
    want = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    off = (K + 1) * 2.0 ** -24 * size                                                # K products added in 32-bit
    got = ops.gemm_tiles(x, w, bias, groups=groups)
    ref = want + bias.double()
    assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + off).all()
    full = ops.gemm_tiles(x, w, out_dtype=torch.float32, groups=groups)
    assert ((full.double() - want).abs() <= off).all()
    assert torch.equal(ops.gemm_tiles(x, w, groups=groups), full.bfloat16())
    # a row's sums do not depend on the tile it lies in
    cut = M // 3
    assert torch.equal(ops.gemm_tiles(x[cut:], w, out_dtype=torch.float32, groups=6 - groups), full[cut:])
    half = N // 2
    for limit, alpha in ((0.0, 0.0), (1.0, 1.7)):
        act = ops.gemm_tiles(x, w, gated=True, groups=groups, limit=limit, alpha=alpha)
        g, u = want[:, :half], want[:, half:]
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            ref = g * torch.sigmoid(alpha * g) * (u + 1)
        else:
            ref = g * torch.sigmoid(g) * u
        slack = 4 * off.amax(-1, keepdim=True) * (2 + g.abs() + u.abs()) + 2.0 ** -21 * ref.abs()   # sums, and the unit's own ulps
        assert ((act.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + slack).all()


def test_when_the_large_product_is_taken():
    """CPU: the ungated rule's rows and sizes, the gated rule's shares on both sides of where they were measured, empty sizes."""
    from ullm_amd.kernels.ops import gemm_tiles_rows
    assert [gemm_tiles_rows(M, 4096, 4096, False) for M in (1, 8192, 8193, 12000, 12288)] == [0, 0, 4, 4, 0]
    assert gemm_tiles_rows(12000, 1024, 4096, False) == 0 and gemm_tiles_rows(12000, 151936, 4096, False) == 0
    assert [gemm_tiles_rows(M, 24576, 4096, True) for M in (0, 159, 192, 256, 350, 450, 1300, 2048, 3000)] == [0, 0, 0, 2, 0, 4, 0, 4, 4]
    assert [gemm_tiles_rows(M, 6144, 1024, True) for M in (256, 700, 1300, 2048, 2600, 4000)] == [0, 2, 4, 4, 2, 2]
    for M in range(0, 20000, 371):
        for N in (0, 8, 2048, 6144, 24576):
            for K in (64, 1024, 12288):
                assert gemm_tiles_rows(M, N, K, False) in (0, 4) and gemm_tiles_rows(M, N, K, True) in (0, 2, 4)


@pytest.mark.gpu
def test_linear_and_gate_up_take_it_where_the_rule_says(ops, monkeypatch):
    from ullm_amd.parts.linear import gate_up, linear
    calls = []
    real = ops.gemm_tiles
    monkeypatch.setattr(ops, "gemm_tiles", lambda *a, **k: calls.append(k) or real(*a, **k))
    x, w, bias = _operands(8200, 4096, 128, 5)
    y = linear(x, w, bias)
    assert calls and (y.float() - (x.float() @ w.float().T + bias)).abs().max() <= 2.0 ** -7 * float(y.float().abs().max())
    z = linear(x, w, bias, out_dtype=torch.float32)
    assert len(calls) == 2 and z.dtype == torch.float32
    x, w, _ = _operands(1000, 6144, 128, 6)
    a = gate_up(x, w)
    h = x.float() @ w.float().T
    want = torch.nn.functional.silu(h[:, :3072]) * h[:, 3072:]
    assert len(calls) == 3 and (a.float() - want).abs().max() <= 2.0 ** -7 * float(want.abs().max())
    linear(x, w)
    gate_up(x[:200], w)
    assert len(calls) == 3
