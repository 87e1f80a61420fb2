"""The panels kernel's shapes at the edges of their tiles: rows and columns past the last tile's, K that no number of parts divides, one
stage a part, against 64-bit results; and the rule by which calls come to it."""
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
@pytest.mark.parametrize("M,N,K", [(1, 16, 256), (31, 48, 320), (33, 176, 256), (97, 208, 576), (129, 272, 1024), (161, 144, 704), (255, 400, 832),
                                   (258, 1040, 1088)])
def test_every_shape_at_tile_edges(ops, M, N, K):
    from ullm_amd.kernels import build, dispatch
    lib = build.load("gemm_panels")
    x, w, bias = _operands(M, N, K, M + N)
    want = x.double() @ w.double().T
    off = (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)             # K products added in 32-bit
    ref, half = want + bias.double(), N // 2
    taken = 0
    for shape in range(lib.ullm_gemm_panels_shapes()):
        takes = lambda mode, slices: lib.ullm_gemm_panels_supports(M, N, K, K + 8, K, mode, shape, slices)      # noqa: B023, E731
        for slices in (1, 2, 3, 8):
            if not takes(dispatch.PANELS_FLOAT, slices):
                continue
            taken += 1
            sums = ops.gemm_panels(x, w, shape | slices << 8, dispatch.PANELS_FLOAT)
            assert sums.shape == (slices, M, N) and ((sums.double().sum(0) - want).abs() <= off).all(), (shape, slices)
            assert torch.equal(ops.gemm_panels(x, w, shape | slices << 8, dispatch.PANELS_FLOAT), sums)          # by no timing
        one = shape | 1 << 8
        if not takes(dispatch.PANELS_STORE, 1):
            continue
        full = ops.gemm_panels(x, w, one, dispatch.PANELS_FLOAT)[0]
        assert torch.equal(ops.gemm_panels(x, w, one, dispatch.PANELS_STORE), full.bfloat16()), shape
        got = ops.gemm_panels(x, w, one, dispatch.PANELS_STORE, bias)
        assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + off + 2.0 ** -23 * ref.abs()).all(), shape
        act = ops.gemm_panels(x, w, one, dispatch.PANELS_STORE, bias, act=ops.ACT_RELU2)
        assert ((act.double() - ref.clamp(min=0) ** 2).abs() <= 2.0 ** -8 * ref ** 2 + 4 * off * (ref.abs() + off)).all(), shape
        if not takes(dispatch.PANELS_GATED, 1):
            continue
        for limit, alpha in ((0.0, 0.0), (1.0, 1.7)):
            unit = ops.gemm_panels(x, w, one, dispatch.PANELS_GATED, limit=limit, alpha=alpha)
            g, u = want[:, :half], want[:, half:]
            if limit:
                g, u = g.clamp(max=limit), u.clamp(-limit, limit)
                expect = g * torch.sigmoid(alpha * g) * (u + 1)
            else:
                expect = g * torch.sigmoid(g) * u
            slack = 4 * off.amax(-1, keepdim=True) * (2 + g.abs() + u.abs()) + 2.0 ** -21 * expect.abs()        # sums, and the unit's own ulps
            assert ((unit.double() - expect).abs() <= 2.0 ** -8 * expect.abs() + slack).all(), (shape, limit)
    assert taken >= (24 if K >= 1024 else 8)


@pytest.mark.gpu
def test_what_it_refuses(ops):
    from ullm_amd.kernels import dispatch
    x, w, bias = _operands(40, 64, 256, 1)
    with pytest.raises(ops.KernelError):
        ops.gemm_panels(x, w, 99 | 1 << 8, dispatch.PANELS_STORE)                    # no such shape
    with pytest.raises(ops.KernelError):
        ops.gemm_panels(x, w, 0 | 2 << 8, dispatch.PANELS_STORE)                     # slices of a rounded result
    with pytest.raises(ops.KernelError):
        ops.gemm_panels(x, w, 1 << 8, dispatch.PANELS_GATED, bias)
    assert not ops.gemm_panels_supports(x[:, 4:], w[:, 4:]) and not ops.gemm_panels_supports(x[:, :128], w)


def test_when_it_is_taken():
    """CPU: sizes on both sides of every line of the rule; every plan is one that the kernel takes, in one round of blocks."""
    from ullm_amd.kernels import build, dispatch
    lib = build.load("gemm_panels")
    P = dispatch.panels
    assert [P(r, 24576, 4096, "gated")[0] >= 0 for r in (16, 17, 256, 257, 3000)] == [False, True, True, False, False]
    assert [P(r, 1024, 3072, "stream")[0] >= 0 for r in (16, 17, 1024, 1025)] == [False, True, True, False]
    assert [P(r, 1024, 3072, "stream", False, True)[0] >= 0 for r in (16, 1025, 1800, 20000)] == [False, True, True, False]
    assert [P(r, 4096, 12288, "stream")[0] >= 0 for r in (17, 1024, 1025)] == [True, True, False]
    assert [P(r, 151936, 1024, "float")[0] >= 0 for r in (16, 17, 256, 257)] == [False, True, True, False]      # in more than one round
    assert [P(r, 2048, 2048, "float")[0] >= 0 for r in (17, 512, 513)] == [True, True, False] and P(600, 4096, 2048, "float")[0] >= 0
    assert P(64, 1000, 1024, "store")[0] < 0 and P(64, 1024, 1024, "store")[0] >= 0            # a smaller matrix than measured
    assert P(64, 2052, 1024, "store")[0] < 0 and P(64, 2048, 1000, "store")[0] < 0 and P(64, 8200, 1024, "gated")[0] < 0
    for rows in list(range(17, 2200, 61)) + [2048]:
        for N, K in ((1024, 1024), (4096, 1024), (6144, 4096), (1024, 3072), (4096, 12288), (24576, 4096), (2048, 2048), (51200, 5120)):
            for role, keep in (("store", False), ("gated", False), ("stream", False), ("stream", True)):
                plan, mode = P(rows, N, K, role, keep)
                if plan < 0:
                    continue
                assert lib.ullm_gemm_panels_supports(rows, N, K, K, K, mode, plan & 255, plan >> 8)
                assert mode == dispatch.PANELS_FLOAT or (not keep and (mode == dispatch.PANELS_GATED) == (role == "gated"))


@pytest.mark.gpu
def test_parts_take_it_where_the_rule_says(ops, monkeypatch):
    from types import SimpleNamespace
    from ullm_amd.kernels import dispatch
    from ullm_amd.parts.linear import gate_up, linear, linear_into_stream
    calls, real = [], ops.gemm_panels
    monkeypatch.setattr(ops, "gemm_panels", lambda *a, **k: calls.append(a[3]) or real(*a, **k))
    ctx = SimpleNamespace(stacked_branches=True)
    for rows in (16, 17, 130):
        x, w, bias = _operands(rows, 1024, 2048, rows)
        want = x.double() @ w.double().T
        close = lambda y, ref: float((y.double() - ref).abs().max()) <= 2.0 ** -7 * float(ref.abs().max())      # noqa: E731
        assert close(linear(x, w, bias), want + bias.double())
        full = linear(x, w, bias, out_dtype=torch.float32)
        assert full.dtype == torch.float32 and float((full.double() - want - bias.double()).abs().max()) <= 1e-5 * float(want.abs().max())
        g, u = want[:, :512], want[:, 512:]
        assert close(gate_up(x, w), g * torch.sigmoid(g) * u)
        y = linear_into_stream(x, w, ctx)
        assert close(y if y.dim() == 2 else y.sum(0), want)
        assert (len(calls) == 4) == (rows > 16) and (rows == 16 or set(calls) >= {dispatch.PANELS_GATED, dispatch.PANELS_FLOAT})
        del calls[:]


# products whose fastest plan without an activation is slices that a kernel adds (at 17 rows; one that fits no round in one slice), and
# one whose plan is whole
@pytest.mark.gpu
@pytest.mark.parametrize("N,K,rows", [(10240, 2560, (17, 32, 40, 64)), (12288, 3072, (17, 24)), (5120, 5120, (17, 64, 130, 400)), (4096, 1024, (17, 100))])
def test_an_activation_sees_the_32_bit_sums(ops, N, K, rows):
    from ullm_amd.kernels import dispatch
    from ullm_amd.parts.linear import linear
    assert any(dispatch.panels(r, N, K, "store")[1] == dispatch.PANELS_FLOAT for r in rows) == (N != 4096)
    for M in rows:
        x, w, bias = _operands(M, N, K, M)
        off = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + bias.double().abs())
        y = x.double() @ w.double().T + bias.double()
        ref = y.clamp(min=0) ** 2
        # one rounding to bfloat16 behind the square: the sums' own rounding would be doubled by it and come on top
        assert ((linear(x, w, bias, act=ops.ACT_RELU2).double() - ref).abs() <= 2.0 ** -8 * ref + 4 * off * (y.abs() + off)).all(), M


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [130, 400])
def test_rows_that_overlap_go_where_they_went(ops, rows):
    """An expanded row, and windows of one buffer, as x and as W: refused by the kernel, so the other products take them."""
    from types import SimpleNamespace
    from ullm_amd.parts.linear import gate_up, linear, linear_into_stream
    x, w, bias = _operands(rows, 2048, 1024, rows)
    x = x.contiguous()
    row, windows = x[:1].expand(rows, 1024), x.flatten()[:1024 + 1016 * (rows - 1)].as_strided((rows, 1024), (1016, 1))
    w_row, ctx = w[:1].expand(2048, 1024), SimpleNamespace(stacked_branches=True)
    for a, b in ((row, w), (windows, w), (x, w_row)):
        assert not ops.gemm_panels_supports(a, b)
        want = a.double() @ b.double().T
        close = lambda y, ref: float((y.double() - ref).abs().max()) <= 2.0 ** -7 * float(ref.abs().max())      # noqa: E731
        y = linear_into_stream(a, b, ctx)
        assert close(y if y.dim() == 2 else y.sum(0), want) and close(linear(a, b, bias), want + bias.double())
        assert b is w_row or close(linear(a, b, out_dtype=torch.float32), want)          # 32-bit results of such a W always were refused
        g, u = want[:, :1024], want[:, 1024:]
        assert close(gate_up(a, b), g * torch.sigmoid(g) * u)


def test_operands_that_are_the_librarys(ops):
    """CPU, with stand-ins for device tensors: a matrix on another device than x is never handed to the kernel (the library refuses it),
    nor is a single vector, which the library takes."""
    from types import SimpleNamespace

    def tensor(device, *shape):
        strides = (shape[-1], 1)[-len(shape):]
        return SimpleNamespace(dtype=torch.bfloat16, device=torch.device(device), is_cuda=device != "cpu", shape=shape, data_ptr=lambda: 0,
                               dim=lambda: len(shape), stride=lambda i: strides[i])
    takes = lambda x, w: ops.gemm_panels_supports(x, w)        # noqa: E731
    x = tensor("cuda:0", 130, 1024)
    assert takes(x, tensor("cuda:0", 2048, 1024))
    assert not takes(x, tensor("cpu", 2048, 1024)) and not takes(x, tensor("cuda:1", 2048, 1024))
    assert not takes(tensor("cpu", 130, 1024), tensor("cpu", 2048, 1024))
    assert not takes(tensor("cuda:0", 1024), tensor("cuda:0", 2048, 1024))


@pytest.mark.gpu
def test_a_vector_and_operands_of_two_devices(ops):
    x, w, _ = _operands(200, 2048, 1024, 3)
    want = x[0].double() @ w.double().T
    assert (ops.gemm_bf16(x[0].contiguous(), w).double() - want).abs().max() <= 2.0 ** -7 * want.abs().max()
    for M in (130, 200):
        with pytest.raises(RuntimeError):
            ops.gemm_bf16(x[:M], w.cpu())


# one slice is ahead of four and the kernel that adds them; slices are ahead
@pytest.mark.gpu
@pytest.mark.parametrize("N,K,rows,sums", [(2048, 2048, (17, 48, 200, 1000), 0), (1024, 2048, (48,), 0), (5120, 17408, (17, 130), 1)])
def test_blocks_that_want_a_branch_whole(ops, monkeypatch, N, K, rows, sums):
    """Where no norm adds slices, a branch is made in one piece unless slices and the kernel that adds them are ahead."""
    from types import SimpleNamespace
    from ullm_amd.parts import LayerCache
    from ullm_amd.parts.block import ParallelBlock, SandwichBlock
    from ullm_amd.parts.decay import SideBySide
    from ullm_amd.parts.linear import linear_into_stream
    launched, real = [], ops.branch_sum
    monkeypatch.setattr(ops, "branch_sum", lambda a, b=None: launched.append(b is None) or real(a, b))
    for M in rows:
        x, w, _ = _operands(M, N, K, M)
        ctx = SimpleNamespace(stacked_branches=True, whole_branch=False, dtype=torch.bfloat16)
        want = x.double() @ w.double().T
        product = SimpleNamespace(forward=lambda h, c, cache=None: linear_into_stream(h, w, c), cache_need=lambda: None,
                                  step_planners={})
        norm = SimpleNamespace(add_norm=lambda branch, residual, rows=None, out_dtype=None: x, kernel_form=lambda: (None, 0.0, 0))
        onto = SimpleNamespace(forward_onto=lambda h, c, base: base)
        branches = [SandwichBlock(norm, product, norm).forward(None, None, ctx, None)[1].branch,
                    SandwichBlock(norm, product, norm, 1.0, norm, product, norm).forward(None, None, ctx, None)[1].branch,
                    ParallelBlock(norm, product, None).forward(None, None, ctx, None)[1].branch,
                    ParallelBlock(norm, product, onto).forward(None, None, ctx, None)[1].branch,
                    *SideBySide(product, product).forward_pair(x, ctx, LayerCache())[::2]]
        assert len(launched) == 7 * sums and not ctx.whole_branch
        for y in branches:
            assert y.dim() == 2 and (y.double() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
        del launched[:]
        stack = linear_into_stream(x, w, ctx)                # a norm adds slices as before
        assert (stack if stack.dim() == 2 else stack.sum(0)).shape == (M, N)
