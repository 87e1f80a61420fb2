"""Rows of a product that the kernels for few rows and the library keep, because they were measured to be ahead of the panels kernel there."""
import json

import pytest
import torch

from ullm_amd.kernels import dispatch


@pytest.fixture
def table(tmp_path, monkeypatch):
    def use(matrices):
        path = tmp_path / "table.json"
        path.write_text(json.dumps({"matrices": matrices}))
        monkeypatch.setattr(dispatch, "TABLE_PATH", str(path))
        monkeypatch.setattr(dispatch, "_table", None)
        dispatch.panels.cache_clear()
    yield use
    monkeypatch.undo()
    dispatch._table = None                                     # the real table again, and nothing remembered of this one
    dispatch.panels.cache_clear()


def _takes(rows, columns, inner, role="store", **more):
    return dispatch.panels(rows, columns, inner, role, **more)[0] >= 0


def test_measured_ranges(table):
    """A range counts for its own kind of product, ends where it ends, and not where launches are what takes the time."""
    table({"7168x5120": {"store_kept": "17-96"}, "8192x4096": {"silu_kept": "300-310", "store_kept": ""}, "5120x17408": {"stream_kept": "41-48"}})
    for role in ("store", "activated"):
        assert [_takes(r, 7168, 5120, role) for r in (17, 96, 97)] == [False, False, True]
    assert _takes(17, 7168, 5120, host_bound=True) and _takes(48, 7168, 5120, "stream") and _takes(48, 7168, 5120, "float")
    assert [_takes(r, 8192, 4096, "gated") for r in (299, 300, 310, 311)] == [True, False, False, True] and _takes(300, 8192, 4096)
    for more in ({}, {"keep_sums": True}, {"whole": True}):
        assert [_takes(r, 5120, 17408, "stream", **more) for r in (40, 41, 48, 49)] == [True, False, False, True]
    table({"7168x5120": {"store_kept": ""}})
    assert _takes(17, 7168, 5120)


def test_rows_for_partial_sums_leave_the_others_to_the_panels_kernel(table):
    """Rows that a table names for the partial sums stay with them unless they were compared with the panels kernel; the others do not: it
    used to be off at every row count."""
    table({"4096x1024": {"sums_from": 33, "sums_to": 256}, "4096x2048": {"sums_from": 33, "sums_to": 256, "store_kept": "33-40"}})
    from ullm_amd.parts.dense import _product
    for rows in (17, 32, 257, 300):
        assert _takes(rows, 4096, 1024) and _product(rows, 4096, 1024, "store", False).tiles == 0
    for rows in (33, 40, 256):
        assert not _takes(rows, 4096, 1024) and _takes(rows, 4096, 1024, "activated") and _takes(rows, 4096, 1024, "stream")
    assert [_takes(rows, 4096, 2048) for rows in (32, 33, 40, 41)] == [True, False, False, True]


@pytest.mark.parametrize("columns,inner,role,rows", [(5632, 5120, "store", (17, 32, 48)), (5120, 3072, "store", (17, 32)), (10240, 2560, "activated", (40, 48)),
                                                     (19456, 2560, "gated", (40, 48))])
def test_matrices_that_were_not_measured(columns, inner, role, rows):
    """Of 24 to 64 M values, up to 48 rows, with units left idle by the plan; not where the rows kernel is not what takes the call."""
    assert getattr(dispatch.limits(columns, inner), "silu_kept" if role == "gated" else "store_kept") is None
    for r in rows:
        assert not _takes(r, columns, inner, role) and (role == "activated" or _takes(r, columns, inner, role, host_bound=True))
    assert _takes(64, columns, inner, role) and _takes(100, columns, inner, role)
    assert _takes(17, 19456, 2560, "gated")                     # the few-rows kernel's call
    assert _takes(40, 4096, 4608) and _takes(40, 16384, 4096, "activated") and _takes(40, 8192, 3584)      # small, large, no unit idle


def test_few_columns_that_were_not_measured(table):
    """From 513 rows on the library's; not with other sizes, an activation, for a stream that adds slices or where launches count."""
    table({"1024x3072": {"stacked_from": 17, "stacked_to": 96}, "1024x2048": {"store_kept": "769-1024"}})
    for columns, inner, last in ((1024, 2560, 512), (1024, 3072, 512), (768, 1536, 512)):
        for role, more in (("store", {}), ("stream", {"whole": True})):
            assert [_takes(r, columns, inner, role, **more) for r in (last, last + 1, 1024)] == [True, False, False]
            assert _takes(900, columns, inner, role, host_bound=True, **more)
        assert _takes(900, columns, inner, "activated") and _takes(900, columns, inner, "stream")
    assert [_takes(r, 1024, 2048) for r in (640, 768, 769)] == [True, True, False]                  # measured
    for columns, inner in ((1024, 1024), (1024, 4096), (1536, 2048), (2048, 2048), (2560, 2560)):
        assert _takes(640, columns, inner) and _takes(640, columns, inner, "stream", whole=True)


def test_ranges_from_times():
    from ullm_amd.kernels.microbench import derive_limits
    rows = [16, 17, 32, 48, 64, 128, 256, 288]
    times = {"library": dict(zip(rows, [20, 20, 20, 20, 20, 20, 29, 22])), "rows": {16: 14, 17: 14, 32: 15, 48: 22},
             "partial sums>sum": {17: 18, 32: 18, 48: 18, 64: 18, 128: 21}, "panels": {17: 16, 32: 17, 48: 19, 64: 20, 128: 20, 256: 28, 288: 24},
             "norm": {}}
    # 17 and 32 the rows kernel, 48 and 64 the partial sums; 288 alone makes no range
    found = derive_limits(times, {"store"}, 0, 0)
    assert found["store_kept"] == [[17, 64]] and (found["rows"], found["sums_from"], found["sums_to"]) == (32, 33, 64)
    times = {"library>norm": {17: 30, 32: 30, 48: 30, 64: 22, 288: 20, 320: 21}, "partial sums>norm": {17: 20, 32: 20, 48: 20},
             "panels>norm": {17: 20, 32: 21, 48: 21, 64: 21, 288: 25, 320: 21}}
    assert derive_limits(times, {"stream"}, 0, 0) == {"stacked_from": 17, "stacked_to": 48, "stream_kept": [[18, 48]]}
    times = {"skinny+silu": {16: 9, 17: 20}, "rows+silu": {16: 12, 17: 12, 32: 13, 64: 30}, "library+silu": {16: 20, 17: 20, 32: 20, 64: 29},
             "panels+silu": {17: 14, 32: 14, 64: 29}, "norm": {}}
    assert derive_limits(times, {"silu"}, 0, 0)["silu_kept"] == [[17, 32]]


def test_written_and_read_back(table):
    table({})
    dispatch.write_entry(778, 64, {"store_kept": [[17, 64], [257, 320]], "silu_kept": []})
    got = dispatch.limits(778, 64)
    assert (got.store_kept, got.silu_kept, got.stream_kept) == (((17, 64), (257, 320)), (), None)


@pytest.mark.gpu
def test_the_kernels_that_keep_them(monkeypatch):
    """q|k|v 7168 x 5120: the rows kernel, partial sums, then panels; gate|up 19456 x 2560: the rows kernel; each against 64 bits."""
    from ullm_amd.kernels import ops
    from ullm_amd.parts.linear import gate_up, linear
    calls = []
    for name in ("gemm_rows", "gemm_partial_sums", "gemm_panels"):
        monkeypatch.setattr(ops, name, lambda *a, _real=getattr(ops, name), _name=name, **k: calls.append(_name) or _real(*a, **k))
    g = torch.Generator(device="cuda").manual_seed(2)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=g).bfloat16()          # noqa: E731
    w, u = draw(7168, 5120) * 5120 ** -0.5, draw(19456, 2560) * 2560 ** -0.5
    for rows, kernel in ((17, "gemm_rows"), (33, "gemm_rows"), (34, "gemm_partial_sums"), (96, "gemm_partial_sums"), (97, "gemm_panels")):
        x = draw(rows, 5120)
        want = x.double() @ w.double().T
        assert (linear(x, w).double() - want).abs().max() <= 2.0 ** -8 * want.abs().max() and calls == [kernel], rows
        del calls[:]
    for rows, kernel in ((33, "gemm_rows"), (48, "gemm_rows"), (49, "gemm_panels")):
        x = draw(rows, 2560)
        gate, up = (x.double() @ u.double().T).chunk(2, 1)
        want = gate * torch.sigmoid(gate) * up
        assert (gate_up(x, u).double() - want).abs().max() <= 2.0 ** -7 * want.abs().max() and calls == [kernel], rows
        del calls[:]
