"""Steps with prompt portions through a run of alike pre-norm layers: every layer's launches from native code.

A step of few tokens is bound by the host: a layer's ten launches cost the interpreter more than its kernels take (0.6B: 160 us,
and 60 us of kernels at 300 tokens).  What a part's ``forward`` decides from sizes alone is decided here once for all layers, and the
launches go out from one call (``kernels/dense.py``).  The kernels, their order and so the results are those of the blocks'
own ``forward`` (but for products that are not worth the library's launch, or a kernel for few rows, here), which takes whatever this does not: float32, steps of single tokens (captured graphs, mostly), up to 16 rows
(the folded kernels), products that the library is ahead for (their kernels then take longer than the host) and parts of
any other kind.
"""
from __future__ import annotations

import operator
from typing import List, Optional, Sequence, Tuple

import torch

from ..kernels import dense, dispatch, ops
from .attention import GQAttention
from .base import Block, LayerCache, StepContext
from .block import PreNormBlock
from .feedforward import SwiGLU
from .norm import RMSNorm


_KINDS = (GQAttention, SwiGLU, RMSNorm, RMSNorm)
_of_block = operator.attrgetter("mixer", "ffn", "mixer_norm", "ffn_norm")
_of_mixer = operator.attrgetter("hidden_size", "nq", "nkv", "hd", "scale", "reach", "bias", "qk_norm_eps")
_of_ffn = operator.attrgetter("hidden_size", "intermediate_size")
_of_norm = operator.attrgetter("eps", "size")


def layer_form(block: Block) -> Optional[tuple]:
    """What has to be alike in a run's layers (None: not a block that a run takes): the numbers its launches are made with.  A part with
    a method of its own for what a run does (a wrapper put on the object) is left to its own forward pass.  Asked of every layer in
    every step: 1.3 us each."""
    if type(block) is not PreNormBlock:
        return None
    m, f, n1, n2 = parts = _of_block(block)
    if tuple(map(type, parts)) != _KINDS or m.general:
        return None
    own = m.__dict__
    if ("forward" in block.__dict__ or "forward" in own or "_attend" in own or "forward" in f.__dict__
            or "add_norm" in n1.__dict__ or "add_norm" in n2.__dict__):
        return None
    return _of_mixer(m), _of_ffn(f), _of_norm(n1), _of_norm(n2)


def alike_layers(blocks: Sequence[Block]) -> int:
    """How many of the first blocks are alike in that."""
    form = layer_form(blocks[0]) if blocks else None
    n = 0
    while form is not None and n < len(blocks) and layer_form(blocks[n]) == form:
        n += 1
    return n


# Up to this many multiplications and additions a layer's kernels take less time than the interpreter's launches (0.6B at 1200 tokens: 130
# us, 140): own products are then worth it also where the library's are a few us ahead.
HOST_BOUND = 19_000_000_000


def _product(rows: int, columns: int, inner: int, role: str, host_bound: bool) -> Optional[dense.Product]:
    """The framework's own product that the parts' ``linear``, ``gate_up`` and ``linear_into_stream`` would take, if it is one for
    many rows; with ``host_bound`` also one that another kernel is ahead of."""
    lim = dispatch.limits(columns, inner)
    plan, mode = dispatch.panels(rows, columns, inner, role, role == "stream" and lim.stacked_from <= rows <= lim.stacked_to, host_bound)
    if plan >= 0:
        return dense.Product(0, mode, plan & 0xff, plan >> 8)
    if role == "gated":
        groups = dispatch.gated_tile_groups(rows, columns, inner)
        return dense.Product(1, ops.TILES_GATED, groups, 1) if groups and rows > max(lim.silu_skinny, lim.silu_rows) else None
    if rows > max(lim.skinny, lim.rows, lim.sums_to, lim.stacked_to) and any(first <= rows <= last for first, last in lim.tiles):
        return dense.Product(1, ops.TILES_STORE, ops.TILES_GROUPS, 1)
    return None


class _Unusual(Exception):
    """A tensor that the blocks' own forward has to take, or to refuse."""


def _bf16(t: torch.Tensor, shape: Tuple[int, ...]) -> int:
    at = t.data_ptr()
    if t.dtype != torch.bfloat16 or t.shape != shape or not t.is_contiguous() or at % 16:
        raise _Unusual
    return at


def _f32(t: Optional[torch.Tensor], n: int) -> int:
    if t is None:
        return 0
    if t.dtype != torch.float32 or t.numel() != n or not t.is_contiguous():
        raise _Unusual
    return t.data_ptr()


def _pools(cache: LayerCache, nkv: int, page_size: int, hd: int) -> Tuple[int, int]:
    k, v = cache.k_pool, cache.v_pool
    if k is None or v is None or k.shape[0] != v.shape[0]:
        raise _Unusual
    return _bf16(k, (k.shape[0], nkv, page_size, hd)), _bf16(v, (v.shape[0], nkv, hd, page_size))


def _layers(blocks: List[Block], caches: List[LayerCache], widths: Tuple[int, int, int, int], page_size: int, rotation: tuple,
            table: torch.Tensor) -> List[tuple]:
    """Every layer's fields (``dense.LAYER_FIELDS``)."""
    H, I, q_width, qkv_width = widths
    table_rows, rot, style = rotation
    out = []
    for block, cache in zip(blocks, caches):
        a, f = block.mixer, block.ffn
        angles, its_rot, its_style = a.position.kernel_args() if a.position is not None else (None, 0, 0)
        if (its_rot, its_style) != (rot, style) or (table_rows and angles.shape != (table_rows, rot)):
            raise _Unusual
        out.append((_f32(block.mixer_norm.gain, H), _f32(a.q_gain, a.hd), _f32(a.k_gain, a.hd),
                    _f32(angles, table_rows * rot) if table_rows else 0, _f32(a.b_qkv, qkv_width), _f32(block.ffn_norm.gain, H),
                    _bf16(a.w_qkv, (qkv_width, H)), _bf16(a.w_o, (H, q_width)), _bf16(f.w_gate_up, (2 * I, H)), _bf16(f.w_down, (H, I)),
                    *_pools(cache, a.nkv, page_size, a.hd), table.data_ptr(), table.stride(0), 1 if cache.owner else 0))
    return out


def run_layers(blocks: List[Block], caches: List[LayerCache], residual: torch.Tensor, ctx: StepContext) -> Optional[torch.Tensor]:
    """Runs a model's first, alike blocks over the batch: the stream ``residual`` is updated in place, and what the last block leaves to
    be added to it is returned, as its ``forward`` would; None (and nothing done) where this way is not taken."""
    T, H = residual.shape
    if T < dispatch.PANELS_MIN_ROWS or alike_layers(blocks) < len(blocks):      # as they are now: parts may have been exchanged
        return None
    first = blocks[0]
    m, I = first.mixer, first.ffn.intermediate_size
    work = ctx.plans["attention"].facts
    group = ctx.groups[caches[0].group]
    if (ctx.dtype != torch.bfloat16 or not work["num_tiles"] or not ctx.stacked_branches
            or H % 64 or I % 64 or m.nq * m.hd % 64 or residual.dtype != torch.float32 or not residual.is_contiguous()
            or any(c.group != caches[0].group for c in caches)
            or not ops.attention_mfma_supports(ctx.dtype, m.hd, group.page_size, m.nq, m.nkv)):
        return None
    q_width, qkv_width = m.nq * m.hd, (m.nq + 2 * m.nkv) * m.hd
    if max(T, 2 * I, qkv_width) * max(H, I, q_width) >= 2 ** 31:
        return None
    host_bound = T * (H * (qkv_width + q_width) + 3 * I * H) <= HOST_BOUND
    into, out, gate_up, down = (_product(T, *product, host_bound) for product in (
        (qkv_width, H, "store"), (H, q_width, "stream"), (2 * I, H, "gated"), (H, I, "stream")))
    if into is None or out is None or gate_up is None or down is None:
        return None
    angles, rot, style = m.position.kernel_args() if m.position is not None else (None, 0, 0)
    table_rows = 0
    if style != 0 and rot > 0:
        if angles is None or angles.dim() != 2:
            return None
        table_rows = angles.shape[0]
    bt, plan = group.block_table, ctx.plans["attention"].arrays
    for t, n in ((ctx.positions, T), (ctx.token_entry, T), (plan["decode_tokens"], work["num_decode"]), (plan["tiles"], 2 * work["num_tiles"]),
                 (plan["wide_tiles"], 2 * work["num_wide"])):
        if t.dtype != torch.int32 or not t.is_contiguous() or t.numel() < n:
            return None
    if bt.dtype != torch.int32 or bt.dim() != 2 or bt.stride(1) != 1 or -(-work["max_decode_kv"] // group.page_size) > bt.shape[1]:
        return None
    try:
        layers = _layers(blocks, caches, (H, I, q_width, qkv_width), group.page_size, (table_rows, rot, style), bt)
    except _Unusual:
        return None
    device = residual.device

    def rows_of(width):
        return torch.empty((T, width), dtype=torch.bfloat16, device=device)

    def branch_of(p):
        return torch.empty((p.slices, T, H), dtype=torch.float32, device=device) if p.mode == dispatch.PANELS_FLOAT else rows_of(H)

    normed, qkv, q, attended, act = (rows_of(n) for n in (H, qkv_width, q_width, q_width, I))
    mixed, fed = branch_of(out), branch_of(down)
    sums = torch.empty((into.slices, T, qkv_width), dtype=torch.float32, device=device) if into.mode == dispatch.PANELS_FLOAT else None
    waves, splits, parts = 1, 1, None
    if work["num_decode"]:
        waves, splits = ops.decode_cuts(work["num_decode"], m.nkv, -(-(m.nq // m.nkv) // 16), work["max_decode_kv"], m.hd, m.reach,
                                        ops.compute_units(device))
        parts = ops.decode_parts(work["num_decode"], m.nq, m.hd, splits, waves, device)
    address = lambda t: 0 if t is None else t.data_ptr()       # noqa: E731
    step = dense.Step(
        residual=residual.data_ptr(), normed=normed.data_ptr(), qkv=qkv.data_ptr(), q=q.data_ptr(), attended=attended.data_ptr(),
        act=act.data_ptr(), sums=address(sums), decode_parts=address(parts), mixed=mixed.data_ptr(), fed=fed.data_ptr(),
        positions=ctx.positions.data_ptr(), token_entry=ctx.token_entry.data_ptr(), decode_tokens=plan["decode_tokens"].data_ptr(),
        prompt_tiles=plan["tiles"].data_ptr(), wide_tiles=plan["wide_tiles"].data_ptr(), tile_keys_total=int(work["tile_keys_total"]),
        wide_keys_total=int(work["wide_keys_total"]), into=into, out=out, gate_up=gate_up, down=down, tokens=T, width=H,
        heads=m.nq, kv_heads=m.nkv, head_dim=m.hd, inner=I, table_rows=table_rows, rot=rot, style=style, page_size=group.page_size,
        window=m.reach, num_decode=work["num_decode"], decode_splits=splits, decode_waves=4 if m.hd == 256 and waves == 8 else waves,
        num_tiles=work["num_tiles"], tile_keys_max=work["tile_keys_max"], num_wide=work["num_wide"], wide_keys_max=work["wide_keys_max"],
        decode_keys_total=work.get("decode_keys", 0), decode_keys_max=work["max_decode_kv"],
        eps1=first.mixer_norm.eps, eps2=first.ffn_norm.eps,
        qk_eps=m.qk_norm_eps if m.qk_norm_eps is not None else 0.0, scale=m.scale)
    dense.dense_layers(step, layers)
    return fed
