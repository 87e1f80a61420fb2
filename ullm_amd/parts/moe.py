"""Routed feed-forward: a router picks ``top`` of several small gated feed-forwards per token.

The router's logits are a 32-bit product of the part's input with a matrix [R, hidden], R = experts with weights +
identity experts.  The scores are the softmax over all R; the choice goes by score + a learned correction per
output (``correction``), the weights by the chosen outputs' scores alone, divided by their sum (+ 1e-20).  The last
``identity`` router outputs stand for experts without tensors whose output is their input.  Every expert is
``down(act(gate(x), up(x)))`` without biases, with the clamped gated unit
``act(g, u) = g' * sigmoid(alpha * g') * (u' + 1)``, ``g' = min(g, limit)``, ``u' = clamp(u, -limit, limit)``.
A shared expert of the same form (sizes and limit of its own) may run for every token and is added.
Two more forms, each a parameter: ``routing="top_logits"`` picks the ``top`` largest of logits + a learned bias per
output (the ``correction`` tensor, then a bias on the logits) and weighs them by the softmax over the picked ones
alone; ``routing="sigmoid"`` scores every output by the sigmoid of its own logit, chooses by score + correction and
weighs by the chosen scores over their sum (+ 1e-20); ``weight_scale`` multiplies every weight; ``limit=None`` makes
every expert the plain gated unit ``silu(g) * u``; ``renormalize=False`` takes the chosen scores as weights as they are;
``groups`` and ``keep_groups``: the router's outputs form that many equal groups of neighbours, and only outputs of the
best ``keep_groups`` can be chosen (a group counts as much as its ``group_top`` largest choice scores together: one or two).

The experts' matrices are stacked ([experts, 2 ff, hidden] with gate rows, then up rows, per expert, and
[experts, hidden, ff]); the loader puts the checkpoint's per-expert tensors into their rows.  A step groups
its (token, expert) pairs by expert on the device and runs the two products over the grouped rows
(``ops.moe_sort``, ``ops.moe_rows``); launches are sized by the step's token count alone, so a step of single
tokens can be replayed from a graph.  The result is 32-bit: ``forward_onto`` adds it onto another branch of
the same block (and that branch's bias) in the kernel that sums the experts.
"""
from __future__ import annotations

import functools
import math
from typing import Dict, List, Optional

import torch

from ..kernels import ops
from .base import FeedForward, NormedBranch, PartEnv, StepContext, SummedBranch, WeightDecl, register_part
from .linear import gate_up, linear

DEFAULT_NAMES = {"router": "router", "correction": "correction", "expert": "e{index}", "gate": "gate", "up": "up",
                 "down": "down", "shared": "shared"}


def _expected_tiles(experts: int, mean: float, rows: int) -> float:
    """Tiles of ``rows`` that ``experts`` experts fill together, whose rows spread around ``mean`` a little more than by chance."""
    spread, per_expert, full = math.sqrt(2.0 * (mean + (0.06 * mean) ** 2)), 1.0, 1
    while full * rows < mean + 4.0 * spread:
        per_expert += 0.5 * math.erfc((full * rows - mean) / spread)
        full += 1
    return experts * per_expert


def _tile_cost(rows: int, tiles: float, experts: int, hidden: int, ff: int) -> float:
    """About the microseconds of gate|up and down over ``tiles`` tiles of ``rows`` (see :func:`tile_rows_for`)."""
    cost = 0.0
    for inner, columns, gated in ((hidden, ff, True), (ff, hidden, False)):
        megabytes = (4e-6 if gated else 2e-6) * experts * columns * inner
        if rows <= 32:
            cost += 4.86 + megabytes * (1.0 / (7.83 if rows == 16 else 6.09) + (tiles / experts - 1.0) / 2.94)
            continue
        per_tile = -(-columns // ((64 if rows == 64 else 128) * (1 if gated else 2)))
        rounds = tiles * per_tile / 256
        whole = int(rounds)
        begun = 1.0 - math.exp(-(rounds - whole) * 256 / per_tile)     # whether some tile makes one more
        full_round = 10.3 + 0.0212 * inner                     # of blocks of 256 rows
        if rows == 64:
            last = (whole + 1 - rounds) * begun * 0.55 * min(1.0, 2.42 / rounds)
            work, read = full_round * max(0.425, (0.249 + 4.33e-5 * inner) * (rounds + last)), megabytes / 5.3
            cost += (work ** 4 + read ** 4) ** 0.25
        else:
            work, read = full_round * (0.674 if rows == 128 else 1.0), megabytes / (5.03 if rows == 128 else 4.54)
            cost += max(1, whole) * (work ** 4 + (read / max(1.0, rounds)) ** 4) ** 0.25 + (work * begun if whole else 0.0)
    return cost


@functools.lru_cache(maxsize=1024, typed=True)
def tile_rows_for(tokens: int, top: int, experts: int, hidden: int = 0, ff: int = 0) -> int:
    """Grouped rows a block of the expert products takes, a function of the step's and the matrices' sizes alone.

    Inner sizes that are multiples of 64 (and rows that 32-bit offsets reach): the tile whose products cost least by an estimate
    from the tiles that the experts fill and the blocks these make.  Tiles of 16 and 32 rows read an expert's matrix again for
    every tile (at 7.8 and 6.1 TB/s the first time, 2.9 after that).  The others are bound by the matrices' bytes (5.3, 5.0 and
    4.5 TB/s) or by rounds of blocks over 256 compute units.  A block of 256 or 128 rows fills a unit, one of 128 takes 0.67 of the
    other's time, and a round with a single block takes as long as a full one: 32 experts make one round of 128 rows until one of
    them has a 129th row, and 145 us of 105.  Several blocks of 64 share a unit (0.3 to 0.45 a block, 0.43 alone), so few experts of few
    columns keep them longest.  Fitted to 454 measured points: eleven shapes (4 to 96 experts, width 1024 to 5120, 512 to 4096
    columns), means of 3 to 800 rows an expert, rows of the experts by chance alone or up to a quarter of the mean beside it.  The
    tile it takes was 0.4 % slower than the best on average; near a round's edge the best goes by the one expert with
    most rows, and the estimate by an even routing, which lost up to 25 % where the routing was not.
    gate|up + down in tiles of 16 / 32 / 64 / 128 / 256, us:
    32 experts, width 2048, 1024 columns at means of 12, 24, 36, 96, 160, 256 and 512 rows 81 / 77 / 94 / 100 / 112,
    130 / 81 / 91 / 98 / 107, 182 / 146 / 92 / 101 / 110, - / - / 113 / 105 / 119, - / - / 155 / 129 / 122, - / - / 223 / 174 / 191,
    - / - / 388 / 288 / 285, and over twelve routings at 44, 50, 56, 104 and 128 - / - / 95 / 102 / 110, - / - / 104 / 102 / 111,
    - / - / 110 / 103 / 112, - / - / 119 / 126 / 119, - / - / 141 / 133 / 120; 8 experts, width 1024, 512 columns at 36, 96, 160, 320, 1024
    19 / 17 / 19 / 26 / 35, 38 / 30 / 20 / 29 / 39, - / - / 21 / 30 / 41, - / - / 29 / 32 / 45, - / - / 56 / 61 / 51; 8 experts, width 4096, 1536
    columns at 24, 36, 128, 320 106 / 68 / 71 / 87 / 125, 146 / 110 / 71 / 90 / 127, - / - / 116 / 102 / 133, - / - / 231 / 168 / 150.
    A prompt of 440 tokens of a stack with six such layer runs took 2.42 ms in tiles of 64, 2.37 in tiles of 128.  (Tiles of 128 and 256
    have become faster since, where the experts' matrices come from memory, by up to a quarter: :func:`product_rows_for`.)"""
    mean = tokens * top / max(1, experts)
    if (mean > 0 and experts > 0 and hidden > 0 and hidden % 64 == 0 and ff > 0 and ff % 64 == 0
            and (tokens * top + 256 * experts) * max(hidden, ff) < 2 ** 31 and 2 * hidden * ff < 2 ** 31):
        return min((16, 32, 64, 128, 256), key=lambda rows: _tile_cost(rows, _expected_tiles(experts, mean, rows), experts, hidden, ff))
    if mean >= 96:
        return 128
    if mean >= 48:
        return 64
    return 32 if mean >= 24 else 16


def product_rows_for(tokens: int, top: int, experts: int, hidden: int = 0, ff: int = 0) -> int:
    """Grouped rows a block of the expert products takes: what :func:`tile_rows_for` says, but where its figures for tiles of 128 and
    256 rows are behind the kernels'.

    From 24 rows an expert on tiles of 128 in place of 32 and 64, where the rows of the matrices are long enough that blocks in step got
    in each other's way (width 2048 and more) and the gate|up of the experts' first tiles fills every compute unit.  us of gate|up +
    down, tiles of 64 and of 128, for routings by chance / unequal experts / very unequal ones: 32 experts, width 2048, 1024 columns at a mean of
    36 92 / 97 / 89 and 80 / 85 / 77; 64 experts of 768 columns at 42 140 / 145 / 127 and 134 / 136 / 122.  Not with fewer blocks or shorter rows (24 experts, width 3072, 1024 columns 1.04 of it, 40 of width 1536 1.13).

    From 250 on tiles of 256, whose blocks take a last tile of 64 rows or less at its own cost, where the experts' first tiles make
    about a round of blocks in each product (256 rows, 128 and 256: 16 experts, width 5120, 1536 columns 322 / 317 / 311 and 274 / 312 / 317; 32
    experts, width 2048, 1024 columns 176 / 170 / 176 and 158 / 183 / 182; 48 experts, width 1024, 1024 columns 135 / 134 / 131 and 120 / 141 / 121).  With fewer
    rows they are ahead only while every expert's last tile is short or long, as none is that is not routed to by chance alone: at
    30 to 55 rows 0.84 to 1.05 of the time of 64 by chance and 0.92 to 1.32 where experts are unequal (16 experts of 1536
    columns, 36 rows 159 / 161 / 161 and 153 / 198 / 197), at 106 to 120 of 128 1.05 to 1.26.  With fewer blocks they leave most units
    idle (8 experts, width 4096, 1536 columns 125 / 120 / 124 and 151 / 142 / 148).

    Over sixteen shapes (8 to 256 experts, width 512 to 5120) and 2 to 750 rows an expert 0.995 / 0.993 / 0.992 of the time by
    :func:`tile_rows_for` alone."""
    rows = tile_rows_for(tokens, top, experts, hidden, ff)
    mean = tokens * top / max(1, experts)
    if (hidden <= 0 or hidden % 64 or ff <= 0 or ff % 64 or (tokens * top + 256 * experts) * max(hidden, ff) >= 2 ** 31
            or 2 * hidden * ff >= 2 ** 31):
        return rows
    first_up, first_down = experts * -(-ff // 128), experts * -(-hidden // 256)          # blocks of the experts' first tiles
    if mean >= 24 and rows < 128 and hidden >= 2048 and first_up >= 256:
        return 128
    if mean >= 250 and first_up + first_down >= 460:
        return 256
    return rows


@register_part("ffn", "routed_experts")
class RoutedExperts(FeedForward):
    def __init__(self, hidden_size: int, experts: int, intermediate_size: int, top: int, limit: Optional[float],
                 prefix: str, identity: int = 0, alpha: float = 1.702, correction: bool = True,
                 shared_size: int = 0, shared_limit: Optional[float] = None, names: Optional[Dict[str, str]] = None,
                 routing: str = "softmax_all", weight_scale: float = 1.0, renormalize: bool = True, groups: int = 1,
                 keep_groups: Optional[int] = None, group_top: int = 1):
        modes = {"softmax_all": ops.ROUTE_SOFTMAX_ALL, "top_logits": ops.ROUTE_TOP_LOGITS, "sigmoid": ops.ROUTE_SIGMOID}
        if routing not in modes:
            raise ValueError(f"routing={routing!r}: one of {sorted(modes)}")
        self.mode, self.weight_scale = modes[routing], float(weight_scale)
        self.raw, self.groups, self.keep_groups = not renormalize, int(groups), int(groups if keep_groups is None else keep_groups)
        if self.raw and routing == "top_logits":
            raise ValueError("routing='top_logits' weighs by a softmax over the chosen: always normalised")
        outputs = experts + identity
        if not 1 <= self.groups <= ops.MOE_MAX_GROUPS or outputs % self.groups or not 1 <= self.keep_groups <= self.groups \
                or top > outputs // self.groups * self.keep_groups:
            raise ValueError(f"{outputs} router outputs in {groups} equal groups (at most {ops.MOE_MAX_GROUPS}) of which "
                             f"{self.keep_groups} are kept, {top} chosen")
        if group_top not in (1, 2):
            raise ValueError(f"group_top={group_top}: a group counts as much as its largest choice score or its two largest")
        self.group_top = int(group_top)
        limit = 0.0 if limit is None else limit            # the kernels read a limit of 0 as the plain unit
        if experts < 0 or identity < 0 or experts + identity < 1:
            raise ValueError(f"{experts} experts and {identity} identity experts: a router needs at least one output")
        if not 1 <= top <= experts + identity:
            raise ValueError(f"top={top} of {experts + identity} router outputs")
        if experts + identity > ops.MOE_MAX_ROUTER or top > ops.MOE_MAX_TOP:
            raise ValueError(f"at most {ops.MOE_MAX_ROUTER} router outputs and a top of {ops.MOE_MAX_TOP}")
        self.hidden_size, self.experts, self.identity, self.top = hidden_size, int(experts), int(identity), int(top)
        self.ff, self.limit, self.alpha = int(intermediate_size), float(limit), float(alpha)
        self.shared_ff = int(shared_size)
        self.shared_limit = float(shared_limit) if shared_limit is not None else self.limit
        self.has_correction = bool(correction)
        self.prefix = prefix
        self.names = {**DEFAULT_NAMES, **(names or {})}
        self.w_router = self.correction = self.w_gate_up = self.w_down = self.w_shared_gate_up = self.w_shared_down = None

    def kernel_families(self, dtype):
        return ("moe",)

    # ------------------------------------------------------------------ weights
    def _expert(self, index: int, role: str) -> str:
        return f"{self.prefix}.{self.names['expert'].format(index=index)}.{self.names[role]}"

    def _shared(self, role: str) -> str:
        return f"{self.prefix}.{self.names['shared']}.{self.names[role]}"

    def weights(self) -> List[WeightDecl]:
        p, H, I, R = self.prefix, self.hidden_size, self.ff, self.experts + self.identity
        out = [WeightDecl(f"{p}.{self.names['router']}", (R, H), keep_fp32=True)]
        if self.has_correction:
            out.append(WeightDecl(f"{p}.{self.names['correction']}", (R,), keep_fp32=True))
        for e in range(self.experts):
            out += [WeightDecl(self._expert(e, "gate"), (I, H), merged_into=f"{p}.experts.gate_up", row_offset=2 * I * e),
                    WeightDecl(self._expert(e, "up"), (I, H), merged_into=f"{p}.experts.gate_up", row_offset=2 * I * e + I),
                    WeightDecl(self._expert(e, "down"), (H, I), merged_into=f"{p}.experts.down", row_offset=H * e)]
        if self.shared_ff:
            S = self.shared_ff
            out += [WeightDecl(self._shared("gate"), (S, H), merged_into=f"{p}.shared.gate_up", row_offset=0),
                    WeightDecl(self._shared("up"), (S, H), merged_into=f"{p}.shared.gate_up", row_offset=S),
                    WeightDecl(self._shared("down"), (H, S))]
        return out

    def bind(self, tensors: Dict[str, torch.Tensor], env: PartEnv) -> None:
        p, H, I = self.prefix, self.hidden_size, self.ff
        self.w_router = tensors[f"{p}.{self.names['router']}"].contiguous()
        self.correction = tensors[f"{p}.{self.names['correction']}"].contiguous() if self.has_correction else None
        if self.experts:
            self.w_gate_up = tensors[f"{p}.experts.gate_up"].contiguous().view(self.experts, 2 * I, H)
            self.w_down = tensors[f"{p}.experts.down"].contiguous().view(self.experts, H, I)
        if self.shared_ff:
            self.w_shared_gate_up = tensors[f"{p}.shared.gate_up"].contiguous()
            self.w_shared_down = tensors[self._shared("down")].contiguous()

    # ------------------------------------------------------------------ the step
    def route(self, x: torch.Tensor):
        """(ids int32 [T, top], weights float32 [T, top]) of the rows of x."""
        if self.hidden_size <= ops.MOE_ROUTER_MAX_WIDTH:
            return ops.moe_router(x, self.w_router, self.correction, self.top, self.mode, self.weight_scale,     # the product and the routing in one
                                  self.groups, self.keep_groups, self.raw, self.group_top)
        logits = ops.gemm_simple(x, self.w_router, out_dtype=torch.float32)       # 32-bit sums in a fixed order
        return ops.moe_route(logits, self.correction, self.top, self.mode, self.weight_scale, self.groups, self.keep_groups,
                             self.raw, self.group_top)

    def forward(self, x: torch.Tensor, ctx: StepContext) -> torch.Tensor:
        return self.forward_onto(x, ctx, None, None)

    def forward_onto(self, x: torch.Tensor, ctx: StepContext, base: Optional[torch.Tensor],
                     bias: Optional[torch.Tensor] = None) -> torch.Tensor:
        """float32 [T, hidden]: ``base`` (another branch's output, or None) + ``bias`` + this feed-forward of x."""
        *products, shared = self._products(x, ctx)
        return ops.moe_combine(*products, base=base, bias=bias, shared=shared)

    def branch_onto(self, x: torch.Tensor, ctx: StepContext, base: Optional[torch.Tensor], mult: float) -> NormedBranch:
        """``forward_onto`` whose last kernel is left to whoever adds the branch to the stream."""
        if type(self).forward_onto is not RoutedExperts.forward_onto:      # a subclass that changes the sum
            return NormedBranch(self.forward_onto(x, ctx, base), None, mult)
        *products, shared = self._products(x, ctx)
        return SummedBranch(lambda: ops.moe_combine(*products, shared=shared, base=base),
                            lambda residual, alpha, gain, shift, m: ops.moe_combine_tanh(*products, residual, alpha, gain, shift, m, base=base,
                                                                                         shared=shared), x.dtype, mult)

    def _products(self, x: torch.Tensor, ctx: StepContext) -> tuple:
        """What the last kernel adds up: the experts' rows, x, ids, weights, every pair's slot, the experts' number, the shared expert's rows."""
        T = x.shape[0]
        ids, weights = self.route(x)
        y = None
        # in 32-bit a row is worked after the other whatever the tile: the fewer a tile, the more of them side by side
        tile_rows = product_rows_for(T, self.top, self.experts, *((self.hidden_size, self.ff) if x.dtype == torch.bfloat16 else (0, 0)))
        slot_of_pair = ids.view(-1)               # read for experts with weights only
        if self.experts:
            slot_of_pair, token_of_slot, tiles, _ = ops.moe_sort(ids, self.experts, tile_rows)
            act = ops.moe_rows(x, token_of_slot, self.w_gate_up, tiles, tile_rows, T * self.top, gated=True,
                               limit=self.limit, alpha=self.alpha)
            y = ops.moe_rows(act, None, self.w_down, tiles, tile_rows, T * self.top, gated=False)
        shared = None
        if self.shared_ff:
            # gate | up with the unit on store where the few-rows kernels take the step, as the dense feed-forward's
            act = gate_up(x, self.w_shared_gate_up, self.shared_limit, self.alpha)
            shared = linear(act, self.w_shared_down)
        return y, x, ids, weights, slot_of_pair, self.experts, shared
