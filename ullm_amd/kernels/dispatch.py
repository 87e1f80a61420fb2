"""Which product kernel a projection takes, by its number of rows and its matrix.

Every choice between the hand-written product kernels and the library is asked here.  All but one are limits of rows: up to how
many (for the large product in which ranges of thousands of) rows of the batch a kernel is ahead for a matrix of
``columns`` x ``inner``; the large product with the gated unit goes by how full its blocks' rounds are
(:func:`gated_tile_groups`).  The limits of a matrix come from a table
of measurements (``tuned_gfx950.json`` beside this file, written by
``python -m ullm_amd.kernels.microbench tune --columns N --inner K``), and for a matrix the table does not hold
from rules in terms of the matrix's size alone.  Parts ask :func:`limits`; none of them names a model or carries
a threshold of its own.  A limit only ever selects among kernels that compute the same function, and every
kernel's own ``*_supports`` check still decides whether it can take the operands at all, so a wrong or missing
entry costs time, never a result.
"""
from __future__ import annotations

import functools
import json
import os
from dataclasses import asdict, dataclass, fields
from typing import Dict, Optional, Tuple

from . import build

TABLE_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuned_gfx950.json")


@dataclass(frozen=True)
class Limits:
    """Row limits of one weight matrix [columns, inner] (for gate|up: columns = 2 x intermediate).  From 17 rows on they say which kernel
    takes a product that the panels kernel (:func:`panels`) does not: inner sizes that are no whole stages of 64, small matrices, the rows
    of the ``kept`` fields and more blocks than fit a round."""
    # y = x W^T in bfloat16: the few-rows kernel up to ``skinny`` rows, then the rows kernel up to ``rows``
    # (0: never), then the library
    skinny: int = 16
    rows: int = 64
    # the RMS norm before the product folded into the few-rows kernel up to this many rows (asked where the product
    # before has not prepared the norm: a model's first layer, a part behind one that adds no result of its own)
    fold_norm: int = 8
    # silu(gate) * up on store: the few-rows kernel up to ``silu_skinny``, the rows kernel up to ``silu_rows``,
    # then the library product and the activation kernel
    silu_skinny: int = 16
    silu_rows: int = 64
    # a product whose result the next norm adds to the stream: as a stack of partial sums over slices of the
    # inner dimension from ``stacked_from`` to ``stacked_to`` rows (0, 0: never)
    stacked_from: int = 17
    stacked_to: int = 256
    # y = x W^T in bfloat16 above ``skinny`` and ``rows``: partial sums over slices of the inner dimension and a
    # kernel that adds them, from ``sums_from`` to ``sums_to`` rows (0, 0: never; only measured matrices have it)
    sums_from: int = 0
    sums_to: int = 0
    # y = x W^T over thousands of rows: the framework's large product (``ops.gemm_tiles``) in these ranges of rows, (first,
    # last) each, where the library's choices fall off (only measured matrices have any)
    tiles: Tuple[Tuple[int, int], ...] = ()
    # ranges of rows, (first, last) each, that the kernels named above keep because they were measured to be ahead of the panels kernel
    # there, for the three kinds of product; None: not measured (the rows of ``sums_from`` .. ``sums_to`` then stay with the partial sums,
    # :func:`_rows_kernel_ahead` and :func:`_library_ahead` answer for the others)
    store_kept: Optional[Tuple[Tuple[int, int], ...]] = None
    silu_kept: Optional[Tuple[Tuple[int, int], ...]] = None
    stream_kept: Optional[Tuple[Tuple[int, int], ...]] = None
    # 32-bit results (the logits head): the few-rows kernel up to here, then the library
    f32_skinny: int = 16


def default_limits(columns: int, inner: int) -> Limits:
    """The rules for a matrix that was not measured, in terms of its size alone.  They follow what the
    measured matrices (2 M to 780 M elements) have in common: the rows kernel needs enough columns to give
    every compute unit a block; a small matrix has few blocks to pay for 32-bit rows of X, so the norm stays
    folded in for every row count the kernel takes; gate|up keeps the few-rows kernel to 32 rows unless the
    matrix is very large, and the rows kernel to 128 rows from 12 288 result columns on; stacks of partial sums outweigh a matrix of a few M elements; the few-rows kernel
    with four tiles a block is ahead of the library up to 32 rows on matrices with very many columns."""
    weight = columns * inner
    return Limits(
        skinny=16,
        rows=64 if columns >= 2048 else 0,
        fold_norm=16 if weight <= (40 << 20) else 8,
        silu_skinny=32 if weight <= 200_000_000 else 16,
        silu_rows=(128 if columns // 2 >= 12288 else 64) if columns // 2 >= 2048 else 0,
        stacked_from=17 if weight >= (8 << 20) else 0,
        stacked_to=256 if weight >= (8 << 20) else 0,
        f32_skinny=32 if columns >= 65536 else 16)


def _ranges(text: str) -> Tuple[Tuple[int, int], ...]:
    """``"8256-8960 11840-12544"`` as ((8256, 8960), (11840, 12544))."""
    return tuple((int(a), int(b)) for a, b in (r.split("-") for r in text.split()))


RANGES = ("tiles", "store_kept", "silu_kept", "stream_kept")          # written as text in the table
_table: Optional[dict] = None


def _load() -> dict:
    global _table
    if _table is None:
        table: Dict[str, Limits] = {}
        if os.path.isfile(TABLE_PATH):
            with open(TABLE_PATH, "r", encoding="utf-8") as f:
                raw = json.load(f)
            names = {f.name for f in fields(Limits)}
            for key, entry in raw.get("matrices", {}).items():
                try:
                    columns, inner = (int(x) for x in key.split("x"))
                except ValueError:
                    raise ValueError(f"{TABLE_PATH}: key {key!r} is not COLUMNSxINNER") from None
                base = asdict(default_limits(columns, inner))
                base.update({k: _ranges(v) if k in RANGES else int(v) for k, v in entry.items() if k in names})
                table[key] = Limits(**base)
        _table = table
    return _table


def limits(columns: int, inner: int) -> Limits:
    """The row limits of a weight matrix [columns, inner]: measured ones where the table has the matrix,
    the size rules otherwise."""
    table = _load()
    found = table.get((columns, inner))                    # by a tuple: this is asked for every projection of every step
    if found is None:
        found = table.get(f"{columns}x{inner}")
        if found is None:
            return default_limits(columns, inner)
        table[(columns, inner)] = found
    return found


def is_tuned(columns: int, inner: int) -> bool:
    return f"{columns}x{inner}" in _load()


def write_entry(columns: int, inner: int, fields_measured: Dict[str, object]) -> None:
    """Put the measured limits of one matrix into the table file (used by ``microbench tune``); fields that
    were not measured for it are left to the size rules."""
    global _table
    names = {f.name for f in fields(Limits)}
    unknown = set(fields_measured) - names
    if unknown:
        raise KeyError(f"no such limits: {sorted(unknown)}")
    raw = {"device": "gfx950", "matrices": {}}
    if os.path.isfile(TABLE_PATH):
        with open(TABLE_PATH, "r", encoding="utf-8") as f:
            raw = json.load(f)
    entry = raw.setdefault("matrices", {}).setdefault(f"{columns}x{inner}", {})
    entry.update({k: " ".join(f"{a}-{b}" for a, b in v) if k in RANGES else int(v) for k, v in fields_measured.items()})
    with open(TABLE_PATH, "w", encoding="utf-8") as f:
        json.dump(raw, f, indent=1, sort_keys=True)
        f.write("\n")
    _table = None
    panels.cache_clear()


PANELS_STORE, PANELS_GATED, PANELS_FLOAT = 0, 1, 2
PANELS_MIN_ROWS = 17          # up to 16 rows the few-rows kernel, which folds what stands around the product into itself
PANELS_MIN_WEIGHT = 1 << 20   # values of the smallest matrix it was measured on
PANELS_MAX_SLICES = 8
SUM_US = 4.0                  # the kernel that adds slices: its launch and the trip to memory


@functools.lru_cache(maxsize=8192)           # of sizes alone, and asked for by every layer of every step
def _panels_plan(rows: int, columns: int, inner: int, mode: int, max_slices: int, rounds: bool = False) -> Tuple[int, float]:
    """The panels kernel's plan and its estimated us; a plan of -1 where it does not take the product or (unless ``rounds``) its
    blocks need more than one round."""
    plan = int(build.load("gemm_panels").ullm_gemm_panels_plan(rows, columns, inner, mode, max_slices))
    if plan < 0 or (plan >> 16 & 1 and not rounds):
        return -1, 0.0
    return plan & 0xffff, (plan >> 17) / 8


ROWS_AHEAD_ROWS, ROWS_AHEAD_WEIGHTS, ROWS_AHEAD_COLUMNS, ROWS_AHEAD_BLOCKS = 48, (13_000_000, 64_000_000), 4096, 230


def _rows_kernel_ahead(rows: int, columns: int, inner: int, plan: int, mode: int) -> bool:
    """Whether the rows kernel, where it is what takes the call, is ahead of the panels kernel's plan in one slice, for matrices that were
    not measured: those of 13 to 64 M values and more than 4096 columns at up to 48 rows whose plan leaves a tenth of the compute units and more
    without a block.
    Such a product is a read of W by the units that have one, while the rows kernel gives every unit as many columns (us, the
    rows kernel and this: 5120 x 5120 at 17 / 32 / 48 rows 14.2 / 14.9 / 19.2 and 15.8 / 17.7 / 20.8, 5120 x 3072 at 17 / 32 9.8 / 10.0 and 11.4 / 11.0, with
    an activation 10240 x 2560 at 36 / 48
    14.5 / 15.6 and 16.5 / 17.3, 11008 x 4096 21.5 / 21.4 and 24.4 / 23.4, 12288 x 3072 18.3 / 18.0 and 19.5 / 19.6; gate|up 19456 x 2560 20.5 /
    21.2 and 22.4 / 23.2).  Smaller matrices are read in time by fewer units (4096 x 4096 at 40 rows 14.6 and 11.5, 5120 x 2048 level, 4096 x
    6144 and 4096 x 8192 at 17 to 48 0.68 to 0.93 of the rows kernel's time), larger ones bound by memory
    either way (gate|up 22016 x 4096 at 48 rows 10 % behind, 16384 x 4096 9 %)."""
    lim, weight = limits(columns, inner), columns * inner
    few, most = (lim.silu_skinny, lim.silu_rows) if mode == PANELS_GATED else (lim.skinny, lim.rows)
    return (few < rows <= min(most, ROWS_AHEAD_ROWS) and ROWS_AHEAD_WEIGHTS[0] <= weight < ROWS_AHEAD_WEIGHTS[1]
            and columns > ROWS_AHEAD_COLUMNS and plan >> 8 == 1
            and build.load("gemm_panels").ullm_gemm_panels_blocks(rows, columns, mode, plan & 0xff, 1) < ROWS_AHEAD_BLOCKS)


def _library_ahead(rows: int, columns: int, inner: int) -> bool:
    """Whether the library is ahead of the panels kernel for a matrix of few columns that was not measured: up to 1024 of them and 1536 to 3072
    values a row, from 513 rows on, where the panels' tiles make one or two hundred blocks that each walk
    half of K or all of it (time of the panels kernel over the library's at 400 / 640 / 900 rows: 768 x 2560 1.03 / 1.12 / 1.23, 1024 x 2048 0.89 / 1.05 /
    1.22; 1024 x 1024 0.69 / 0.87 / 0.94, 1024 x 4096 0.86 / 0.99 / 1.03, 2048 x 2048 0.88 / 0.92 / 1.06).  1536 x 2048 (1.10 / 1.17 / 1.07) and
    sums that the stream adds (1024 x 2048 0.98 / 1.11 / 1.20) are left as they are: alike layers launched together take the panels kernel there,
    as launches are what takes the time, and have the bits of the layers one by one."""
    return columns <= 1024 and 1536 <= inner <= 3072 and rows > 512


@functools.lru_cache(maxsize=8192)
def panels(rows: int, columns: int, inner: int, role: str, keep_sums: bool = False, host_bound: bool = False,
           whole: bool = False) -> Tuple[int, int]:
    """The plan by which the panels kernel (``ops.gemm_panels``) takes x [rows, inner] times W [columns, inner], and its mode; a plan of -1
    where another product is ahead.  Roles: ``store`` (a bfloat16 result; in float mode the slices are added by a kernel),
    ``activated`` (the same with an activation on store), ``gated`` (W is gate | up), ``stream`` (a result that the next norm adds: bfloat16, or slices' 32-bit sums; with
    ``keep_sums`` always the sums; where what follows wants it ``whole``, slices only if they make up for the kernel that adds them: 48 x
    2048 x 2048 in one slice 5.0 us, in four 4.4 and 4.8 to add them) and ``float`` (the 32-bit sums as they are, one slice: logits, branches).

    It is taken from 17 rows on while its blocks fit one round of the chip: there its tiles fill it (us, what took the calls
    before and this: gate|up 24576 x 4096 at 17 / 64 / 256 rows 36 / 43 / 64 and 32 / 36 / 58; 6144 x 1024 at 40 / 256 / 800 7.9 / 15.1 / 17.3 and
    5.8 / 9.6 / 15.0; 4096 x 12288 into the stream at 130 / 512 / 1024 30.6 / 83 / 118 and 26.4 / 51 / 94; 6144 x 4096 at 64 / 256 / 1024 17.8 / 31 / 53
    and 16.8 / 25.7 / 53.3).  In two rounds the library's tiles are ahead (6144 x 4096 at 1300 rows 65 and 83, gate|up 24576 x 4096 at 320
    79 and 87), and from 1025 rows on also in one (1024 x 3072 at 1300 / 2048 rows 17.2 / 20.0 and 20.4 / 24.1, 2048 x 2048 at 2048 / 3000
    21.0 / 26.5 and 23.0 / 27.6; inside a prompt of 1064 rows 6144 x 4096 59 and 63, 4096 x 4096 and 4096 x 12288 183 and 189 together,
    the prompt 17.9 and 18.4 ms; level at 2048).  Rows for which the kernels that took the calls before were measured to be ahead, or
    for matrices that were not measured are expected to be (:func:`_rows_kernel_ahead`, :func:`_library_ahead`), are left to them.  Neither holds where ``host_bound``
    says that launches are what takes the time."""
    if rows < PANELS_MIN_ROWS or columns * inner < PANELS_MIN_WEIGHT or (rows > 1024 and not host_bound):
        return -1, 0
    plan, mode = _panels_of_role(rows, columns, inner, role, keep_sums, whole)
    if plan < 0 or host_bound or role == "float":
        return plan, mode
    lim = limits(columns, inner)
    kept = getattr(lim, {"gated": "silu_kept", "stream": "stream_kept"}.get(role, "store_kept"))
    if any(first <= rows <= last for first, last in kept or ()):
        return -1, 0
    if kept is None and role == "store" and lim.sums_from > 0 and lim.sums_from <= rows <= lim.sums_to:
        return -1, 0                                       # named for the partial sums, not compared with this kernel
    if kept is None and role != "stream" and mode != PANELS_FLOAT and _rows_kernel_ahead(rows, columns, inner, plan, mode):
        return -1, 0
    if kept is None and (role == "store" or role == "stream" and whole) and _library_ahead(rows, columns, inner):
        return -1, 0
    return plan, mode


def _panels_of_role(rows: int, columns: int, inner: int, role: str, keep_sums: bool, whole: bool) -> Tuple[int, int]:
    """The panels kernel's fastest plan for a role, and its mode."""
    if role == "float":
        # logits heads are read once at these rows, in however many rounds (library and this: 151936 x 4096 at 17 / 64 / 128 rows 266 / 270 /
        # 290 and 192 / 223 / 268, 151936 x 1024 at 101 91 and 81, 32768 x 2048 at 48 / 256 37 / 46 and 25 / 41); smaller matrices go to the
        # library sooner than where the result is rounded (2048 x 2048 at 300 / 600 / 1024 rows 10.8 / 13.1 / 15.4 and 10.3 / 13.2 / 17.2, 4096 x 2048
        # at 600 / 1024 23 / 26 and 18 / 23)
        if rows <= (256 if columns >= 16384 else 1024 if columns >= 4096 else 512):
            return _panels_plan(rows, columns, inner, PANELS_FLOAT, 1, columns >= 16384)[0], PANELS_FLOAT
        return -1, 0
    if role == "gated":
        return _panels_plan(rows, columns, inner, PANELS_GATED, 1)[0], PANELS_GATED
    if role == "activated":                          # the 32-bit sums are one block's: an activation of added slices would see them rounded
        return _panels_plan(rows, columns, inner, PANELS_STORE, 1)[0], PANELS_STORE
    sums, sums_us = _panels_plan(rows, columns, inner, PANELS_FLOAT, PANELS_MAX_SLICES)
    one, one_us = _panels_plan(rows, columns, inner, PANELS_FLOAT, 1) if whole else (-1, 0.0)
    added = one if 0 <= one and one_us <= sums_us + SUM_US else sums          # as 32-bit sums
    if role == "stream" and keep_sums:
        return added, PANELS_FLOAT
    stored, stored_us = _panels_plan(rows, columns, inner, PANELS_STORE, 1)
    stored_us += rows * columns * 2 / 5e6 if role == "stream" else 0.0
    if sums >= 0 and sums_us + (SUM_US if role == "store" else 0.0) < stored_us or stored < 0:
        return added, PANELS_FLOAT
    return stored, PANELS_STORE


def gated_tile_groups(rows: int, columns: int, inner: int) -> int:
    """The 64-row groups a block of the large product should take for x [rows, inner] times gate|up [columns, inner] with the
    unit on store (``ops.gemm_tiles``), or 0 where the library's product and the activation kernel behind it are ahead.

    The activation's pass is saved, worth the more the shorter ``inner`` is, and what decides is how full the rounds of blocks
    over 256 compute units are, rows and columns of the last tiles included (a round of 128-row tiles takes 0.65 of one of 256
    rows).  The lines are laid through eleven matrices (inner sizes of 1024 to 8192) at 160 to 8000 rows, library and this,
    us, with the share of the rounds: 24576 x 4096 at 256 / 300 / 1024 / 1150 / 2048 / 3000 / 6000 rows 67 / 76 / 169 / 190 / 292 / 593 / 853
    and 66 / 91 / 170 / 189 / 293 / 445 / 858, shares of 0.58, 0.44, 0.75 (two rounds), 0.84, 1, 0.88, 0.98; 12288 x 2048 at 450 /
    768 / 850 / 1150 35 / 44 / 48 / 58 and 31 / 49 / 47 / 50, 0.51, 0.56, 0.62, 0.84; 9728 x 2560 at 1150 / 1300 59 / 67 and 63 / 65,
    0.67, 0.75; 6144 x 1024 at 512 / 700 / 1300 / 3000 / 4096 17 / 20 / 26 / 48 / 61 and 17 / 17 / 25 / 48 / 51, 0.29, 0.39, 0.48, 0.56 (two
    rounds), 0.77; 8192 x 8192 at 2048 / 6000 187 / 547 and 198 / 578: the pass is 5 % of the product there, and the library's
    product alone 5 to 10 % ahead.  Whole prompts of an 8B model whose gate|up takes the one and the other: 512 rows 10.33 and
    10.36 ms, 2048 27.0 and 26.4, 3000 43.7 and 39.1, 6000 80.3 and 80.3."""
    if rows < 160 or columns < 1 or inner > 6144:
        return 0

    def rounds(groups):
        return -(-(-(-rows // (64 * groups)) * -(-columns // 256)) // 256)
    groups, cost = min(((4, rounds(4)), (2, 0.65 * rounds(2))), key=lambda c: c[1])
    short = min(1.0, 1024 / inner)
    if rounds(groups) > 1:
        least = 0.84 - 0.27 * short
    else:
        least = 0.62 - 0.27 * short if groups == 2 else min(0.72, 0.3 + 0.15 * inner / 1024)
    return groups if rows * columns / (2 ** 24 * cost) >= least else 0
