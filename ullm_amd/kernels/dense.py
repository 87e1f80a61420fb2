"""The Python face of ``csrc/dense_layers.hip``: the launches of a run of alike layers from one native call."""
from __future__ import annotations

import ctypes
from typing import Dict, Sequence

import numpy as np

from . import build, ops

_ptr, _int, _float, _long = ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_longlong
# the entry points the run calls, in the order of the structure's first fields
LAUNCHERS = (("elementwise", "ullm_add_rmsnorm"), ("elementwise", "ullm_sum_stacks"), ("elementwise", "ullm_qk_norm_rope_write"),
             ("elementwise", "ullm_qk_norm_rope_write_sums"), ("gemm_panels", "ullm_gemm_panels"), ("gemm_tiles", "ullm_gemm_tiles"),
             ("attention_mfma", "ullm_attention_decode"), ("attention_mfma", "ullm_attention_prefill"),
             ("attention_mfma", "ullm_attention_mixed"))
LAYER_FIELDS = ("norm1", "q_gain", "k_gain", "cos_sin", "b_qkv", "norm2", "w_qkv", "w_o", "w_gate_up", "w_down", "k_pool", "v_pool",
                "block_table", "bt_stride", "write_kv")          # of 8 bytes each


class Product(ctypes.Structure):
    """``tiles``: 0 the panels kernel in ``shape`` and ``slices``, 1 the large tiles of ``shape`` 64-row groups."""
    _fields_ = [("tiles", _int), ("mode", _int), ("shape", _int), ("slices", _int)]


class Step(ctypes.Structure):
    _fields_ = ([(name, _ptr) for _, name in LAUNCHERS]
                + [(name, _ptr) for name in ("residual", "normed", "qkv", "q", "attended", "act", "sums", "decode_parts", "mixed", "fed",
                                             "positions", "token_entry", "decode_tokens", "prompt_tiles", "wide_tiles")]
                + [("tile_keys_total", _long), ("wide_keys_total", _long), ("decode_keys_total", _long)]
                + [(name, Product) for name in ("into", "out", "gate_up", "down")]
                + [(name, _int) for name in ("tokens", "width", "heads", "kv_heads", "head_dim", "inner",
                                             "table_rows", "rot", "style", "page_size", "window", "num_decode", "decode_splits",
                                             "decode_waves", "num_tiles", "tile_keys_max", "num_wide", "wide_keys_max", "decode_keys_max")]
                + [(name, _float) for name in ("eps1", "eps2", "qk_eps", "scale")])


_addresses: Dict[str, int] = {}


def dense_layers(step: Step, layers: Sequence[Sequence[int]]) -> None:
    """Launches the layers' work on torch's current stream.  ``layers``: every layer's fields as LAYER_FIELDS has them.  What the
    fields point to is the caller's to check; it must stay alive until the launches are queued, as for any launch."""
    if not _addresses:
        _addresses.update({name: ctypes.cast(getattr(build.load(family), name), _ptr).value for family, name in LAUNCHERS})
    for name, address in _addresses.items():
        setattr(step, name, address)
    table = np.array(layers, dtype=np.int64)
    if table.ndim != 2 or table.shape[1] != len(LAYER_FIELDS):
        raise ops.KernelError("every layer has one number a field")
    ops._check(build.load("dense_layers").ullm_dense_layers(ctypes.byref(step), _ptr(table.ctypes.data), table.shape[0], ops._stream()),
               "dense_layers")
