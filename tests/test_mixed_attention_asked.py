"""Which steps ask for decoded tokens and prompt portions in one attention launch: those with heads that the launch takes."""
from types import SimpleNamespace

import pytest
import torch

from ullm_amd.kernels import ops


@pytest.mark.parametrize("hd,nq,nkv,asked", [(128, 16, 8, 1), (128, 32, 2, 1), (128, 17, 1, 0), (64, 16, 8, 0), (96, 4, 4, 0), (256, 8, 2, 0)])
def test_only_heads_that_it_takes(hd, nq, nkv, asked, monkeypatch):
    """CPU: the others go straight to the two launches."""
    calls = []
    monkeypatch.setattr(ops, "attention_mixed_mfma", lambda *a, **k: calls.append("mixed"))
    monkeypatch.setattr(ops, "attention_decode_mfma", lambda *a, **k: calls.append("decode"))
    monkeypatch.setattr(ops, "attention_prefill_mfma", lambda *a, **k: calls.append("prefill"))
    facts = dict(num_decode=3, num_tiles=2, decode_keys=30, max_decode_kv=20, tile_keys_total=64, tile_keys_max=32)
    plan = SimpleNamespace(facts=facts, arrays=dict(decode_tokens=None, tiles=None))
    q = torch.empty(8, nq * hd, dtype=torch.bfloat16)
    ops.paged_attention(q, None, None, SimpleNamespace(positions=None, token_entry=None), SimpleNamespace(block_table=None, page_size=16), nq, nkv, hd,
                        1.0, 0, plan=plan)
    assert calls == ["mixed"] * asked + ["decode", "prefill"]
