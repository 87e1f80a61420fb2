"""Steps with prompt portions whose layers are launched from native code: the bits of the blocks' own forward passes, over every way
their products, attention and branches go; and what is left to the blocks."""
import ctypes

import pytest
import torch

DEV = "cuda:0"
# width, heads, kv heads, head size, inner size, bias, window
SIZES = {"plain": (1024, 8, 4, 128, 1024, False, 0), "wide": (1024, 16, 8, 128, 3072, True, 0), "window": (2048, 8, 8, 64, 1024, True, 40)}
LARGE = (4096, 32, 8, 128, 12288, True, 0)


def test_the_structures_agree():
    """CPU: the step and the layers as the caller lays them out are as long as the callee's."""
    from ullm_amd.kernels import build, dense
    lib = build.load("dense_layers")
    assert lib.ullm_dense_step_bytes() == ctypes.sizeof(dense.Step)
    assert lib.ullm_dense_layer_bytes() == 8 * len(dense.LAYER_FIELDS)


def test_which_layers_are_alike():
    """CPU: layers of other sizes, windows or kinds end a run."""
    from ullm_amd.models import build_model
    from ullm_amd.parts.dense import alike_layers, layer_form
    cfg = dict(architectures=["Qwen3ForCausalLM"], hidden_size=64, num_hidden_layers=4, num_attention_heads=4, num_key_value_heads=2,
               head_dim=32, intermediate_size=128, vocab_size=256, rope_theta=10000.0, rms_norm_eps=1e-6, max_position_embeddings=128)
    blocks = build_model(cfg)[1].blocks
    assert alike_layers(blocks) == 4 and alike_layers(blocks[:1]) == 1 and alike_layers([]) == 0
    blocks[2].mixer.reach = 16
    assert alike_layers(blocks) == 2
    blocks[1].ffn.__class__ = type("Other", (type(blocks[1].ffn),), {})
    assert layer_form(blocks[1]) is None and alike_layers(blocks) == 1
    blocks[0].mixer_norm.add_norm = blocks[0].mixer_norm.add_norm              # a method of the part's own
    assert alike_layers(blocks) == 0


def _runner(size, seed):
    from ullm_amd.engine.loading import make_env
    from ullm_amd.engine.runner import ModelRunner
    from ullm_amd.models import build_model
    from ullm_amd.weights.random_init import bind_random_weights
    H, nq, nkv, hd, inner, bias, window = LARGE if size == "large" else SIZES[size]
    cfg = dict(architectures=["Qwen3ForCausalLM"], hidden_size=H, num_hidden_layers=3, num_attention_heads=nq, num_key_value_heads=nkv,
               head_dim=hd, intermediate_size=inner, vocab_size=512, rope_theta=10000.0, rms_norm_eps=1e-6, max_position_embeddings=4096,
               tie_word_embeddings=False, attention_bias=bias, use_sliding_window=window > 0, sliding_window=window or None,
               max_window_layers=0)
    _, model = build_model(cfg)
    env = make_env("bfloat16", DEV, 2048)
    bind_random_weights(model, env, seed)
    return ModelRunner(model, env, 16, 600, 24)


def _steps(runner, seed):
    """The logits of steps of prompts, of portions beside single tokens, and of what is left of the portions."""
    from ullm_amd.engine.runner import StepEntry
    g = torch.Generator().manual_seed(seed)
    draw = lambda n: torch.randint(0, 512, (n,), generator=g).tolist()      # noqa: E731
    cache, out = runner.cache, []

    def step(work):
        entries = []
        for rc, n in work:
            assert cache.reserve(rc, n)
            entries.append(StepEntry(rc, draw(n), [0, n - 1] if n > 1 else [0]))
        out.append(runner.step(entries).clone())
    live = [cache.admit(f"r{i}") for i in range(20)]
    step([(live[0], 17)])                                                   # the fewest rows
    step([(live[1], 130), (live[2], 3)])
    step([(live[3], 700), (live[4], 250)])                                  # as many rows as some products are ahead for
    step([(rc, 1) for rc in live[:3]] + [(live[5], 40)])
    step([(rc, 1) for rc in live[:5]] + [(live[5], 300)] + [(rc, 2) for rc in live[6:20]])
    step([(rc, 1) for rc in live[6:20]] + [(live[3], 33), (live[5], 9)])
    for rc in live:
        cache.release(rc)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("size", sorted(SIZES))
def test_the_blocks_bits(size, monkeypatch):
    from ullm_amd.kernels import dense
    from ullm_amd.models import model as models
    calls, real = [], dense.dense_layers
    monkeypatch.setattr(dense, "dense_layers", lambda step, layers: calls.append((step.tokens, step.into.mode, step.down.mode)) or real(step, layers))
    got = _steps(_runner(size, 5), 9)
    # the few kernels of the smallest product's matrix size aside, every step's layers were launched at once
    assert [t for t, _, _ in calls] == [17, 133, 950, 43, 333, 56]
    assert {mode for _, _, mode in calls} >= {2}
    monkeypatch.setattr(models, "run_layers", lambda *a: None)
    want = _steps(_runner(size, 5), 9)
    assert len(calls) == 6 and all(torch.isfinite(w).all() for w in want)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def _logits(runner, *steps):
    """The last tokens' logits of steps of as many tokens for one request each."""
    from ullm_amd.engine.runner import StepEntry
    cache, out, entries = runner.cache, [], []
    for counts in steps:
        entries = [StepEntry(cache.admit(f"r{i}"), [(13 * j + i) % 512 for j in range(n)], [n - 1]) for i, n in enumerate(counts)]
        assert all(cache.reserve(e.cache, len(e.tokens)) for e in entries)
        out.append(runner.step(entries).clone())
        for e in entries:
            cache.release(e.cache)
    return out


@pytest.mark.gpu
def test_the_blocks_bits_by_every_way_of_the_products(monkeypatch):
    """A width of 4096 with biases: q|k|v in slices that a kernel adds with the bias, gate|up by the large tiles beside panels, all four
    products by the large tiles."""
    from ullm_amd.kernels import dense
    from ullm_amd.models import model as models
    ways, real = [], dense.dense_layers
    monkeypatch.setattr(dense, "dense_layers", lambda step, layers: ways.append([(p.tiles, p.mode) for p in (
        step.into, step.out, step.gate_up, step.down)]) or real(step, layers))
    steps = ([90, 40], [512], [2040] * 4 + [200])
    got = _logits(_runner("large", 6), *steps)
    store, gated, sums = ((0, mode) for mode in range(3))
    assert ways == [[sums, sums, gated, sums], [store, sums, (1, 1), sums], [(1, 0), (1, 0), (1, 1), (1, 0)]]
    monkeypatch.setattr(models, "run_layers", lambda *a: None)
    for a, b in zip(got, _logits(_runner("large", 6), *steps)):
        assert torch.isfinite(b).all() and torch.equal(a, b)


@pytest.mark.gpu
def test_launches_that_take_longer_than_the_products(monkeypatch):
    """Steps of 1025 to about 1200 rows of a small width take panels that the blocks leave to the library: not its bits, so against the
    blocks' with the roundings of three layers of bfloat16 between them (2^-9 each of q|k|v, heads, activation, branch: a dozen of 2^-9
    at most add up to 2.4 %, by chance 0.7 %)."""
    from ullm_amd.kernels import dense
    from ullm_amd.models import model as models
    rows, real = [], dense.dense_layers
    monkeypatch.setattr(dense, "dense_layers", lambda step, layers: rows.append((step.tokens, step.into.tiles)) or real(step, layers))
    steps = ([1025], [700, 500])
    got = _logits(_runner("wide", 7), *steps)
    assert rows == [(1025, 0), (1200, 0)]
    monkeypatch.setattr(models, "run_layers", lambda *a: None)
    for a, b in zip(got, _logits(_runner("wide", 7), *steps)):
        assert (a - b).norm() <= 2.4e-2 * b.norm()


@pytest.mark.gpu
def test_what_is_left_to_the_blocks(monkeypatch):
    """16 rows, single tokens, a step whose branches are not to come as sums, a matrix that lies off 16 bytes: the blocks' own forward passes."""
    from ullm_amd.engine.runner import StepEntry
    from ullm_amd.kernels import dense
    calls, real = [], dense.dense_layers
    monkeypatch.setattr(dense, "dense_layers", lambda step, layers: calls.append(step.tokens) or real(step, layers))
    runner = _runner("plain", 3)
    cache = runner.cache
    rcs = [cache.admit(f"r{i}") for i in range(5)]

    def step(*counts):
        entries = [StepEntry(rc, [7] * n, [n - 1]) for rc, n in zip(rcs, counts) if n]
        assert all(cache.reserve(e.cache, len(e.tokens)) for e in entries)
        return runner.step(entries).clone()
    step(16)
    step(1, 0, 0, 0)
    assert not calls
    runner._stacked_branches = False
    step(0, 0, 0, 0, 40)
    assert not calls
    runner._stacked_branches = True
    step(0, 40)
    assert calls == [40]
    mixer = runner.model.blocks[1].mixer
    room = torch.empty(mixer.w_o.numel() + 1, dtype=torch.bfloat16, device=DEV)
    room[1:] = mixer.w_o.flatten()
    aligned, mixer.w_o = mixer.w_o, room[1:].view_as(mixer.w_o)
    a = step(0, 0, 40)
    assert calls == [40]
    mixer.w_o = aligned
    b = step(0, 0, 0, 40)
    assert calls == [40, 40] and (a - b).abs().max() <= 3e-2 * b.abs().max()
    for rc in rcs:
        cache.release(rc)


def _scaled(model):
    model.blocks[1].mixer.scale *= 2.0


def _narrowed(model):
    model.blocks[2].mixer.reach = 24


def _other_eps(model):
    model.blocks[1].ffn_norm.eps = 1.0


def _wrapped(model):
    part = model.blocks[1].ffn
    real = part.forward
    part.forward = lambda x, ctx: real(x * 2, ctx)


def _shorter(model):
    model.run_order = model.run_order[:2]


@pytest.mark.gpu
@pytest.mark.parametrize("change", [_scaled, _narrowed, _other_eps, _wrapped, _shorter])
def test_layers_changed_after_the_model_was_built(change, monkeypatch):
    """A run takes the layers as they are when the step comes: what was exchanged in one of them is not run with the first one's numbers."""
    from ullm_amd.engine.runner import StepEntry
    from ullm_amd.models import model as models

    def logits():
        runner = _runner("plain", 4)
        rc, out = runner.cache.admit("r"), []
        for k in range(2):
            assert runner.cache.reserve(rc, 60)
            out.append(runner.step([StepEntry(rc, [(11 * i + k) % 512 for i in range(60)], [59])]).clone())
            if k == 0:
                change(runner.model)
        return out
    got = logits()
    monkeypatch.setattr(models, "run_layers", lambda *a: None)
    want = logits()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
