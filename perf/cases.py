"""The workloads this engine's speed is judged on, each one pass through the step function that generation and trace
replay drive: requests admitted to the cache manager, `ModelRunner.step` over their tokens, logits out, requests released.

Models are the named sizes of `ullm_amd/config/presets` at full depth with weights drawn here: Qwen3 dense, which the
benchmark is quoted on, and the two stacks that between them use routed feed-forwards, every recurrence that keeps a
matrix state, and attention under windows, chunks and sinks.  Four kinds of pass:

  prompts   new requests' prompts, all in one step; the logits behind each prompt's last token (scoring, time to first token)
  decode    live requests (their prompts' pages shared through the prefix tree) for some steps of one token each
  mixed     steps that hold one token of every live request beside a portion of a new request's long prompt
  serve     new requests from their prompts through some steps of one token each (models whose state is no page to share)

Tokens are given, not sampled, so that two implementations that round differently still walk the same path.  Routers are
drawn so that a token's experts stand clear of the others, as a trained router's do: else the choice would hang on rounding.
"""
import json
import math
import os
import zlib

import torch

import ullm_amd
from ullm_amd.engine.loading import make_env
from ullm_amd.engine.runner import ModelRunner, StepEntry
from ullm_amd.models import build_model
from ullm_amd.weights.loader import merged_tensors, unique_decls

PAGE = 16
DEVICE = "cuda:0"
F = torch.float64
STEP_TOKENS = 8192          # prompts ahead of the measured steps go in steps of at most this many tokens


def listed():
    return [
        # one user waiting for the next token of a small model: launches and latency
        dict(name="decode_small_b1", kind="decode", model="qwen3-0.6b", dtype="bfloat16", batch=1, context=1024, steps=16),
        # the benchmark's headline: eight conversations of a thousand tokens
        dict(name="decode_b8", kind="decode", model="qwen3-8b", dtype="bfloat16", batch=8, context=1024, steps=8),
        # a busy server's decode step: ragged contexts, the weights shared by 64 rows
        dict(name="decode_b64", kind="decode", model="qwen3-8b", dtype="bfloat16", batch=64, context=768, steps=4),
        # long documents: the cache outweighs the weights
        dict(name="decode_long", kind="decode", model="qwen3-0.6b", dtype="bfloat16", batch=15, context=8192, steps=8),
        # a few short chat turns at once: rows between the few-rows kernels and the large products
        dict(name="prompts_short", kind="prompts", model="qwen3-8b", dtype="bfloat16", count=3, tokens=130),
        # the benchmark's prompt
        dict(name="prompt_2048", kind="prompts", model="qwen3-8b", dtype="bfloat16", count=1, tokens=2048),
        # a long document read in one step
        dict(name="prompt_long", kind="prompts", model="qwen3-8b", dtype="bfloat16", count=1, tokens=12000),
        # continuous batching: decoding requests beside portions of a newcomer's prompt
        dict(name="mixed_b100", kind="mixed", model="qwen3-0.6b", dtype="bfloat16", batch=100, context=640, portion=700, steps=4),
        # the 32-bit engine scoring a prompt
        dict(name="prompt_float32", kind="prompts", model="qwen3-0.6b", dtype="float32", count=1, tokens=500),
        # prompts of stacks with recurrences and routed feed-forwards: one of the benchmark's length, several ragged ones
        dict(name="kumudra_prompt", kind="prompts", model="kumudra-2048", dtype="bfloat16", count=1, tokens=2048),
        dict(name="risolorn_prompts", kind="prompts", model="risolorn-2048", dtype="bfloat16", count=5, tokens=3000),
        # short requests of such a stack from prompt to last token
        dict(name="risolorn_serve", kind="serve", model="risolorn-2048", dtype="bfloat16", batch=48, context=60, steps=24),
    ]


def draw(rng):
    """One more case of the same ranges: sizes over their logarithm, odd ones among them."""
    def between(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    kind = rng.choice(("decode", "decode", "prompts", "prompts", "mixed", "serve", "stack", "float32"))
    if kind == "decode":
        model = rng.choice(("qwen3-0.6b", "qwen3-8b"))
        batch = between(1, 64)
        most = (120000 if model == "qwen3-0.6b" else 40000) // batch
        return dict(kind=kind, model=model, dtype="bfloat16", batch=batch, context=between(64, min(8192, most)), steps=4)
    if kind == "prompts":
        count = rng.choice((1, 1, 2, 4, 7))
        return dict(kind=kind, model=rng.choice(("qwen3-0.6b", "qwen3-8b")), dtype="bfloat16", count=count,
                    tokens=between(20 * count, 11000))
    if kind == "mixed":
        return dict(kind=kind, model="qwen3-0.6b", dtype="bfloat16", batch=between(4, 100), context=between(64, 640),
                    portion=between(40, 1500), steps=4)
    if kind == "serve":
        return dict(kind=kind, model=rng.choice(("kumudra-2048", "risolorn-2048")), dtype="bfloat16", batch=between(1, 48),
                    context=between(16, 60), steps=24)
    if kind == "stack":
        count = rng.choice((1, 2, 5))
        return dict(kind="prompts", model=rng.choice(("kumudra-2048", "risolorn-2048")), dtype="bfloat16", count=count,
                    tokens=between(40 * count, 3000))
    return dict(kind="prompts", model="qwen3-0.6b", dtype="float32", count=rng.choice((1, 2)), tokens=between(40, 500))


# ----------------------------------------------------------------------------- what a case's requests are

def config_of(case):
    folder = os.path.join(os.path.dirname(ullm_amd.__file__), "config", "presets")
    with open(os.path.join(folder, case["model"] + ".json"), encoding="utf-8") as f:
        return json.load(f)


def vocabulary(cfg):
    return cfg.get("vocab") or cfg["vocab_size"]


def lengths(case):
    """Tokens of every request's prompt (decode: whole pages and one token more, so that the first step brings one)."""
    if case["kind"] == "prompts":
        n, total = case["count"], case["tokens"]
        shares = [1.0 + 0.5 * math.cos(2.3 * i) if n > 1 else 1.0 for i in range(n)]
        cut = [max(1, int(total * s / sum(shares))) for s in shares]
        cut[0] += total - sum(cut)
        return cut
    raw = [case["context"] * (1.0 - 0.45 * ((7 * b) % 16) / 16) for b in range(case["batch"])]
    if case["kind"] == "serve":
        return [max(1, int(r)) for r in raw]
    return [PAGE * max(1, int(r) // PAGE) + 1 for r in raw]


def requests_of(case, seed):
    """Every live request's tokens: its prompt and what the steps bring after it (mixed: the newcomer's prompt last)."""
    V = vocabulary(config_of(case))
    gen = torch.Generator().manual_seed(1000003 * int(seed) + 17)
    more = {"prompts": 0, "decode": case.get("steps", 0) - 1, "mixed": case.get("steps", 0) - 1, "serve": case.get("steps", 0)}[case["kind"]]
    sizes = [n + more for n in lengths(case)] + ([case["portion"] * case["steps"]] if case["kind"] == "mixed" else [])
    return [torch.randint(0, V, (n,), generator=gen).tolist() for n in sizes]


# ----------------------------------------------------------------------------- weights, the same for the engine and for exact()

class Weights:
    """Checkpoint tensors by name, drawn on the device from the seed and the name, in bfloat16 as a checkpoint holds them."""

    def __init__(self, cfg, seed):
        self.cfg, self.seed = cfg, int(seed)

    def _gen(self, name):
        return torch.Generator(device=DEVICE).manual_seed(self.seed * 1000003 + zlib.crc32(name.encode()))

    def _normal(self, name, shape):
        return torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(0.0, 1.0, generator=self._gen(name))

    def _directions(self, n, width):
        return torch.sign(torch.randn(n, width, device=DEVICE, generator=self._gen("expert directions")))

    def __call__(self, name, *shape):
        """Large matrices in bfloat16, in place; the rest in float32 with bfloat16 values."""
        last = name.rsplit(".", 1)[-1]
        if "vocab_size" in self.cfg:
            if name.endswith("norm.weight") or name.endswith("layernorm.weight"):
                return (1.0 + 0.1 * self._normal(name, shape).float()).bfloat16()
            std = 0.5 if "embed" in name else (0.6 if "o_proj" in name or "down_proj" in name else 1.0) / math.sqrt(shape[-1])
            return self._normal(name, shape).mul_(std)
        if name == "embed":
            return self._embedding(shape)
        if last == "router":
            return self._router(name, shape)
        r = self._normal(name, shape).float() if len(shape) < 2 or ".hc" in name or last in ("conv", "u") else None
        if last == "alpha":
            t = 0.7 + 0.1 * r
        elif last in ("norm1", "norm2", "norm") and len(shape) == 1:
            t = 1.0 + 0.1 * r
        elif ".hc" in name:
            S = shape[0]
            t = (torch.eye(S, device=DEVICE) * 0.9 + 0.1 / S + 0.03 * r if last == "mix" else 1.0 / S + 0.05 * r if last == "in"
                 else 1.0 + 0.1 * r)
        elif ".mu." in name:
            t = torch.sigmoid(r)
        elif last == "w0":
            t = -2.5 + 1.5 * r
        elif last == "u":
            t = 0.5 * r
        elif last == "conv":
            t = r / math.sqrt(shape[-1])
        elif name.endswith("a2.b"):
            t = 3.0 + 2.0 * r
        elif name.endswith(".f.b"):
            t = 4.0 + 1.5 * r
        elif last == "A_log":
            t = torch.log(torch.sigmoid(r) * 2 + 0.05)
        elif last == "dt_bias":
            t = -3.0 + 1.5 * r
        elif last == "correction":
            t = 0.01 * r
        elif len(shape) == 1:
            t = 0.2 * r                                        # biases, sinks
        else:
            return self._normal(name, shape).mul_((0.5 if last in ("o", "down") else 1.0) / math.sqrt(shape[-1]))
        return t.bfloat16()

    def _embedding(self, shape):
        """Token rows with a part along four experts' directions, no two groups of eight experts holding three of them."""
        V, W = shape
        n = next(L["mlp"]["router"]["experts"] for L in self.cfg["layers"] if "router" in L["mlp"])
        size = n // 4
        g = self._gen("token experts")
        groups = torch.rand(V, 4, device=DEVICE, generator=g).argsort(-1)[:, :3]
        within = torch.rand(V, 3, size, device=DEVICE, generator=g).argsort(-1)
        experts = torch.stack((groups[:, 0] * size + within[:, 0, 0], groups[:, 0] * size + within[:, 0, 1],
                               groups[:, 1] * size + within[:, 1, 0], groups[:, 2] * size + within[:, 2, 0]), -1)
        amounts = 0.55 + 0.3 * torch.rand(V, 4, device=DEVICE, generator=g)
        along = torch.zeros(V, n, device=DEVICE).scatter_(1, experts, amounts)
        return (self._normal("embed", shape).float() * 0.8 + along @ self._directions(n, W)).bfloat16()

    def _router(self, name, shape):
        n, W = shape
        turn = (zlib.crc32(name.encode()) % 4) * (n // 4)         # another layer, other experts; groups stay groups
        order = (torch.arange(n, device=DEVICE) + turn) % n
        return (self._directions(n, W)[order] * (9.0 / W) + self._normal(name, shape).float() * (0.1 / math.sqrt(W))).bfloat16()


def bound_model(case, seed, context_len):
    cfg = config_of(case)
    weights = Weights(cfg, seed)
    _, model = build_model(cfg)
    env = make_env(case["dtype"], DEVICE, context_len)
    decls = model.weight_decls()
    merged, tensors, aliases = merged_tensors(decls), {}, []
    for d in unique_decls(decls).values():
        if d.alias_of is not None:
            aliases.append(d)
            continue
        dtype = torch.float32 if d.keep_fp32 else env.dtype
        drawn = weights(d.name, *d.shape)
        if d.merged_into is not None:
            m = merged[d.merged_into]
            if m.name not in tensors:
                tensors[m.name] = torch.empty(m.shape, dtype=dtype, device=DEVICE)
            tensors[m.name][d.row_offset:d.row_offset + d.shape[0]].copy_(drawn)
        else:
            tensors[d.name] = drawn.to(dtype)
    for d in aliases:
        tensors[d.name] = tensors[d.alias_of]
    model.bind(tensors, env)
    return model, env


# ----------------------------------------------------------------------------- the pass

def prepare(case, seed):
    tokens = requests_of(case, seed)
    kind = case["kind"]
    longest = max(len(t) for t in tokens) + PAGE
    # the prompt's pages stay with the prefix tree; the steps' own pages come and go
    per_request = [-(-len(t) // PAGE) + 2 for t in tokens]
    context_len = PAGE * -(-longest // PAGE)
    model, env = bound_model(case, seed, context_len)
    runner = ModelRunner(model, env, PAGE, sum(per_request), len(tokens), enable_prefix_cache=kind in ("decode", "mixed"))
    state = {"case": case, "runner": runner, "tokens": tokens, "lengths": lengths(case)}
    if kind in ("decode", "mixed"):
        _read_prompts(state)
    if kind in ("decode", "serve"):
        run(state)                                 # a server's decode graphs are captured by the time a request arrives
    return state


def _read_prompts(state):
    """The live requests' prompts (all but the first decoded token) into pages that the prefix tree keeps."""
    cache, runner = state["runner"].cache, state["runner"]
    batch, n = [], 0

    def flush():
        if batch:
            runner.step([StepEntry(rc, part, []) for rc, part, _ in batch])
            for rc, part, _ in batch:
                cache.release(rc, part)
            del batch[:]
    for i, length in enumerate(state["lengths"]):
        part = state["tokens"][i][:length - 1]
        if n + len(part) > STEP_TOKENS:
            flush()
            n = 0
        rc = cache.admit(f"prompt {i}")
        _reserve(cache, rc, len(part))
        batch.append((rc, part, i))
        n += len(part)
    flush()


def _reserve(cache, rc, n):
    if not cache.reserve(rc, n):
        raise RuntimeError("the pool has too few pages for this case")


def run(state):
    case, runner, tokens, sizes = state["case"], state["runner"], state["tokens"], state["lengths"]
    cache, kind = runner.cache, case["kind"]
    shared = kind in ("decode", "mixed")
    live = [cache.admit(f"r{i}", tokens[i][:n]) if shared else cache.admit(f"r{i}") for i, n in enumerate(sizes)]
    newcomer = cache.admit("newcomer") if kind == "mixed" else None
    out = []
    if kind in ("prompts", "serve"):
        for rc, n in zip(live, sizes):
            _reserve(cache, rc, n)
        out.append(runner.step([StepEntry(rc, t[:n], [n - 1]) for rc, t, n in zip(live, tokens, sizes)]).clone())
    if kind != "prompts":
        for _ in range(case["steps"]):
            entries = []
            for rc, t in zip(live, tokens):
                at = rc.num_computed
                _reserve(cache, rc, 1)
                entries.append(StepEntry(rc, t[at:at + 1], [0]))
            if newcomer is not None:
                at, n = newcomer.num_computed, case["portion"]
                _reserve(cache, newcomer, n)
                entries.append(StepEntry(newcomer, tokens[-1][at:at + n], [n - 1]))
            out.append(runner.step(entries).clone())      # a graph's logits last until the next step
    for rc in live + ([newcomer] if newcomer is not None else []):
        cache.release(rc)
    return out


# ----------------------------------------------------------------------------- what a pass cannot do without

def _passes(case):
    """[(new tokens, keys already there) of every request] per step."""
    sizes, steps = lengths(case), case.get("steps", 0)
    if case["kind"] == "prompts":
        return [[(n, 0) for n in sizes]]
    if case["kind"] == "serve":
        return [[(n, 0) for n in sizes]] + [[(1, n + s) for n in sizes] for s in range(steps)]
    return [[(1, n - 1 + s) for n in sizes] + ([(case["portion"], case["portion"] * s)] if case["kind"] == "mixed" else [])
            for s in range(steps)]


def work(case):
    cfg = config_of(case)
    size = 4 if case["dtype"] == "float32" else 2
    V = vocabulary(cfg)
    nbytes = flops = 0.0
    for step in _passes(case):
        tokens, rows = sum(n for n, _ in step), len(step)
        keys = sum(n + old for n, old in step)
        pairs = sum(n * old + n * (n + 1) // 2 for n, old in step)
        if "vocab_size" in cfg:
            W, H, G, D, I, L = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim",
                                                 "intermediate_size", "num_hidden_layers"))
            per = W * (H + 2 * G) * D + H * D * W + 3 * W * I
            nbytes += size * (L * per + V * W + L * 2 * G * D * keys) + 4 * rows * V
            flops += 2 * L * per * tokens + 4 * L * H * D * pairs + 2 * V * W * rows
        else:
            W = cfg["width"]
            loop = cfg.get("loop") or {"start": 0, "stop": 0, "times": 1}
            for i, L in enumerate(cfg["layers"]):
                times = loop["times"] if loop["start"] <= i < loop["stop"] else 1
                for m in ((L["mixer"]["left"], L["mixer"]["right"]) if L["type"] == "parallel" else (L["mixer"],)):
                    H, G, d, dv = m["heads"], m.get("kv_heads", m["heads"]), m["dim"], m.get("vdim", m["dim"])
                    attends = "scale" in m
                    q = (H if L["type"] != "delta" else G) * d
                    mat = W * (q + G * d + (G if attends else H) * dv + 2 * H * dv - (H * dv if attends else 0))
                    window = (m.get("mask") or {}).get("size") or 1 << 60
                    seen = sum(min(window, n + old) for n, old in step)
                    kv = seen * G * (d + dv) * 2 if attends else 2 * 4 * rows * H * d * dv
                    mix = 2 * sum(n * min(window, old + (n + 1) // 2) for n, old in step) * H * (d + dv) if attends else 6 * tokens * H * d * dv
                    nbytes += times * (2 * mat + kv)
                    flops += times * (2 * mat * tokens + mix)
                f = L["mlp"]
                if "router" in f:
                    n, top, ff = f["router"]["experts"], f["router"]["top"], f["expert"]["ff"]
                    used = n * (1 - (1 - top / n) ** tokens)
                    nbytes += times * (2 * used * 3 * W * ff)
                    flops += times * 2 * tokens * top * 3 * W * ff
                else:
                    nbytes += times * 2 * 3 * W * f["ff"]
                    flops += times * 2 * tokens * 3 * W * f["ff"]
            nbytes += 2 * V * W + 4 * rows * V
            flops += 2 * V * W * rows
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the error against exact(): sums in another order in 32-bit, rounding of the products' inputs over the
    layers in bfloat16 (a stack whose logits hold more of the token's own row shows less of it)."""
    if case["dtype"] == "float32":
        return {"rel": 1.2e-5, "max": 2e-4}
    rel = {"kumudra-2048": 2.5e-3, "risolorn-2048": 1.2e-2}.get(case["model"], 2.5e-2)
    return {"rel": rel, "max": 12 * rel}


# ----------------------------------------------------------------------------- the same in 64 bits, in plain torch

def exact(case, seed):
    cfg, tokens, sizes = config_of(case), requests_of(case, seed), lengths(case)
    if work(case)["flops"] * (sum(len(t) for t in tokens) / max(1, sum(n for s in _passes(case) for n, _ in s))) > 1.5e15:
        return None
    w = Weights(cfg, seed)
    spans, at = [], 0
    for t in tokens:
        spans.append((at, at + len(t)))
        at += len(t)
    ids = torch.tensor([t for seq in tokens for t in seq], device=DEVICE)
    x, head = (_qwen3 if "vocab_size" in cfg else _kumudra if cfg["architecture"] == "Kumudra" else _risolorn)(cfg, w, ids, spans)
    rows = []
    for step in range(1 if case["kind"] == "prompts" else case["steps"] + (case["kind"] == "serve")):
        here = [a + n - 1 + step for (a, _), n in zip(spans, sizes)]
        if case["kind"] == "mixed":
            here.append(spans[-1][0] + case["portion"] * (step + 1) - 1)
        rows.append(here)
    return [(x[torch.tensor(r, device=DEVICE)] @ head.double().T) * cfg.get("logit_scale", 1.0) for r in rows]


def _linear(x, weight):
    weight = weight.double()
    return torch.cat([part @ weight.T for part in x.split(8192)])


def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _attend(q, k, v, spans, scale, sees=None, sink=None):
    """Causal attention of every sequence alone; q [N, H, d], k and v [N, G, .]; sees(query, key positions) narrows it."""
    out = torch.empty(q.shape[0], q.shape[1], v.shape[-1], dtype=F, device=q.device)
    per = q.shape[1] // k.shape[1]
    for a, b in spans:
        for first in range(a, b, 2048):
            last = min(b, first + 2048)
            i, j = torch.arange(first - a, last - a, device=q.device)[:, None], torch.arange(last - a, device=q.device)[None]
            seen = (j <= i) if sees is None else (j <= i) & sees(i, j)
            for g in range(k.shape[1]):
                s = (q[first:last, g * per:(g + 1) * per].transpose(0, 1) @ k[a:last, g].T) * scale
                s = s.masked_fill(~seen, -math.inf)
                if sink is not None:
                    extra = sink[g * per:(g + 1) * per].double()[:, None, None].expand(per, last - first, 1)
                    p = torch.softmax(torch.cat((s, extra), -1), -1)[..., :-1]
                else:
                    p = torch.softmax(s, -1)
                out[first:last, g * per:(g + 1) * per] = (p @ v[a:last, g]).transpose(0, 1)
    return out


def _positions(spans):
    return torch.cat([torch.arange(b - a, device=DEVICE) for a, b in spans])


def _turn(x, first, second, angle, size=1.0):
    c, s = (angle.double().cos() * size)[:, None], (angle.double().sin() * size)[:, None]
    out = x.clone()
    a, b = x[..., first], x[..., second]
    out[..., first], out[..., second] = a * c - b * s, b * c + a * s
    return out


def _qwen3(cfg, w, ids, spans):
    W, H, G, D, I, V, eps = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim",
                                              "intermediate_size", "vocab_size", "rms_norm_eps"))
    table = w("model.embed_tokens.weight", V, W)
    x = table[ids].double()
    # the model's angles are products of 32-bit numbers
    freq = 1.0 / (cfg["rope_theta"] ** (torch.arange(0, D, 2, dtype=torch.float) / D))
    angle = _positions(spans).float()[:, None] * freq.to(DEVICE)
    half = torch.arange(D // 2, device=DEVICE)
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * w(p + "input_layernorm.weight", W).double()
        q = _linear(h, w(p + "self_attn.q_proj.weight", H * D, W)).view(-1, H, D)
        k = _linear(h, w(p + "self_attn.k_proj.weight", G * D, W)).view(-1, G, D)
        v = _linear(h, w(p + "self_attn.v_proj.weight", G * D, W)).view(-1, G, D)
        q = _turn(_rms(q, eps) * w(p + "self_attn.q_norm.weight", D).double(), half, half + D // 2, angle)
        k = _turn(_rms(k, eps) * w(p + "self_attn.k_norm.weight", D).double(), half, half + D // 2, angle)
        o = _attend(q, k, v, spans, D ** -0.5).reshape(-1, H * D)
        x = x + _linear(o, w(p + "self_attn.o_proj.weight", W, H * D))
        h = _rms(x, eps) * w(p + "post_attention_layernorm.weight", W).double()
        up = _silu(_linear(h, w(p + "mlp.gate_proj.weight", I, W))) * _linear(h, w(p + "mlp.up_proj.weight", I, W))
        x = x + _linear(up, w(p + "mlp.down_proj.weight", W, I))
    head = table if cfg["tie_word_embeddings"] else w("lm_head.weight", V, W)
    return _rms(x, eps) * w("model.norm.weight", W).double(), head


def _gated(h, w, p, ff):
    W = h.shape[1]
    return _linear(_silu(_linear(h, w(p + ".gate", ff, W))) * _linear(h, w(p + ".up", ff, W)), w(p + ".down", W, ff))


def _routed(h, w, p, f, normed):
    r, W = f["router"], h.shape[1]
    n, top = r["experts"], r["top"]
    s = torch.sigmoid(_linear(h, w(p + ".router", n, W)))
    choice = s + w(p + ".correction", n).double()
    if "groups" in r:
        count, keep = r["groups"]["count"], r["groups"]["keep"]
        worth = choice.view(-1, count, n // count).topk(2, -1).values.sum(-1)
        kept = torch.zeros_like(worth).scatter_(1, worth.topk(keep, -1).indices, 1.0)
        choice = choice.masked_fill(kept.repeat_interleave(n // count, 1) == 0, -math.inf)
    picked = choice.topk(top, -1).indices
    weight = s.gather(1, picked)
    if normed:
        weight = weight / (weight.sum(-1, keepdim=True) + 1e-20) * r.get("scale", 1.0)
    out = torch.zeros_like(h)
    for e in range(n):
        rows, place = (picked == e).nonzero(as_tuple=True)
        if rows.numel():
            out.index_add_(0, rows, _gated(h[rows], w, f"{p}.e{e}", f["expert"]["ff"]) * weight[rows, place][:, None])
    return out


class _Side:
    """Sequences side by side: [N, ...] rows to [sequences, longest, ...] and back."""

    def __init__(self, spans):
        self.longest = max(b - a for a, b in spans)
        self.seq = torch.cat([torch.full((b - a,), i, device=DEVICE) for i, (a, b) in enumerate(spans)])
        self.pos, self.n = _positions(spans), len(spans)

    def apart(self, x):
        out = torch.zeros((self.n, self.longest) + x.shape[1:], dtype=F, device=DEVICE)
        out[self.seq, self.pos] = x.double()
        return out

    def back(self, x):
        return x[self.seq, self.pos]


def _before(x, spans, back):
    """Every row's predecessor `back` tokens earlier in its own sequence, zeros ahead of the first."""
    side = _Side(spans)
    y = side.apart(x)
    return side.back(torch.cat((torch.zeros_like(y[:, :back]), y[:, :y.shape[1] - back]), 1)) if back < y.shape[1] else torch.zeros_like(x)


def _decayed(q, k, v, decay, spans, bonus=None):
    side = _Side(spans)
    q, k, v, decay = (side.apart(t) for t in (q, k, v, decay))
    S = torch.zeros(side.n, q.shape[2], q.shape[3], v.shape[3], dtype=F, device=DEVICE)
    out = torch.zeros_like(v)
    for t in range(side.longest):
        kv = k[:, t, :, :, None] * v[:, t, :, None, :]
        if bonus is None:
            S = torch.addcmul(kv, S, decay[:, t, :, :, None])
            out[:, t] = (S * q[:, t, :, :, None]).sum(2)
        else:
            out[:, t] = ((S + bonus[:, :, None] * kv) * q[:, t, :, :, None]).sum(2)
            S = torch.addcmul(kv, S, decay[:, t, :, :, None])
    return side.back(out)


def _kumudra(cfg, w, ids, spans):
    W, V, eps, mult, S = cfg["width"], cfg["vocab"], cfg["norm"]["eps"], cfg["residual_mult"], cfg["streams"]
    pos = _positions(spans)

    def norm(u, name):
        d = u - u.mean(-1, keepdim=True)
        return d * torch.rsqrt(d.square().mean(-1, keepdim=True) + eps) * w(name, W).double()

    def lightning(h, p, m):
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        q, k = (_silu(_linear(h, w(f"{p}.{s}", H * d, W))).view(-1, H, d) for s in "qk")
        v = _silu(_linear(h, w(p + ".v", H * dv, W))).view(-1, H, dv)
        decay = torch.tensor(m["decay"], dtype=F, device=DEVICE)[None, :, None].expand(h.shape[0], H, d)
        o = _rms(_decayed(q, k, v, decay, spans).reshape(-1, H * dv), eps) * w(p + ".norm", H * dv).double()
        return _linear(o * torch.sigmoid(_linear(h, w(p + ".g", H * dv, W))), w(p + ".o", W, H * dv))

    def gla(h, p, m):
        H, d, dv, rank = m["heads"], m["dim"], m["vdim"], m.get("rank", 16)
        q, k = (_linear(h, w(f"{p}.{s}", H * d, W)).view(-1, H, d) for s in "qk")
        v = _linear(h, w(p + ".v", H * dv, W)).view(-1, H, dv)
        z = _linear(_linear(h, w(p + ".a1", rank, W)), w(p + ".a2", H * d, rank)) + w(p + ".a2.b", H * d).double()
        o = _decayed(q * d ** -0.5, k, v, torch.sigmoid(z).pow(1.0 / m["tau"]).view(-1, H, d), spans)
        o = (_rms(o, eps) * w(p + ".norm", dv).double()).reshape(-1, H * dv)
        return _linear(o * _silu(_linear(h, w(p + ".g", H * dv, W))), w(p + ".o", W, H * dv))

    def windowed(h, p, m):
        H, G, d, dv, rot = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]
        q, k, v = ((_linear(h, w(f"{p}.{s}", n, W)) + w(f"{p}.{s}.b", n).double()).view(h.shape[0], -1, e)
                   for s, n, e in (("q", H * d, d), ("k", G * d, d), ("v", G * dv, dv)))
        sc, half = rot["scaling"], rot["dims"] // 2
        f = float(rot["base"]) ** (-2.0 * torch.arange(half, dtype=F) / rot["dims"])
        length = 2 * math.pi / f
        blend = ((sc["original"] / length - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        angle = pos.double()[:, None] * ((1 - blend) * f / sc["factor"] + blend * f).to(DEVICE)
        i = torch.arange(half, device=DEVICE)
        o = _attend(_turn(q, i, i + half, angle), _turn(k, i, i + half, angle), v, spans, m["scale"],
                    lambda a, b: a - b < m["mask"]["size"])
        return _linear(o.reshape(-1, H * dv), w(p + ".o", W, H * dv))

    def mixing(h, p, m):
        H, d, rank = m["heads"], m["dim"], m.get("rank", 16)
        prev = _before(h, spans, 1)
        mix = {s: h + (prev - h) * w(f"{p}.mu.{s}", W).double() for s in "rkvgw"}
        r, k, v = (_linear(mix[s], w(f"{p}.{s}", H * d, W)).view(-1, H, d) for s in "rkv")
        z = _linear(torch.tanh(_linear(mix["w"], w(p + ".w1", rank, W))), w(p + ".w2", H * d, rank)) + w(p + ".w0", H * d).double()
        o = _decayed(r, k, v, torch.exp(-torch.exp(z)).view(-1, H, d), spans, w(p + ".u", H, d).double())
        o = _rms(o, eps).reshape(-1, H * d) * w(p + ".norm", H * d).double() * _silu(_linear(mix["g"], w(p + ".g", H * d, W)))
        return _linear(o, w(p + ".o", W, H * d))

    def parallel(h, p, m):
        return m["left_scale"] * windowed(h, p + ".left", m["left"]) + m["right_scale"] * mixing(h, p + ".right", m["right"])

    def sublayer(xs, p, q, fn):
        y = fn(torch.einsum("s,snd->nd", w(f"{p}.hc{q}.in", S).double(), xs))
        return torch.einsum("sr,snd->rnd", w(f"{p}.hc{q}.mix", S, S).double(), xs) + mult * w(f"{p}.hc{q}.out", S).double()[:, None, None] * y

    embed = w("embed", V, W)
    xs = (embed[ids].double() * cfg["embedding"]["scale"])[None].repeat(S, 1, 1)
    mixers = {"lightning": lightning, "gla": gla, "parallel": parallel}
    a, b, times = (cfg["loop"][k] for k in ("start", "stop", "times"))
    n = len(cfg["layers"])
    for i in list(range(a)) + list(range(a, b)) * times + list(range(b, n)):
        L, p = cfg["layers"][i], f"l{i}"
        xs = sublayer(xs, p, 1, lambda u: mixers[L["type"]](norm(u, p + ".norm1"), p + ".mix", L["mixer"]))
        f = L["mlp"]
        xs = sublayer(xs, p, 2, lambda u: _gated(norm(u, p + ".norm2"), w, p + ".mlp", f["ff"]) if f["kind"] == "dense"
                      else _routed(norm(u, p + ".norm2"), w, p + ".mlp", f, True))
    return norm(xs.sum(0), "final.norm"), embed


def _risolorn(cfg, w, ids, spans):
    W, V, eps = cfg["width"], cfg["vocab"], cfg["norm"]["eps"]
    pos, side = _positions(spans), _Side(spans)

    def softplus(z):
        return torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs()))

    def normed(x, name):
        return torch.tanh(w(name + ".alpha").double() * x) * w(name, W).double() + w(name + ".b", W).double()

    def delta(h, p, m):
        H, G, d, dv, taps = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"]

        def conv(s, n):
            u, c = _linear(h, w(f"{p}.{s}", n, W)), w(f"{p}.{s}.conv", n, taps).double()
            return _silu(sum(c[:, j] * (_before(u, spans, taps - 1 - j) if j < taps - 1 else u) for j in range(taps)))

        def unit(x):
            return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)
        q = unit(conv("q", G * d).view(-1, G, d)) * d ** -0.5
        k, v = unit(conv("k", G * d).view(-1, G, d)), conv("v", H * dv).view(-1, H, dv)
        beta = torch.sigmoid(_linear(h, w(p + ".b", H, W)))
        g = torch.exp(-torch.exp(w(p + ".A_log", H).double()) * softplus(_linear(h, w(p + ".a", H, W)) + w(p + ".dt_bias", H).double()))
        q, k = (side.apart(t.repeat_interleave(H // G, 1)) for t in (q, k))
        v, g, beta = side.apart(v), side.apart(g), side.apart(beta)
        S = torch.zeros(side.n, H, d, dv, dtype=F, device=DEVICE)
        out = torch.zeros_like(v)
        for t in range(side.longest):
            S = g[:, t, :, None, None] * S
            u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
            S = torch.addcmul(S, k[:, t, :, :, None], u[:, :, None, :])
            out[:, t] = (S * q[:, t, :, :, None]).sum(2)
        o = (_rms(side.back(out), eps) * w(p + ".norm", dv).double()).reshape(-1, H * dv)
        return _linear(o * _silu(_linear(h, w(p + ".g", H * dv, W))), w(p + ".o", W, H * dv))

    def mlstm(h, p, m):
        H, d, dv, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k = (side.apart(_linear(h, w(f"{p}.{s}", H * d, W)).view(-1, H, d)) for s in "qk")
        v = side.apart(_linear(h, w(p + ".v", H * dv, W)).view(-1, H, dv))
        i, f = (side.apart(cap * torch.tanh((_linear(h, w(f"{p}.{s}", H, W)) + w(f"{p}.{s}.b", H).double()) / cap)) for s in "if")
        f = -softplus(-f)
        S = torch.zeros(side.n, H, d, dv, dtype=F, device=DEVICE)
        n, top, out = torch.zeros_like(S[..., 0]), torch.zeros(side.n, H, dtype=F, device=DEVICE), torch.zeros_like(v)
        for t in range(side.longest):
            now = torch.maximum(f[:, t] + top, i[:, t])
            keep, take = torch.exp(f[:, t] + top - now), torch.exp(i[:, t] - now)
            kt = take[..., None] * k[:, t]
            S = torch.addcmul(keep[..., None, None] * S, kt[..., None], v[:, t, :, None, :])
            n, top = keep[..., None] * n + kt, now
            qt = q[:, t] * d ** -0.5
            out[:, t] = (S * qt[..., None]).sum(2) / (torch.maximum((n * qt).sum(-1).abs(), torch.exp(-top)) + 1e-6)[..., None]
        o = _rms(side.back(out), eps).reshape(-1, H * dv) * w(p + ".norm", H * dv).double()
        return _linear(o * torch.sigmoid(_linear(h, w(p + ".g", H * dv, W))), w(p + ".o", W, H * dv))

    def attention(h, p, m):
        H, G, d, dv, rot = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]
        q, k, v = ((_linear(h, w(f"{p}.{s}", n, W)) + w(f"{p}.{s}.b", n).double()).view(h.shape[0], -1, e)
                   for s, n, e in (("q", H * d, d), ("k", G * d, d), ("v", G * dv, dv)))
        sc, dims, base = rot["scaling"], rot["dims"], rot["base"]
        f = float(base) ** (-2.0 * torch.arange(dims // 2, dtype=F) / dims)
        lo, hi = (dims * math.log(sc["original"] / (2 * math.pi * sc[s])) / (2 * math.log(base)) for s in ("fast", "slow"))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
        slow = ((torch.arange(dims // 2, dtype=F) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        angle = pos.double()[:, None] * (f / sc["factor"] * slow + f * (1 - slow)).to(DEVICE)
        i, size = torch.arange(dims // 2, device=DEVICE) * 2, 0.1 * math.log(sc["factor"]) + 1.0
        o = _attend(_turn(q, i, i + 1, angle, size), _turn(k, i, i + 1, angle, size), v, spans, m["scale"],
                    lambda a, b: a // m["mask"]["size"] == b // m["mask"]["size"], w(p + ".sink", H))
        return _linear(o.reshape(-1, H * dv), w(p + ".o", W, H * dv))

    mixers = {"delta": delta, "mlstm": mlstm, "attention": attention}
    x = w("embed", V, W)[ids].double() * cfg["embedding"]["scale"]
    for i, L in enumerate(cfg["layers"]):
        p = f"l{i}"
        h = normed(x, p + ".norm1")
        x = x + mixers[L["type"]](h, p + ".mix", L["mixer"]) + _routed(h, w, p + ".mlp", L["mlp"], False)
    return normed(x, "final.norm"), w("head", V, W)
