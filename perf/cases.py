"""Performance cases of this framework: what a program that serves models through HipModel asks of it.

The models are the repository's own configurations (uzu_amd.synthetic presets; the layer sizes that bench.py gives the f32-stream designs) with random weights in the formats
of real checkpoints.  A process loads a model once and keeps it; what differs from request to request -- tokens, sequence states -- is made by `prepare` from the seed.

The random weights are scaled the way a trained model's are: a sublayer adds a small part to the residual stream, attention scores are peaked, routers decide clearly, and the
read-out has one clear winner (the tied model repeats its token, the untied ones walk a permutation of the vocabulary).  So a logit is a smooth function of the arithmetic and
results of two correct implementations can be compared, which a stack of unscaled random layers does not allow.
"""
from __future__ import annotations

import json
import math
import os
import random
import tempfile
from dataclasses import replace
from types import SimpleNamespace

import numpy as np
import torch

from uzu_amd import desc as D
from uzu_amd import loader
from uzu_amd import rilavik
from uzu_amd import synthetic as S
from uzu_amd.backend import Context
from uzu_amd.engine import MODEL_BATCH, MODEL_DEFAULT, MODEL_FULL_F32, HipModel

QWEN, LLAMA, RILAVIK = "qwen3.5-0.8b", "llama-3-8b", "rilavik"
MAX_CONTEXT = {QWEN: 4096, LLAMA: 2304, RILAVIK: 4096}
LLAMA_SEQUENCES, RILAVIK_SEQUENCES = 4, 12  # sequences a batched pass may carry
STEP_A, STEP_B = 4099, 13                   # successor of token t in the untied models: (STEP_A t + STEP_B) mod vocabulary


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # the greedy loop of a chat request on the small quantized model: 16 chained tokens (one round trip of LanguageModel.generate) behind a cached 2 k prompt
        dict(name="qwen decode at 2k", model=QWEN, bits=4, kind="decode", context=2040, steps=16),
        # the same early in a conversation, where attention is a single pass over a short cache
        dict(name="qwen decode at 131", model=QWEN, bits=4, kind="decode", context=131, steps=8),
        # time to the first token: a short question, an ordinary prompt, a long document
        dict(name="qwen prompt of 37", model=QWEN, bits=4, kind="prefill", tokens=37),
        dict(name="qwen prompt of 517", model=QWEN, bits=4, kind="prefill", tokens=517),
        dict(name="qwen prompt of 2043", model=QWEN, bits=4, kind="prefill", tokens=2043),
        # one round of speculative decoding: a tree of 13 drafted tokens checked in one pass, a path of it accepted
        dict(name="qwen verify 13", model=QWEN, bits=4, kind="verify", context=1500, nodes=13),
        # a larger model, weights in 8 bits, one user
        dict(name="llama int8 decode at 2k", model=LLAMA, bits=8, kind="decode", context=2000, steps=4),
        # the largest: four prompts prefilled together, then each sequence's first decoded token
        dict(name="llama int4 4 x 1021", model=LLAMA, bits=4, kind="batch", sequences=4, tokens=1021),
        # an f32-stream design: several prompts of unequal length in one step, wide and narrow
        dict(name="rilavik w2048 prompts", model=RILAVIK, width=2048, products="bf16", kind="prompts", lengths="1000,531,517"),
        # ... one user's chained decode
        dict(name="rilavik w1024 decode", model=RILAVIK, width=1024, products="bf16", kind="decode", context=1333, steps=16),
        # ... and a server's: eight sequences of unequal length, four steps, each fed with the token sampled before it
        dict(name="rilavik w2048 8 users", model=RILAVIK, width=2048, products="bf16", kind="users", lengths="40,300,555,700,901,1203,1500,1999", steps=4),
        # the design's other precision: products on f32 operands
        dict(name="rilavik w1024 f32 prompt", model=RILAVIK, width=1024, products="f32", kind="prompts", lengths="300"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.randrange(7)
    if what == 0:
        return dict(model=QWEN, bits=4, kind="decode", context=_log_uniform(rng, 16, 4000), steps=rng.randint(4, 16))
    if what == 1:
        return dict(model=QWEN, bits=4, kind="prefill", tokens=_log_uniform(rng, 5, 3000))
    if what == 2:
        return dict(model=QWEN, bits=4, kind="verify", context=_log_uniform(rng, 64, 3000), nodes=rng.randint(2, 16))
    if what == 3:
        return dict(model=LLAMA, bits=rng.choice((4, 8)), kind="decode", context=_log_uniform(rng, 64, 2200), steps=rng.randint(2, 6))
    if what == 4:
        return dict(model=LLAMA, bits=4, kind="batch", sequences=rng.randint(1, LLAMA_SEQUENCES), tokens=_log_uniform(rng, 24, 1021))
    width = rng.choice((1024, 2048))
    if what == 5:
        f32 = rng.random() < 0.25
        lengths = [_log_uniform(rng, 8, 300 if f32 else 1300) for _ in range(rng.randint(1, 2 if f32 else 4))]
        return dict(model=RILAVIK, width=width, products="f32" if f32 else "bf16", kind="prompts", lengths=",".join(map(str, lengths)))
    if rng.random() < 0.3:
        return dict(model=RILAVIK, width=width, products="bf16", kind="decode", context=_log_uniform(rng, 16, 3000), steps=rng.randint(4, 16))
    lengths = [_log_uniform(rng, 16, 2000) for _ in range(rng.randint(2, RILAVIK_SEQUENCES))]
    return dict(model=RILAVIK, width=width, products="bf16", kind="users", lengths=",".join(map(str, lengths)), steps=rng.randint(2, 6))


def _lengths(case):
    return [int(v) for v in case["lengths"].split(",")]


# ------------------------------------------------------------------------------------------------ models: made once per process from a fixed seed, kept
_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _context():
    return _keep("context", lambda: Context.new(0))


def _generator(*key):
    g = torch.Generator(device="cuda")
    g.manual_seed(random.Random(repr(key)).randrange(1 << 62))
    return g


def _bf16_bits(t):
    return t.to(torch.bfloat16).contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _quantized(cfg, name, n, k, gain=1.0, row_gain=None):
    """A random matrix [n, k] in the quantized layout (scale + bias per group), dequantized entries of standard deviation gain / sqrt(k); row_gain: [(rows, factor)], in order."""
    g = _generator(cfg.name, cfg.bits, name)
    levels, groups = 1 << cfg.bits, k // cfg.group_size
    codes = torch.randint(0, 256, (n, k * cfg.bits // 8), dtype=torch.uint8, device="cuda", generator=g)
    base = gain / (math.sqrt(k) * math.sqrt((levels * levels - 1) / 12.0))
    scales = base * (0.6 + 0.8 * torch.rand((n, groups), device="cuda", generator=g))
    if row_gain:
        scales *= torch.cat([torch.full((rows, 1), float(f), device="cuda") for rows, f in row_gain])
    scales = scales.to(torch.bfloat16)
    biases = (-(levels - 1) / 2.0 + 0.24 * (torch.rand((n, groups), device="cuda", generator=g) - 0.5)) * scales.float()
    return D.LinearWeights(n, k, cfg.bits, cfg.group_size, D.QUANT_SCALE_BIAS, codes.cpu().numpy(), _bf16_bits(scales), _bf16_bits(biases))


def _successor_rows(lw):
    """The same table with row t moved to row (STEP_A t + STEP_B) mod n: as a read-out it answers token t with its successor."""
    at = np.empty(lw.n, dtype=np.int64)
    at[(np.arange(lw.n, dtype=np.int64) * STEP_A + STEP_B) % lw.n] = np.arange(lw.n)
    return D.LinearWeights(lw.n, lw.k, lw.bits, lw.group_size, lw.method, np.ascontiguousarray(lw.weights[at]), np.ascontiguousarray(lw.scales[at]), np.ascontiguousarray(lw.biases[at]))


def _quantized_bundle(model, bits):
    cfg = replace(S.PRESETS[model](max_context_length=MAX_CONTEXT[model]), bits=bits)
    d = cfg.model_dim
    out = 1.0 / math.sqrt(2.0 * cfg.num_layers * d)  # what one of the 2 L sublayers adds to a stream whose embedding rows have entries of 1 / sqrt(d)
    layers = []
    for i, kind in enumerate(cfg.layer_kinds):
        p = f"layers.{i}."
        lw = D.LayerWeights(mixer_kind=kind, hidden_dim=cfg.hidden_dim, activation=D.ACT_SILU, pre_mixer_norm=S.make_norm(cfg, p + "pre_mixer_norm", d),
                            pre_mlp_norm=S.make_norm(cfg, p + "pre_mlp_norm", d), up_projection=_quantized(cfg, p + "up", 2 * cfg.hidden_dim, d),
                            down_projection=_quantized(cfg, p + "down", d, cfg.hidden_dim, gain=2.0 * out))
        if kind == D.MIXER_ATTENTION:
            q, kv = cfg.num_heads * cfg.head_dim, cfg.num_groups * cfg.head_dim
            lw.num_heads, lw.num_groups, lw.head_dim, lw.has_gate, lw.use_rope = cfg.num_heads, cfg.num_groups, cfg.head_dim, cfg.has_gate, True
            lw.qkv_projection = _quantized(cfg, p + "qkv", q + 2 * kv, d, row_gain=None if cfg.qk_norm else [(q + kv, 1.4), (kv, 1.0)])
            if cfg.has_gate:
                lw.gate_projection = _quantized(cfg, p + "gate", q, d)
            lw.out_projection = _quantized(cfg, p + "out", d, q, gain=2.0 * out)
            if cfg.qk_norm:
                lw.query_norm, lw.key_norm = S.make_norm(cfg, p + "query_norm", cfg.head_dim), S.make_norm(cfg, p + "key_norm", cfg.head_dim)
                for norm in (lw.query_norm, lw.key_norm):
                    norm.scales += np.float32(0.5)
        else:
            H, G, dk, dv = cfg.dn_num_heads, cfg.dn_num_groups, cfg.dn_head_dim, cfg.dn_value_head_dim
            conv = 2 * G * dk + H * dv
            r = np.random.default_rng(1000 + i)
            lw.dn_num_heads, lw.dn_num_groups, lw.dn_head_dim, lw.dn_value_head_dim, lw.dn_kernel_size, lw.dn_norm_epsilon = H, G, dk, dv, cfg.dn_kernel_size, cfg.norm_epsilon
            lw.dn_in_proj, lw.dn_out_proj = _quantized(cfg, p + "in", conv + H * dv + 2 * H, d), _quantized(cfg, p + "out", d, H * dv, gain=2.0 * out)
            lw.dn_conv_weights = r.uniform(-0.6, 0.6, (conv, cfg.dn_kernel_size)).astype(np.float32)
            lw.dn_a_log, lw.dn_dt_bias = r.uniform(-3.0, 0.5, H).astype(np.float32), r.uniform(-1.0, 1.0, H).astype(np.float32)
            lw.dn_norm_scales = (1.0 + r.uniform(-0.1, 0.1, dv)).astype(np.float32)
        layers.append(lw)
    embedding = _quantized(cfg, "embedding", cfg.vocab_size, d)
    return D.ModelBundle(name=cfg.name, vocab_size=cfg.vocab_size, model_dim=d, max_context_length=cfg.max_context_length, rope=cfg.rope, embedding=embedding,
                         output_norm=S.make_norm(cfg, "output_norm", d), layers=layers, tied_embeddings=cfg.tied_embeddings,
                         output_embedding=None if cfg.tied_embeddings else _successor_rows(embedding))


def _rilavik_config(width):
    """The layer sizes of bench.py's side run of this design."""
    heads = width // 128
    mlp = rilavik.moe_mlp(8, 2, width)
    pair = rilavik.parallel_layer(rilavik.attention_half(heads, heads // 4, 128, 128, 1024), rilavik.state_space_half(width // 64, 64, 128, 2, 2), mlp=mlp)
    return rilavik.config(32768, width, [pair, pair, pair, rilavik.gla_layer(heads, 128, 128, mlp=mlp)])


def _rilavik_tensors(width):
    """bf16 tensors on the GPU by name.  The first 8 coordinates of an embedding row name the token's two experts, and a router reads mostly those."""
    cfg = _rilavik_config(width)
    t = {}

    def lin(name, n, k, gain=1.0):
        t[name] = (torch.randn((n, k), device="cuda", generator=_generator(width, name)) * (gain / math.sqrt(k))).to(torch.bfloat16)

    def vec(name, n, centre, spread):
        t[name] = (centre + spread * (torch.rand(n, device="cuda", generator=_generator(width, name)) - 0.5)).to(torch.bfloat16)

    def taps(name, channels, n):
        w = torch.randn((channels, n), device="cuda", generator=_generator(width, name)) * 0.4
        w[:, -1] += 0.6
        t[name] = w.to(torch.bfloat16)

    vocab = cfg["vocab"]
    lin("embed", vocab, width, math.sqrt(width))
    token = torch.arange(vocab, device="cuda")
    first, second = token * 5 % 8, (token * 5 + 1 + token // 8 % 7) % 8
    t["embed"][:, :8] = -6.0
    t["embed"][token, first] = t["embed"][token, second] = 6.0
    for i, lc in enumerate(cfg["layers"]):
        p, mx = f"l{i}.", lc["mixer"]
        m, f = p + "mix.", p + "mlp."
        for s in (1, 2):
            vec(f"{p}norm{s}", width, 1.0, 0.4), vec(f"{p}norm{s}b", width, 1.0, 0.4), vec(f"{p}ls{s}", width, 0.5, 0.4)
        if lc["type"] == "gla":
            H, dk, dv, rank = mx["heads"], mx["dim"], mx["vdim"], mx["rank"]
            lin(m + "q", H * dk, width), lin(m + "k", H * dk, width), lin(m + "v", H * dv, width), lin(m + "g", H * dv, width)
            lin(m + "a1", rank, width), lin(m + "a2", H * dk, rank), vec(m + "a2.b", H * dk, 1.0, 4.0), vec(m + "norm", dv, 1.0, 0.4), lin(m + "o", width, H * dv)
        else:
            L, R = mx["left"], mx["right"]
            for n, ch, gain in (("q", L["heads"] * L["dim"], 2.0), ("k", L["kv_heads"] * L["dim"], 2.0), ("v", L["kv_heads"] * L["vdim"], 1.0)):
                lin(f"{m}left.{n}", ch, width, gain), taps(f"{m}left.{n}.conv", ch, L["conv"])
            lin(m + "left.o", width, L["heads"] * L["vdim"])
            H, inner, mixed = R["heads"], R["heads"] * R["vdim"], R["heads"] * R["vdim"] + 2 * R["groups"] * R["state"]
            lin(m + "right.in", inner + mixed + H, width), lin(m + "right.o", width, inner), taps(m + "right.conv", mixed, R["conv"])
            vec(m + "right.conv.b", mixed, 0.0, 0.4), vec(m + "right.dt_bias", H, -2.0, 3.0), vec(m + "right.A_log", H, 0.5, 2.0), vec(m + "right.D", H, 0.5, 1.0)
            vec(m + "right.norm", inner, 1.0, 0.4)
        E, ff = lc["mlp"]["router"]["experts"], lc["mlp"]["expert"]["ff"]
        router = torch.randn((E, width), device="cuda", generator=_generator(width, f + "router")) * (0.05 / math.sqrt(width))
        router[:, :8] = 0.5 * torch.eye(8, device="cuda")
        t[f + "router"] = router.to(torch.bfloat16)
        for e in range(E):
            lin(f"{f}e{e}.gate", ff, width), lin(f"{f}e{e}.up", ff, width), lin(f"{f}e{e}.down", width, ff)
    vec("final.norm", width, 1.0, 0.4)
    head = torch.empty_like(t["embed"])
    head[(token * STEP_A + STEP_B) % vocab] = t["embed"]
    t["head"] = (head.float() / math.sqrt(width)).to(torch.bfloat16)
    t["head"][:, :8] = 0.0
    return cfg, t


def _rilavik_bundle(width):
    cfg, t = _rilavik_tensors(width)
    full = json.loads(json.dumps(cfg))
    full["architecture"] = rilavik.ARCHITECTURE
    for lc in full["layers"]:
        lc["mixer"].pop("rank", None)
    with tempfile.TemporaryDirectory() as tmp:
        with open(os.path.join(tmp, "config.json"), "w", encoding="utf-8") as f:
            json.dump(full, f)
        loader.write_safetensors(os.path.join(tmp, "model.safetensors"), {k: ("BF16", _bf16_bits(v)) for k, v in t.items()}, {})
        return loader.load_model_dir(tmp, max_context_length=MAX_CONTEXT[RILAVIK])


def _bundle(case):
    if case["model"] == RILAVIK:
        return _keep(("bundle", RILAVIK, case["width"]), lambda: _rilavik_bundle(case["width"]))
    return _keep(("bundle", case["model"], case["bits"]), lambda: _quantized_bundle(case["model"], case["bits"]))


def _model(case):
    if case["model"] == RILAVIK:
        flags = MODEL_BATCH(RILAVIK_SEQUENCES) | (MODEL_FULL_F32 if case["products"] == "f32" else 0)
    else:
        flags = MODEL_BATCH(LLAMA_SEQUENCES) if case["model"] == LLAMA else MODEL_DEFAULT
    key = ("model", case["model"], case.get("bits"), case.get("width"), case.get("products"))
    return _keep(key, lambda: HipModel(_context(), _bundle(case), flags))


# ------------------------------------------------------------------------------------------------ prepare / run
def _requests(case, seed):
    """The prompts of a case, token ids in [0, vocabulary)."""
    vocab = 32768 if case["model"] == RILAVIK else S.PRESETS[case["model"]]().vocab_size
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    lengths = _lengths(case) if "lengths" in case else [case["tokens"]] * case.get("sequences", 1) if "tokens" in case else [case["context"]]
    prompts = [rng.integers(0, vocab, n, dtype=np.uint32) for n in lengths]
    if kind != "verify":
        return prompts, None
    # a drafted tree in depth-first order: most nodes extend the node before them, some open a branch further up
    heights = [0]
    for _ in range(case["nodes"] - 1):
        heights.append(heights[-1] + 1 if rng.random() < 0.6 else int(rng.integers(1, heights[-1] + 2)))
    n = len(heights)
    ends = [next((j - 1 for j in range(i + 1, n) if heights[j] <= heights[i]), n - 1) for i in range(n)]
    nodes = np.array([[i, ends[i], heights[i]] for i in range(n)], dtype=np.uint32)
    path = [i for i in range(n) if all(heights[j] == j for j in range(i + 1))]
    return prompts, (rng.integers(0, vocab, n, dtype=np.uint32), nodes, path)


def prepare(case, seed):
    model = _model(case)
    prompts, tree = _requests(case, seed)
    kind = case["kind"]
    st = SimpleNamespace(model=model, kind=kind, prompts=prompts, steps=case.get("steps", 0), states=[model.new_state() for _ in prompts], prefixes=None)
    if kind in ("decode", "verify", "users"):  # the prompts' states are in hand: a pass continues copies of them
        st.prefixes = [model.new_state() for _ in prompts]
        if kind == "users":
            _, st.first = model.step_batch(st.prefixes, prompts, None, sample=True)
        else:
            model.bind(st.prefixes[0])
            model.prefill(prompts[0])
            model.bind(None)
    if tree is not None:
        st.tree_tokens, st.tree_nodes, st.tree_path = tree
    return st


def _logits(model):
    if model.f32_stream:
        return torch.from_numpy(model.read_logits_f32())
    return torch.from_numpy(model.read_logits().view(np.int16)).view(torch.bfloat16)


def run(st):
    model = st.model
    if st.kind == "prefill":
        model.bind(st.states[0])
        model.reset()
        token = model.prefill(st.prompts[0])
        return {"logits": _logits(model), "token": token}
    if st.kind == "decode":  # a cached prompt continued: its state is copied, then chained greedy steps
        st.states[0].copy_from(st.prefixes[0])
        model.bind(st.states[0])
        tokens, _ = model.decode(st.steps)
        return {"logits": _logits(model), "tokens": tokens}
    if st.kind == "verify":
        st.states[0].copy_from(st.prefixes[0])
        model.bind(st.states[0])
        tokens = model.verify_tree(st.tree_tokens, st.tree_nodes)
        hidden = model.final_hidden_rows()
        model.accept(st.tree_path)
        return {"hidden": torch.from_numpy(hidden.view(np.int16)).view(torch.bfloat16), "tokens": tokens}
    if st.kind == "batch":
        for s in st.states:
            s.reset()
        first = model.prefill_batch(st.states, np.stack(st.prompts))
        logits, tokens = [], []
        for s in st.states:
            model.bind(s)
            token, _ = model.decode(1)
            tokens.append(int(token[0]))
            logits.append(_logits(model))
        return {"first": first, "logits": torch.stack(logits), "tokens": np.array(tokens)}
    if st.kind == "prompts":
        for s in st.states:
            s.reset()
        logits, tokens = model.step_batch(st.states, st.prompts, [[len(p) - 1] for p in st.prompts], sample=True)
        return {"logits": logits, "tokens": tokens}
    tokens, out = st.first, []  # users
    for s, prefix in zip(st.states, st.prefixes):
        s.copy_from(prefix)
    for step in range(st.steps):
        last = step == st.steps - 1
        logits, tokens = model.step_batch(st.states, [[int(t)] for t in tokens], [[0]] * len(tokens) if last else None, sample=True)
        out.append(tokens)
    return {"logits": logits, "tokens": np.stack(out)}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _matrix_sizes(case):
    """(entries of the layers' matrices that one row multiplies, bytes of all layers' matrices, entries of the read-out, bytes of the read-out)"""
    if case["model"] == RILAVIK:
        w = case["width"]
        heads, expert = w // 128, 3 * w * w
        pair = w * (w + 2 * (heads // 4) * 128) + w * w + w * (2 * w + 2 * 2 * 128 + w // 64) + w * w
        gla = w * 4 * w + 16 * 2 * w + w * w
        dense = 3 * pair + gla + 4 * 8 * w
        return dense + 4 * 2 * expert, 2 * (dense + 4 * 8 * expert), 32768 * w, 2 * 32768 * w
    cfg = S.PRESETS[case["model"]]()
    d, per = cfg.model_dim, case["bits"] / 8.0 + 4.0 / cfg.group_size
    entries = 0
    for kind in cfg.layer_kinds:
        entries += 3 * d * cfg.hidden_dim
        if kind == D.MIXER_ATTENTION:
            q, kv = cfg.num_heads * cfg.head_dim, cfg.num_groups * cfg.head_dim
            entries += d * (q + 2 * kv + (q if cfg.has_gate else 0)) + q * d
        else:
            conv = 2 * cfg.dn_num_groups * cfg.dn_head_dim + cfg.dn_num_heads * cfg.dn_value_head_dim
            v = cfg.dn_num_heads * cfg.dn_value_head_dim
            entries += d * (conv + v + 2 * cfg.dn_num_heads) + v * d
    return entries, entries * per, cfg.vocab_size * d, cfg.vocab_size * d * per


def _sequence_cost(case, before, count):
    """(flops, bytes) of the token mixing of `count` new positions behind `before` cached ones, without matrices: scores and sums over the visible keys, the recurrences' state."""
    if case["model"] == RILAVIK:
        w = case["width"]
        heads, window = w // 128, 1024
        seen = sum(min(window, before + i + 1) for i in range(count))
        state = (w // 64) * 64 * 128
        flops = 3 * (4.0 * heads * 128 * seen + 4.0 * state * count) + 4.0 * heads * 128 * 128 * count
        cached = min(window, before) + count
        return flops, 3 * (cached * 2 * (heads // 4) * 128 * 2 + 2 * state * 4) + 2 * heads * 128 * 128 * 4
    cfg = S.PRESETS[case["model"]]()
    seen = count * before + count * (count + 1) / 2.0
    flops = nbytes = 0.0
    for kind in cfg.layer_kinds:
        if kind == D.MIXER_ATTENTION:
            flops += 4.0 * cfg.num_heads * cfg.head_dim * seen
            nbytes += 4.0 * cfg.num_groups * cfg.head_dim * (before + count)
        else:
            state = cfg.dn_num_heads * cfg.dn_value_head_dim * cfg.dn_head_dim
            flops += 6.0 * state * count
            nbytes += 8.0 * state
    return flops, nbytes


def work(case):
    entries, layer_bytes, head, head_bytes = _matrix_sizes(case)
    kind = case["kind"]
    if kind in ("decode", "users"):
        at = _lengths(case) if kind == "users" else [case["context"]]
        passes = [[(c + s, 1) for c in at] for s in range(case["steps"])]
        logit_rows = [len(at)] * case["steps"]
    elif kind == "verify":
        passes, logit_rows = [[(case["context"], case["nodes"])]], [case["nodes"]]
    elif kind == "batch":
        passes = [[(0, case["tokens"])] * case["sequences"]] + [[(case["tokens"], 1)]] * case["sequences"]
        logit_rows = [case["sequences"]] + [1] * case["sequences"]
    else:
        lengths = _lengths(case) if kind == "prompts" else [case["tokens"]]
        passes, logit_rows = [[(0, n) for n in lengths]], [len(lengths)]
    flops = nbytes = 0.0
    for sequences, out_rows in zip(passes, logit_rows):
        rows = sum(c for _, c in sequences)
        streamed = layer_bytes
        if case["model"] == RILAVIK:  # experts that no row chose are not read
            expert = 4 * 3 * case["width"] ** 2 * 2.0
            streamed -= expert * 8 * (1.0 - 2.0 / 8.0) ** rows
        flops += 2.0 * entries * rows + 2.0 * head * out_rows
        nbytes += streamed + head_bytes
        for before, count in sequences:
            f, b = _sequence_cost(case, before, count)
            flops, nbytes = flops + f, nbytes + b
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Four times (bf16 products) what the path was measured to be off its 64-bit results: 2.5e-6 with f32 products, 6e-3 with bf16 products on an f32 stream, 1.6e-2 .. 2e-2 where
    the stream itself is rounded to bf16 after every sublayer (there two correct orders of summation share most of that error: less than twice it)."""
    if case["model"] == RILAVIK:
        return {"rel": 1e-5, "max": 2e-4} if case["products"] == "f32" else {"rel": 0.025, "max": 0.25}
    return {"rel": 0.03, "max": 0.3}


# ------------------------------------------------------------------------------------------------ the same results in 64 bits
F64 = torch.float64


def _f64_bits(bits):
    return torch.from_numpy(np.ascontiguousarray(bits).view(np.int16)).cuda().view(torch.bfloat16).to(F64)


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().to(F64)


def _dequantize(lw, rows=None):
    take = (lambda a: a) if rows is None else (lambda a: a[rows])
    codes = torch.from_numpy(np.ascontiguousarray(take(lw.weights))).cuda()
    if lw.bits == 4:
        codes = torch.stack([codes & 15, codes >> 4], dim=-1).reshape(codes.shape[0], lw.k)
    w = codes.to(F64).view(codes.shape[0], lw.k // lw.group_size, lw.group_size)
    return (w * _f64_bits(take(lw.scales))[:, :, None] + _f64_bits(take(lw.biases))[:, :, None]).view(codes.shape[0], lw.k)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, freq):
    """x [B, T, heads, width]: the coordinates (i, i + half) of every head turn by position * freq[i]."""
    half = freq.numel()
    angle = torch.arange(x.shape[1], device=x.device, dtype=F64)[:, None] * freq
    c, s = angle.cos()[:, None, :], angle.sin()[:, None, :]
    u, v = x[..., :half], x[..., half:2 * half]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * half:]], dim=-1)


def _attend(q, k, v, scale, window=0):
    """q [B, T, H, d], k and v [B, T, G, d], causal, the last `window` positions (0: all) -> [B, T, H dv]"""
    B, T, H, _ = q.shape
    G = k.shape[2]
    at = torch.arange(T, device=q.device)
    far = at[:, None] - at[None, :]
    hidden = (far < 0) | (far >= (window or T + 1))
    out = torch.empty((B, T, H, v.shape[3]), device=q.device, dtype=F64)
    for b in range(B):
        for h in range(H):
            g = h // (H // G)
            s = (q[b, :, h] @ k[b, :, g].T) * scale
            out[b, :, h] = torch.softmax(s.masked_fill_(hidden, -math.inf), dim=-1) @ v[b, :, g]
    return out.reshape(B, T, -1)


def _causal_conv(x, w, bias=None):
    """x [B, T, C], w [C, taps]: the last tap weighs the current position"""
    taps = w.shape[1]
    padded = torch.cat([x.new_zeros((x.shape[0], taps - 1, x.shape[2])), x], dim=1)
    y = sum(padded[:, j:j + x.shape[1]] * w[:, j] for j in range(taps))
    return y if bias is None else y + bias


def _rope_frequencies(r):
    i = torch.arange(r.head_dim // 2, device="cuda", dtype=F64)
    f = r.base ** (-2.0 * i / r.head_dim)
    if r.kind == D.ROPE_LLAMA:
        wavelength = 2.0 * math.pi / f
        low, high = r.original_context_length / r.low_frequency_factor, r.original_context_length / r.high_frequency_factor
        s = (r.original_context_length / wavelength - r.low_frequency_factor) / (r.high_frequency_factor - r.low_frequency_factor)
        f = torch.where(wavelength < high, f, torch.where(wavelength > low, f / r.scaling_factor, s * f + (1.0 - s) * f / r.scaling_factor))
    return f


def _delta_net(x, lw):
    B, T, _ = x.shape
    H, G, dk, dv = lw.dn_num_heads, lw.dn_num_groups, lw.dn_head_dim, lw.dn_value_head_dim
    key, value = G * dk, H * dv
    y = x @ _dequantize(lw.dn_in_proj).T
    mixed, z, beta, a = torch.split(y, [2 * key + value, value, H, H], dim=-1)
    mixed = _silu(_causal_conv(mixed, _f64(lw.dn_conv_weights)))
    q, k, v = torch.split(mixed, [key, key, value], dim=-1)
    unit = lambda u: u * torch.rsqrt(u.square().sum(-1, keepdim=True) + 1e-6)
    q = unit(q.view(B, T, G, dk)).repeat_interleave(H // G, dim=2) * dk ** -0.5
    k = unit(k.view(B, T, G, dk)).repeat_interleave(H // G, dim=2)
    v = v.view(B, T, H, dv)
    decay = torch.exp(-torch.exp(_f64(lw.dn_a_log)) * torch.nn.functional.softplus(a + _f64(lw.dn_dt_bias), threshold=100.0))
    beta = torch.sigmoid(beta)
    q, k, v = (u.permute(1, 0, 2, 3).reshape(T, B * H, -1) for u in (q, k, v))
    decay, beta = (u.permute(1, 0, 2).reshape(T, B * H, 1) for u in (decay, beta))
    state, out = x.new_zeros((B * H, dv, dk)), x.new_empty((T, B * H, dv))
    for t in range(T):
        kt = k[t].unsqueeze(-1)
        state *= decay[t].unsqueeze(-1)
        change = beta[t] * (v[t] - torch.bmm(state, kt).squeeze(-1))
        torch.baddbmm(state, change.unsqueeze(-1), k[t].unsqueeze(1), out=state)
        out[t] = torch.bmm(state, q[t].unsqueeze(-1)).squeeze(-1)
    out = out.view(T, B, H, dv).permute(1, 0, 2, 3)
    out = _rms(out, _f64(lw.dn_norm_scales), lw.dn_norm_epsilon) * _silu(z).view(B, T, H, dv)
    return out.reshape(B, T, value) @ _dequantize(lw.dn_out_proj).T


def _quantized_forward(bundle, tokens):
    """tokens [B, T] -> the rows behind the output norm [B, T, d]"""
    B, T = tokens.shape
    weight = lambda n: _f64(n.scales) + n.scale_offset
    x = _dequantize(bundle.embedding, tokens.reshape(-1).astype(np.int64)).view(B, T, -1)
    freq = _rope_frequencies(bundle.rope)
    for lw in bundle.layers:
        h = _rms(x, weight(lw.pre_mixer_norm), lw.pre_mixer_norm.epsilon)
        if lw.mixer_kind == D.MIXER_ATTENTION:
            H, G, hd = lw.num_heads, lw.num_groups, lw.head_dim
            q, k, v = torch.split((h @ _dequantize(lw.qkv_projection).T).view(B, T, H + 2 * G, hd), [H, G, G], dim=2)
            if lw.query_norm.present:
                q, k = _rms(q, weight(lw.query_norm), lw.query_norm.epsilon), _rms(k, weight(lw.key_norm), lw.key_norm.epsilon)
            o = _attend(_turn(q, freq), _turn(k, freq), v, hd ** -0.5)
            if lw.has_gate:
                o = o * torch.sigmoid(h @ _dequantize(lw.gate_projection).T)
            x = x + o @ _dequantize(lw.out_projection).T
        else:
            x = x + _delta_net(h, lw)
        h = _rms(x, weight(lw.pre_mlp_norm), lw.pre_mlp_norm.epsilon)
        up, gate = (h @ _dequantize(lw.up_projection).T).chunk(2, dim=-1)
        x = x + (up * _silu(gate)) @ _dequantize(lw.down_projection).T
    return _rms(x, weight(bundle.output_norm), bundle.output_norm.epsilon)


def _quantized_head(bundle, rows):
    lw = bundle.embedding if bundle.tied_embeddings else bundle.output_embedding
    return torch.cat([rows @ _dequantize(lw, slice(i, i + 32768)).T for i in range(0, lw.n, 32768)], dim=-1)


def _rilavik_forward(cfg, t, tokens):
    """tokens [T] -> the last row's logits"""
    w = lambda name: t[name].to(F64)
    eps = float(cfg["norm"]["eps"])
    x = t["embed"][torch.from_numpy(tokens.astype(np.int64)).cuda()].to(F64)[None]
    T = x.shape[1]

    def decayed(q, k, v, decay):  # [T, heads, *]: S <- decay S + k v^T, o = S^T q
        state, out = x.new_zeros((q.shape[1], q.shape[2], v.shape[2])), x.new_empty((T, q.shape[1], v.shape[2]))
        for i in range(T):
            state *= decay[i].unsqueeze(-1)
            torch.baddbmm(state, k[i].unsqueeze(-1), v[i].unsqueeze(1), out=state)
            out[i] = torch.bmm(q[i].unsqueeze(1), state).squeeze(1)
        return out

    def attention(h, p, mx):
        H, G, dk, dv = mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"]
        q, k, v = (_causal_conv(h @ w(p + n).T, w(p + n + ".conv")) for n in ("q", "k", "v"))
        rot = mx["rot"]
        freq = rot["base"] ** (-2.0 * torch.arange(rot["dims"] // 2, device="cuda", dtype=F64) / rot["dims"])
        o = _attend(_turn(q.view(1, T, H, dk), freq), _turn(k.view(1, T, G, dk), freq), v.view(1, T, G, dv), mx["scale"], mx["mask"]["size"])
        return o @ w(p + "o").T

    def state_space(h, p, mx):
        H, dv, N, G = mx["heads"], mx["vdim"], mx["state"], mx["groups"]
        inner = H * dv
        z, xbc, dt = torch.split(h @ w(p + "in").T, [inner, inner + 2 * G * N, H], dim=-1)
        u, B, C = torch.split(_silu(_causal_conv(xbc, w(p + "conv"), w(p + "conv.b"))), [inner, G * N, G * N], dim=-1)
        dt = torch.nn.functional.softplus(dt + w(p + "dt_bias"), threshold=100.0)[0]
        u = u.view(T, H, dv)
        B, C = (a.view(T, G, N).repeat_interleave(H // G, dim=1) for a in (B, C))
        decay = torch.exp(-torch.exp(w(p + "A_log")) * dt)
        y = decayed(C, dt.unsqueeze(-1) * B, u, decay.unsqueeze(-1)) + w(p + "D")[:, None] * u
        parts = mx["norm_groups"]
        y = (y.reshape(T, inner) * _silu(z[0])).view(T, parts, inner // parts)
        y = _rms(y, 1.0, eps).reshape(1, T, inner) * w(p + "norm")
        return y @ w(p + "o").T

    def linear_attention(h, p, mx):
        H, dk, dv = mx["heads"], mx["dim"], mx["vdim"]
        q, k, v = ((h @ w(p + n).T).view(T, H, -1) for n in ("q", "k", "v"))
        decay = torch.exp(torch.nn.functional.logsigmoid(h @ w(p + "a1").T @ w(p + "a2").T + w(p + "a2.b")) / mx["tau"]).view(T, H, dk)
        o = _rms(decayed(q * dk ** -0.5, k, v, decay), w(p + "norm"), eps).reshape(1, T, H * dv)
        return (o * _silu(h @ w(p + "g").T)) @ w(p + "o").T

    def experts(h, p, ml):
        h = h[0]
        score, chosen = torch.sigmoid(h @ w(p + "router").T).topk(ml["router"]["top"], dim=-1)
        out = torch.zeros_like(h)
        for e in range(ml["router"]["experts"]):
            at, which = (chosen == e).nonzero(as_tuple=True)
            if at.numel():
                u = score[at, which].unsqueeze(-1) * h[at]
                out[at] += (_silu(u @ w(f"{p}e{e}.gate").T) * (u @ w(f"{p}e{e}.up").T)) @ w(f"{p}e{e}.down").T
        return out[None]

    for i, lc in enumerate(cfg["layers"]):
        p, mx = f"l{i}.", lc["mixer"]
        h = _rms(x, w(p + "norm1"), eps)
        if lc["type"] == "gla":
            o = linear_attention(h, p + "mix.", mx)
        else:
            o = mx["left_scale"] * attention(h, p + "mix.left.", mx["left"]) + mx["right_scale"] * state_space(h, p + "mix.right.", mx["right"])
        x = x + _rms(o, w(p + "norm1b"), eps) * w(p + "ls1")
        x = x + _rms(experts(_rms(x, w(p + "norm2"), eps), p + "mlp.", lc["mlp"]), w(p + "norm2b"), eps) * w(p + "ls2")
    return _rms(x[:, -1], w("final.norm"), eps)[0] @ w("head").T


def _chain(case, token, n):
    """The n tokens that follow `token`: what the read-out's construction makes the greedy choice."""
    out, vocab = [], 32768 if case["model"] == RILAVIK else S.PRESETS[case["model"]]().vocab_size
    for _ in range(n):
        token = token if case["model"] == QWEN else (STEP_A * int(token) + STEP_B) % vocab
        out.append(int(token))
    return np.array(out, dtype=np.uint32)


def exact(case, seed):
    prompts, tree = _requests(case, seed)
    kind, steps = case["kind"], case.get("steps", 0)
    if case["model"] == RILAVIK:
        cfg, t = _keep(("tensors", case["width"]), lambda: _rilavik_tensors(case["width"]))
        logits, tokens = [], []
        for p in prompts:
            chain = _chain(case, p[-1], steps + 1)
            logits.append(_rilavik_forward(cfg, t, np.concatenate([p, chain[:steps]])))
            tokens.append(chain[1:] if steps else chain)
        if kind == "decode":
            return {"logits": logits[0], "tokens": tokens[0]}
        return {"logits": torch.stack(logits).cpu().numpy(), "tokens": np.stack(tokens, axis=1) if kind == "users" else np.concatenate(tokens)}
    bundle = _bundle(case)
    if kind == "verify":  # every root-to-leaf path as a sequence of its own, padded behind its end
        ids, nodes, _ = tree
        n, paths = len(ids), {}
        for i in range(n):
            paths[i] = [j for j in range(i + 1) if nodes[j, 0] <= i <= nodes[j, 1]]
        leaves = [i for i in range(n) if nodes[i, 1] == i]
        depth = max(len(paths[i]) for i in leaves)
        rows = np.stack([np.concatenate([prompts[0], ids[paths[i]], np.zeros(depth - len(paths[i]), dtype=np.uint32)]) for i in leaves])
        h = _quantized_forward(bundle, rows)
        at = {j: (leaf, len(prompts[0]) + k) for leaf, i in enumerate(leaves) for k, j in enumerate(paths[i])}
        return {"hidden": torch.stack([h[at[i]] for i in range(n)]), "tokens": ids}
    more = {"prefill": 0, "decode": steps, "batch": 1}[kind]
    chains = [_chain(case, p[-1], more + 1) for p in prompts]
    h = _quantized_forward(bundle, np.stack([np.concatenate([p, c[:more]]) for p, c in zip(prompts, chains)]))
    logits = _quantized_head(bundle, h[:, -1])
    if kind == "batch":
        return {"first": np.array([c[0] for c in chains]), "logits": logits, "tokens": np.array([c[1] for c in chains])}
    return {"logits": logits[0], "token": int(chains[0][0])} if kind == "prefill" else {"logits": logits[0], "tokens": chains[0][1:]}
