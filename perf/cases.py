"""The work a serving program has this framework do, as cases that can be timed and compared.

A case is one pass through the public entry points (``ferrisinfer_amd.Context``,
``ferrisinfer_amd.runtime.Runtime``): the attention ops of a ragged batch, the blocks of a
decoder layer, the heads that end a step, and a whole generation through the scheduler.  The
shapes are the repository's own configurations: the tiny Llama, the Qwen2-0.5B and the
Llama-3-8B shaped decoders and the standalone 32/8-head attention batches.

  op        one pass
  decode    paged decode attention, one new token per sequence
  prefill   varlen causal attention of prompt chunks over the paged pool
  layer     one decoder layer: q|k|v, RoPE and KV append, attention, wo, SwiGLU MLP, both norms
  mlp       the MLP block alone: up/gate + SwiGLU, down projection, residual and next norm
  head      the greedy head over the vocabulary
  sample    temperature / top-k / top-p sampling of a batch's logits
  serve     prompts submitted to the runtime, run to the end through its scheduler
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ferrisinfer_amd import DTYPE_BF16, DTYPE_F32, Context
from ferrisinfer_amd.runtime import Runtime

BLOCK = 16
EPS = 1e-6

# hidden, intermediate, layers, query heads, kv heads, vocabulary, rope theta
MODELS = {
    "tiny": (256, 688, 4, 8, 2, 4096, 10000.0),
    "qwen2": (896, 4864, 24, 14, 2, 151936, 1000000.0),
    "llama3": (4096, 14336, 32, 32, 8, 128256, 500000.0),
}

_CONTEXT = None


def _ctx() -> Context:
    """A program keeps one context per GPU."""
    global _CONTEXT
    if _CONTEXT is None:
        _CONTEXT = Context(0)
    return _CONTEXT


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one chat user, a short history: what a single token's attention costs
        dict(name="decode-1-qwen2", op="decode", heads=14, kv_heads=2, dim=64, kv="f32", seqs=1, min_ctx=700,
             max_ctx=700),
        # the standalone ragged batch: 64 users, histories between 128 and 2048 tokens
        dict(name="decode-64-f32", op="decode", heads=32, kv_heads=8, dim=128, kv="f32", seqs=64, min_ctx=128,
             max_ctx=2048),
        # a full server with long histories over a bf16 pool
        dict(name="decode-256-bf16", op="decode", heads=32, kv_heads=8, dim=128, kv="bf16", seqs=256, min_ctx=512,
             max_ctx=8192),
        # prompts of mixed length arriving together, some behind a shared prefix, exact pool
        dict(name="prefill-16-f32", op="prefill", heads=32, kv_heads=8, dim=128, kv="f32", seqs=16, min_new=32,
             max_new=1024, max_prefix=512),
        # the second chunk of a long prompt over a bf16 pool
        dict(name="prefill-chunk-bf16", op="prefill", heads=32, kv_heads=8, dim=128, kv="bf16", seqs=1,
             min_new=2048, max_new=2048, max_prefix=2048),
        # one layer of the decode step of a 64-user batch, f32 weights
        dict(name="layer-decode-64", op="layer", model="qwen2", weights="f32", kv="f32", phase="decode", seqs=64,
             min_ctx=64, max_ctx=2048),
        # one layer of a mixed prefill step at the scheduler's 1024-token budget, odd chunk sizes
        dict(name="layer-prefill-1k", op="layer", model="qwen2", weights="f32", kv="f32", phase="prefill", seqs=4,
             min_new=201, max_new=256, max_prefix=1792),
        # the MLP of a 16-user decode step over bf16 weights: the weights are what is read
        dict(name="mlp-16-bf16", op="mlp", model="llama3", weights="bf16", rows=16),
        # the MLP of a step with a 2048-token chunk and 256 decode tokens, bf16 weights
        dict(name="mlp-2304-bf16", op="mlp", model="llama3", weights="bf16", rows=2304),
        # the greedy head of a 64-user batch over the largest vocabulary
        dict(name="head-64-f32", op="head", model="qwen2", weights="f32", rows=64),
        # chat sampling of a 64-user batch
        dict(name="sample-64", op="sample", rows=64, vocab=151936, temperature=0.7, top_k=20, top_p=0.9),
        # 16 prompts answered with 8 sampled tokens each through the scheduler
        dict(name="serve-16", op="serve", model="qwen2", weights="f32", kv="f32", prompts=16, min_prompt=24,
             max_prompt=160, tokens=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _attention_shape(rng):
    h, _, _, hq, hkv, _, _ = MODELS[rng.choice(sorted(MODELS))]
    return dict(heads=hq, kv_heads=hkv, dim=h // hq, kv=rng.choice(["f32", "bf16"]))


def draw(rng):
    op = rng.choice(["decode", "decode", "prefill", "prefill", "layer", "layer", "mlp", "mlp", "head", "sample",
                     "serve"])
    if op == "decode":
        c = dict(op=op, **_attention_shape(rng))
        c["seqs"] = _log(rng, 1, 256)
        c["max_ctx"] = _log(rng, 16, 8192)
        c["min_ctx"] = max(1, int(c["max_ctx"] * rng.uniform(0.05, 1.0)))
        limit = 4.2e9 / (c["kv_heads"] * c["dim"] * (8 if c["kv"] == "f32" else 4))
        c["seqs"] = max(1, min(c["seqs"], int(2 * limit / (c["min_ctx"] + c["max_ctx"]))))
        return c
    if op == "prefill":
        c = dict(op=op, **_attention_shape(rng))
        c["seqs"] = _log(rng, 1, 16)
        c["max_new"] = _log(rng, 8, 2048 // c["seqs"])
        c["min_new"] = max(1, int(c["max_new"] * rng.uniform(0.1, 1.0)))
        c["max_prefix"] = rng.choice([0, _log(rng, 16, 2048)])
        c["f32_math"] = c["kv"] == "f32" or rng.random() < 0.5  # over a bf16 pool the caller chooses
        return c
    if op == "layer":
        model, weights = rng.choice([("tiny", "f32"), ("qwen2", "f32"), ("qwen2", "bf16"), ("llama3", "bf16")])
        c = dict(op=op, model=model, weights=weights, kv="bf16" if model == "llama3" else rng.choice(["f32", "bf16"]),
                 phase=rng.choice(["decode", "prefill"]))
        if c["phase"] == "decode":
            c["seqs"] = _log(rng, 1, 128)
            c["max_ctx"] = _log(rng, 16, 4096)
            c["min_ctx"] = max(1, int(c["max_ctx"] * rng.uniform(0.05, 1.0)))
        else:
            c["seqs"] = _log(rng, 1, 8)
            c["max_new"] = _log(rng, 8, 1024 // c["seqs"])
            c["min_new"] = max(1, int(c["max_new"] * rng.uniform(0.3, 1.0)))
            c["max_prefix"] = rng.choice([0, _log(rng, 16, 2048)])
        return c
    if op in ("mlp", "head"):
        model, weights = rng.choice([("tiny", "f32"), ("qwen2", "f32"), ("qwen2", "bf16"), ("llama3", "bf16"),
                                     ("llama3", "bf16")])
        return dict(op=op, model=model, weights=weights, rows=_log(rng, 1, 2304 if op == "mlp" else 257))
    if op == "sample":
        return dict(op=op, rows=_log(rng, 1, 257), vocab=rng.choice([4096, 32000, 32003, 128256, 151936]),
                    temperature=round(rng.uniform(0.3, 1.5), 3), top_k=_log(rng, 2, 256),
                    top_p=round(rng.uniform(0.5, 1.0), 3))
    c = dict(op="serve", model=rng.choice(["tiny", "qwen2"]), weights=rng.choice(["f32", "bf16"]), kv="f32",
             prompts=_log(rng, 1, 16), tokens=rng.randint(2, 8))
    c["max_prompt"] = _log(rng, 8, 160)
    c["min_prompt"] = max(1, int(c["max_prompt"] * rng.uniform(0.2, 1.0)))
    return c


# ---------------------------------------------------------------- sizes of a case

def _spread(n, lo, hi):
    """n ragged lengths in [lo, hi], the ends among them, in a fixed mixed order."""
    if n == 1:
        return [hi]
    return [lo + (hi - lo) * ((i * 7919) % n) // (n - 1) for i in range(n)]  # 7919: a prime above any n


def _sequences(case):
    """(cached prefix, new tokens) of every sequence of an attention or layer case."""
    if case["op"] == "decode" or case.get("phase") == "decode":
        return [(c - 1, 1) for c in _spread(case["seqs"], case["min_ctx"], case["max_ctx"])]
    new = _spread(case["seqs"], case["min_new"], case["max_new"])
    prefix = _spread(case["seqs"], 0, case["max_prefix"])
    return [(prefix[-1 - i], n) for i, n in enumerate(new)]


def _heads(case):
    if "model" in case:
        h, _, _, hq, hkv, _, _ = MODELS[case["model"]]
        return hq, hkv, h // hq
    return case["heads"], case["kv_heads"], case["dim"]


# ---------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype).mul_(std)


def _metadata(case, seed):
    """Block tables, slots and positions of the case's sequences over a pool handed out in a
    random order, as a paged server's are after a while."""
    seqs = _sequences(case)
    lens = [p + n for p, n in seqs]
    blocks = [-(-x // BLOCK) for x in lens]
    pool = sum(blocks) + 8
    perm = np.random.RandomState(seed % (1 << 31)).permutation(pool)
    tables = np.zeros((len(seqs), max(blocks)), np.int32)
    at, slots, positions, cu = 0, [], [], [0]
    for i, ((prefix, new), k) in enumerate(zip(seqs, blocks)):
        tables[i, :k] = perm[at:at + k]
        at += k
        p = np.arange(prefix, prefix + new)
        positions.append(p)
        slots.append(tables[i, p // BLOCK].astype(np.int64) * BLOCK + p % BLOCK)
        cu.append(cu[-1] + new)
    to = lambda a, t: torch.from_numpy(np.ascontiguousarray(a, t)).cuda()  # noqa: E731
    return dict(seqs=seqs, pool=pool, tables=to(tables, np.int32), lens=to(lens, np.int32), cu=to(cu, np.int32),
                positions=to(np.concatenate(positions), np.int32), slots=to(np.concatenate(slots), np.int64),
                max_ctx=max(lens), max_new=max(n for _, n in seqs), rows=cu[-1])


def _pools(case, meta, g):
    _, hkv, d = _heads(case)
    dtype = torch.float32 if case["kv"] == "f32" else torch.bfloat16
    return [_normal(g, meta["pool"], hkv, BLOCK, d, dtype=dtype) for _ in range(2)]


def _attention_inputs(case, seed):
    hq, hkv, d = _heads(case)
    g = _generator(seed)
    m = _metadata(case, seed)
    k, v = _pools(case, m, g)
    return dict(m, k=k, v=v, q=_normal(g, m["rows"], hq, d))


def _rope_tables(positions, d, theta):
    inv = theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device="cuda") / d)
    angle = torch.arange(positions, dtype=torch.float64, device="cuda")[:, None] * inv
    return angle.cos().float().contiguous(), angle.sin().float().contiguous()


def _layer_weights(case, g, names):
    h, f, _, hq, hkv, _, _ = MODELS[case["model"]]
    shapes = dict(wq=(h, h), wk=(h, hkv * (h // hq)), wv=(h, hkv * (h // hq)), wo=(h, h), w1=(h, f), w3=(h, f),
                  w2=(f, h))
    dtype = torch.float32 if case["weights"] == "f32" else torch.bfloat16
    w = {n: _normal(g, *shapes[n], std=0.02, dtype=dtype) for n in names}
    for n in ("norm1", "norm2"):
        w[n] = 1.0 + _normal(g, h, std=0.1)
    return w


def _mlp_inputs(case, seed):
    h = MODELS[case["model"]][0]
    g = _generator(seed)
    w = _layer_weights(case, g, ("w1", "w3", "w2"))
    x = _normal(g, case["rows"], h)
    return w, (x.bfloat16() if case["weights"] == "bf16" else x), _normal(g, case["rows"], h)


def _layer_inputs(case, seed):
    h, _, _, hq, hkv, _, theta = MODELS[case["model"]]
    g = _generator(seed)
    m = _metadata(case, seed)
    k, v = _pools(case, m, g)
    w = _layer_weights(case, g, ("wq", "wk", "wv", "wo", "w1", "w3", "w2"))
    x = _normal(g, m["rows"], h)
    biases = [_normal(g, n, std=0.02) for n in (h, hkv * (h // hq), hkv * (h // hq))]
    cos, sin = _rope_tables(m["max_ctx"], h // hq, theta)
    return dict(m, k=k, v=v, w=w, x=x.bfloat16() if case["weights"] == "bf16" else x,
                residual=_normal(g, m["rows"], h), biases=biases, cos=cos, sin=sin)


def _head_inputs(case, seed):
    h, vocab = MODELS[case["model"]][0], MODELS[case["model"]][5]
    g = _generator(seed)
    dtype = torch.float32 if case["weights"] == "f32" else torch.bfloat16
    w = _normal(g, vocab, h, std=0.02, dtype=dtype)
    return w, _normal(g, case["rows"], h).to(dtype)


def _sample_inputs(case, seed):
    g = _generator(seed)
    logits = _normal(g, case["rows"], case["vocab"], std=2.0)
    states = np.random.RandomState(seed % (1 << 31)).randint(1, 1 << 62, case["rows"], dtype=np.int64)
    return logits, torch.from_numpy(states).cuda()


def _prompts(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    vocab = MODELS[case["model"]][5]
    return [r.randint(0, vocab, n).astype(np.uint32)
            for n in _spread(case["prompts"], case["min_prompt"], case["max_prompt"])]


def _runtime(case, seed):
    h, f, layers, hq, hkv, vocab, theta = MODELS[case["model"]]
    rt = Runtime(h, f, layers, hq, hkv, vocab, max_pos=4096, theta=theta, tie=True, max_batch=16, max_seq=1024,
                 num_blocks=512, kv_dtype=case["kv"], weight_dtype=case["weights"], graph_decode=True,
                 sampler=(0.7, 20, 0.9, 42))
    g = _generator(seed)
    kvw = hkv * (h // hq)
    put = lambda n, *shape: rt.set_weight_device(n, _normal(g, *shape, std=0.02))  # noqa: E731
    one = torch.ones(h, device="cuda")
    put("tok_embeddings.weight", vocab, h)
    for i in range(layers):
        p = "layers.%d." % i
        rt.set_weight_device(p + "attention_norm.weight", one)
        rt.set_weight_device(p + "ffn_norm.weight", one)
        for n, shape in (("attention.wq", (h, h)), ("attention.wk", (h, kvw)), ("attention.wv", (h, kvw)),
                         ("attention.wo", (h, h)), ("feed_forward.w1", (h, f)), ("feed_forward.w3", (h, f)),
                         ("feed_forward.w2", (f, h))):
            put(p + n + ".weight", *shape)
    rt.set_weight_device("norm.weight", one)
    return rt


def prepare(case, seed):
    c, op = _ctx(), case["op"]
    if op in ("decode", "prefill"):
        s = _attention_inputs(case, seed)
        s["out"] = torch.empty_like(s["q"])
    elif op == "layer":
        s = _layer_inputs(case, seed)
        _pack_layer(c, case, s)
    elif op == "mlp":
        w, x, residual = _mlp_inputs(case, seed)
        s = dict(w=w, x=x, residual=residual, rows=case["rows"])
        _pack_mlp(c, case, s)
    elif op == "head":
        h, vocab = MODELS[case["model"]][0], MODELS[case["model"]][5]
        w, x = _head_inputs(case, seed)
        bf16 = case["weights"] == "bf16"
        s = dict(x=x, token=torch.empty(case["rows"], dtype=torch.int32, device="cuda"),
                 prob=torch.empty(case["rows"], device="cuda"),
                 w=c.weight_pack_bf16(w, h, vocab, src_layout=1) if bf16 else c.weight_pack(w, h, vocab, 2, src_layout=1))
    elif op == "sample":
        logits, states = _sample_inputs(case, seed)
        full = lambda v, t: torch.full((case["rows"],), v, dtype=t, device="cuda")  # noqa: E731
        s = dict(logits=logits, states=states, temperature=full(case["temperature"], torch.float32),
                 top_k=full(case["top_k"], torch.int32), top_p=full(case["top_p"], torch.float32),
                 token=full(0, torch.int32), prob=full(0.0, torch.float32))
    else:
        s = dict(rt=_runtime(case, seed), prompts=_prompts(case, seed))
    return dict(s, case=dict(case))


def _pack_mlp(c, case, s):
    h, f = MODELS[case["model"]][:2]
    w, rows, bf16 = s["w"], s["rows"], case["weights"] == "bf16"
    act = torch.bfloat16 if bf16 else torch.float32
    if bf16:
        s["w13"], s["w2"] = c.weight_pack_bf16_pair(w["w1"], w["w3"], h, f), c.weight_pack_bf16(w["w2"], f, h)
        s["s_w2"] = c.gemm_bf16_splits(rows, f, h)
    else:
        s["w13"], s["w2"] = c.weight_pack_pair(w["w1"], w["w3"], h, f), c.weight_pack(w["w2"], f, h, 32)
        s["s_w2"] = c.gemm_packed_splits(rows, f, h, 32)
    s["norm2"] = w["norm2"]
    s["act"] = torch.empty(rows, f, dtype=act, device="cuda")
    s["mlp_parts"] = torch.empty(s["s_w2"], rows, h, device="cuda")
    s["sum"] = torch.empty(rows, h, device="cuda")
    s["out"] = torch.empty(rows, h, dtype=act, device="cuda")
    if "q" not in s:
        del s["w"]


def _pack_layer(c, case, s):
    h, f, _, hq, hkv, _, _ = MODELS[case["model"]]
    w, rows, bf16, n = s["w"], s["rows"], case["weights"] == "bf16", (hq + 2 * hkv) * (h // hq)
    if bf16:
        s["wqkv"], s["wo"] = c.weight_pack_bf16_columns([w["wq"], w["wk"], w["wv"]], h), c.weight_pack_bf16(w["wo"], h, h)
        s["s_qkv"], s["s_wo"] = c.gemm_bf16_splits(rows, h, n), c.gemm_bf16_splits(rows, h, h)
        s["attn16"] = torch.empty(rows, h, dtype=torch.bfloat16, device="cuda")
    else:
        s["wqkv"], s["wo"] = c.weight_pack_columns([w["wq"], w["wk"], w["wv"]], h, 32), c.weight_pack(w["wo"], h, h, 32)
        s["s_qkv"], s["s_wo"] = c.gemm_packed_splits(rows, h, n, 32), c.gemm_packed_splits(rows, h, h, 32)
    s["norm1"] = w["norm1"]
    s["qkv_parts"] = torch.empty(s["s_qkv"], rows, n, device="cuda")
    s["wo_parts"] = torch.empty(s["s_wo"], rows, h, device="cuda")
    s["q"] = torch.empty(rows, hq, h // hq, device="cuda")
    s["attn"] = torch.empty(rows, hq, h // hq, device="cuda")
    s["mid"] = torch.empty(rows, h, device="cuda")
    s["normed"] = torch.empty(rows, h, dtype=torch.bfloat16 if bf16 else torch.float32, device="cuda")
    _pack_mlp(c, case, s)
    del s["w"]


# ---------------------------------------------------------------- one pass

def run(state):
    c, case = _ctx(), state["case"]
    return _RUN[case["op"]](c, case, state)


def _kv_dtype(case):
    return DTYPE_F32 if case["kv"] == "f32" else DTYPE_BF16


def _run_decode(c, case, s):
    c.attn_decode_paged(s["q"], s["k"], s["v"], _kv_dtype(case), s["tables"], s["lens"], s["max_ctx"],
                        case["kv_heads"], BLOCK, s["pool"], case["dim"] ** -0.5, s["out"])
    return s["out"]


def _prefill(c, case, s, q, out, hkv, scale):
    args = (s["tables"], s["cu"], s["lens"], s["max_new"], hkv, BLOCK, s["pool"], scale, out)
    if case["kv"] == "bf16" and not case.get("f32_math"):
        c.attn_prefill_paged_bf16(q, s["k"], s["v"], *args)
    else:
        c.attn_prefill_paged(q, s["k"], s["v"], _kv_dtype(case), *args)


def _run_prefill(c, case, s):
    _prefill(c, case, s, s["q"], s["out"], case["kv_heads"], case["dim"] ** -0.5)
    return s["out"]


def _mlp(c, case, s, x, residual):
    h, f = MODELS[case["model"]][:2]
    if case["weights"] == "bf16":
        c.gemm_bf16_swiglu(x, s["w13"], h, f, s["act"])
        c.gemm_bf16(s["act"], s["w2"], f, h, s["s_w2"], s["mlp_parts"])
    else:
        c.gemm_packed_swiglu(x, s["w13"], h, f, s["act"])
        c.gemm_packed(s["act"], s["w2"], f, h, 32, s["s_w2"], s["mlp_parts"])
    c.splitk_residual_rms_norm(s["mlp_parts"], s["s_w2"], None, residual, s["sum"], s["norm2"], s["out"], EPS)


def _run_mlp(c, case, s):
    _mlp(c, case, s, s["x"], s["residual"])
    return s["sum"], s["out"]


def _run_layer(c, case, s):
    h, _, _, hq, hkv, _, _ = MODELS[case["model"]]
    d, bf16 = h // hq, case["weights"] == "bf16"
    n, scale, positions = (hq + 2 * hkv) * d, d ** -0.5, int(s["cos"].shape[0])
    if bf16:
        c.gemm_bf16(s["x"], s["wqkv"], h, n, s["s_qkv"], s["qkv_parts"])
    else:
        c.gemm_packed(s["x"], s["wqkv"], h, n, 32, s["s_qkv"], s["qkv_parts"])
    if case["phase"] == "decode":
        c.attn_decode_paged_qkv(s["qkv_parts"], s["s_qkv"], s["biases"], s["positions"], s["cos"], s["sin"], d,
                                positions, s["slots"], s["k"], s["v"], _kv_dtype(case), s["tables"], s["lens"],
                                s["max_ctx"], hq, hkv, d, BLOCK, s["pool"], scale, s["attn"], s["q"])
    else:
        c.qkv_rope_append(s["qkv_parts"], s["s_qkv"], s["biases"], s["positions"], s["cos"], s["sin"], d, positions,
                          s["slots"], s["k"], s["v"], _kv_dtype(case), s["pool"], BLOCK, hq, hkv, d, s["q"])
        _prefill(c, case, s, s["q"], s["attn"], hkv, scale)
    attn = s["attn"].view(s["rows"], h)
    if bf16:
        c.convert_f32_to_bf16(attn, s["attn16"])
        c.gemm_bf16(s["attn16"], s["wo"], h, h, s["s_wo"], s["wo_parts"])
    else:
        c.gemm_packed(attn, s["wo"], h, h, 32, s["s_wo"], s["wo_parts"])
    c.splitk_residual_rms_norm(s["wo_parts"], s["s_wo"], None, s["residual"], s["mid"], s["norm1"], s["normed"], EPS)
    _mlp(c, case, s, s["normed"], s["mid"])
    return s["attn"], s["sum"], s["out"], s["k"], s["v"]


def _run_head(c, case, s):
    vocab = MODELS[case["model"]][5]
    (c.lm_head_argmax_bf16 if case["weights"] == "bf16" else c.lm_head_argmax_packed)(
        s["x"], s["w"], vocab, s["token"], s["prob"])
    return s["token"], s["prob"]


def _run_sample(c, case, s):
    c.sample_tokens(s["logits"], s["temperature"], s["top_k"], s["top_p"], s["states"], s["token"], s["prob"])
    return s["token"], s["prob"], s["states"]


def _run_serve(c, case, s):
    rt, order, got = s["rt"], {}, {}
    for p in s["prompts"]:
        order[rt.submit(p, max_new_tokens=case["tokens"])] = len(order)
    logits = None
    while rt.has_pending():
        _, updates = rt.execute_next_tick()
        for u in updates:
            if u["token"] is not None:
                got.setdefault(order[u["sequence_id"]], []).append((u["token"], u["probability"]))
        if logits is None:
            logits = rt.last_logits()  # the program scores the first answers' distributions
    tokens = np.array([[t for t, _ in got[i]] for i in range(len(order))], np.int64)
    probs = np.array([[p for _, p in got[i]] for i in range(len(order))], np.float32)
    return logits, probs, tokens


_RUN = dict(decode=_run_decode, prefill=_run_prefill, layer=_run_layer, mlp=_run_mlp, head=_run_head,
            sample=_run_sample, serve=_run_serve)


# ---------------------------------------------------------------- what a pass cannot do without

def _attention_work(case):
    hq, hkv, d = _heads(case)
    seqs = _sequences(case)
    size = 4 if case["kv"] == "f32" else 2
    kv = sum(p + n for p, n in seqs) * hkv * d * 2 * size
    flops = sum(4 * hq * d * (n * p + n * (n + 1) // 2) for p, n in seqs)
    return dict(bytes=kv + 8 * sum(n for _, n in seqs) * hq * d, flops=flops)


def _mlp_work(model, size, rows):
    h, f = MODELS[model][:2]
    return dict(bytes=3 * h * f * size + rows * h * (size + 4 + 4 + size), flops=6 * rows * h * f)


def work(case):
    op = case["op"]
    size = 4 if case.get("weights") == "f32" else 2
    if op in ("decode", "prefill"):
        return _attention_work(case)
    if op == "mlp":
        return _mlp_work(case["model"], size, case["rows"])
    if op == "layer":
        h, _, _, hq, hkv, _, _ = MODELS[case["model"]]
        rows, n = sum(k for _, k in _sequences(case)), (hq + 2 * hkv) * (h // hq)
        a, m = _attention_work(case), _mlp_work(case["model"], size, rows)
        return dict(bytes=a["bytes"] + m["bytes"] + h * (n + h) * size, flops=a["flops"] + m["flops"] + 2 * rows * h * (n + h))
    if op == "head":
        h, vocab = MODELS[case["model"]][0], MODELS[case["model"]][5]
        return dict(bytes=h * vocab * size + case["rows"] * h * size, flops=2 * case["rows"] * h * vocab)
    if op == "sample":
        return dict(bytes=4 * case["rows"] * case["vocab"], flops=2 * case["rows"] * case["vocab"])
    h, f, layers, hq, hkv, vocab, _ = MODELS[case["model"]]
    params = layers * (h * (hq + 2 * hkv) * (h // hq) + h * h + 3 * h * f)
    head, rows = h * vocab, sum(_spread(case["prompts"], case["min_prompt"], case["max_prompt"]))
    passes = case["tokens"]  # the prompts' pass gives the first token
    return dict(bytes=passes * (params + head) * size,
                flops=2 * params * (rows + (passes - 1) * case["prompts"]) + 2 * head * passes * case["prompts"])


def tolerance(case):
    """About four times the distance from the 64-bit result, or from the same sums in another
    order, over seeds and drawn sizes."""
    op = case["op"]
    bf16 = case.get("weights") == "bf16"
    if op == "decode":
        return {"rel": 2e-6, "max": 5e-5}
    if op == "prefill":  # the bf16 path rounds queries and probabilities to 8 bits
        if case["kv"] == "bf16" and not case.get("f32_math"):
            return {"rel": 1e-2, "max": 0.2}
        return {"rel": 2e-6, "max": 5e-5}
    if op in ("layer", "mlp"):
        if bf16 or case.get("kv") == "bf16":
            return {"rel": 1e-2, "max": 0.2}
        return {"rel": 2e-6, "max": 5e-5}
    if op == "head":
        return {"rel": 2e-3 if bf16 else 4e-6, "max": 2e-2 if bf16 else 1e-4}
    if op == "sample":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 2e-2, "max": 0.5} if bf16 else {"rel": 3e-5, "max": 1e-3}


# ---------------------------------------------------------------- the same in 64 bits

def exact(case, seed):
    op = case["op"]
    if op in ("decode", "prefill"):
        s = _attention_inputs(case, seed)
        return _attention64(s, s["q"].double(), s["k"], s["v"])
    if op == "mlp":
        w, x, residual = _mlp_inputs(case, seed)
        return _mlp64(w, x.double(), residual.double())
    if op == "layer":
        return _layer64(case, seed)
    if op == "head":
        w, x = _head_inputs(case, seed)
        best, total, token = None, None, None
        for at in range(0, w.shape[0], 16384):
            logits = x.double() @ w[at:at + 16384].double().t()
            m, i = logits.max(dim=1)
            e = (logits - m[:, None]).exp().sum(dim=1)
            if best is None:
                best, total, token = m, e, i
                continue
            top = torch.maximum(best, m)
            total = total * (best - top).exp() + e * (m - top).exp()
            token = torch.where(m > best, i + at, token)
            best = top
        return token.int(), 1.0 / total
    if op == "sample":
        return _sample64(case, seed)
    return None  # a whole generation: its tokens decide what it computes next


def _attention64(s, q, k, v):
    """Causal attention of every sequence's new rows over its own blocks, one kv head at a time."""
    hq, d = q.shape[1:]
    hkv = k.shape[1]
    out = torch.empty_like(q)
    at = 0
    for i, (prefix, new) in enumerate(s["seqs"]):
        n = prefix + new
        ids = s["tables"][i, :-(-n // BLOCK)].long()
        mask = torch.arange(n, device="cuda")[None, :] > prefix + torch.arange(new, device="cuda")[:, None]
        for j in range(hkv):
            keys = k[ids, j].reshape(-1, d)[:n].double()
            values = v[ids, j].reshape(-1, d)[:n].double()
            for head in range(j * (hq // hkv), (j + 1) * (hq // hkv)):
                scores = (q[at:at + new, head] @ keys.t()) * d ** -0.5
                out[at:at + new, head] = torch.softmax(scores.masked_fill(mask, -math.inf), dim=1) @ values
        at += new
    return out


def _norm64(x, w):
    return x / (x.square().mean(dim=1, keepdim=True) + EPS).sqrt() * w.double()


def _mlp64(w, x, residual):
    act = (x @ w["w1"].double()) * torch.nn.functional.silu(x @ w["w3"].double())
    total = residual + act @ w["w2"].double()
    return total, _norm64(total, w["norm2"])


def _layer64(case, seed):
    s = _layer_inputs(case, seed)
    w, x = s["w"], s["x"].double()
    h, _, _, hq, hkv, _, _ = MODELS[case["model"]]
    rows, d = x.shape[0], h // hq
    q, k, v = (x @ w[n].double() + b.double() for n, b in zip(("wq", "wk", "wv"), s["biases"]))
    at = s["positions"].long()
    cos, sin = s["cos"].double()[at][:, None], s["sin"].double()[at][:, None]

    def rope(t):
        a, b = t.view(rows, -1, d).chunk(2, dim=2)
        return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=2)

    block, offset = s["slots"] // BLOCK, s["slots"] % BLOCK
    pools = []
    for pool, new in ((s["k"], rope(k)), (s["v"], v.view(rows, hkv, d))):
        wide = pool.double()
        wide[block, :, offset] = new if pool.dtype == torch.float32 else new.to(pool.dtype).double()
        pools.append(wide)
    attn = _attention64(s, rope(q), *pools)
    mid = s["residual"].double() + attn.reshape(rows, h) @ w["wo"].double()
    total, out = _mlp64(w, _norm64(mid, w["norm1"]), mid)
    return attn, total, out, pools[0], pools[1]


def _sample64(case, seed):
    logits, states = _sample_inputs(case, seed)
    k = min(case["top_k"], case["vocab"])
    top, ids = torch.topk(logits, k, dim=1)
    top, ids, states = top.double().cpu().numpy(), ids.cpu().numpy(), states.cpu().numpy().astype(np.uint64)
    temperature, top_p = float(np.float32(case["temperature"])), float(np.float32(case["top_p"]))
    tokens, probs = np.zeros(len(ids), np.int32), np.zeros(len(ids))
    after = np.zeros(len(ids), np.int64)
    for r in range(len(ids)):
        weight = np.exp((top[r] - top[r, 0]) / temperature)
        sums = np.cumsum(weight)
        kept = min(k, int(np.searchsorted(sums, sums[-1] * min(top_p, 1.0))) + 1)
        x = int(states[r])
        x ^= x >> 12
        x = (x ^ (x << 25)) & ((1 << 64) - 1)
        x ^= x >> 27
        after[r] = x - (1 << 64) if x >> 63 else x
        u = (((x * 0x2545F4914F6CDD1D) & ((1 << 64) - 1)) >> 40) / float(1 << 24)
        at = min(int(np.searchsorted(sums[:kept], u * sums[kept - 1])), kept - 1)
        tokens[r], probs[r] = ids[r, at], weight[at] / sums[kept - 1]
    return tokens, probs, after
