"""Performance cases of the embedding engine, through its public entry points.

A case is one call a program makes again and again:

* kind "model": texts through a loaded encoder (Model.embed with host ids,
  Model.embed_tokens for per-token vectors, Model.embed_device with ids and
  vectors in HBM);
* kind "linear": one dense layer (tensor.Linear, bias and activation fused);
* kind "attention": one attention layer over packed texts (tensor.Attention).

Model shapes are the synthetic.py configurations. Where a case names fewer
layers than the model has, they are whole layers of that model: a forward
repeats them. Embedding tables are cut to VOCAB rows (only the rows a batch
names are read). Weights are N(0, 1/K), so activations stay O(1) through the
layers and attention is neither flat nor one-hot.
"""
import dataclasses
import math
import random

import numpy as np
import torch

VOCAB = 16384
# mode names -> RH_QUANT_* / RH_MODE_* values (the two enumerations agree)
QUANT = {"fp32": 0, "w8": 1, "int8": 2}
ACT = {"none": 0, "gelu": 1}
BERT_FAMILY = ("minilm", "bert", "distilbert", "mpnet")
FAMILIES = BERT_FAMILY + ("nomic", "modernbert", "qwen3", "gemma")


def _model(name, family, quant, entry, layers, batch, len_lo, len_hi):
    return {"name": name, "kind": "model", "family": family, "quant": quant, "entry": entry,
            "layers": layers, "batch": batch, "len_lo": len_lo, "len_hi": len_hi}


def listed():
    return [
        # A search query against a small index: one short text, weight-only
        # int8 MiniLM, whole model. The smallest call there is; latency counts.
        _model("minilm-w8-query", "minilm", "w8", "embed", 6, 1, 11, 11),
        # A question to a BERT-base index, full int8, whole model.
        _model("bert-int8-query", "bert", "int8", "embed", 12, 1, 28, 28),
        # A query with its instruction prefix through the decoder embedder,
        # four of its layers.
        _model("qwen3-w8-query", "qwen3", "w8", "embed", 4, 1, 45, 45),
        # A page of search results or chat turns re-embedded at once, at the
        # default fp32 precision.
        _model("mpnet-fp32-turns", "mpnet", "fp32", "embed", 4, 8, 9, 70),
        # Per-token vectors (late interaction, highlighting) of passages.
        _model("minilm-fp32-tokens", "minilm", "fp32", "embed_tokens", 6, 32, 16, 128),
        # Index building: the 64 x 256 document batch of the benchmark, whole
        # model, ids and vectors resident on the device.
        _model("bert-int8-docs", "bert", "int8", "embed_device", 12, 64, 64, 256),
        # Long documents: two texts near the 8192-token limit, one global and
        # one local layer.
        _model("modernbert-w8-long", "modernbert", "w8", "embed_device", 2, 2, 5003, 8192),
        # Documents through the decoder embedder at the default fp32 precision.
        _model("qwen3-fp32-docs", "qwen3", "fp32", "embed_device", 2, 12, 97, 512),
        # Documents through the bidirectional Gemma embedder: default fp32,
        # and the 16 x 2048 weight-only int8 batch of the benchmark (one local
        # and one global layer each).
        _model("gemma-fp32-docs", "gemma", "fp32", "embed_device", 2, 6, 300, 2048),
        _model("gemma-w8-docs", "gemma", "w8", "embed_device", 2, 16, 2048, 2048),
        # One dense layer with its GELU on a ragged number of rows, full int8.
        {"name": "linear-int8-gelu", "kind": "linear", "mode": "int8", "act": "gelu",
         "m": 1213, "k": 768, "n": 3072},
        # One attention layer on fp32 rows at fp32-grade precision, ragged
        # passages, 16 heads of 64.
        {"name": "attention-fp32", "kind": "attention", "dh": 64, "heads": 16, "kv_heads": 16,
         "causal": False, "window": 0, "precision": 3, "batch": 24, "len_lo": 33,
         "len_hi": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    if pick < 0.65:
        family = rng.choice(FAMILIES)
        quant = rng.choice(list(QUANT))
        entry = rng.choice(("embed", "embed_tokens", "embed_device"))
        longest = {"modernbert": 4096, "nomic": 2048, "qwen3": 2048, "gemma": 2048}.get(family, 512)
        hi = _log_int(rng, 4, longest)
        lo = max(1, int(hi * rng.uniform(0.15, 1.0)))
        batch = _log_int(rng, 1, max(1, min(48, 12288 // hi)))
        return {"kind": "model", "family": family, "quant": quant, "entry": entry, "layers": 2,
                "batch": batch, "len_lo": lo, "len_hi": hi}
    if pick < 0.85:
        return {"kind": "linear", "mode": rng.choice(list(QUANT)),
                "act": rng.choice(list(ACT)), "m": _log_int(rng, 1, 12288),
                "k": _log_int(rng, 200, 3200), "n": 16 * _log_int(rng, 20, 256)}
    dh = rng.choice((32, 64, 128, 256))
    kv = rng.choice((1, 2, 4)) * (2 if dh < 128 else 1)
    # 4 is the reference's own order: full attention with as many kv heads
    precision = rng.choice((1, 3, 3, 4) if dh < 256 else (1, 3))
    group = 1 if precision == 4 else rng.choice((1, 2, 3))
    hi = _log_int(rng, 8, 2048)
    plain = precision == 4
    return {"kind": "attention", "dh": dh, "heads": kv * group, "kv_heads": kv,
            "causal": False if plain else rng.random() < 0.3,
            "window": 0 if plain else rng.choice((0, 0, 65, 257)), "precision": precision,
            "batch": _log_int(rng, 1, max(1, min(48, 12288 // hi))),
            "len_lo": max(1, int(hi * rng.uniform(0.15, 1.0))), "len_hi": hi}


# ---- inputs -------------------------------------------------------------------------

def _shape(case):
    from rembed_amd import synthetic as S
    base = {"minilm": S.MINILM_L6, "bert": S.BERT_BASE, "distilbert": S.DISTILBERT_BASE,
            "mpnet": S.MPNET_BASE, "nomic": S.NOMIC_V15, "modernbert": S.MODERNBERT_BASE,
            "qwen3": S.QWEN3_0_6B, "gemma": S.GEMMA3_300M}[case["family"]]
    more = {"layers": case["layers"], "vocab": VOCAB}
    if case["family"] == "gemma" and case["layers"] < base.sliding_pattern:
        more["sliding_pattern"] = case["layers"]  # the last layer is the global one
    return dataclasses.replace(base, **more)


def _lens(case):
    """The texts' lengths: part of the case, not of the seed."""
    r = random.Random("%d %d %d" % (case["batch"], case["len_lo"], case["len_hi"]))
    lens = [r.randint(case["len_lo"], case["len_hi"]) for _ in range(case["batch"])]
    lens[0] = case["len_hi"]
    return lens


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _tensors(case, seed):
    """HF-named float32 tensors of the case's model, on the GPU."""
    s, g = _shape(case), _gen(2 * seed)
    fam, H, I = case["family"], s.hidden, s.intermediate

    def mat(n, k):
        return torch.randn(n, k, generator=g, device="cuda") * (1.0 / math.sqrt(k))

    def vec(n, at=0.0):
        return torch.randn(n, generator=g, device="cuda") * 0.05 + at

    def table(n):
        return torch.randn(n, H, generator=g, device="cuda") * (1.0 / math.sqrt(H))

    t = {}
    if fam in BERT_FAMILY:
        t["embeddings.word_embeddings.weight"] = table(s.vocab)
        t["embeddings.position_embeddings.weight"] = table(s.max_position)
        if s.type_vocab:
            t["embeddings.token_type_embeddings.weight"] = table(s.type_vocab)
        t["embeddings.LayerNorm.weight"], t["embeddings.LayerNorm.bias"] = vec(H, 1.0), vec(H)
        for l in range(s.layers):
            for nm, (n, k) in zip(_bert_names(fam, l), ((H, H),) * 4 + ((I, H), (H, I))):
                t[nm + ".weight"], t[nm + ".bias"] = mat(n, k), vec(n)
            for nm in _bert_norms(fam, l):
                t[nm + ".weight"], t[nm + ".bias"] = vec(H, 1.0), vec(H)
        if s.rel_buckets:
            t["encoder.relative_attention_bias.weight"] = torch.randn(
                s.rel_buckets, s.heads, generator=g, device="cuda") * 0.5
    elif fam == "nomic":
        t["embeddings.word_embeddings.weight"] = table(s.vocab)
        t["embeddings.token_type_embeddings.weight"] = table(2)
        t["emb_ln.weight"], t["emb_ln.bias"] = vec(H, 1.0), vec(H)
        for l in range(s.layers):
            p = f"encoder.layers.{l}."
            t[p + "attn.Wqkv.weight"], t[p + "attn.out_proj.weight"] = mat(3 * H, H), mat(H, H)
            t[p + "mlp.fc11.weight"], t[p + "mlp.fc12.weight"] = mat(I, H), mat(I, H)
            t[p + "mlp.fc2.weight"] = mat(H, I)
            for nm in ("norm1", "norm2"):
                t[p + nm + ".weight"], t[p + nm + ".bias"] = vec(H, 1.0), vec(H)
    elif fam == "modernbert":
        t["embeddings.tok_embeddings.weight"] = table(s.vocab)
        t["embeddings.norm.weight"], t["final_norm.weight"] = vec(H, 1.0), vec(H, 1.0)
        for l in range(s.layers):
            p = f"layers.{l}."
            if l:
                t[p + "attn_norm.weight"] = vec(H, 1.0)
            t[p + "attn.Wqkv.weight"], t[p + "attn.Wo.weight"] = mat(3 * H, H), mat(H, H)
            t[p + "mlp_norm.weight"] = vec(H, 1.0)
            t[p + "mlp.Wi.weight"], t[p + "mlp.Wo.weight"] = mat(2 * I, H), mat(H, I)
    else:
        gemma = fam == "gemma"
        one = 0.0 if gemma else 1.0  # Gemma's checkpoints hold the weight less one
        qd, kvd = s.heads * s.head_dim, s.kv_heads * s.head_dim
        t["embed_tokens.weight"], t["norm.weight"] = table(s.vocab), vec(H, one)
        for l in range(s.layers):
            p = f"layers.{l}."
            t[p + "input_layernorm.weight"] = vec(H, one)
            t[p + "self_attn.q_proj.weight"] = mat(qd, H)
            t[p + "self_attn.k_proj.weight"] = mat(kvd, H)
            t[p + "self_attn.v_proj.weight"] = mat(kvd, H)
            t[p + "self_attn.o_proj.weight"] = mat(H, qd)
            t[p + "self_attn.q_norm.weight"] = vec(s.head_dim, one)
            t[p + "self_attn.k_norm.weight"] = vec(s.head_dim, one)
            t[p + "post_attention_layernorm.weight"] = vec(H, one)
            if gemma:
                t[p + "pre_feedforward_layernorm.weight"] = vec(H, one)
                t[p + "post_feedforward_layernorm.weight"] = vec(H, one)
            t[p + "mlp.gate_proj.weight"], t[p + "mlp.up_proj.weight"] = mat(I, H), mat(I, H)
            t[p + "mlp.down_proj.weight"] = mat(H, I)
        if gemma:
            t["2_Dense.linear.weight"] = mat(s.dense_hidden, H)
            t["3_Dense.linear.weight"] = mat(H, s.dense_hidden)
    return t


def _bert_names(fam, l):
    """q, k, v, o, FFN1 and FFN2 of one BERT-family layer."""
    if fam == "distilbert":
        p = f"transformer.layer.{l}."
        return [p + "attention.%s_lin" % n for n in ("q", "k", "v", "out")] + [p + "ffn.lin1",
                                                                               p + "ffn.lin2"]
    p = f"encoder.layer.{l}."
    if fam == "mpnet":
        a = [p + "attention.attn.%s" % n for n in ("q", "k", "v", "o")]
    else:
        a = [p + "attention.self.%s" % n for n in ("query", "key", "value")]
        a.append(p + "attention.output.dense")
    return a + [p + "intermediate.dense", p + "output.dense"]


def _bert_norms(fam, l):
    if fam == "distilbert":
        return [f"transformer.layer.{l}.sa_layer_norm", f"transformer.layer.{l}.output_layer_norm"]
    p = f"encoder.layer.{l}."
    return [p + ("attention.LayerNorm" if fam == "mpnet" else "attention.output.LayerNorm"),
            p + "output.LayerNorm"]


def _ids(case, seed):
    r = np.random.default_rng(seed)
    lens = np.array(_lens(case), np.int32)
    ids = np.zeros((len(lens), int(lens.max())), np.int64)
    for b, n in enumerate(lens):
        ids[b, :n] = r.integers(4, VOCAB, size=n)
    return ids, lens


def _linear_inputs(case, seed):
    g = _gen(2 * seed + 1)
    m, k, n = case["m"], case["k"], case["n"]
    a = torch.randn(m, k, generator=g, device="cuda")
    # a few strong features, as normalized activations have
    a[:, :: max(1, k // 6)] *= 4.0
    w = torch.randn(n, k, generator=g, device="cuda") * (1.0 / math.sqrt(k))
    b = torch.randn(n, generator=g, device="cuda") * 0.05
    return a, w, b


def _attention_inputs(case, seed):
    lens = _lens(case)
    width = (case["heads"] + 2 * case["kv_heads"]) * case["dh"]
    rows = torch.randn(sum(lens), width, generator=_gen(2 * seed + 1), device="cuda")
    if case["precision"] == 1:
        rows = rows.to(torch.bfloat16)
    return rows, lens


class _Dev:
    """A torch tensor where the entry points take a device buffer."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


_context = []


def _ctx():
    """The program's one context (one stream), as a server holds it."""
    from rembed_amd import tensor as T
    if not _context:
        _context.append(T.Context(0))
    return _context[0]


def prepare(case, seed):
    from rembed_amd import tensor as T
    from rembed_amd.model import Model
    ctx = _ctx()
    if case["kind"] == "model":
        host = {k: v.cpu().numpy() for k, v in _tensors(case, seed).items()}
        st = {"model": Model(ctx, _shape(case), host, QUANT[case["quant"]]),
              "entry": case["entry"]}
        st["ids"], st["lens"] = _ids(case, seed)
        if case["entry"] == "embed_device":
            st["ids_dev"] = _Dev(torch.from_numpy(st["ids"].astype(np.int32)).cuda())
            st["out"] = _Dev(torch.empty(len(st["lens"]), st["model"].shape.hidden,
                                         device="cuda"))
    elif case["kind"] == "linear":
        a, w, b = _linear_inputs(case, seed)
        m, k, n = case["m"], case["k"], case["n"]
        st = {"ctx": ctx, "m": m, "act": ACT[case["act"]], "a": _Dev(a),
              "w": T.PackedWeight(ctx, QUANT[case["mode"]], w.cpu().numpy(), k, n,
                                  b.cpu().numpy()),
              "dst": _Dev(torch.empty(m, n, device="cuda"))}
        if case["mode"] == "int8":
            st["ldq"] = T.ldq_for(k)
            st["qa"] = _Dev(torch.empty(m, st["ldq"], dtype=torch.uint8, device="cuda"))
            st["rs"] = _Dev(torch.empty(m, device="cuda"))
    else:
        rows, lens = _attention_inputs(case, seed)
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        st = {"ctx": ctx, "case": case, "rows": _Dev(rows), "max_len": max(lens),
              "cu": _Dev(torch.from_numpy(cu).cuda()),
              "out": _Dev(torch.empty(sum(lens), case["heads"] * case["dh"], device="cuda"))}
    torch.cuda.synchronize()  # the context's stream does not wait for torch's
    return st


def run(st):
    from rembed_amd import tensor as T
    if "model" in st:
        if st["entry"] == "embed":
            return st["model"].embed(st["ids"], st["lens"])
        if st["entry"] == "embed_tokens":
            return st["model"].embed_tokens(st["ids"], st["lens"])
        batch, stride = st["ids"].shape
        st["model"].embed_device(st["ids_dev"], st["lens"], batch, stride, st["out"])
        return st["out"].tensor
    if "w" in st:
        T.Linear(st["ctx"], st["dst"], st["a"], st["w"], st["m"], st["act"], st.get("qa"),
                 st.get("ldq", 0), st.get("rs"))
        return st["dst"].tensor
    c = st["case"]
    q, kv = c["heads"] * c["dh"], c["kv_heads"] * c["dh"]
    T.Attention(st["ctx"], st["out"], q, st["rows"], c["precision"] == 1, q + 2 * kv, 0, q,
                q + kv, st["cu"], c["batch"], st["max_len"], c["heads"], c["kv_heads"], c["dh"],
                1.0 / math.sqrt(c["dh"]), c["causal"], c["window"], c["precision"])
    return st["out"].tensor


# ---- what a pass cannot do without ----------------------------------------------------

def _pairs(n, causal, window):
    """(query, key) pairs that attend in a text of n tokens."""
    left = min(n, window) if window else n
    tri = left * (left + 1) // 2 + (n - left) * left  # keys at or before the query
    return tri if causal else 2 * tri - n


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        each = {"fp32": 4, "w8": 1, "int8": 1}[case["mode"]]
        return {"bytes": 4 * m * k + each * n * k + 8 * n + 4 * m * n, "flops": 2 * m * k * n}
    lens = _lens(case)
    if case["kind"] == "attention":
        c, each = case, 2 if case["precision"] == 1 else 4
        rows = sum(lens)
        pairs = sum(_pairs(n, c["causal"], c["window"]) for n in lens)
        return {"bytes": rows * c["dh"] * (each * (c["heads"] + 2 * c["kv_heads"])
                                           + 4 * c["heads"]),
                "flops": 4 * pairs * c["dh"] * c["heads"]}
    s, fam, M = _shape(case), case["family"], sum(lens)
    H, I = s.hidden, s.intermediate
    dh = getattr(s, "head_dim", H // s.heads)
    qd, kvd = s.heads * dh, getattr(s, "kv_heads", s.heads) * dh
    per = H * (qd + 2 * kvd) + qd * H + (2 if fam in BERT_FAMILY else 3) * H * I
    flops = 2 * M * per * s.layers
    for l in range(s.layers):
        window = 0
        if fam == "gemma" and (l + 1) % s.sliding_pattern:
            window = s.sliding_window
        if fam == "modernbert" and l % s.global_every:
            window = s.local_attention // 2 + 1
        flops += 4 * qd * sum(_pairs(n, fam == "qwen3", window) for n in lens)
    rows = M if case["entry"] == "embed_tokens" else len(lens)
    each = 4 if case["quant"] == "fp32" else 1
    return {"bytes": each * per * s.layers + 4 * M * H + 8 * M + 4 * rows * H, "flops": flops}


def tolerance(case):
    """About four times what each path is off its value in 64 bits: sums in
    another order stay well inside. In whole models a rounding that differs in
    one layer (of bf16 operands, or of int8 rows at a tie) moves the rest."""
    if case["kind"] == "linear":
        return {"rel": {"fp32": 4e-5, "w8": 8e-3, "int8": 1e-6}[case["mode"]]}
    if case["kind"] == "attention":
        return {"rel": {1: 1e-2, 3: 3e-5, 4: 4e-6}[case["precision"]]}
    return {"rel": {"fp32": 8e-5, "w8": 1e-2, "int8": 3e-2}[case["quant"]]}


# ---- the same in 64 bits ----------------------------------------------------------------

def _dense(quant, x, w, b=None):
    """x·wᵀ + b in 64 bits. The integers of "w8" and "int8" are part of what the
    modes mean: per output channel for the weights, per row ("int8") for x,
    their scales held in 32 bits."""
    w = w.double()
    if quant != "fp32":
        s = w.abs().amax(1, keepdim=True) / 127
        s = torch.where(s == 0, torch.ones_like(s), s)
        if quant == "w8":
            s = s.float().double()
        w = torch.round(w / s).clamp(-127, 127) * s.float().double()
    if quant == "int8":
        r = x.float()
        s = r.abs().amax(1, keepdim=True) / 127
        s = torch.where(s == 0, torch.ones_like(s), s)
        x = torch.round(r * (1 / s)).clamp(-128, 127).double() * s.double()
    y = x @ w.t()
    return y if b is None else y + b.double()


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def _layer_norm(x, w, b, eps):
    x = x - x.mean(1, keepdim=True)
    x = x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * w.double()
    return x if b is None else x + b.double()


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, theta):
    n, dh = x.shape
    f = theta ** (-torch.arange(0, dh, 2, dtype=torch.float64, device=x.device) / dh)
    a = torch.arange(n, dtype=torch.float64, device=x.device)[:, None] * f[None]
    c, s = torch.cos(a), torch.sin(a)
    u, v = x[:, : dh // 2], x[:, dh // 2:]
    return torch.cat([u * c - v * s, v * c + u * s], 1)


def _attend(q, k, v, scale, causal=False, window=0, bias=None):
    """One head of one text, [n][dh] each."""
    n = q.shape[0]
    i = torch.arange(n, device=q.device)
    out = torch.empty_like(q)
    for r in range(0, n, 2048):  # bounded score rows
        s = (q[r:r + 2048] @ k.t()) * scale
        if bias is not None:
            s = s + bias[r:r + 2048]
        d = i[r:r + 2048, None] - i[None, :]
        if causal:
            s = s.masked_fill(d < 0, -math.inf)
        if window:
            s = s.masked_fill(d.abs() >= window, -math.inf)
        out[r:r + 2048] = torch.softmax(s, 1) @ v
    return out


def _heads(rows, lens, heads, kv, dh, scale, causal=False, window=0, bias=None, prep=None):
    """Attention over packed q|k|v rows; prep(x, is_query) treats each head's rows."""
    out = torch.empty(rows.shape[0], heads * dh, dtype=rows.dtype, device=rows.device)
    r0 = 0
    for n in lens:
        t = rows[r0:r0 + n]
        for h in range(heads):
            g = h // (heads // kv)
            q = t[:, h * dh:(h + 1) * dh]
            k = t[:, (heads + g) * dh:(heads + g + 1) * dh]
            v = t[:, (heads + kv + g) * dh:(heads + kv + g + 1) * dh]
            if prep is not None:
                q, k = prep(q, True), prep(k, False)
            out[r0:r0 + n, h * dh:(h + 1) * dh] = _attend(
                q, k, v, scale, causal, window, None if bias is None else bias(n, h))
        r0 += n
    return out


def _mpnet_bias(table, buckets):
    half = buckets // 2
    small = half // 2

    def bucket(d):  # d: query less key
        at, a = (half if d < 0 else 0), abs(d)
        if a >= small:
            a = min(half - 1, small + int(math.log(a / small) / math.log(128.0 / small)
                                          * (half - small)))
        return at + a

    made = {}

    def bias(n, h):
        if n not in made:
            i = torch.arange(n, device=table.device)
            row = torch.tensor([bucket(d) for d in range(1 - n, n)], device=table.device)
            made[n] = row[i[:, None] - i[None, :] + n - 1]
        return table.double()[made[n], h]
    return bias


def _exact_bert(case, s, t, ids, lens, q):
    fam, eps, dh = case["family"], s.eps, s.hidden // s.heads
    at = torch.cat([torch.arange(n, device="cuda") for n in lens])
    x = t["embeddings.word_embeddings.weight"].double()[ids]
    x = x + t["embeddings.position_embeddings.weight"].double()[at + s.position_offset]
    if s.type_vocab:
        x = x + t["embeddings.token_type_embeddings.weight"][0].double()
    x = _layer_norm(x, t["embeddings.LayerNorm.weight"], t["embeddings.LayerNorm.bias"], eps)
    bias = None
    if s.rel_buckets:
        bias = _mpnet_bias(t["encoder.relative_attention_bias.weight"], s.rel_buckets)
    for l in range(s.layers):
        wq, wk, wv, wo, w1, w2 = [(t[n + ".weight"], t[n + ".bias"]) for n in _bert_names(fam, l)]
        n1, n2 = [(t[n + ".weight"], t[n + ".bias"]) for n in _bert_norms(fam, l)]
        rows = torch.cat([_dense(q, x, *w) for w in (wq, wk, wv)], 1)
        c = _heads(rows, lens, s.heads, s.heads, dh, 1 / math.sqrt(dh), bias=bias)
        x = _layer_norm(x + _dense(q, c, *wo), *n1, eps)
        x = _layer_norm(x + _dense(q, _gelu(_dense(q, x, *w1)), *w2), *n2, eps)
    return x


def _exact_rope(case, s, t, ids, lens, q):
    fam, eps, H, I = case["family"], s.eps, s.hidden, s.intermediate
    dh, heads = s.head_dim, s.heads
    if fam in ("nomic", "modernbert"):
        word = "word" if fam == "nomic" else "tok"
        x = t["embeddings.%s_embeddings.weight" % word].double()[ids]
        if fam == "nomic":
            x = x + t["embeddings.token_type_embeddings.weight"][0].double()
            x = _layer_norm(x, t["emb_ln.weight"], t["emb_ln.bias"], eps)
        else:
            x = _layer_norm(x, t["embeddings.norm.weight"], None, eps)
        for l in range(s.layers):
            p = ("encoder.layers.%d." if fam == "nomic" else "layers.%d.") % l
            local = fam == "modernbert" and l % s.global_every
            theta = s.rope_local_theta if local else s.rope_theta
            h = x
            if fam == "modernbert" and l:
                h = _layer_norm(x, t[p + "attn_norm.weight"], None, eps)
            c = _heads(_dense(q, h, t[p + "attn.Wqkv.weight"]), lens, heads, heads, dh,
                       1 / math.sqrt(dh), window=s.local_attention // 2 + 1 if local else 0,
                       prep=lambda y, _: _rope(y, theta))
            if fam == "nomic":
                x = _layer_norm(x + _dense(q, c, t[p + "attn.out_proj.weight"]),
                                t[p + "norm1.weight"], t[p + "norm1.bias"], eps)
                m = _dense(q, x, t[p + "mlp.fc11.weight"])
                g = _dense(q, x, t[p + "mlp.fc12.weight"])
                m = m * g * torch.sigmoid(g)
                x = _layer_norm(x + _dense(q, m, t[p + "mlp.fc2.weight"]),
                                t[p + "norm2.weight"], t[p + "norm2.bias"], eps)
            else:
                x = x + _dense(q, c, t[p + "attn.Wo.weight"])
                u = _dense(q, _layer_norm(x, t[p + "mlp_norm.weight"], None, eps),
                           t[p + "mlp.Wi.weight"])
                x = x + _dense(q, _gelu(u[:, :I]) * u[:, I:], t[p + "mlp.Wo.weight"])
        return x if fam == "nomic" else _layer_norm(x, t["final_norm.weight"], None, eps)
    gemma = fam == "gemma"
    one = 1.0 if gemma else 0.0
    scale = 1 / math.sqrt(s.query_pre_attn_scalar if gemma else dh)
    x = t["embed_tokens.weight"].double()[ids]
    if gemma:
        x = x * float(np.float32(math.sqrt(H)))
    for l in range(s.layers):
        p = f"layers.{l}."
        def norm(y, name):
            return _rms(y, t[p + name + ".weight"].double() + one, eps)
        local = gemma and (l + 1) % s.sliding_pattern
        theta = s.rope_local_theta if local else s.rope_theta
        h = norm(x, "input_layernorm")
        rows = torch.cat([_dense(q, h, t[p + f"self_attn.{n}_proj.weight"]) for n in "qkv"], 1)
        c = _heads(rows, lens, heads, s.kv_heads, dh, scale, causal=not gemma,
                   window=s.sliding_window if local else 0,
                   prep=lambda y, is_q: _rope(norm(y, "self_attn.q_norm" if is_q
                                                   else "self_attn.k_norm"), theta))
        c = _dense(q, c, t[p + "self_attn.o_proj.weight"])
        x = x + (norm(c, "post_attention_layernorm") if gemma else c)
        h = norm(x, "pre_feedforward_layernorm" if gemma else "post_attention_layernorm")
        g = _dense(q, h, t[p + "mlp.gate_proj.weight"])
        u = _dense(q, h, t[p + "mlp.up_proj.weight"])
        if gemma:
            g = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))
        else:
            g = g * torch.sigmoid(g)
        c = _dense(q, g * u, t[p + "mlp.down_proj.weight"])
        x = x + (norm(c, "post_feedforward_layernorm") if gemma else c)
    return _rms(x, t["norm.weight"].double() + one, eps)


def exact(case, seed):
    if case["kind"] == "linear":
        a, w, b = _linear_inputs(case, seed)
        y = _dense(case["mode"], a.double(), w, b)
        return _gelu(y) if case["act"] == "gelu" else y
    if case["kind"] == "attention":
        c = case
        rows, lens = _attention_inputs(c, seed)
        return _heads(rows.double(), lens, c["heads"], c["kv_heads"], c["dh"],
                      1 / math.sqrt(c["dh"]), c["causal"], c["window"])
    s, t = _shape(case), _tensors(case, seed)
    padded, lens = _ids(case, seed)
    lens = [int(n) for n in lens]
    ids = torch.from_numpy(np.concatenate([padded[b, :n] for b, n in enumerate(lens)])).cuda()
    body = _exact_bert if case["family"] in BERT_FAMILY else _exact_rope
    texts = torch.split(body(case, s, t, ids, lens, case["quant"]), lens)
    if case["entry"] == "embed_tokens":
        return list(texts)
    pool = {0: lambda y: y.mean(0), 1: lambda y: y[0], 2: lambda y: y[-1]}[s.pooling]
    v = torch.stack([pool(y) for y in texts])
    if case["family"] == "gemma":
        v = v @ t["2_Dense.linear.weight"].double().t() @ t["3_Dense.linear.weight"].double().t()
    if s.normalize:
        v = v / v.norm(dim=1, keepdim=True)
    v = v.cpu().numpy() if case["entry"] == "embed" else v
    return v
