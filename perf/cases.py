"""The work that is timed: whole decode steps, and the single layers a program composes from the device-pointer
launches.

Each case is a dict of plain values; its ``op`` names one of four kinds of work:

* ``decode``: an ``Engine`` over a model file, a fresh sequence, one ``step`` per token.  ``logits`` "last" is a prompt
  fed without waiting (and, since a step is the same launch, generation over the same contexts), whose last step
  returns its logits; "every" is the perplexity loop through the C entry point, which collects every step's logits in
  the program's own buffer.
* ``mlp``: a stack of feed-forward blocks (norm, gate_up with SwiGLU, down onto the residual stream).
* ``matvec``: one projection per layer of a stack, each layer with weights of its own.
* ``attention``: single-token attention over each layer's fp16 KV cache, with the caller's scratch or the library's.

A stack has one set of weights (or caches) per layer, as a model does, so a layer's bytes come from memory and not from
the cache that its last pass left.
"""
import ctypes
import functools
import math
import tempfile

import numpy as np
import torch

from cudallm_amd import engine as E
from cudallm_amd import format as fmt

EPS = 1e-5
HEAD_DIM = 64
GROUP = 128  # columns of an int4 scale
HIDDEN, INTER, LAYERS, HEADS, KV_HEADS, VOCAB = 2048, 8192, 16, 32, 8, 128256  # the engine's one model shape
QKV = (HEADS + 2 * KV_HEADS) * HEAD_DIM
MODEL_SEED = 29  # a program serves one model: the seed of a case picks its tokens
MAX_SEQ = 4096


def listed():
    return [
        # A chat turn: a short prompt and its continuation, contexts 1 to 272 (the benchmark's 16 + 256 tokens).
        dict(name="decode_bf16", op="decode", wtype="bf16", tokens=272, logits="last"),
        # Scoring text: the logits of every position go back to the host.
        dict(name="score_int4", op="decode", wtype="int4", tokens=96, logits="every"),
        # The smallest call: one key projection, alone.
        dict(name="key_bf16", op="matvec", wtype="bf16", rows=512, cols=2048, epilogue="store", norm=True, layers=1),
        # The fused query, key and value projection of 16 layers.
        dict(name="qkv_int8", op="matvec", wtype="int8", rows=3072, cols=2048, epilogue="store", norm=True, layers=16),
        # The feed-forward blocks of 16 layers, most of a model's bytes, in each weight type.
        dict(name="mlp_bf16", op="mlp", wtype="bf16", hidden=2048, inter=8192, layers=16),
        dict(name="mlp_int8", op="mlp", wtype="int8", hidden=2048, inter=8192, layers=16),
        dict(name="mlp_int4", op="mlp", wtype="int4", hidden=2048, inter=8192, layers=16),
        # The output projection: one call over the whole vocabulary.
        dict(name="head_int8", op="matvec", wtype="int8", rows=128256, cols=2048, epilogue="store", norm=True, layers=1),
        # A wider model's feed-forward blocks, at widths that are not 2048 or 8192.
        dict(name="mlp_wide_int4", op="mlp", wtype="int4", hidden=4096, inter=12288, layers=4),
        # Attention early in a chat, late in a long one, and at the longest context.
        dict(name="attention_100", op="attention", kv_heads=8, ctx=100, max_seq=4096, layers=16, scratch="library"),
        dict(name="attention_8000", op="attention", kv_heads=8, ctx=8000, max_seq=8192, layers=16, scratch="library"),
        dict(name="attention_131071", op="attention", kv_heads=8, ctx=131071, max_seq=131072, layers=2, scratch="caller"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(("decode", "mlp", "matvec", "matvec", "attention", "attention"))
    wtype = rng.choice(("bf16", "int8", "int4"))
    if op == "decode":
        if rng.random() < 0.5:
            return dict(op=op, wtype=wtype, tokens=_log_int(rng, 8, 272), logits="last")
        return dict(op=op, wtype=wtype, tokens=_log_int(rng, 4, 96), logits="every")
    if op == "mlp":
        hidden = rng.choice((1024, 2048, 2048, 3072, 4096))
        inter = rng.choice((3072, 4096, 8192, 8192, 11264, 12288))
        return dict(op=op, wtype=wtype, hidden=hidden, inter=inter, layers=rng.randint(1, 16))
    if op == "matvec":
        epilogue = rng.choice(("store", "add", "swiglu"))
        rows = _log_int(rng, 64, 32768)
        if epilogue == "swiglu":
            rows += rows % 2
        cols = 1024 * rng.choice((1, 2, 2, 2, 3, 4, 5, 6, 8, 8, 10, 12))
        return dict(op=op, wtype=wtype, rows=rows, cols=cols, epilogue=epilogue, norm=rng.random() < 0.5,
                    layers=rng.randint(1, 16))
    ctx = _log_int(rng, 1, 131072)
    max_seq = -(-ctx // 128) * 128 if rng.random() < 0.5 else min(131072, max(4096, 2 ** math.ceil(math.log2(ctx))))
    kv_heads = rng.choice((1, 2, 4, 8, 8, 8, 16))
    scratch = "library" if 4 * kv_heads * (max_seq // 128) <= 8192 and rng.random() < 0.5 else "caller"
    return dict(op=op, kv_heads=kv_heads, ctx=ctx, max_seq=max_seq, layers=rng.randint(1, 16 if max_seq <= 16384 else 2),
                scratch=scratch)


# ---- weights: N(0, 0.02) rounded to bf16, and quantised from that ----------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _norm_weight(g, n):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float32) + 0.5


def _matrix(g, wtype, rows, cols):
    """(stored weight, stored scales or None): bf16; int8 and a scale per row; int4 pairs and an fp16 scale per group."""
    w = _normal(g, rows, cols).mul_(0.02).to(torch.bfloat16)
    if wtype == "bf16":
        return w, None
    w = w.float()
    if wtype == "int8":
        s = w.abs().amax(1) / 127
        s = torch.where(s == 0, torch.ones_like(s), s)
        return torch.round(w / s[:, None]).clamp_(-127, 127).to(torch.int8), s
    w = w.view(rows, cols // GROUP, GROUP)
    s = w.abs().amax(2) / 7
    s = torch.where(s == 0, torch.ones_like(s), s).to(torch.float16)
    q = (torch.round(w / s.float()[:, :, None]).clamp_(-8, 7) + 8).to(torch.uint8).view(rows, cols // 2, 2)
    return (q[:, :, 0] | (q[:, :, 1] << 4)).contiguous(), s.contiguous()


def _dense(wtype, w, s):
    """The stored matrix's values in 64 bits."""
    if wtype == "bf16":
        return w.double()
    if wtype == "int8":
        return w.double() * s.double()[:, None]
    q = torch.stack((w & 15, w >> 4), dim=2).view(w.shape[0], -1, GROUP).double() - 8
    return (q * s.double()[:, :, None]).view(w.shape[0], -1)


def _matrix_bytes(wtype, rows, cols):
    per_row = {"bf16": 2 * cols, "int8": cols + 4, "int4": cols // 2 + 2 * (cols // GROUP)}[wtype]
    return rows * per_row


def _ptr(t):
    return None if t is None else t.data_ptr()


# ---- whole decode steps ----------------------------------------------------------------------------------------------


def _model_tensors(wtype):
    """The model's (name, kind, stored tensors) in file order; the same every time."""
    g = _generator(MODEL_SEED)
    i = torch.arange(HEAD_DIM // 2, dtype=torch.float64)
    yield "rope.inv_freq", "vector", ((500000.0 ** (-2 * i / HEAD_DIM)).float(),)
    yield "tok_embeddings", "matrix", _matrix(g, wtype, VOCAB, HIDDEN)
    yield "norm.weight", "vector", (_norm_weight(g, HIDDEN),)
    for layer in range(LAYERS):
        p = f"layers.{layer}."
        yield p + "attn_norm.weight", "vector", (_norm_weight(g, HIDDEN),)
        yield p + "wqkv", "matrix", _matrix(g, wtype, QKV, HIDDEN)
        yield p + "wo", "matrix", _matrix(g, wtype, HIDDEN, HIDDEN)
        yield p + "ffn_norm.weight", "vector", (_norm_weight(g, HIDDEN),)
        yield p + "w_gate_up", "matrix", _matrix(g, wtype, 2 * INTER, HIDDEN)
        yield p + "w_down", "matrix", _matrix(g, wtype, HIDDEN, INTER)


def _model_specs(wtype):
    def matrix(name, rows, cols):
        dtype = {"bf16": fmt.BF16, "int8": fmt.I8, "int4": fmt.I4X2}[wtype]
        scales = {"bf16": [], "int8": [(fmt.F32, 1)], "int4": [(fmt.F16, cols // GROUP)]}[wtype]
        return [(name + ".weight", dtype, rows, cols)] + [(name + ".scales", d, rows, c) for d, c in scales]

    specs = [("rope.inv_freq", fmt.F32, HEAD_DIM // 2, 1)] + matrix("tok_embeddings", VOCAB, HIDDEN)
    specs.append(("norm.weight", fmt.F32, HIDDEN, 1))
    for layer in range(LAYERS):
        p = f"layers.{layer}."
        specs.append((p + "attn_norm.weight", fmt.F32, HIDDEN, 1))
        specs += matrix(p + "wqkv", QKV, HIDDEN) + matrix(p + "wo", HIDDEN, HIDDEN)
        specs.append((p + "ffn_norm.weight", fmt.F32, HIDDEN, 1))
        specs += matrix(p + "w_gate_up", 2 * INTER, HIDDEN) + matrix(p + "w_down", HIDDEN, INTER)
    return specs


@functools.lru_cache(maxsize=None)
def _model_file(wtype):
    """An open file without a name that holds the model; it goes with the process."""
    f = tempfile.TemporaryFile()
    header = dict(hidden_size=HIDDEN, intermediate_size=INTER, n_layers=LAYERS, n_heads=HEADS, n_kv_heads=KV_HEADS,
                  head_dim=HEAD_DIM, vocab_size=VOCAB, max_seq_len=MAX_SEQ, rms_eps=EPS, rope_theta=500000.0,
                  weight_dtype={"bf16": fmt.WEIGHT_BF16, "int8": fmt.WEIGHT_INT8, "int4": fmt.WEIGHT_INT4}[wtype],
                  group_size=GROUP if wtype == "int4" else 0)
    w = fmt.Writer(f"/proc/self/fd/{f.fileno()}", header, _model_specs(wtype))
    for _, _, tensors in _model_tensors(wtype):
        for t in tensors:
            if t is not None:
                t = t.view(torch.int16) if t.dtype == torch.bfloat16 else t
                w.write(t.cpu().numpy().reshape(-1))
    w.close()
    return f


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, VOCAB, case["tokens"]).tolist()


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _exact_decode(case, seed):
    """Every position at once, in 64 bits but for what the cache holds: rotated k and v rounded to fp16, and the
    rotation's angle, which is the 32-bit product of the position and the stored frequency."""
    wtype, tokens = case["wtype"], torch.tensor(_tokens(case, seed), device="cuda")
    n = len(tokens)
    tensors = _model_tensors(wtype)

    def vector():
        return next(tensors)[2][0].cuda()

    def matrix():
        return next(tensors)[2]

    angle = (torch.arange(n, device="cuda", dtype=torch.float32)[:, None] * vector()[None, :]).double()
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]

    def rotate(t):
        a, b = t[..., :HEAD_DIM // 2], t[..., HEAD_DIM // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)

    emb = matrix()
    final_norm = vector()
    x = _dense(wtype, emb[0][tokens], None if emb[1] is None else emb[1][tokens])
    causal = torch.ones(n, n, device="cuda", dtype=torch.bool).tril()
    for _ in range(LAYERS):
        h = _rms(x, vector())
        qkv = (h @ _dense(wtype, *matrix()).T).view(n, HEADS + 2 * KV_HEADS, HEAD_DIM)
        q = rotate(qkv[:, :HEADS])
        k = rotate(qkv[:, HEADS:HEADS + KV_HEADS]).to(torch.float16).double()
        v = qkv[:, HEADS + KV_HEADS:].to(torch.float16).double()
        heads = []
        for i in range(HEADS):
            s = (q[:, i] @ k[:, i // 4].T.contiguous()) * 0.125
            heads.append(torch.softmax(s.masked_fill(~causal, -math.inf), dim=-1) @ v[:, i // 4].contiguous())
        x = x + torch.cat(heads, dim=1) @ _dense(wtype, *matrix()).T
        gu = _rms(x, vector()) @ _dense(wtype, *matrix()).T
        x = x + (torch.nn.functional.silu(gu[:, :INTER]) * gu[:, INTER:]) @ _dense(wtype, *matrix()).T
    x = _rms(x if case["logits"] == "every" else x[-1:], final_norm)
    logits = torch.cat([x @ _dense(wtype, emb[0][r:r + 16032], None if emb[1] is None else emb[1][r:r + 16032]).T
                        for r in range(0, VOCAB, 16032)], dim=1)
    return logits if case["logits"] == "every" else logits[0]


def _run_decode(state):
    engine, tokens = state["engine"], state["tokens"]
    engine.reset()
    if state["logits"] is not None:
        best = ctypes.c_int()
        for t, row in zip(tokens, state["logits"]):
            E.call("cudallm_step", engine.handle, t, row.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), ctypes.byref(best))
        return state["logits"]
    for t in tokens[:-1]:
        engine.step_async(t)
    return engine.step(tokens[-1], want_logits=True)[1]


# ---- layers ----------------------------------------------------------------------------------------------------------


def _mlp_layer(g, case):
    hidden, inter, wtype = case["hidden"], case["inter"], case["wtype"]
    return _norm_weight(g, hidden), _matrix(g, wtype, 2 * inter, hidden), _matrix(g, wtype, hidden, inter)


def _run_mlp(state):
    c, stream = state["case"], torch.cuda.current_stream().cuda_stream
    hidden, inter, wtype = c["hidden"], c["inter"], c["wtype"]
    x, act = state["x"].clone(), state["act"]
    for norm, (wg, sg), (wd, sd) in state["layers"]:
        E.launch_matvec(wtype, "swiglu", 0, _ptr(wg), _ptr(sg), _ptr(x), _ptr(norm), EPS, _ptr(act), 2 * inter, hidden, stream)
        E.launch_matvec(wtype, "add", 0, _ptr(wd), _ptr(sd), _ptr(act), None, EPS, _ptr(x), hidden, inter, stream)
    return x


def _exact_mlp(case, seed):
    g, inter = _generator(seed), case["inter"]
    x = _normal(g, case["hidden"]).double()
    for _ in range(case["layers"]):
        norm, gate_up, down = _mlp_layer(g, case)
        gu = _dense(case["wtype"], *gate_up) @ _rms(x, norm)
        x = x + _dense(case["wtype"], *down) @ (torch.nn.functional.silu(gu[:inter]) * gu[inter:])
    return x


def _matvec_layer(g, case):
    out = case["rows"] // 2 if case["epilogue"] == "swiglu" else case["rows"]
    x, y = _normal(g, case["cols"]), _normal(g, out)
    norm = _norm_weight(g, case["cols"]) if case["norm"] else None
    return x, y, norm, _matrix(g, case["wtype"], case["rows"], case["cols"])


def _run_matvec(state):
    c, stream = state["case"], torch.cuda.current_stream().cuda_stream
    wtype, epilogue, rows, cols = c["wtype"], c["epilogue"], c["rows"], c["cols"]
    out = state["y"].clone() if epilogue == "add" else torch.empty_like(state["y"])
    for i, (x, norm, w, s) in enumerate(state["layers"]):
        E.launch_matvec(wtype, epilogue, 0, _ptr(w), _ptr(s), _ptr(x), _ptr(norm), EPS, out.data_ptr() + i * out.stride(0) * 4,
                        rows, cols, stream)
    return out[:, :state["n"]]


def _exact_matvec(case, seed):
    g, outs = _generator(seed), []
    for _ in range(case["layers"]):
        x, y, norm, (w, s) = _matvec_layer(g, case)
        x = x.double() if norm is None else _rms(x.double(), norm)
        d = torch.cat([_dense(case["wtype"], w[r:r + 16384], None if s is None else s[r:r + 16384]) @ x
                       for r in range(0, case["rows"], 16384)])
        if case["epilogue"] == "swiglu":
            d = torch.nn.functional.silu(d[:len(y)]) * d[len(y):]
        outs.append(y.double() + d if case["epilogue"] == "add" else d)
    return torch.stack(outs)


def _attention_layer(g, case):
    cache = (case["kv_heads"], case["max_seq"], HEAD_DIM)
    q = _normal(g, 4 * case["kv_heads"] * HEAD_DIM)
    return q, _normal(g, *cache).to(torch.float16), _normal(g, *cache).to(torch.float16)


def _run_attention(state):
    c, stream, out = state["case"], torch.cuda.current_stream().cuda_stream, torch.empty_like(state["out"])
    nh, nkv, max_seq, pos = 4 * c["kv_heads"], c["kv_heads"], c["max_seq"], _ptr(state["pos"])
    for i, (q, k, v) in enumerate(state["layers"]):
        o = out.data_ptr() + i * out.stride(0) * 4
        if c["scratch"] == "library":
            E.launch_attention_static(_ptr(q), _ptr(k), _ptr(v), pos, o, nh, nkv, HEAD_DIM, max_seq, stream)
        else:
            E.launch_attention(_ptr(q), _ptr(k), _ptr(v), pos, _ptr(state["part_o"]), _ptr(state["part_ml"]), o, nh, nkv,
                               HEAD_DIM, max_seq, stream)
    return out


def _exact_attention(case, seed):
    g, outs = _generator(seed), []
    for _ in range(case["layers"]):
        q, k, v = _attention_layer(g, case)
        heads = []
        for i in range(case["kv_heads"]):
            s = q.double().view(-1, 4, HEAD_DIM)[i] @ k[i, :case["ctx"]].double().T.contiguous() * 0.125
            heads.append((torch.softmax(s, dim=-1) @ v[i, :case["ctx"]].double()).view(-1))
        outs.append(torch.cat(heads))
    return torch.stack(outs)


# ---- what the measurement calls --------------------------------------------------------------------------------------


def prepare(case, seed):
    if case["op"] == "decode":
        engine = E.Engine(f"/proc/self/fd/{_model_file(case['wtype']).fileno()}")
        rows = np.zeros((case["tokens"], VOCAB), np.float32) if case["logits"] == "every" else None
        return dict(op="decode", engine=engine, tokens=_tokens(case, seed), logits=rows)
    g, state = _generator(seed), dict(op=case["op"], case=case)
    if case["op"] == "mlp":
        state["x"] = _normal(g, case["hidden"])
        state["act"] = torch.empty(case["inter"], device="cuda")
        state["layers"] = [_mlp_layer(g, case) for _ in range(case["layers"])]
    elif case["op"] == "matvec":
        made = [_matvec_layer(g, case) for _ in range(case["layers"])]
        n = state["n"] = len(made[0][1])
        state["y"] = torch.zeros(len(made), -(-n // 4) * 4, device="cuda")  # a layer's outputs start at 16 bytes
        for row, (_, y, _, _) in zip(state["y"], made):
            row[:n] = y
        state["layers"] = [(x, norm, w, s) for x, _, norm, (w, s) in made]
    else:
        nh = 4 * case["kv_heads"]
        state["layers"] = [_attention_layer(g, case) for _ in range(case["layers"])]
        state["pos"] = torch.tensor([case["ctx"] - 1], device="cuda", dtype=torch.int32)
        state["out"] = torch.empty(case["layers"], nh * HEAD_DIM, device="cuda")
        slots = nh * (case["max_seq"] // 128)
        state["part_o"] = torch.empty(slots * HEAD_DIM, device="cuda") if case["scratch"] == "caller" else None
        state["part_ml"] = torch.empty(slots * 2, device="cuda") if case["scratch"] == "caller" else None
    return state


def run(state):
    return {"decode": _run_decode, "mlp": _run_mlp, "matvec": _run_matvec, "attention": _run_attention}[state["op"]](state)


def work(case):
    if case["op"] == "decode":
        # A step knows nothing of the next token, so each reads every weight and the cache so far.
        n, wtype = case["tokens"], case["wtype"]
        shapes = [(VOCAB, HIDDEN)] + LAYERS * [(QKV, HIDDEN), (HIDDEN, HIDDEN), (2 * INTER, HIDDEN), (HIDDEN, INTER)]
        params = sum(r * c for r, c in shapes)
        kv = LAYERS * 2 * KV_HEADS * HEAD_DIM * 2 * n * (n + 1) / 2
        out = 4 * VOCAB * (n if case["logits"] == "every" else 1)
        return {"bytes": n * sum(_matrix_bytes(wtype, r, c) for r, c in shapes) + kv + out,
                "flops": 2 * n * params + LAYERS * 4 * HEADS * HEAD_DIM * n * (n + 1) / 2}
    layers = case["layers"]
    if case["op"] == "mlp":
        h, i = case["hidden"], case["inter"]
        weights = _matrix_bytes(case["wtype"], 2 * i, h) + _matrix_bytes(case["wtype"], h, i)
        return {"bytes": layers * (weights + 4 * h) + 8 * h, "flops": layers * 6 * h * i}
    if case["op"] == "matvec":
        rows, cols = case["rows"], case["cols"]
        out = rows // 2 if case["epilogue"] == "swiglu" else rows
        vectors = cols * (2 if case["norm"] else 1) + out * (2 if case["epilogue"] == "add" else 1)
        return {"bytes": layers * (_matrix_bytes(case["wtype"], rows, cols) + 4 * vectors), "flops": layers * 2 * rows * cols}
    nkv, ctx = case["kv_heads"], case["ctx"]
    return {"bytes": layers * (2 * 2 * nkv * ctx * HEAD_DIM + 2 * 4 * 4 * nkv * HEAD_DIM),
            "flops": layers * 4 * 4 * nkv * HEAD_DIM * ctx}


def tolerance(case):
    # Four times the largest error seen against 64 bits: 2.6e-6 in the layers (sums in 32 bits), 2.9e-4 in the logits,
    # where a difference in the last bits now and then rounds a cached k or v to the other fp16 neighbour.
    return {"rel": 1e-3 if case["op"] == "decode" else 1e-5}


def exact(case, seed):
    return {"decode": _exact_decode, "mlp": _exact_mlp, "matvec": _exact_matvec,
            "attention": _exact_attention}[case["op"]](case, seed)
