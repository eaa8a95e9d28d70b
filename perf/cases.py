"""The framework's work as its users call it, sized over the range they use.

A text-to-speech program runs four things through this library, for one voice
(a desktop or browser app) up to a few hundred (a server): the prefill of the
voice-clone prompts, the greedy frame loop, the codec decoder that turns the
frames' codes into sound, and -- where it drives the layers itself -- the
kernel-level ring append, attention and projection calls.  The listed cases
take each of them at its smallest, its usual and its large sizes, in both K/V
storage types; draw() gives sizes in between and odd ones.

Every case goes through mockbird_amd.Context.  Inputs come from the seed alone.
exact() restates each path in float64 torch, with K and V rounded to bf16
where the ring stores bf16 (the caller chose that) and the rotary angle formed
in fp32 (the exported graph defines it so).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import mockbird_amd as mb
from mockbird_amd import synth

D, H, HD, QKV, FFN, NVQ, CODES, PAD = 768, 12, 64, 2304, 3072, 16, 1024, 1024
LAYERS, VOCAB, CAPACITY = 12, 32000, 1024
ASSISTANT, AUDIO_END = 9, 7
PENALTY = 1.2
KV = {"f32": mb.MB_KV_F32, "bf16": mb.MB_KV_BF16}


def listed():
    return [
        # The ring append + decode attention of one decode step's 12 layers:
        # one voice of an interactive program, and 64 voices on long texts
        # whose rings have mostly wrapped (the isolated attention workload of
        # bench.py).
        {"name": "attend_1_f32", "op": "attend", "voices": 1, "capacity": 1024, "kv": "f32"},
        {"name": "attend_64_bf16", "op": "attend", "voices": 64, "capacity": 2048, "kv": "bf16"},
        # One layer's ring write + causal prefill attention: the server's batch
        # of full prompts on the bf16 path, and a few ragged prompts in fp32.
        {"name": "prompt_attention_16x512_bf16", "op": "prompt_attention", "voices": 16,
         "rows": 512, "shortest": 512, "past": 0, "kv": "bf16", "q": "bf16"},
        {"name": "prompt_attention_5x333_f32", "op": "prompt_attention", "voices": 5, "rows": 333,
         "shortest": 97, "past": 0, "kv": "f32", "q": "f32"},
        # One projection: c_attn over the rows of one voice's prompt in fp32,
        # and fc_in with its GELU over a server's prompt batch in the
        # split-bf16 form that bf16-K/V contexts run.
        {"name": "linear_281_c_attn_f32", "op": "linear", "rows": 281, "n": QKV, "k": D,
         "gelu": False, "split": False},
        {"name": "linear_8192_fc_in_split", "op": "linear", "rows": 8192, "n": FFN, "k": D,
         "gelu": True, "split": True},
        # The whole prompt pass: one voice-clone prompt of 150 reference
        # frames and 128 text ids (281 rows) with every row's hidden state,
        # and 48 voices of 64 to 400 rows.
        {"name": "prefill_1x281_f32", "op": "prefill", "voices": 1, "rows": 281, "shortest": 281,
         "kv": "f32", "all_rows": True},
        {"name": "prefill_48x400_bf16", "op": "prefill", "voices": 48, "rows": 400, "shortest": 64,
         "kv": "bf16", "all_rows": False},
        # The greedy frame loop after the prompt: one voice, and 64 voices with
        # the many-voice storage options (bf16 K/V and bf16 weights).
        {"name": "frames_1_f32", "op": "frames", "voices": 1, "frames": 8, "pos": 300, "kv": "f32",
         "weights": "f32"},
        {"name": "frames_64_bf16", "op": "frames", "voices": 64, "frames": 4, "pos": 300,
         "kv": "bf16", "weights": "bf16"},
        # The codec decoder in mid-stream, its longest windows full: one voice
        # played as it is made (host buffers, 4 frames = 0.32 s a call), and
        # 256 voices of a server on device buffers.
        {"name": "codec_1_f32", "op": "codec", "voices": 1, "frames": 4, "warm": 110, "kv": "f32",
         "host": True},
        {"name": "codec_256_bf16", "op": "codec", "voices": 256, "frames": 4, "warm": 110,
         "kv": "bf16", "host": False},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(("attend", "prompt_attention", "linear", "prefill", "frames", "codec"))
    kv = rng.choice(("f32", "bf16"))
    if op == "attend":
        voices = log(1, 256)
        return {"op": op, "voices": voices, "capacity": log(64, min(4096, 131072 // voices)),
                "kv": kv}
    if op == "prompt_attention":
        voices, rows = log(1, 16), log(16, 512)
        return {"op": op, "voices": voices, "rows": rows, "shortest": rng.randint(1, rows),
                "past": rng.choice((0, 0, log(8, 500))), "kv": kv,
                "q": "bf16" if kv == "bf16" and rng.random() < 0.5 else "f32"}
    if op == "linear":
        n, k = rng.choice(((QKV, D), (D, D), (FFN, D), (D, FFN), (D, 256), (256, 256),
                           (1024, 256), (256, 1024)))
        rows = log(1, 8192)
        return {"op": op, "rows": rows, "n": n, "k": k, "gelu": rng.random() < 0.3,
                "split": rows > 8 and rng.random() < 0.5}
    if op == "prefill":
        voices, rows = log(1, 48), log(64, 400)
        return {"op": op, "voices": voices, "rows": rows, "shortest": rng.randint(16, rows),
                "kv": kv, "all_rows": voices <= 4 and rng.random() < 0.5}
    if op == "frames":
        voices = log(1, 64)
        return {"op": op, "voices": voices, "frames": rng.randint(1, max(1, min(8, 256 // voices))),
                "pos": log(70, 900), "kv": kv, "weights": rng.choice(("f32", "bf16"))}
    voices = log(1, 256)
    return {"op": op, "voices": voices, "frames": rng.randint(1, 4), "warm": log(4, 110), "kv": kv,
            "host": voices <= 8}


# ------------------------------------------------------------------- inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0):
    x = torch.randn(shape, generator=g, device="cuda")
    return x.mul_(std) if std != 1.0 else x


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()


def _lengths(case, seed):
    """Prompt rows per voice, the first voice the longest."""
    n = np.random.default_rng([seed, 1]).integers(case["shortest"], case["rows"] + 1,
                                                  size=case["voices"])
    n[0] = case["rows"]
    return n.astype(np.int32)


def _model_tensors(seed):
    """(name, tensor) of a random-init model: matrices N(0, 0.02), LayerNorm
    scales 1, small biases.  The text head's two decision columns are alike,
    so that every voice goes on (a tie continues)."""
    g = _generator(seed)
    for name, shape, kind in synth.tensor_specs(LAYERS, VOCAB):
        if kind == "ln_w":
            t = torch.ones(shape, device="cuda")
        else:
            t = _randn(g, *shape, std=0.02)
        if name == "model.text_lm_head.weight":
            t[:, AUDIO_END] = t[:, ASSISTANT]
        yield name, t


def _codec_tensors(seed):
    g = _generator(seed)
    for name, shape, kind, scale in synth.codec_specs(mb.CODEC_LAYERS):
        t = _randn(g, *shape)
        if kind == "ln_w":
            t = 1 + t * scale
        elif kind == "scale":
            t = scale * (1 + 0.25 * t)
        else:
            t = t * scale
        yield name, t


def _upload(ctx, tensors):
    for name, t in tensors:
        ctx.upload(name, t.cpu().numpy())


def _prompt_ids(case, n, seed):
    """Voice-clone prompts [B][rows][17]: half reference frames, half text."""
    B, R = case["voices"], case["rows"]
    g = np.random.default_rng([seed, 2])
    ids = np.full((B, R, NVQ + 1), PAD, np.int32)
    ids[:, :, 0] = g.integers(0, VOCAB, size=(B, R))
    codes = g.integers(0, CODES, size=(B, R, NVQ))
    for b in range(B):
        half = int(n[b]) // 2
        ids[b, 1:half, 0] = synth.USER_SLOT
        ids[b, 1:half, 1:] = codes[b, 1:half]
    return ids


def _context(**kw):
    ctx = mb.Context(**kw)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    return ctx


# ---------------------------------------------- ring rows of earlier positions

CHUNK = 128  # rows of one write


def _history(g, voices, first, count):
    """Chunks (c0, qkv [voices][CHUNK][2304], rows of this chunk, first positions)
    that fill each voice's ring from position first[b], count[b] rows."""
    for c0 in range(0, int(count.max()), CHUNK):
        yield (c0, _randn(g, voices, CHUNK, QKV), np.clip(count - c0, 0, CHUNK).astype(np.int32),
               (first + c0).astype(np.int32))


def _fill(ctx, layer, g, voices, first, count):
    for _, qkv, rows, p0 in _history(g, voices, first, count):
        n, p = _i32(rows), _i32(p0)
        ctx.ring_write_rows_dev(layer, voices, CHUNK, qkv.data_ptr(), p.data_ptr(), n.data_ptr(), 0)
        torch.cuda.current_stream().synchronize()


def _attend_positions(case, seed):
    B, C = case["voices"], case["capacity"]
    pos = np.random.default_rng([seed, 3]).integers(1, 3 * C, size=B)
    first = np.maximum(0, pos - C + 1)
    return pos.astype(np.int32), first.astype(np.int32), (pos - first).astype(np.int32)


# ------------------------------------------------------------------- prepare

def prepare(case, seed):
    return globals()["_prepare_" + case["op"]](case, seed)


def _prepare_attend(case, seed):
    B, C = case["voices"], case["capacity"]
    ctx = _context(n_layers=LAYERS, capacity=C, max_seqs=B, max_rows=CHUNK, kv_dtype=KV[case["kv"]])
    pos, first, count = _attend_positions(case, seed)
    g = _generator(seed)
    qkv = _randn(g, LAYERS, B, QKV)
    for layer in range(LAYERS):
        _fill(ctx, layer, g, B, first, count)
    return {"case": case, "ctx": ctx, "qkv": qkv, "pos": _i32(pos), "max_pos": int(pos.max()),
            "out": torch.zeros((LAYERS, B, D), device="cuda")}


def _prepare_prompt_attention(case, seed):
    B, R, past = case["voices"], case["rows"], case["past"]
    ctx = _context(n_layers=1, capacity=CAPACITY, max_seqs=B, max_rows=max(R, CHUNK),
                   kv_dtype=KV[case["kv"]])
    n = _lengths(case, seed)
    g = _generator(seed)
    dtype = torch.bfloat16 if case["q"] == "bf16" else torch.float32
    qkv = _randn(g, B, R, QKV).to(dtype)
    zero = np.zeros(B, np.int32)
    if past:
        _fill(ctx, 0, g, B, zero, zero + past)
    return {"case": case, "ctx": ctx, "qkv": qkv, "n": _i32(n), "pos0": _i32(zero + past),
            "q": torch.zeros((B, R, D), device="cuda", dtype=dtype),
            "out": torch.zeros((B, R, D), device="cuda")}


def _linear_inputs(case, seed):
    g = _generator(seed)
    return (_randn(g, case["rows"], case["k"]), _randn(g, case["k"], case["n"], std=0.02),
            _randn(g, case["n"], std=0.02))


def _prepare_linear(case, seed):
    M, N, K = case["rows"], case["n"], case["k"]
    ctx = _context(n_layers=1, capacity=8, max_seqs=1, max_rows=8, vocab=16)
    a, w, bias = _linear_inputs(case, seed)
    if case["split"]:
        wx = torch.empty(2 * K * N, dtype=torch.bfloat16, device="cuda")
        ctx.split_weights_dev(w.data_ptr(), K, N, wx.data_ptr())
        torch.cuda.current_stream().synchronize()
        w = wx
    return {"case": case, "ctx": ctx, "a": a, "w": w, "bias": bias,
            "c": torch.zeros((M, N), device="cuda")}


def _prepare_prefill(case, seed):
    n = _lengths(case, seed)
    ctx = _context(n_layers=LAYERS, capacity=CAPACITY, max_seqs=case["voices"],
                   max_rows=case["rows"], kv_dtype=KV[case["kv"]], vocab=VOCAB)
    _upload(ctx, _model_tensors(seed))
    return {"case": case, "ctx": ctx, "ids": _prompt_ids(case, n, seed), "n": n}


def _frames_inputs(case, seed):
    """Positions (within 64 of case["pos"]) and the hidden rows the prompts left."""
    B = case["voices"]
    g = np.random.default_rng([seed, 4])
    pos = (case["pos"] + g.integers(0, 64, size=B)).astype(np.int32)
    return pos, g.standard_normal((B, D), dtype=np.float32)


def _prepare_frames(case, seed):
    B = case["voices"]
    ctx = _context(n_layers=LAYERS, capacity=CAPACITY, max_seqs=B, max_rows=CHUNK,
                   kv_dtype=KV[case["kv"]], vocab=VOCAB)
    _upload(ctx, _model_tensors(seed))
    if case["weights"] == "bf16":
        ctx.set_weight_storage(mb.MB_W_BF16)
    pos, hidden = _frames_inputs(case, seed)
    g = _generator(seed + 1)
    for layer in range(LAYERS):
        _fill(ctx, layer, g, B, np.zeros(B, np.int32), pos)
    return {"case": case, "ctx": ctx, "pos": pos, "hidden": hidden}


def _codec_codes(case, seed):
    g = np.random.default_rng([seed, 5])
    return g.integers(0, CODES, size=(case["warm"] + case["frames"], case["voices"], NVQ),
                      dtype=np.int32)


def _prepare_codec(case, seed):
    B, n = case["voices"], case["frames"]
    ctx = _context(n_layers=1, capacity=16, max_seqs=1, max_rows=16, vocab=16)
    _upload(ctx, _codec_tensors(seed))
    ctx.codec_init(B, kv_dtype=KV[case["kv"]])
    codes = _codec_codes(case, seed)
    warm = _i32(codes[:case["warm"]])
    pcm = torch.zeros((B, 2, case["warm"] * mb.CODEC_SAMPLES), device="cuda")
    ctx.codec_decode_dev(B, case["warm"], warm.data_ptr(), pcm.data_ptr())
    torch.cuda.current_stream().synchronize()
    state = {"case": case, "ctx": ctx}
    if case["host"]:
        state["codes"] = codes[case["warm"]:]
    else:
        state["codes"] = _i32(codes[case["warm"]:])
        state["pcm"] = torch.zeros((B, 2, n * mb.CODEC_SAMPLES), device="cuda")
    return state


# ----------------------------------------------------------------------- run

def run(state):
    return globals()["_run_" + state["case"]["op"]](state, state["case"], state["ctx"])


def _run_attend(s, case, ctx):
    for layer in range(LAYERS):
        ctx.append_attend_dev(layer, case["voices"], s["qkv"][layer].data_ptr(), s["pos"].data_ptr(),
                              s["max_pos"], s["out"][layer].data_ptr())
    return s["out"]


def _run_prompt_attention(s, case, ctx):
    dtype = mb.MB_DT_BF16 if case["q"] == "bf16" else mb.MB_DT_F32
    args = (s["pos0"].data_ptr(), s["n"].data_ptr())
    ctx.ring_write_rows_dev(0, case["voices"], case["rows"], s["qkv"].data_ptr(), *args,
                            s["q"].data_ptr(), qkv_dtype=dtype, q_dtype=dtype)
    ctx.prefill_attention_dev(0, case["voices"], case["rows"], s["q"].data_ptr(), *args,
                              s["out"].data_ptr(), q_dtype=dtype)
    return [s["q"], s["out"]]


def _run_linear(s, case, ctx):
    call = ctx.linear_split_dev if case["split"] else ctx.linear_dev
    call(case["rows"], case["n"], case["k"], s["a"].data_ptr(), case["k"], s["w"].data_ptr(),
         s["bias"].data_ptr(), s["c"].data_ptr(), case["n"],
         mb.MB_EPI_GELU if case["gelu"] else mb.MB_EPI_STORE)
    return s["c"]


def _run_prefill(s, case, ctx):
    if case["all_rows"]:
        return ctx.prefill_rows(s["ids"], s["n"])
    return ctx.prefill(s["ids"], s["n"])


def _run_frames(s, case, ctx):
    codes, cont, hidden, pos = ctx.decode_frames(s["hidden"], s["pos"], case["frames"])
    return {"codes": codes, "cont": cont.astype(np.int32), "hidden": hidden, "pos": pos}


def _run_codec(s, case, ctx):
    if case["host"]:
        return ctx.codec_decode(s["codes"])
    ctx.codec_decode_dev(case["voices"], case["frames"], s["codes"].data_ptr(), s["pcm"].data_ptr())
    return s["pcm"]


# ---------------------------------------------------------------------- work

LAYER_WEIGHTS = D * QKV + D * D + 2 * D * FFN


def work(case):
    op, e = case["op"], 2 if case.get("kv") == "bf16" else 4
    if op == "attend":
        # the windows' expected slots: positions U[1, 3C), two thirds full rings
        B, C = case["voices"], case["capacity"]
        slots = B * C * 5 / 6
        return {"bytes": LAYERS * (slots * 2 * D * e + B * (QKV + D) * 4),
                "flops": LAYERS * slots * 4 * D}
    if op == "prompt_attention":
        B, past, s = case["voices"], case["past"], 4 if case["q"] == "f32" else 2
        n = (case["rows"] + case["shortest"]) / 2
        return {"bytes": B * (n * (QKV * s + 2 * D * e + D * s + D * 4) + past * 2 * D * e),
                "flops": B * 4 * D * (n * (n + 1) / 2 + n * past)}
    if op == "linear":
        M, N, K = case["rows"], case["n"], case["k"]
        return {"bytes": 4 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    if op == "prefill":
        B = case["voices"]
        n = (case["rows"] + case["shortest"]) / 2
        rows = B * n
        return {"bytes": LAYERS * (LAYER_WEIGHTS * 4 + rows * 2 * D * e) + rows * 17 * 4
                + (rows if case["all_rows"] else B) * D * 4,
                "flops": LAYERS * (2 * rows * LAYER_WEIGHTS + B * 4 * D * n * (n + 1) / 2)}
    if op == "frames":
        # per frame: every layer's weights and window, the local layer 17 times
        # (read once from memory) and the 16 heads
        B, w = case["voices"], 2 if case["weights"] == "bf16" else 4
        pos = case["pos"] + 32
        weights = (LAYERS + 1) * LAYER_WEIGHTS + NVQ * D * CODES
        passes = (LAYERS + 17) * LAYER_WEIGHTS + NVQ * D * CODES
        return {"bytes": case["frames"] * (weights * w + B * LAYERS * pos * 2 * D * e),
                "flops": case["frames"] * B * (2 * passes + LAYERS * pos * 4 * D)}
    B, F = case["voices"], case["frames"]
    nbytes = flops = 0
    for s, (layers, window) in enumerate(zip(mb.CODEC_LAYERS, mb.CODEC_CONTEXT)):
        n, layer_w = 4 << s, 4 * 256 * 256 + 2 * 256 * 1024
        slots = min(window, n * case["warm"]) + n
        edge = (192 if s == 0 else 384) * 256 + 256 * (240 if s == 3 else 768)
        nbytes += layers * (B * slots * 2 * 256 * e + layer_w * 4) + edge * 4
        flops += B * n * (layers * (2 * layer_w + 4 * 256 * slots) + 2 * edge)
    return {"bytes": F * (nbytes + B * 2 * mb.CODEC_SAMPLES * 4), "flops": F * flops}


def tolerance(case):
    """About four times the error that these paths show against exact(): fp32
    sums in another order; on bf16 rings a K or V element that rounds the
    other way; bf16 queries and probabilities; split-bf16 products."""
    op, f32 = case["op"], case.get("kv") == "f32"
    if op == "attend":
        return {"rel": 1e-6 if f32 else 8e-5}
    if op == "prompt_attention":
        return {"rel": 8e-3 if case["q"] == "bf16" else 1.5e-6 if f32 else 3e-5}
    if op == "linear":
        return {"rel": 2e-5 if case["split"] else 2e-6}
    if op == "prefill":
        return {"rel": 4e-6 if f32 else 8e-4}
    if op == "frames":
        # a code may change at a near tie of two logits, and then its voice
        return {"rel": 5e-6 if f32 else 1e-3, "differ": 0.01}
    return {"rel": 2e-6 if f32 else 5e-5}


# --------------------------------------------------------------------- exact

def exact(case, seed):
    return globals()["_exact_" + case["op"]](case, seed)


def _rope(x, pos):
    """x [..., heads, 64] in float64 at positions pos [...]: the angle is the
    fp32 product of the position and the graph's fp32 frequencies."""
    inv = (1.0 / (10000 ** (torch.arange(0, HD, 2).float() / HD))).to(x.device)
    a = (pos.to(torch.float32)[..., None] * inv).double()[..., None, :]
    c, s = a.cos(), a.sin()
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * c - x1 * s, x1 * c + x0 * s), -1).flatten(-2)


def _stored(x, kv):
    """x as a ring of that storage holds it (float64)."""
    return x.float().to(torch.bfloat16).double() if kv == "bf16" else x


def _softmax_attention(q, k, v, seen):
    """q [B, H, n, 64], k and v [B, H, m, 64], seen [B, n, m]; rows that see
    nothing are zero."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * 0.125
    s = s.masked_fill(~seen[:, None], float("-inf"))
    p = torch.nan_to_num(torch.softmax(s, -1))
    return torch.matmul(p, v)


def _norm(x, w, b):
    m = x.mean(-1, keepdim=True)
    v = (x - m).square().mean(-1, keepdim=True)
    return (x - m) / (v + 1e-5).sqrt() * w + b


def _gelu_tanh(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _heads(x):
    """[B, n, heads * 64] -> [B, heads, n, 64]"""
    return x.unflatten(-1, (-1, HD)).transpose(1, 2).contiguous()


def _exact_history(g, voices, first, count, kv):
    """Roped K and V [B, H, rows, 64] of _fill's rows, their positions [B, rows]
    (-1 past each voice's last)."""
    ks, vs, ps = [], [], []
    for _, qkv, rows, p0 in _history(g, voices, first, count):
        p = torch.from_numpy(p0.astype(np.int64)).cuda()[:, None] + torch.arange(CHUNK, device="cuda")
        live = torch.arange(CHUNK, device="cuda") < torch.from_numpy(rows.astype(np.int64)).cuda()[:, None]
        x = qkv.double().unflatten(-1, (3, H, HD))
        ks.append(_stored(_rope(x[:, :, 1], p), kv))
        vs.append(_stored(x[:, :, 2], kv))
        ps.append(torch.where(live, p, -1))
    if not ks:
        none = torch.zeros((voices, H, 0, HD), dtype=torch.float64, device="cuda")
        return none, none, torch.zeros((voices, 0), dtype=torch.int64, device="cuda")
    return (torch.cat(ks, 1).transpose(1, 2).contiguous(),
            torch.cat(vs, 1).transpose(1, 2).contiguous(), torch.cat(ps, 1))


def _exact_attend(case, seed):
    B, C, kv = case["voices"], case["capacity"], case["kv"]
    pos, first, count = _attend_positions(case, seed)
    g = _generator(seed)
    qkv = _randn(g, LAYERS, B, QKV)
    cur = torch.from_numpy(pos.astype(np.int64)).cuda()
    out = []
    for layer in range(LAYERS):
        k, v, p = _exact_history(g, B, first, count, kv)
        x = qkv[layer].double().unflatten(-1, (3, H, HD))
        kn = _stored(_rope(x[:, 1], cur), kv)
        k = torch.cat((k, kn[:, :, None]), 2)
        v = torch.cat((v, _stored(x[:, 2], kv)[:, :, None]), 2)
        p = torch.cat((p, cur[:, None]), 1)
        seen = (p >= 0) & (cur[:, None] - p < C)
        out.append(_softmax_attention(_rope(x[:, 0], cur)[:, :, None], k, v, seen[:, None])
                   .reshape(B, D))
    return torch.stack(out)


def _exact_prompt_attention(case, seed):
    B, R, past, kv = case["voices"], case["rows"], case["past"], case["kv"]
    n = torch.from_numpy(_lengths(case, seed).astype(np.int64)).cuda()
    g = _generator(seed)
    qkv = _randn(g, B, R, QKV)
    if case["q"] == "bf16":
        qkv = qkv.to(torch.bfloat16)
    zero = np.zeros(B, np.int32)
    k0, v0, p0 = _exact_history(g, B, zero, zero + past, kv)
    row = torch.arange(R, device="cuda").expand(B, R)
    cur, live = past + row, row < n[:, None]
    x = qkv.double().unflatten(-1, (3, H, HD))
    q = _rope(x[:, :, 0], cur) * live[..., None, None]
    if case["q"] == "bf16":
        q = q.float().to(torch.bfloat16).double()  # the roped rows are stored so
    k = torch.cat((k0, _stored(_rope(x[:, :, 1], cur), kv).transpose(1, 2)), 2)
    v = torch.cat((v0, _stored(x[:, :, 2], kv).transpose(1, 2)), 2)
    p = torch.cat((p0, torch.where(live, cur, -1)), 1)
    seen = (p[:, None] >= 0) & (p[:, None] <= cur[..., None]) & live[..., None]
    out = _softmax_attention(q.transpose(1, 2).contiguous(), k, v, seen)
    return [q.reshape(B, R, D), out.transpose(1, 2).reshape(B, R, D)]


def _exact_linear(case, seed):
    a, w, bias = (t.double() for t in _linear_inputs(case, seed))
    y = a @ w + bias
    return _gelu_tanh(y) if case["gelu"] else y


class _Model:
    """The decoder in float64 (ref-decode.mjs:162-286), every matrix rounded to
    bf16 first where the weights are stored so."""

    def __init__(self, seed, weights="f32"):
        self.t = {}
        for name, t in _model_tensors(seed):
            matrix = t.ndim == 2 and (".attn." in name or ".mlp." in name or "audio_lm_heads" in name)
            self.t[name] = t.to(torch.bfloat16).float() if matrix and weights == "bf16" else t

    def __getitem__(self, name):
        return self.t[name].double()

    def norm(self, p, x):
        return _norm(x, self[p + ".weight"], self[p + ".bias"])

    def linear(self, p, x):
        return x @ self[p + ".weight"] + self[p + ".bias"]

    def embed(self, ids):
        """ids [..., 17]"""
        x = self.t["core.model.transformer.wte.weight"][ids[..., 0]].double()
        for k in range(NVQ):
            c = ids[..., k + 1]
            row = self.t[f"core.model.audio_embeddings.{k}.weight"][c.clamp(max=CODES - 1)].double()
            x = x + row * (c < CODES)[..., None]
        return x

    def layer(self, p, x, pos, k0, v0, seen, kv):
        """x [B, n, 768] at pos [B, n] after the rows k0, v0 [B, H, m, 64];
        seen [B, n, m + n].  Returns x, k, v."""
        y = self.linear(p + "attn.c_attn", self.norm(p + "ln_1", x)).unflatten(-1, (3, H, HD))
        k = torch.cat((k0, _stored(_rope(y[:, :, 1], pos), kv).transpose(1, 2)), 2)
        v = torch.cat((v0, _stored(y[:, :, 2], kv).transpose(1, 2)), 2)
        q = _rope(y[:, :, 0], pos).transpose(1, 2).contiguous()
        a = _softmax_attention(q, k, v, seen).transpose(1, 2).flatten(-2)
        x = x + self.linear(p + "attn.c_proj", a)
        m = _gelu_tanh(self.linear(p + "mlp.fc_in", self.norm(p + "ln_2", x)))
        return x + self.linear(p + "mlp.fc_out", m), k, v


def _no_rows(B):
    return torch.zeros((B, H, 0, HD), dtype=torch.float64, device="cuda")


def _exact_prefill(case, seed):
    n = _lengths(case, seed)
    ids = torch.from_numpy(_prompt_ids(case, n, seed).astype(np.int64)).cuda()
    m = _Model(seed)
    B, R = case["voices"], case["rows"]
    out = torch.zeros((B, R, D), dtype=torch.float64, device="cuda")
    x = [m.embed(ids[b:b + 1, :n[b]]) for b in range(B)]
    for layer in range(LAYERS):
        for b in range(B):
            pos = torch.arange(int(n[b]), device="cuda")[None]
            seen = pos[:, None] <= pos[..., None]
            x[b] = m.layer(f"core.model.transformer.h.{layer}.", x[b], pos, _no_rows(1), _no_rows(1),
                           seen, case["kv"])[0]
    for b in range(B):
        out[b, :n[b]] = m.norm("core.model.transformer.ln_f", x[b][0])
    if case["all_rows"]:
        return out
    return torch.stack([out[b, n[b] - 1] for b in range(B)])


def _exact_frames(case, seed):
    # bf16 rings: a greedy choice follows the last bits of every layer before
    # it, so the frames of two correct programs part within a few
    if case["kv"] == "bf16":
        return None
    B = case["voices"]
    m = _Model(seed, case["weights"])
    pos, hidden = _frames_inputs(case, seed)
    hidden, cur = torch.from_numpy(hidden).cuda().double(), torch.from_numpy(pos.astype(np.int64)).cuda()
    g = _generator(seed + 1)
    past = [_exact_history(g, B, np.zeros(B, np.int32), pos, "f32") for _ in range(LAYERS)]
    used = torch.zeros((NVQ, B, CODES), dtype=torch.bool, device="cuda")
    who = torch.arange(B, device="cuda")
    for _ in range(case["frames"]):
        ids = torch.full((B, NVQ + 1), ASSISTANT, dtype=torch.int64, device="cuda")
        x, k, v = hidden, _no_rows(B), _no_rows(B)
        for step in range(NVQ + 1):
            at = torch.full((B, 1), step, device="cuda")
            all_seen = torch.ones((B, 1, step + 1), dtype=torch.bool, device="cuda")
            y, k, v = m.layer("model.local_transformer.h.0.", x[:, None], at, k, v, all_seen, "f32")
            if step == 0:
                x = m["core.model.transformer.wte.weight"][ASSISTANT].expand(B, D)
                continue
            ch = step - 1
            s = m.norm("model.local_transformer.ln_f", y[:, 0]) @ m[f"model.audio_lm_heads.{ch}.weight"]
            s = torch.where(used[ch], torch.where(s < 0, s * PENALTY, s / PENALTY), s)
            ids[:, step] = s.argmax(-1)
            used[ch, who, ids[:, step]] = True
            x = m[f"core.model.audio_embeddings.{ch}.weight"][ids[:, step]]
        x = m.embed(ids)[:, None]
        for layer in range(LAYERS):
            k, v, p = past[layer]
            p = torch.cat((p, cur[:, None]), 1)
            x, k, v = m.layer(f"core.model.transformer.h.{layer}.", x, cur[:, None], k, v,
                              ((p >= 0) & (cur[:, None] - p < CAPACITY))[:, None], "f32")
            past[layer] = (k, v, p)
        hidden, cur = m.norm("core.model.transformer.ln_f", x[:, 0]), cur + 1
    return {"codes": None, "cont": None, "hidden": hidden, "pos": None}


def _exact_codec(case, seed):
    w = {name: t.double() for name, t in _codec_tensors(seed)}
    codes = torch.from_numpy(_codec_codes(case, seed).astype(np.int64)).cuda()
    F, B, kv = codes.shape[0], case["voices"], case["kv"]
    acc = 0
    for k in range(NVQ):
        p = f"model.quantizer.quantizers.{k}."
        acc = acc + w[p + "codebook.weight"][codes[:, :, k]] @ w[p + "out_proj.weight"].T \
            + w[p + "out_proj.bias"]
    y = acc @ w["model.quantizer.output_proj.weight"].T + w["model.quantizer.output_proj.bias"]
    x = y.unflatten(-1, (192, 4)).transpose(-1, -2).transpose(0, 1).reshape(B, F * 4, 192)
    for s in range(4):
        p = f"model.decoder.{synth.CODEC_DECODER_INDEX[s]}."
        x = x @ w[p + "input_proj.weight"]
        pos = torch.arange(x.shape[1], device="cuda")
        back = pos[:, None] - pos
        seen = ((back >= 0) & (back < mb.CODEC_CONTEXT[s]))[None]
        for i in range(mb.CODEC_LAYERS[s]):
            q = p + f"transformer.layers.{i}."
            for b in range(0, B, 8):  # 8 voices' score matrices at a time
                z = x[b:b + 8]
                y = (_norm(z, w[q + "norm1.weight"], w[q + "norm1.bias"])
                     @ w[q + "self_attn.in_proj.weight"]).unflatten(-1, (3, 4, HD))
                qr, kr = _rope(y[:, :, 0], pos), _stored(_rope(y[:, :, 1], pos), kv)
                a = _softmax_attention(_heads(qr.flatten(-2)), _heads(kr.flatten(-2)),
                                       _heads(_stored(y[:, :, 2], kv).flatten(-2)), seen)
                z = z + w[q + "layer_scale_1.scale"] * (
                    a.transpose(1, 2).flatten(-2) @ w[q + "self_attn.out_proj.weight"])
                f = _norm(z, w[q + "norm2.weight"], w[q + "norm2.bias"]) @ w[q + "ffn.0.weight"]
                f = 0.5 * f * (1 + torch.erf(f / math.sqrt(2.0)))
                x[b:b + 8] = z + w[q + "layer_scale_2.scale"] * (f @ w[q + "ffn.2.weight"])
        x = x @ w[p + "output_proj.weight"]
        if s < 3:  # row t becomes rows 2t and 2t + 1: new[2t + r][m] = old[t][2m + r]
            x = x.unflatten(-1, (384, 2)).transpose(-1, -2).reshape(B, -1, 384)
    # audio[c][t * 120 + j] = latent[t][2j + c]
    pcm = x.unflatten(-1, (120, 2)).permute(0, 3, 1, 2).reshape(B, 2, F * mb.CODEC_SAMPLES)
    return pcm[:, :, case["warm"] * mb.CODEC_SAMPLES:].contiguous()
