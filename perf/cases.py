"""The work a user of this framework has it do, as measurable cases.

Every case goes through the public C-ABI entry points on device memory, on one
stream, the way a serving program calls them.  The listed cases cover the
decode step, the prefill, whole attention layers, MLP layers and a model's
forward; draw() gives more of the same ranges.

The head shapes are the benchmark's: 8 query / 2 kv heads of 64 (the small
parity shape), 32 / 8 of 128 (the 8B class) and 64 / 8 of 128 (the 70B class).
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from tailorquantkernel_amd import attn, native

QK = 32
PAGE = native.PAGE_TOKENS
SHAPES = {"small": (8, 2, 64, 512, 1408), "8b": (32, 8, 128, 4096, 14336), "70b": (64, 8, 128, 8192, 28672)}
THETA = 500000.0
EPS = 1e-6
STEP_ROWS = 8192      # cache rows appended at a time while a cache is filled
VOCAB = 128256


# ---- the cases -------------------------------------------------------------

def listed():
    return [
        # one short conversation on the smallest shape: one launch's latency
        {"name": "step-small", "path": "step", "shape": "small", "n": 1, "low": 256, "high": 256, "outliers": False},
        # one 4k conversation, one layer's step
        {"name": "step-8b-4k", "path": "step", "shape": "8b", "n": 1, "low": 4096, "high": 4096, "outliers": False},
        # a serving batch: 64 conversations of very different lengths
        {"name": "step-8b-batch64", "path": "step", "shape": "8b", "n": 64, "low": 512, "high": 8192,
         "outliers": False},
        # long contexts on the large shape, keys and values with outliers
        {"name": "step-70b-32k", "path": "step", "shape": "70b", "n": 16, "low": 32768, "high": 32768,
         "outliers": True},
        # a whole prompt at once
        {"name": "prefill-8b-2k", "path": "prefill", "shape": "8b", "pos": 0, "n": 2048},
        # the next turn of a conversation: a ragged chunk after earlier context
        {"name": "prefill-8b-turn", "path": "prefill", "shape": "8b", "pos": 1000, "n": 333},
        # an attention layer of one decode step
        {"name": "layer-8b-step", "path": "layer", "shape": "8b", "format": "q8", "n": 1, "low": 4096, "high": 4096},
        # an attention layer over a prompt
        {"name": "layer-8b-prompt", "path": "layer_batch", "shape": "8b", "format": "q8", "pos": 0, "n": 2048},
        # an MLP of one decode step
        {"name": "mlp-8b-step", "path": "mlp", "hidden": 4096, "inter": 14336, "format": "q8", "n": 1},
        # an MLP over a prompt
        {"name": "mlp-8b-prompt", "path": "mlp", "hidden": 4096, "inter": 14336, "format": "q8", "n": 2048},
        # an MLP over a batch of conversations or a short prompt, 4-bit weights
        {"name": "mlp-8b-q4-rows", "path": "mlp", "hidden": 4096, "inter": 14336, "format": "q4", "n": 100},
        # a model: a prompt, then the next token
        {"name": "model-8b-2layer", "path": "model", "shape": "8b", "layers": 2, "format": "q8", "n": 300},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["step", "step", "prefill", "layer", "layer_batch", "mlp", "mlp", "model"])
    shape = rng.choice(["small", "8b", "70b"])
    fmt = rng.choice(["q8", "q8", "q4"])
    if path in ("step", "layer"):
        n = _log_int(rng, 1, 64)
        high = _log_int(rng, 64, min(32768, 524288 // n))
        low = high if rng.random() < 0.4 else rng.randint(max(1, high // 16), high)
        if path == "step":
            return {"path": path, "shape": shape, "n": n, "low": low, "high": high, "outliers": rng.random() < 0.3}
        high = min(high, 65536 // n)
        return {"path": path, "shape": shape, "format": fmt, "n": n, "low": min(low, high), "high": high}
    if path in ("prefill", "layer_batch"):
        big = shape == "70b"
        n = _log_int(rng, 2, 1024 if big else 2048)
        pos = 0 if rng.random() < 0.5 else rng.randint(1, 1024 if big else 2048)
        if path == "prefill":
            return {"path": path, "shape": shape, "pos": pos, "n": n}
        return {"path": path, "shape": shape, "format": fmt, "pos": pos, "n": min(n, 512) if big else n}
    if path == "mlp":
        hidden, inter = rng.choice([(512, 1408), (2048, 5632), (4096, 14336), (8192, 28672),
                                    (QK * rng.randint(16, 128), QK * rng.randint(32, 448))])
        return {"path": path, "hidden": hidden, "inter": inter, "format": fmt,
                "n": _log_int(rng, 1, 2048 * 4096 * 14336 // max(4096 * 14336, hidden * inter))}
    shape = rng.choice(["small", "8b"])
    return {"path": "model", "shape": shape, "layers": rng.randint(1, 2), "format": fmt, "n": _log_int(rng, 2, 300)}


# ---- inputs ----------------------------------------------------------------

def _generator(seed, *part):
    return torch.Generator(device="cuda").manual_seed(hash((int(seed),) + part) & 0x7FFFFFFFFFFF)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


_stream = None


def _user_stream():
    """The one stream this program works on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream.cuda_stream


def _lengths(case):
    """Tokens each sequence holds after its step: the case's own, for every seed."""
    if case["low"] == case["high"]:
        return [case["high"]] * case["n"]
    r = random.Random(case["n"] * 1000003 + case["low"] * 101 + case["high"])
    return [case["high"]] + [r.randint(case["low"], case["high"]) for _ in range(case["n"] - 1)]


def _rope(pos, hd):
    """cos and sin rows [len(pos)][hd/2] of the given positions."""
    i = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    angle = torch.as_tensor(pos, device="cuda", dtype=torch.float64)[:, None] * THETA ** (-2.0 * i / hd)
    return angle.cos().float().contiguous(), angle.sin().float().contiguous()


def _cached(seed, seq, row0, rows, width, outliers):
    """Keys (rotated) and values of rows already in a sequence's cache."""
    g = _generator(seed, 1, seq, row0)
    kv = [_randn(g, rows, width) for _ in range(2)]
    if outliers:
        for t in kv:
            u = torch.rand(rows, width, generator=g, device="cuda")
            t.copy_(torch.where(u < 0.01, torch.where(u < 0.005, -8.0, 8.0), t))
    return kv


def _chunks(rows):
    return [(r, min(STEP_ROWS, rows - r)) for r in range(0, rows, STEP_ROWS)]


class _Pool:
    """A paged cache's device memory, seen by torch."""

    def __init__(self, kv):
        base, nbytes, _ = kv.pool()
        self.kv = kv
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (base, False), "version": 2}


def _cache(shape, seed, filled, capacity, outliers=False):
    """A paged cache whose sequence i holds filled[i] tokens on scattered pages."""
    nq, nkv, hd = SHAPES[shape][:3]
    pages = [-(-c // PAGE) for c in capacity]
    kv = native.PagedKV(nq, nkv, hd, sum(pages), len(pages), max(pages))
    ids = np.random.RandomState(seed & 0x7FFFFFFF).permutation(sum(pages)).astype(np.int32)
    at = 0
    for s, p in enumerate(pages):
        kv.set_pages(s, ids[at:at + p])
        at += p
    stream = _user_stream()
    for s, rows in enumerate(filled):
        for r0, n in _chunks(rows):
            k, v = _cached(seed, s, r0, n, nkv * hd, outliers)
            seq = torch.full((n,), s, dtype=torch.int32, device="cuda")
            pos = torch.arange(r0, r0 + n, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            native.check(kv.lib.tq_hip_kv_append_async(kv.h, n, seq.data_ptr(), pos.data_ptr(), k.data_ptr(),
                                                       v.data_ptr(), None, None, stream), "append")
            torch.cuda.synchronize()
    return kv


def _blocks(kv):
    """The cache's codes and scales, views of its memory."""
    b = torch.as_tensor(_Pool(kv), device="cuda").view(-1, 36)
    return b[:, 4:].view(torch.int8), b[:, :4].view(torch.float32)


def _weight_values(g, rows, cols, fmt, std=None):
    """Codes [rows][cols/32][32] and scales of a packed matrix, the packer's rules."""
    top = 127.0 if fmt == "q8" else 7.0
    codes = torch.empty(rows, cols // QK, QK, dtype=torch.int8, device="cuda")
    scales = torch.empty(rows, cols // QK, device="cuda")
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        w = _randn(g, min(step, rows - r), cols // QK, QK) * (std if std else cols ** -0.5)
        d = w.abs().amax(-1) / top
        d = torch.where(d == 0, torch.ones_like(d), d)
        x = w * (1.0 / d)[..., None]
        codes[r:r + step] = (x.sign() * (x.abs() + 0.5).floor()).clamp(-top, top).to(torch.int8)
        scales[r:r + step] = d
    return codes, scales


def _pack(codes, scales, fmt):
    """The matrix on the device in the layout the matmuls read."""
    lib = native.load()
    rows, nb = scales.shape
    if fmt == "q8":
        body = codes.view(torch.uint8)
    else:
        u = (codes + 8).view(torch.uint8)
        body = u[..., :16] | (u[..., 16:] << 4)
    src = torch.cat([scales.view(torch.uint8).view(rows, nb, 4), body], -1).contiguous()
    dst = torch.empty(src.numel(), dtype=torch.uint8, device="cuda")
    pack = lib.tq_hip_q8_pack if fmt == "q8" else lib.tq_hip_q4_pack
    torch.cuda.synchronize()
    native.check(pack(dst.data_ptr(), src.data_ptr(), rows, nb * QK, _user_stream()), "pack")
    torch.cuda.synchronize()
    return dst


def _format(fmt):
    return native.FORMAT_Q8 if fmt == "q8" else native.FORMAT_Q4


def _attn_shapes(shape):
    nq, nkv, hd, hidden = SHAPES[shape][:4]
    return [("wq", nq * hd, hidden), ("wk", nkv * hd, hidden), ("wv", nkv * hd, hidden), ("wo", hidden, nq * hd)]


def _mlp_shapes(hidden, inter):
    return [("wgate", inter, hidden), ("wup", inter, hidden), ("wdown", hidden, inter)]


def _matrices(shapes, seed, layer, fmt):
    return {name: _weight_values(_generator(seed, 2, layer, i), rows, cols, fmt)
            for i, (name, rows, cols) in enumerate(shapes)}


def _norm(seed, layer, which, n):
    return 1.0 + 0.1 * _randn(_generator(seed, 3, layer, which), n)


def _attn_weights(shape, seed, layer, fmt):
    nq, nkv, hd, hidden = SHAPES[shape][:4]
    m = {k: _pack(*v, fmt) for k, v in _matrices(_attn_shapes(shape), seed, layer, fmt).items()}
    m["q_norm"], m["k_norm"] = _norm(seed, layer, 0, hd), _norm(seed, layer, 1, hd)
    w = native.AttnWeights(*(m[k].data_ptr() for k in ("wq", "wk", "wv", "wo", "q_norm", "k_norm")), hidden, EPS,
                           _format(fmt))
    return w, m


def _mlp_weights(hidden, inter, seed, layer, fmt):
    m = {k: _pack(*v, fmt) for k, v in _matrices(_mlp_shapes(hidden, inter), seed, 100 + layer, fmt).items()}
    w = native.MlpWeights(m["wgate"].data_ptr(), m["wup"].data_ptr(), m["wdown"].data_ptr(), hidden, inter,
                          _format(fmt))
    return w, m


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _step_rows(case):
    """Lengths, and the cos and sin rows of each sequence's new token."""
    lens = _lengths(case)
    return (lens,) + _rope([n - 1 for n in lens], SHAPES[case["shape"]][2])


def _inputs(case, seed):
    """The fp32 rows the call is given."""
    g = _generator(seed, 4)
    n = case["n"]
    if case["path"] in ("step", "prefill"):
        nq, nkv, hd = SHAPES[case["shape"]][:3]
        return {"q": _randn(g, n, nq * hd), "k": _randn(g, n, nkv * hd), "v": _randn(g, n, nkv * hd)}
    hidden = case["hidden"] if case["path"] == "mlp" else SHAPES[case["shape"]][3]
    return {"x": _randn(g, n, hidden)}


def prepare(case, seed):
    native.init(0)
    s = {"lib": native.load(), "path": case["path"], "n": case["n"], "stream": _user_stream()}
    if case["path"] == "model":
        _prepare_model(s, case, seed)
        torch.cuda.synchronize()
        return s
    s.update(_inputs(case, seed))
    n = case["n"]
    if case["path"] == "mlp":
        s["w"], s["weights"] = _mlp_weights(case["hidden"], case["inter"], seed, 0, case["format"])
        s["ws"] = torch.empty(s["lib"].tq_hip_mlp_ws_bytes(C.byref(s["w"]), n), dtype=torch.uint8, device="cuda")
        s["out"] = torch.zeros(n, case["hidden"], device="cuda")
        torch.cuda.synchronize()
        return s
    nq, nkv, hd, hidden = SHAPES[case["shape"]][:4]
    if case["path"] in ("step", "layer"):
        lens, s["cos"], s["sin"] = _step_rows(case)
        s["pos"], s["max_pos"] = _int32([m - 1 for m in lens]), max(lens) - 1
        s["kv"] = _cache(case["shape"], seed, [m - 1 for m in lens], lens, case.get("outliers", False))
    else:
        s["cos"], s["sin"] = _rope(range(case["pos"], case["pos"] + n), hd)
        s["pos0"] = case["pos"]
        s["kv"] = _cache(case["shape"], seed, [case["pos"]], [case["pos"] + n])
    s["codes"], s["scales"] = _blocks(s["kv"])
    if case["path"] in ("layer", "layer_batch"):
        s["w"], s["weights"] = _attn_weights(case["shape"], seed, 0, case["format"])
        s["ws"] = torch.empty(s["lib"].tq_hip_attention_layer_ws_bytes(s["kv"].h, C.byref(s["w"]), n),
                              dtype=torch.uint8, device="cuda")
        s["out"] = torch.zeros(n, hidden, device="cuda")
    else:
        s["out"] = torch.zeros(n, nq * hd, device="cuda")
    torch.cuda.synchronize()
    return s


def _prepare_model(s, case, seed):
    lib, fmt = attn.load(), case["format"]
    nq, nkv, hd, hidden, inter = SHAPES[case["shape"]]
    keep, layers = [], (attn.DevLayerWeights * case["layers"])()
    for i in range(case["layers"]):
        aw, am = _attn_weights(case["shape"], seed, i, fmt)
        mw, mm = _mlp_weights(hidden, inter, seed, i, fmt)
        n1, n2 = _norm(seed, i, 2, hidden), _norm(seed, i, 3, hidden)
        layers[i] = attn.DevLayerWeights(n1.data_ptr(), aw, n2.data_ptr(), mw)
        keep += [am, mm, n1, n2]
    embed = _pack(*_weight_values(_generator(seed, 5), VOCAB, hidden, fmt, 0.05), fmt)
    final = _norm(seed, 1000, 4, hidden)
    m = attn.DevModel(attn.AttnConfig(nq, nkv, hd, hidden, THETA, EPS), case["layers"], inter, VOCAB,
                      embed.data_ptr(), final.data_ptr(), layers, _format(fmt))
    ctx, ws = attn.DevCtx(), attn.DevBatchWs()
    native.check(lib.tq_dev_ctx_init(C.byref(ctx), C.byref(m), case["n"] + 1), "tq_dev_ctx_init")
    native.check(lib.tq_dev_batch_ws_init(C.byref(ws), C.byref(m), case["n"]), "tq_dev_batch_ws_init")
    s.update(alib=lib, model=_Model(lib, m, ctx, ws, keep + [layers, embed, final]), tokens=_tokens(case, seed))
    s["logits"] = np.empty((2, VOCAB), np.float32)


def _tokens(case, seed):
    return np.random.RandomState(seed & 0x7FFFFFFF).randint(0, VOCAB, case["n"] + 1).astype(np.int32)


class _Model:
    """A device model and its context; frees them with the state."""

    def __init__(self, lib, m, ctx, ws, keep):
        self.lib, self.m, self.ctx, self.ws, self.keep = lib, m, ctx, ws, keep

    def __del__(self):
        self.lib.tq_dev_batch_ws_free(C.byref(self.ws))
        self.lib.tq_dev_ctx_free(C.byref(self.ctx))


# ---- one pass --------------------------------------------------------------

def run(state):
    s, lib = state, state["lib"]
    if s["path"] == "step":
        native.check(lib.tq_hip_decode_step_async(
            s["kv"].h, s["n"], None, s["pos"].data_ptr(), s["max_pos"], s["q"].data_ptr(), s["k"].data_ptr(),
            s["v"].data_ptr(), s["cos"].data_ptr(), s["sin"].data_ptr(), s["out"].data_ptr(), s["stream"]), "step")
    elif s["path"] == "prefill":
        native.check(lib.tq_hip_prefill_async(
            s["kv"].h, 0, s["pos0"], s["n"], s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
            s["cos"].data_ptr(), s["sin"].data_ptr(), s["out"].data_ptr(), s["stream"]), "prefill")
    elif s["path"] == "layer":
        native.check(lib.tq_hip_attention_layer_async(
            s["kv"].h, C.byref(s["w"]), s["n"], None, s["pos"].data_ptr(), s["max_pos"], s["x"].data_ptr(),
            s["cos"].data_ptr(), s["sin"].data_ptr(), s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(),
            s["stream"]), "layer")
    elif s["path"] == "layer_batch":
        native.check(lib.tq_hip_attention_layer_batch_async(
            s["kv"].h, C.byref(s["w"]), 0, s["pos0"], s["n"], s["x"].data_ptr(), s["cos"].data_ptr(),
            s["sin"].data_ptr(), s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(), s["stream"]), "layer batch")
    elif s["path"] == "mlp":
        native.check(lib.tq_hip_mlp_layer_async(
            C.byref(s["w"]), s["n"], s["x"].data_ptr(), s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(),
            s["stream"]), "mlp")
        return {"out": s["out"]}
    else:
        m, alib, tok, logits = s["model"], s["alib"], s["tokens"], s["logits"]
        m.ctx.pos = 0     # a new prompt
        native.check(alib.tq_dev_forward_batch(C.byref(m.ctx), C.byref(m.ws), tok.ctypes.data, s["n"], 1), "prompt")
        native.check(alib.tq_dev_logits(C.byref(m.ctx), logits[0].ctypes.data), "logits")
        native.check(alib.tq_dev_forward_token(C.byref(m.ctx), int(tok[-1])), "token")
        native.check(alib.tq_dev_logits(C.byref(m.ctx), logits[1].ctypes.data), "logits")
        return {"logits": logits}
    return {"out": s["out"], "codes": s["codes"], "scales": s["scales"]}


# ---- what a pass cannot do without -----------------------------------------

def _matrix_bytes(shapes, fmt):
    return sum(r * c for _, r, c in shapes) // QK * (36 if fmt == "q8" else 20)


def _params(shapes):
    return sum(r * c for _, r, c in shapes)


def _attn_work(shape, new, pairs, kv_tokens):
    """Bytes and operations of attention: `new` rows in and out, `pairs` (query, key) pairs, cached rows read."""
    nq, nkv, hd = SHAPES[shape][:3]
    row = nkv * (hd // QK) * 36 * 2
    return (new * (2 * nq * hd + 2 * nkv * hd + hd) * 4 + (kv_tokens + new) * row, 4.0 * hd * nq * pairs)


def work(case):
    n, path = case["n"], case["path"]
    if path in ("step", "layer"):
        lens = _lengths(case)
        b, f = _attn_work(case["shape"], n, sum(lens), sum(lens) - n)
    elif path in ("prefill", "layer_batch"):
        b, f = _attn_work(case["shape"], n, n * case["pos"] + n * (n + 1) / 2, case["pos"])
    if path in ("step", "prefill"):
        return {"bytes": b, "flops": f}
    if path in ("layer", "layer_batch"):
        nq, nkv, hd, hidden = SHAPES[case["shape"]][:4]
        m = _attn_shapes(case["shape"])
        b += _matrix_bytes(m, case["format"]) + n * (2 * hidden - 2 * nq * hd - 2 * nkv * hd) * 4
        return {"bytes": b, "flops": f + 2.0 * n * _params(m)}
    if path == "mlp":
        m = _mlp_shapes(case["hidden"], case["inter"])
        return {"bytes": _matrix_bytes(m, case["format"]) + 8 * n * case["hidden"], "flops": 2.0 * n * _params(m)}
    nq, nkv, hd, hidden, inter = SHAPES[case["shape"]]
    m = _attn_shapes(case["shape"]) + _mlp_shapes(hidden, inter)
    head = [("embed", VOCAB, hidden)]
    kv = nkv * (hd // QK) * 36 * 2
    # every matrix is read for the prompt and again for the token
    b = case["layers"] * (2 * _matrix_bytes(m, case["format"]) + (2 * n + 2) * kv) + 2 * _matrix_bytes(
        head, case["format"]) + 8 * VOCAB + (n + 1) * hidden * 4
    f = 2.0 * (n + 1) * case["layers"] * _params(m) + 4.0 * VOCAB * hidden
    return {"bytes": b, "flops": f + case["layers"] * 4.0 * hd * nq * (n * (n + 1) / 2 + n + 1)}


def tolerance(case):
    """About four times what the paths show against the 64-bit evaluation: the
    attention core sums in fp32, and past a projection a last-bit difference
    moves an activation code by one now and then."""
    if case["path"] in ("step", "prefill"):
        return {"rel": 4e-5, "max": 8e-3}
    if case["path"] == "mlp":
        return {"rel": 4e-4, "max": 2.5e-2}
    if case["path"] in ("layer", "layer_batch"):
        return {"rel": 2e-3, "max": 5e-2, "differ": 1e-3}
    return {"rel": 6e-2, "max": 0.4}


# ---- the same in 64 bits ---------------------------------------------------

def _quantize(x):
    """Activation blocks as the format defines them: fp32 scale and rounded codes, as 64-bit values."""
    b = x.float().reshape(*x.shape[:-1], -1, QK)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d == 0, torch.zeros_like(d), 1.0 / d)
    return ((b * inv).round().double() * d.double()).reshape(x.shape)


def _rotate(x, cos, sin):
    """RoPE of rows [n][heads][hd] in fp32, half-split pairs."""
    x, cos, sin = x.float(), cos[:, None, :], sin[:, None, :]
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _matmul(x, w):
    """Rows x (quantized here) times a packed matrix, in row pieces."""
    codes, scales = w
    xq = _quantize(x)
    step = max(1, (1 << 27) // (codes.shape[1] * QK))
    return torch.cat([xq @ (codes[r:r + step].double() * scales[r:r + step].double()[..., None]).flatten(1).t()
                      for r in range(0, codes.shape[0], step)], -1)


def _rmsnorm(x, w):
    return (x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()).float()


def _attend(q, k, v, first):
    """Causal attention of rows q [n][nq][hd] over k, v [len][nkv][hd]; row i sees first + i + 1 keys."""
    n, nq, hd = q.shape
    nkv, g = k.shape[1], q.shape[1] // k.shape[1]
    scale = float(np.float32(1.0) / np.sqrt(np.float32(hd)))
    qd = _quantize(q)
    out = torch.empty(n, nq, hd, dtype=torch.float64, device="cuda")
    mask = torch.arange(k.shape[0], device="cuda")[None, :] > first + torch.arange(n, device="cuda")[:, None]
    for h in range(nq):
        s = (qd[:, h] @ k[:, h // g].t()) * scale
        out[:, h] = s.masked_fill_(mask, -math.inf).softmax(-1) @ v[:, h // g]
    return out.flatten(1)


def _exact_core(case, seed, q, k, v, seq_rows):
    """The attention core of every sequence: (rows of the call, cached rows, first position) each."""
    nq, nkv, hd = SHAPES[case["shape"]][:3]
    out = torch.empty(q.shape[0], nq * hd, dtype=torch.float64, device="cuda")
    for seq, (rows, cached) in enumerate(seq_rows):
        cos, sin = _rope(range(cached, cached + (rows.stop - rows.start)), hd)
        qr = _rotate(q[rows].reshape(-1, nq, hd), cos, sin)
        kr = _rotate(k[rows].reshape(-1, nkv, hd), cos, sin)
        ks, vs = [], []
        for r0, n in _chunks(cached):
            kc, vc = _cached(seed, seq, r0, n, nkv * hd, case.get("outliers", False))
            ks.append(_quantize(kc))
            vs.append(_quantize(vc))
        ks = torch.cat(ks + [_quantize(kr.flatten(1))]).reshape(-1, nkv, hd)
        vs = torch.cat(vs + [_quantize(v[rows])]).reshape(-1, nkv, hd)
        out[rows] = _attend(qr, ks, vs, cached)
    return out


def _exact_layer(case, seed, layer, x, seq_rows):
    nq, nkv, hd = SHAPES[case["shape"]][:3]
    w = _matrices(_attn_shapes(case["shape"]), seed, layer, case["format"])
    q, k, v = (_matmul(x, w[m]) for m in ("wq", "wk", "wv"))
    q = _rmsnorm(q.reshape(-1, nq, hd), _norm(seed, layer, 0, hd)).flatten(1)
    k = _rmsnorm(k.reshape(-1, nkv, hd), _norm(seed, layer, 1, hd)).flatten(1)
    return _matmul(_exact_core(case, seed, q, k, v.float(), seq_rows), w["wo"])


def _exact_mlp(hidden, inter, seed, layer, fmt, x):
    w = _matrices(_mlp_shapes(hidden, inter), seed, 100 + layer, fmt)
    g = _matmul(x, w["wgate"])
    return _matmul(g * torch.sigmoid(g) * _matmul(x, w["wup"]), w["wdown"])


def exact(case, seed):
    path, n = case["path"], case["n"]
    if path == "model":
        return {"logits": _exact_model(case, seed)}
    x = _inputs(case, seed)
    if path == "mlp":
        return {"out": _exact_mlp(case["hidden"], case["inter"], seed, 0, case["format"], x["x"])}
    if path in ("step", "layer"):
        seq_rows = [(slice(i, i + 1), m - 1) for i, m in enumerate(_lengths(case))]
    else:
        seq_rows = [(slice(0, n), case["pos"])]
    if path in ("step", "prefill"):
        out = _exact_core(case, seed, x["q"], x["k"], x["v"], seq_rows)
    else:
        out = _exact_layer(case, seed, 0, x["x"], seq_rows)
    return {"out": out, "codes": None, "scales": None}


def _exact_model(case, seed):
    """Logits after the prompt and after the next token: one pass over all positions gives both."""
    hidden, inter = SHAPES[case["shape"]][3:]
    n = case["n"] + 1
    codes, scales = _weight_values(_generator(seed, 5), VOCAB, hidden, case["format"], 0.05)
    tok = torch.as_tensor(_tokens(case, seed), device="cuda").long()
    x = (codes[tok].double() * scales[tok].double()[..., None]).flatten(1)
    for i in range(case["layers"]):
        x = x + _exact_layer(case, seed, i, _rmsnorm(x, _norm(seed, i, 2, hidden)), [(slice(0, n), 0)])
        x = x + _exact_mlp(hidden, inter, seed, i, case["format"], _rmsnorm(x, _norm(seed, i, 3, hidden)))
    return _matmul(_rmsnorm(x[-2:], _norm(seed, 1000, 4, hidden)), (codes, scales))
