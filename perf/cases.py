"""The performance cases: what a user of this framework has it do, through its
public entry points, over the range of sizes those entry points serve.

listed() names twelve cases, draw() gives further ones of the same ranges,
prepare() makes what the user's program holds before the call, run() is one
pass, work() the bytes and operations the pass cannot do without, tolerance()
and exact() what its outputs are compared with.

Every float operation of this framework has one fixed order (its outputs are
bit-identical to its CPU oracle and to themselves), so every case is "exact".
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import rustyneedle_amd as rn
from rustyneedle_amd import needle3

DEVICE = "cuda"
INT8_COLUMNS = (384, 512, 1024, 1536, 2048)  # the row widths the int8 matrices take


def listed():
    return [
        # one token through one int8 layer matrix: the smallest call, all latency
        dict(name="vector_2048x512", op="int8", tokens=1, rows=2048, columns=512, plane=0),
        # a long prompt's rows through the gate/up matrix of the decoder
        dict(name="batch_600x4096x512", op="int8", tokens=600, rows=4096, columns=512, plane=0),
        # one token's logits in the archive format: 4-bit embedding, input rotated first
        dict(name="codebook_logits_8192x768", op="codebook", tokens=1, rows=8192, columns=768, bits=4, group=128),
        # a prompt chunk through the stacked q/k/v/gate rows of an archive layer (2-bit)
        dict(name="codebook_256x2048x768", op="codebook", tokens=256, rows=2048, columns=768, bits=2, group=128),
        # attention over caller-held fp16 caches: 64 sequences of 8 heads, ragged lengths
        dict(name="attend_512_heads", op="attend", heads=512, longest=512),
        # the interactive token loop: 64 greedy tokens after a 256-position cache
        dict(name="decode_256", op="decode", context=256, steps=64),
        # the prompt of an ordinary request, and one that fills most of the position table
        dict(name="prefill_256", op="prefill", tokens=256),
        dict(name="prefill_1000", op="prefill", tokens=1000),
        # serving: 64 ragged sequences decoded together
        dict(name="batch_decode_64", op="batch_decode", sequences=64, longest=512, steps=32),
        # a chat turn over an archive model: the system prompt's session cloned, the
        # turn's prompt fed, an answer decoded
        dict(name="needle3_turn_600", op="needle3", prefix=600, prompt=24, steps=16),
        # a long document fed into a new archive session, its first answer token
        dict(name="needle3_feed_2000", op="needle3", prefix=0, prompt=2000, steps=1),
        # 30 s of 16 kHz audio to text: front end, encoder, 48 tokens
        dict(name="speech_30s", op="speech", samples=480000, steps=48),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    op = rng.choice(("int8", "codebook", "attend", "decode", "prefill", "batch_decode", "needle3", "speech"))
    if op == "int8":
        return dict(op=op, tokens=1 if rng.random() < 0.3 else _log(rng, 2, 2048), rows=_log(rng, 48, 8192),
                    columns=rng.choice(INT8_COLUMNS), plane=rng.randrange(2))
    if op == "codebook":
        return dict(op=op, tokens=1 if rng.random() < 0.3 else _log(rng, 2, 512), rows=_log(rng, 48, 8192),
                    columns=_log(rng, 64, 4096), bits=rng.choice((2, 4, 5)), group=rng.choice((64, 128, 256)))
    if op == "attend":
        return dict(op=op, heads=_log(rng, 1, 1024), longest=_log(rng, 8, 1024))
    if op == "decode":
        return dict(op=op, context=_log(rng, 1, 900), steps=_log(rng, 1, 64))
    if op == "prefill":
        return dict(op=op, tokens=_log(rng, 4, 1000))
    if op == "batch_decode":
        return dict(op=op, sequences=_log(rng, 2, 96), longest=_log(rng, 32, 700), steps=_log(rng, 1, 12))
    if op == "needle3":
        return dict(op=op, prefix=rng.choice((0, _log(rng, 4, 1200))), prompt=_log(rng, 1, 1200),
                    steps=_log(rng, 1, 8))
    return dict(op=op, samples=_log(rng, 4000, 480000), steps=_log(rng, 1, 48))  # windows of 25 to 3000 frames


# ---- what a program keeps between calls ------------------------------------------

@functools.lru_cache(maxsize=None)
def _decoder():
    """The 20-layer decoder (d_model 512, 8 heads of 64, FFN 2048, vocab 8192)."""
    return rn.Model(dict(rn.NEEDLE_DECODER))


@functools.lru_cache(maxsize=None)
def _needle3():
    """A model of the documented Needle 3 geometry from a synthetic archive."""
    return needle3.Model(needle3.synthetic_archive(needle3.NEEDLE3))


@functools.lru_cache(maxsize=4)
def _speech(frames):
    """The speech model (6 + 4 layers of 384) for a window of `frames` mel frames, and its log-mel front end."""
    return (rn.Whistle(dict(rn.WHISTLE, frames=frames)),
            rn.Frontend(80, 512, 400, 160, rn.synthetic_mel_filters(80, 512)))


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32).to(dtype)


def _tokens(rng, vocab, n):
    return rng.integers(0, vocab, n, dtype=np.uint32)


def _lengths(rng, longest, n):
    """Ragged cache lengths of [longest / 16, longest], one of them the longest."""
    out = rng.integers(max(1, longest // 16), longest + 1, n).astype(np.int32)
    out[rng.integers(0, n)] = longest
    return out


def _blob(rng, c):
    """A codebook record's bytes: packed indices, then fp16 group norms."""
    padded = _padded(c)
    index_bits = 2 if c["bits"] == 5 else c["bits"]
    packed = rng.integers(0, 256, c["rows"] * padded * index_bits // 8, dtype=np.uint8)
    norms = rng.uniform(0.5, 2.0, c["rows"] * (padded // c["group"])).astype(np.float16)
    return packed, norms


def _padded(c):
    return -(-c["columns"] // c["group"]) * c["group"]


def _int8_inputs(c, seed):
    rng = np.random.default_rng(seed)
    codes = rng.integers(-127, 128, (c["rows"], c["columns"]), dtype=np.int8)
    scales = rng.uniform(1e-3, 1e-2, (c["rows"], c["columns"] // 32)).astype(np.float32)
    return codes, scales, _normal(_generator(seed), (c["tokens"], c["columns"]))


def _codebook_inputs(c, seed):
    packed, norms = _blob(np.random.default_rng(seed), c)
    return packed, norms, _normal(_generator(seed), (c["tokens"], c["columns"]))


def _attend_inputs(c, seed):
    g = _generator(seed)
    n, longest = c["heads"], c["longest"]
    lengths = _lengths(np.random.default_rng(seed), longest, n)
    return (_normal(g, (n, 64)), _normal(g, (n, longest, 64), torch.float16), _normal(g, (n, longest, 64), torch.float16),
            torch.from_numpy(lengths).to(DEVICE))


def prepare(case, seed):
    c, op = dict(case), case["op"]
    rng = np.random.default_rng(seed)
    if op == "int8":
        codes, scales, x = _int8_inputs(c, seed)
        m = rn.QuantisedMatrix(codes, scales, rn.FORM_PLANE if c["plane"] else rn.FORM_PANEL)
        return dict(c, matrix=m, x=x, y=torch.empty((c["tokens"], c["rows"]), device=DEVICE))
    if op == "codebook":
        packed, norms, x = _codebook_inputs(c, seed)
        m = rn.CodebookMatrix(np.concatenate([packed, norms.view(np.uint8)]), c["rows"], c["columns"], c["group"],
                              c["bits"], rn.synthetic_codebook(c["group"]))
        return dict(c, matrix=m, x=x, rotated=torch.empty((c["tokens"], m.padded), device=DEVICE),
                    y=torch.empty((c["tokens"], c["rows"]), device=DEVICE))
    if op == "attend":
        q, k, v, lengths = _attend_inputs(c, seed)
        return dict(c, q=q, k=k, v=v, lengths=lengths, out=torch.empty_like(q))
    if op in ("decode", "prefill", "batch_decode"):
        model = _decoder()
        cfg = model.config
        vocab = cfg["vocab"]

        def cache(g, length):
            shape = (cfg["layers"], cfg["heads"], length, cfg["head_dim"])
            return [_normal(g, shape, torch.float16).cpu().numpy() for _ in range(2)]

        if op == "decode":
            s = model.session(c["context"] + c["steps"])
            s.set_cache(*cache(_generator(seed), c["context"]))
            return dict(c, session=s, first=int(_tokens(rng, vocab, 1)[0]))
        if op == "prefill":
            return dict(c, session=model.session(c["tokens"]), ids=_tokens(rng, vocab, c["tokens"]))
        lengths = _lengths(rng, c["longest"], c["sequences"])
        b = rn.Batch(model, c["sequences"], c["longest"] + c["steps"])
        g = _generator(seed)
        for i, n in enumerate(lengths):
            b.set_cache(i, *cache(g, int(n)))
        return dict(c, batch=b, lengths=lengths, first=_tokens(rng, vocab, c["sequences"]))
    if op == "needle3":
        model = _needle3()
        vocab = model.geometry["vocab"]
        capacity = c["prefix"] + c["prompt"] + c["steps"]
        base = None
        if c["prefix"]:
            base = model.session(capacity)
            base.feed(_tokens(rng, vocab, c["prefix"]))
        return dict(c, model=model, base=base, capacity=capacity, ids=_tokens(rng, vocab, c["prompt"]))
    whistle, frontend = _speech(c["samples"] // 160)  # a front-end hop is 160 samples
    # speech-like samples: a few gliding tones under a slow envelope, and noise
    t = np.arange(c["samples"]) / 16000.0
    x = 0.02 * rng.standard_normal(c["samples"])
    for _ in range(4):
        f0, f1, a = rng.uniform(100, 3000), rng.uniform(-80, 80), rng.uniform(0.02, 0.1)
        x += a * np.sin(2 * np.pi * (f0 * t + 0.5 * f1 * t * np.sin(t))) * (1 + np.sin(rng.uniform(2, 20) * t))
    return dict(c, whistle=whistle, frontend=frontend, samples=x.astype(np.float32),
                first=int(_tokens(rng, whistle.config["vocab"], 1)[0]))


def run(s):
    op = s["op"]
    if op == "int8":
        if s["tokens"] == 1:
            s["matrix"].multiply_vector(s["x"].data_ptr(), s["y"].data_ptr())
        else:
            rn.check(rn.lib.rn_matrix_multiply_batch(s["matrix"].handle, s["x"].data_ptr(), s["tokens"],
                                                     s["y"].data_ptr(), None, None))
        return s["y"]
    if op == "codebook":
        m = s["matrix"]
        m.prepare(s["x"].data_ptr(), s["tokens"], s["rotated"].data_ptr())
        if s["tokens"] == 1:
            rn.check(rn.lib.rn_matrix_multiply_vector(m.handle, s["rotated"].data_ptr(), s["y"].data_ptr(), None, None))
        else:
            rn.check(rn.lib.rn_matrix_multiply_batch(m.handle, s["rotated"].data_ptr(), s["tokens"],
                                                     s["y"].data_ptr(), None, None))
        return dict(rotated=s["rotated"], y=s["y"])
    if op == "attend":
        rn.check(rn.lib.rn_attend_heads(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                        s["lengths"].data_ptr(), s["heads"], s["longest"], 64, s["out"].data_ptr(),
                                        None))
        return s["out"]
    if op == "decode":
        s["session"].truncate(s["context"])
        ids = s["session"].decode_greedy(s["first"], s["steps"])
        return dict(ids=ids.astype(np.int64), logits=s["session"].logits())
    if op == "prefill":
        s["session"].truncate(0)
        s["session"].feed(s["ids"])
        return dict(hidden=s["session"].hidden(), logits=s["session"].logits())
    if op == "batch_decode":
        s["batch"].truncate(s["lengths"])
        ids = s["batch"].decode_greedy(s["first"], s["steps"])
        return dict(ids=ids.astype(np.int64), logits=s["batch"].logits())
    if op == "needle3":
        session = s["base"].clone() if s["base"] is not None else s["model"].session(s["capacity"])
        session.feed(s["ids"])
        ids = session.decode_greedy(int(s["ids"][-1]), s["steps"])
        return dict(ids=ids.astype(np.int64), hidden=session.hidden(), logits=session.logits())
    w = s["whistle"]
    encoded, spread = w.encode_samples(s["frontend"], s["samples"])
    ids = w.decode_greedy(s["first"], s["steps"])
    return dict(encoded=encoded, spread=float(spread), ids=ids.astype(np.int64), logits=w.logits())


# ---- the work of a pass -----------------------------------------------------------

def _int8_bytes(rows, columns):
    return rows * columns + 4 * rows * (columns // 32)


def _decoder_layer_bytes(cfg):
    d, f = cfg["d_model"], cfg["ffn"]
    return _int8_bytes(3 * d, d) + _int8_bytes(d, d) + _int8_bytes(2 * f, d) + _int8_bytes(d, f)


def _decoder_flops(cfg, tokens):
    """The layers' products of `tokens` tokens (two operations a weight)."""
    d, f = cfg["d_model"], cfg["ffn"]
    return 2 * tokens * cfg["layers"] * (4 * d * d + 3 * d * f)


def _needle3_layer(g):
    """(bytes of one layer's weights, multiplications of one token through it)."""
    d, heads, kv = g["d_model"], g["num_heads"] * 64, g["num_kv_heads"] * 64
    lanes, n = g["mhc_lanes"], g["hada_n"]
    weights = (2 * heads + 2 * kv) * d + heads * d + (2 * lanes + lanes * lanes) * lanes * d
    floats = 6 * 1024 + 5 * n + 16 * d + g["qkv_conv_taps"] * (heads + 2 * kv)
    return weights // 4 + weights // 64 + 4 * floats, weights + 6 * n * 32 + 8 * (d + n)


def work(case):
    c, op = case, case["op"]
    if op == "int8":
        return dict(bytes=_int8_bytes(c["rows"], c["columns"]) + 4 * c["tokens"] * (c["rows"] + c["columns"]),
                    flops=2 * c["tokens"] * c["rows"] * c["columns"])
    if op == "codebook":
        padded, index_bits = _padded(c), 2 if c["bits"] == 5 else c["bits"]
        packed = c["rows"] * padded * index_bits // 8 + 2 * c["rows"] * (padded // c["group"])
        return dict(bytes=packed + 4 * c["tokens"] * (c["rows"] + c["columns"] + padded),
                    flops=2 * c["tokens"] * c["rows"] * padded)
    if op == "attend":
        rows = c["heads"] * c["longest"] * 17 // 32  # the mean of the ragged lengths
        return dict(bytes=256 * rows + 2 * 256 * c["heads"], flops=4 * 64 * rows)
    if op in ("decode", "prefill", "batch_decode"):
        cfg = rn.NEEDLE_DECODER
        d, layers, vocab = cfg["d_model"], cfg["layers"], cfg["vocab"]
        weights, logits = layers * _decoder_layer_bytes(cfg), _int8_bytes(vocab, d)
        row = 4 * d * layers  # one position's fp16 keys and values
        if op == "prefill":
            n = c["tokens"]
            return dict(bytes=weights + logits + row * n + 4 * vocab + 4 * d,
                        flops=_decoder_flops(cfg, n) + 2 * vocab * d + 2 * d * layers * n * (n + 1))
        n = c["sequences"] if op == "batch_decode" else 1
        cached = c["longest"] * 17 // 32 if op == "batch_decode" else c["context"]
        per_step = weights + logits + n * row * (cached + c["steps"] // 2 + 1)
        flops = _decoder_flops(cfg, n) + 2 * n * vocab * d + 4 * n * d * layers * (cached + c["steps"] // 2 + 1)
        return dict(bytes=c["steps"] * per_step + 4 * n * vocab, flops=c["steps"] * flops)
    if op == "needle3":
        g = needle3.NEEDLE3
        layer_bytes, per_token = _needle3_layer(g)
        layers, window = g["num_layers"], g["sliding_window"]
        fed, first = c["prompt"], c["prefix"]
        kv, heads = 2 * g["num_kv_heads"] * 64, g["num_heads"] * 64
        end = first + fed + c["steps"]
        pairs = sum(min(p + 1, window) for p in range(first, end)) * 16 + sum(p + 1 for p in range(first, end)) * 4
        logits = g["vocab"] * g["d_model"] // 2 + g["vocab"] * g["d_model"] // 64
        passes = 1 + c["steps"]  # the weights are read once by the feed and once a decoded token
        cache = layers * kv * (first + fed) + c["steps"] * layers * kv * min(first + fed, window)
        return dict(bytes=passes * layers * layer_bytes + (c["steps"] + 1) * logits + cache,
                    flops=2 * (fed + c["steps"]) * layers * per_token + 4 * heads * pairs
                    + 2 * (c["steps"] + 1) * g["vocab"] * g["d_model"])
    w = rn.WHISTLE
    d, f, vocab, frames = w["d_model"], w["ffn"], w["vocab"], (c["samples"] // 160 - 1) // 2 + 1
    enc = _int8_bytes(4 * d, d) + _int8_bytes(2 * f, d) + _int8_bytes(d, f)
    dec = enc + _int8_bytes(2 * d, d)
    memory = w["dec_layers"] * 2 * frames * d
    enc_flops = 2 * frames * w["enc_layers"] * (4 * d * d + 3 * d * f) + 4 * d * w["enc_layers"] * frames * frames
    stem = 4 * frames * 3 * w["mels"] * d + 2 * frames * 3 * d * d + 2 * frames * w["dec_layers"] * 2 * d * d
    dec_flops = w["dec_layers"] * (2 * (6 * d * d + 3 * d * f) + 4 * frames * d) + 2 * vocab * d
    return dict(bytes=4 * c["samples"] + 4 * frames * d + w["enc_layers"] * enc + 2 * memory
                + c["steps"] * (w["dec_layers"] * dec + _int8_bytes(vocab, d) + memory),
                flops=enc_flops + stem + c["steps"] * dec_flops)


def tolerance(case):
    return "exact"


# ---- the same outputs in 64 bits ----------------------------------------------------

def _codes(x, limit):
    """Codes and scales of rows of float64 values: scale = peak / 127 (1 for a zero peak)."""
    peak = x.abs().amax(-1, keepdim=True)
    scale = torch.where(peak > 0, peak / 127.0, torch.ones_like(peak))
    return torch.clamp(torch.round(x / scale), -limit, 127.0), scale


def _hadamard(n):
    h = torch.ones((1, 1), dtype=torch.float64, device=DEVICE)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(n)


def _level_table(bits, group):
    """The float levels of a width, as int8 entries and their scale."""
    if bits == 5:
        a = 1.2240064 / math.sqrt(group)
        levels = torch.tensor([0.0, a, 0.0, -a], dtype=torch.float64)
    else:
        at = {2: (0, 4), 4: (12, 28)}[bits]
        levels = torch.from_numpy(rn.synthetic_codebook(group)[at[0]:at[1]].astype(np.float64))
    scale = levels.abs().max() / 127.0
    return torch.round(levels / scale).to(DEVICE), float(scale)


def exact(case, seed):
    """In 64 bits: the products and the attention. A whole model has no such
    value: it requantises every layer's input to int8 codes, so that a rounding in
    the last place flips a code now and then, which moves the logits by about 1e-2
    and a greedy continuation altogether."""
    c, op = case, case["op"]
    if op == "int8":
        codes, scales, x = _int8_inputs(c, seed)
        q, sx = _codes(x.double(), 128.0)
        w = torch.from_numpy(codes).to(DEVICE).double()
        w = w * torch.from_numpy(scales).to(DEVICE).double().repeat_interleave(32, dim=1)
        return (q @ w.T.contiguous()) * sx
    if op == "codebook":
        packed, norms, x = _codebook_inputs(c, seed)
        rows, group, padded, tokens = c["rows"], c["group"], _padded(c), c["tokens"]
        index_bits = 2 if c["bits"] == 5 else c["bits"]
        rotated = torch.zeros((tokens, padded), dtype=torch.float64, device=DEVICE)
        rotated[:, :c["columns"]] = x.double()
        rotated = (rotated.reshape(-1, group) @ _hadamard(group)).reshape(tokens, -1, group)
        q, sx = _codes(rotated, 127.0)
        table, level_scale = _level_table(c["bits"], group)
        shifts = torch.arange(0, 8, index_bits, device=DEVICE)
        index = (torch.from_numpy(packed).to(DEVICE).long()[:, None] >> shifts) & ((1 << index_bits) - 1)
        w = table[index.reshape(rows, -1, group)] * torch.from_numpy(norms).to(DEVICE).double().reshape(rows, -1, 1)
        y = ((q * sx).reshape(tokens, -1) @ w.reshape(rows, -1).T.contiguous()) * level_scale
        return dict(rotated=rotated.reshape(tokens, padded), y=y)
    if op == "attend":
        q, k, v, lengths = _attend_inputs(c, seed)
        scores = torch.sum(k.double() * q.double()[:, None, :], -1) / 8.0
        past = torch.arange(c["longest"], device=DEVICE)[None, :] >= lengths[:, None]
        p = torch.softmax(scores.masked_fill(past, float("-inf")), -1)
        return torch.sum(p[:, :, None] * v.double(), 1)
    return None
