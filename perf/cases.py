"""The work a user of this library has it do, as cases that can be timed and compared.

Each case goes through the public entry points the way kore's own call sites do: one token's or one
chunk's attention over every layer of a cache, one weight matrix against a chunk, whole layers, a
whole engine over a GGUF file.  Sizes are the Qwen2.5 widths of the benchmark and the tests, and
ragged ones between them; weights and activations are synthetic.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import struct
import tempfile

import numpy as np
import torch

import kore_amd
from kore_amd import hip, layer, model, qmv

Q4K, Q6K = qmv.KORE_QMV_Q4_K, qmv.KORE_QMV_Q6_K
ROPE_BASE = 1e6
EPS = 1e-6

# (n_embd, n_ff, n_head, n_head_kv) of the 7B, 3B and 1.5B models
WIDTHS = {"7b": (3584, 18944, 28, 4), "3b": (2048, 11008, 16, 2), "1.5b": (1536, 8960, 12, 2)}
# attention geometries of the same family: the 0.5B, 1.5B, 3B and 7B models
FAMILY = [(14, 2, 64), (12, 2, 128), (16, 2, 128), (28, 4, 128)]


def listed():
    return [
        # one decode step's attention on one layer of the smallest model: all latency and launches
        {"name": "decode_small", "kind": "decode", "nh": 14, "nkv": 2, "hd": 64, "layers": 1, "pos": 511, "window": 0},
        # one token's attention over every layer at an ordinary context
        {"name": "decode_4k", "kind": "decode", "nh": 28, "nkv": 4, "hd": 128, "layers": 28, "pos": 4111, "window": 0},
        # the same at the longest context the models take
        {"name": "decode_32k", "kind": "decode", "nh": 16, "nkv": 2, "hd": 128, "layers": 36, "pos": 32700, "window": 0},
        # a decode of a geometry outside the Qwen2.5 family, which kore accepts as well
        {"name": "decode_other_geometry", "kind": "decode", "nh": 33, "nkv": 3, "hd": 96, "layers": 8, "pos": 2000,
         "window": 0},
        # a long prompt's attention in one call
        {"name": "prefill_2048", "kind": "prefill", "nh": 28, "nkv": 4, "hd": 128, "rows": 2048, "pos0": 0},
        # the ragged end of a long prompt, over a long cache
        {"name": "prefill_tail", "kind": "prefill", "nh": 12, "nkv": 2, "hd": 128, "rows": 333, "pos0": 7001},
        # a prompt of a geometry outside the family
        {"name": "prefill_other_geometry", "kind": "prefill", "nh": 33, "nkv": 3, "hd": 96, "rows": 700, "pos0": 100},
        # kore with only its attention replaced: host buffers in and out, layer by layer, a 64-row chunk
        {"name": "host_chunk", "kind": "host", "nh": 28, "nkv": 4, "hd": 128, "layers": 4, "rows": 64, "pos0": 448},
        # one Q6_K matrix against the last, short chunk of a prompt
        {"name": "matmul_short_chunk", "kind": "matmul", "rows": 3584, "cols": 18944, "type": Q6K, "nb": 19},
        # four layers of a decode step: matvecs, attention and everything between them
        {"name": "layers_decode", "kind": "layers", "width": "7b", "layers": 4, "rows": 1, "pos0": 4100},
        # four layers of a full 64-row prompt chunk
        {"name": "layers_chunk", "kind": "layers", "width": "7b", "layers": 4, "rows": 64, "pos0": 448},
        # the engine: a prompt in chunks (the last one ragged), then tokens one by one, logits each time
        {"name": "engine", "kind": "engine", "width": "1.5b", "layers": 12, "vocab": 151936, "prompt": 150, "tokens": 8},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "host", "matmul", "layers", "layers", "engine"])
    if kind in ("decode", "prefill") and rng.random() < 0.3:
        nkv = rng.randint(1, 8)
        nh, hd = nkv * rng.randint(1, 12), 2 * rng.randint(8, 128)
        other = True
    else:
        nh, nkv, hd = rng.choice(FAMILY)
        other = False
    if kind == "decode":
        pos = _log_int(rng, 1, 6000 if other else 32767)
        window = 0 if rng.random() < 0.8 else rng.choice([512, 1024, 4096])
        return {"kind": kind, "nh": nh, "nkv": nkv, "hd": hd, "layers": _log_int(rng, 1, 4 if window else 8 if other else 28),
                "pos": pos, "window": window}
    if kind == "prefill":
        return {"kind": kind, "nh": nh, "nkv": nkv, "hd": hd, "rows": _log_int(rng, 1, 500 if other else 2048),
                "pos0": rng.choice([0, _log_int(rng, 1, 1000 if other else 8000)])}
    if kind == "host":
        return {"kind": kind, "nh": nh, "nkv": nkv, "hd": hd, "layers": rng.randint(1, 8),
                "rows": rng.choice([1, 64, rng.randint(2, 63)]), "pos0": _log_int(rng, 1, 4000)}
    if kind == "matmul":
        return {"kind": kind, "rows": _log_int(rng, 64, 20000), "cols": 256 * _log_int(rng, 2, 74),
                "type": rng.choice([Q4K, Q6K]), "nb": rng.choice([64, rng.randint(1, 64)])}
    if kind == "layers":
        return {"kind": kind, "width": rng.choice(sorted(WIDTHS)), "layers": rng.randint(1, 4),
                "rows": rng.choice([1, 1, 64, rng.randint(2, 63)]), "pos0": _log_int(rng, 1, 6000)}
    return {"kind": "engine", "width": rng.choice(["1.5b", "3b"]), "layers": rng.randint(2, 8),
            "vocab": _log_int(rng, 1000, 40000), "prompt": _log_int(rng, 2, 150), "tokens": rng.randint(1, 8)}


# ---- inputs ------------------------------------------------------------------

_streams = []


def _stream():
    """The program's one stream: a pass starts when the one before it has ended."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _acts(g, rows, heads, hd):
    """Rows of q or k: N(0, 1) with about one channel in a hundred six times as large, as activations have."""
    x = torch.randn(rows, heads * hd, generator=g, device="cuda")
    big = torch.rand(heads * hd, generator=g, device="cuda") < 0.01
    return x * torch.where(big, 6.0, 1.0)


def _normal(g, rows, n):
    return torch.randn(rows, n, generator=g, device="cuda")


def _blocks(g, wtype, rows, cols, size=1.0):
    """GGUF blocks [rows][cols / 256][144 or 210] of weights with a mean near zero and a deviation of about 0.02 * size."""
    nb = cols // 256
    w = torch.randint(0, 256, (rows, nb, 144 if wtype == Q4K else 210), generator=g, device="cuda", dtype=torch.uint8)
    s = size * (0.5 + torch.rand(rows, nb, 1, generator=g, device="cuda"))
    if wtype == Q4K:
        w[:, :, 0:2] = (8e-5 * s).half().view(torch.uint8)
        w[:, :, 2:4] = (6e-4 * s).half().view(torch.uint8)
    else:
        w[:, :, 208:210] = (1.46e-5 * s).half().view(torch.uint8)
    return w


def _qmat(wtype, w, rows, cols):
    return qmv.QMat(wtype, rows, cols, device_ptr=w.data_ptr())


class _State:
    """What the program keeps between calls; closes its handles when it goes."""

    def __init__(self):
        self.closing = []

    def __del__(self):
        try:
            torch.cuda.synchronize()
            for c in reversed(self.closing):
                c.close()
        except Exception:
            pass


def _attn(s, c, n_layer, ctx, nh, nkv, hd, window=0):
    s.attn = kore_amd.KoreAttn(n_layer, ctx, nh, nkv, hd, ROPE_BASE, window)
    s.closing.append(s.attn)


def _cache_rows(c):
    """Positions already in the cache before the pass: [first, first + n)."""
    pos = c["pos"] if c["kind"] == "decode" else c["pos0"]
    w = c.get("window", 0)
    return (max(0, pos - w), min(pos, w)) if w else (0, pos)


def _cache(c, seed, l, nkv, hd):
    g = _gen(seed * 1000 + 17 * l + 5)
    n = max(1, _cache_rows(c)[1])
    return _acts(g, n, nkv, hd), _normal(g, n, nkv * hd)


def _fill(s, c, seed, n_layer, nkv, hd):
    """The cache of earlier positions; a ring that has wrapped gets its last rows."""
    first, n = _cache_rows(c)
    if n == 0:
        return
    w = c.get("window", 0)
    for l in range(n_layer):
        k, v = _cache(c, seed, l, nkv, hd)
        if w and first + n > w:
            # K of position p carries the RoPE of p: rows past the window can only be written by decodes
            q = torch.zeros(s.attn.E, device="cuda")
            o = torch.empty(s.attn.E, device="cuda")
            torch.cuda.synchronize()
            for i in range(n):
                s.attn.decode_dev(l, first + i, q.data_ptr(), k[i].data_ptr(), v[i].data_ptr(), o.data_ptr())
        else:
            torch.cuda.synchronize()
            s.attn.append_dev(l, 0, n, k.data_ptr(), v.data_ptr())
        s.attn.sync()


def _step_inputs(c, seed):
    g = _gen(seed)
    L, n = c.get("layers", 1), c.get("rows", 1)
    nh, nkv, hd = c["nh"], c["nkv"], c["hd"]
    return [(_acts(g, n, nh, hd), _acts(g, n, nkv, hd), _normal(g, n, nkv * hd)) for _ in range(L)]


SHAPES = [("wq", "E", "E"), ("wk", "KV", "E"), ("wv", "KV", "E"), ("wo", "E", "E"), ("w_gate", "FF", "E"),
          ("w_up", "FF", "E"), ("w_down", "E", "FF")]


def _layer_weights(g, width, l):
    """One layer's raw weights: Q4_K, with wv and w_down in Q6_K in every other layer (a Q4_K_M file's mix).  The two
    that write the residual stream are smaller, so that a layer adds a fraction of the stream, as in a trained model
    (were it all of it, one changed Q8_K rounding of a decode would be the whole difference after some layers)."""
    E, FF, nh, nkv = WIDTHS[width]
    dims = {"E": E, "FF": FF, "KV": E // nh * nkv}
    mats = []
    for name, r, k in SHAPES:
        t = Q6K if l % 2 == 0 and name in ("wv", "w_down") else Q4K
        mats.append((t, dims[r], dims[k], _blocks(g, t, dims[r], dims[k], 0.25 if name in ("wo", "w_down") else 1.0)))
    vecs = {"attn_norm": 1 + 0.1 * _normal(g, 1, E)[0], "ffn_norm": 1 + 0.1 * _normal(g, 1, E)[0],
            "bq": 0.5 * _normal(g, 1, E)[0], "bk": 0.5 * _normal(g, 1, dims["KV"])[0],
            "bv": 0.1 * _normal(g, 1, dims["KV"])[0]}
    return mats, vecs


def _write_gguf(path, c, seed):
    """A GGUF file of the engine case: written a tensor at a time."""
    E, FF, nh, nkv = WIDTHS[c["width"]]

    def text(v):
        return struct.pack("<Q", len(v)) + v.encode()

    meta = [text("general.architecture") + struct.pack("<I", 8) + text("qwen2")]
    for key, v in (("block_count", c["layers"]), ("context_length", 4096), ("embedding_length", E),
                   ("feed_forward_length", FF), ("attention.head_count", nh), ("attention.head_count_kv", nkv)):
        meta.append(text("qwen2." + key) + struct.pack("<II", 4, v))
    meta.append(text("qwen2.rope.freq_base") + struct.pack("<If", 6, ROPE_BASE))
    meta.append(text("qwen2.attention.layer_norm_rms_epsilon") + struct.pack("<If", 6, EPS))
    meta.append(text("tokenizer.ggml.tokens") + struct.pack("<IIQ", 9, 8, c["vocab"]) +
                (struct.pack("<Q", 1) + b"t") * c["vocab"])
    names, arrays = [], []
    for name, t, dims, a in _engine_tensors(c, seed):
        raw = a.contiguous().view(torch.uint8).reshape(-1).cpu().numpy()
        names.append((name, t, dims))
        arrays.append(raw)
    head, off = b"", 0
    for (name, t, dims), a in zip(names, arrays):
        head += text(name) + struct.pack("<I", len(dims)) + struct.pack("<%dQ" % len(dims), *dims) + struct.pack("<IQ", t, off)
        off += -(-a.size // 32) * 32
    head = b"GGUF" + struct.pack("<IQQ", 3, len(names), len(meta)) + b"".join(meta) + head
    with open(path, "wb") as f:
        f.write(head + bytes(-len(head) % 32))
        for a in arrays:
            a.tofile(f)
            f.write(bytes(-a.size % 32))


def _engine_tensors(c, seed):
    E, V = WIDTHS[c["width"]][0], c["vocab"]
    g = _gen(seed)
    yield "token_embd.weight", Q4K, (E, V), _blocks(g, Q4K, V, E, 25.0)
    yield "output.weight", Q6K, (E, V), _blocks(g, Q6K, V, E)
    yield "output_norm.weight", 0, (E,), 1 + 0.1 * _normal(g, 1, E)[0]
    file_names = dict(wq="attn_q", wk="attn_k", wv="attn_v", wo="attn_output", w_gate="ffn_gate", w_up="ffn_up",
                      w_down="ffn_down")
    for l in range(c["layers"]):
        mats, vecs = _layer_weights(g, c["width"], l)
        for (name, _, _), (t, r, k, a) in zip(SHAPES, mats):
            yield "blk.%d.%s.weight" % (l, file_names[name]), t, (k, r), a
        for name, v in vecs.items():
            fn = {"bq": "attn_q.bias", "bk": "attn_k.bias", "bv": "attn_v.bias"}.get(name, name + ".weight")
            yield "blk.%d.%s" % (l, fn), 0, (v.numel(),), v


def _tokens(c, seed):
    r = np.random.default_rng(seed)
    t = r.integers(0, c["vocab"], c["prompt"] + c["tokens"]).astype(np.int32)
    chunks = [(p, np.ascontiguousarray(t[p:min(p + 64, c["prompt"])])) for p in range(0, c["prompt"], 64)]
    return chunks, [int(x) for x in t[c["prompt"]:]]


def prepare(case, seed):
    c, s = case, _State()
    s.case, kind = c, c["kind"]
    s.stream = _stream()
    if kind in ("decode", "prefill", "host"):
        nh, nkv, hd = c["nh"], c["nkv"], c["hd"]
        L, n = c.get("layers", 1), c.get("rows", 1)
        ctx = c.get("window", 0) or (c["pos"] + 1 if kind == "decode" else c["pos0"] + n)
        _attn(s, c, L, ctx, nh, nkv, hd, c.get("window", 0))
        _fill(s, c, seed, L, nkv, hd)
        s.inputs = _step_inputs(c, seed)
        if kind == "host":
            s.inputs = [tuple(t.cpu().numpy() for t in x) for x in s.inputs]
        else:
            s.out = torch.empty(L, n, nh * hd, device="cuda")
    elif kind == "matmul":
        g = _gen(seed)
        w = _blocks(g, c["type"], c["rows"], c["cols"])
        s.x = _normal(g, c["nb"], c["cols"])
        s.out = torch.empty(c["nb"], c["rows"], device="cuda")
        torch.cuda.synchronize()
        s.w = _qmat(c["type"], w, c["rows"], c["cols"])
        s.closing.append(s.w)
        torch.cuda.synchronize()
    elif kind == "layers":
        E, FF, nh, nkv = WIDTHS[c["width"]]
        hd, n = E // nh, c["rows"]
        _attn(s, c, c["layers"], c["pos0"] + n, nh, nkv, hd)
        _fill(s, c, seed, c["layers"], nkv, hd)
        s.layer = layer.Layer(E, FF, nh, nkv, EPS)
        s.closing.append(s.layer)
        s.weights = []
        g = _gen(seed)
        for l in range(c["layers"]):
            mats, vecs = _layer_weights(g, c["width"], l)
            w = layer.LayerWeights()
            torch.cuda.synchronize()
            w.mats = [_qmat(t, a, r, k) for t, r, k, a in mats]
            w.bufs = {name: hip.DeviceBuffer.from_array(v.cpu().numpy()) for name, v in vecs.items()}
            torch.cuda.synchronize()
            s.weights.append(w)
            s.closing.append(w)
        s.x0 = _normal(_gen(seed + 1), n, E)
        s.x = torch.empty(n, E, device="cuda")
    else:
        fd, path = tempfile.mkstemp(suffix=".gguf", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
        os.close(fd)
        try:
            _write_gguf(path, c, seed)
            s.model = model.Model(path, c["prompt"] + c["tokens"], avx2=True)
        finally:
            os.unlink(path)
        s.closing.append(s.model)
        s.chunks, s.tokens = _tokens(c, seed)
        E, V = WIDTHS[c["width"]][0], c["vocab"]
        s.rows = torch.empty(c["prompt"], E, device="cuda")
        s.logits = torch.empty(1 + c["tokens"], V, device="cuda")
    torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------

def run(state):
    s, c = state, state.case
    kind, st = c["kind"], state.stream.cuda_stream
    if kind == "decode":
        for l, (q, k, v) in enumerate(s.inputs):
            s.attn.decode_dev(l, c["pos"], q.data_ptr(), k.data_ptr(), v.data_ptr(), s.out[l].data_ptr(), st)
        return s.out
    if kind == "prefill":
        q, k, v = s.inputs[0]
        s.attn.prefill_dev(0, c["pos0"], c["rows"], q.data_ptr(), k.data_ptr(), v.data_ptr(), s.out.data_ptr(), st)
        return s.out
    if kind == "host":
        if c["rows"] == 1:
            return [s.attn.decode(l, c["pos0"], q, k, v) for l, (q, k, v) in enumerate(s.inputs)]
        return [s.attn.prefill(l, c["pos0"], q, k, v) for l, (q, k, v) in enumerate(s.inputs)]
    if kind == "matmul":
        s.w.matmul_batch_dev(s.x.data_ptr(), c["nb"], s.out.data_ptr(), st)
        return s.out
    if kind == "layers":
        with torch.cuda.stream(s.stream):
            s.x.copy_(s.x0)
        for l, w in enumerate(s.weights):
            if c["rows"] == 1:
                s.layer.decode_dev(w, s.attn, l, c["pos0"], s.x.data_ptr(), True, st)
            else:
                s.layer.prefill_dev(w, s.attn, l, c["pos0"], c["rows"], s.x.data_ptr(), st)
        return s.x
    # the engine, through its C entry points: the results stay in device memory
    L, m = model.lib(), s.model
    E, V = WIDTHS[c["width"]][0], c["vocab"]

    def keep(dst, src, floats):
        hip.check(hip.lib().hipMemcpyAsync(dst.data_ptr(), src, 4 * floats, hip.D2D, st))

    for pos0, t in s.chunks:
        last = pos0 + t.size == c["prompt"]
        m._check(L.kore_model_prefill_dev(m._h, t.ctypes.data, t.size, pos0, int(last), st))
        keep(s.rows[pos0], L.kore_model_rows_dev(m._h), t.size * E)
    keep(s.logits[0], L.kore_model_logits_dev(m._h), V)
    for i, t in enumerate(s.tokens):
        m._check(L.kore_model_decode_dev(m._h, t, c["prompt"] + i, 1, st))
        keep(s.logits[i + 1], L.kore_model_logits_dev(m._h), V)
    return {"rows": s.rows, "logits": s.logits}


# ---- what a pass cannot do without -------------------------------------------

def _wbytes(t, rows, cols):
    return rows * (cols // 256) * (144 if t == Q4K else 210)


def _attn_work(n, pos0, nh, nkv, hd, rows_before):
    pairs = sum(min(pos0 + i, rows_before + i) + 1 for i in range(n))
    return (2 * (rows_before + n) * nkv * hd * 4 + 2 * n * nh * hd * 4 + 2 * n * nkv * hd * 4, 4 * nh * hd * pairs)


def _layer_work(width, l, n, pos0):
    E, FF, nh, nkv = WIDTHS[width]
    hd = E // nh
    dims = {"E": E, "FF": FF, "KV": hd * nkv}
    b, f = _attn_work(n, pos0, nh, nkv, hd, pos0)
    for name, r, k in SHAPES:
        t = Q6K if l % 2 == 0 and name in ("wv", "w_down") else Q4K
        b += _wbytes(t, dims[r], dims[k])
        f += 2 * n * dims[r] * dims[k]
    return b + 2 * n * E * 4, f


def work(case):
    c, kind = case, case["kind"]
    if kind in ("decode", "prefill", "host"):
        pos0 = c["pos"] if kind == "decode" else c["pos0"]
        b, f = _attn_work(c.get("rows", 1), pos0, c["nh"], c["nkv"], c["hd"], _cache_rows(c)[1])
        return {"bytes": b * c.get("layers", 1), "flops": f * c.get("layers", 1)}
    if kind == "matmul":
        return {"bytes": _wbytes(c["type"], c["rows"], c["cols"]) + 4 * c["nb"] * (c["rows"] + c["cols"]),
                "flops": 2 * c["nb"] * c["rows"] * c["cols"]}
    if kind == "layers":
        parts = [_layer_work(c["width"], l, c["rows"], c["pos0"]) for l in range(c["layers"])]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    E = WIDTHS[c["width"]][0]
    calls = [(p, min(64, c["prompt"] - p)) for p in range(0, c["prompt"], 64)]
    calls += [(c["prompt"] + i, 1) for i in range(c["tokens"])]
    parts = [_layer_work(c["width"], l, n, p) for p, n in calls for l in range(c["layers"])]
    heads = 1 + c["tokens"]
    return {"bytes": sum(p[0] for p in parts) + heads * (_wbytes(Q6K, c["vocab"], E) + 4 * c["vocab"]),
            "flops": sum(p[1] for p in parts) + heads * 2 * c["vocab"] * E}


def tolerance(case):
    """About four times what the path differs from `exact` by, at worst, over the listed and forty drawn cases.

    Decode attention sums its scores in 64 bits (rel 5e-7, max 1.2e-5 measured), prefill attention in 32 (2.2e-6,
    8e-5; a host call may be either).  A batched matmul measures 1.9e-7 and 1e-6, a layer of a chunk 6.5e-7 and 4e-6.
    A layer of a decode is 3e-7 off unless a Q8_K rounding of an activation falls the other way, which changes its
    result by some 1e-3; in an engine's decode one such rounding travels through every later layer (1.1e-2 and 7e-2
    over twelve of them, the same however the first one came about).
    """
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 2e-6, "max": 5e-5}
    if kind in ("prefill", "host"):
        return {"rel": 1e-5, "max": 3e-4}
    if kind == "matmul":
        return {"rel": 2e-6, "max": 1e-5}
    if kind == "layers":
        return {"rel": 1e-2, "max": 5e-2} if case["rows"] == 1 else {"rel": 3e-6, "max": 2e-5}
    return {"rel": 3e-2, "max": 0.3}


# ---- the same in 64 bits -----------------------------------------------------

def _deq(t, w):
    """GGUF blocks [rows][blocks][bytes] -> float64 [rows][cols]."""
    rows, nb = w.shape[:2]

    def f16(a):
        return a.contiguous().view(torch.float16)[..., 0].double()

    out = torch.empty(rows, nb, 256, dtype=torch.float64, device=w.device)
    if t == Q4K:
        d, dmin, s, q = f16(w[:, :, 0:2]), f16(w[:, :, 2:4]), w[:, :, 4:16].int(), w[:, :, 16:144]
        for j in range(8):
            if j < 4:
                sc, mn = s[..., j] & 63, s[..., j + 4] & 63
            else:
                sc = (s[..., j + 4] & 15) | ((s[..., j - 4] >> 6) << 4)
                mn = (s[..., j + 4] >> 4) | ((s[..., j] >> 6) << 4)
            n = q[:, :, 32 * (j // 2):32 * (j // 2) + 32]
            n = (n & 15) if j % 2 == 0 else (n >> 4)
            out[:, :, 32 * j:32 * j + 32] = (d * sc)[..., None] * n.double() - (dmin * mn)[..., None]
    else:
        d, sc = f16(w[:, :, 208:210]), w[:, :, 192:208].contiguous().view(torch.int8).double()
        for h in range(2):
            qh = w[:, :, 128 + 32 * h:160 + 32 * h].int()
            for k in range(4):
                ql = w[:, :, 64 * h + 32 * (k % 2):64 * h + 32 * (k % 2) + 32].int()
                q = ((ql & 15) if k < 2 else (ql >> 4)) | (((qh >> (2 * k)) & 3) << 4)
                scale = (d[..., None] * sc[:, :, 8 * h + 2 * k:8 * h + 2 * k + 2]).repeat_interleave(16, -1)
                out[:, :, 128 * h + 32 * k:128 * h + 32 * k + 32] = scale * (q - 32).double()
    return out.reshape(rows, nb * 256)


def _rope(x, pos, heads, hd):
    """x [n][heads * hd] in float64, positions [n]: pairs (i, i + hd / 2) turned by pos * inv_freq (a float, as kore has it)."""
    i = torch.arange(hd // 2, dtype=torch.float64, device=x.device)
    inv = torch.pow(torch.tensor(ROPE_BASE, dtype=torch.float64, device=x.device), -2.0 * i / hd).float().double()
    a = pos.double()[:, None, None] * inv
    x = x.reshape(x.shape[0], heads, 2, hd // 2)
    lo, hi = x[:, :, 0], x[:, :, 1]
    return torch.stack([lo * a.cos() - hi * a.sin(), lo * a.sin() + hi * a.cos()], 2).reshape(x.shape[0], heads, hd)


def _attend(q, k, v, nkv, first_own):
    """q [n][nh][hd], k/v [m][nkv][hd]: row i sees the first first_own + i + 1 rows."""
    n, nh, hd = q.shape
    m = k.shape[0]
    mask = torch.arange(m, device=q.device)[None, :] > first_own + torch.arange(n, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(nh):
        g = h // (nh // nkv)
        s = (q[:, h].contiguous() @ k[:, g].t().contiguous()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), 1) @ v[:, g].contiguous()
    return out.reshape(n, nh * hd)


def _exact_attn(q, k, v, old, pos0, first, nh, nkv, hd):
    """Attention of n new rows at pos0.. over the old (pre-RoPE) rows of positions first.. and themselves."""
    n = q.shape[0]
    at = torch.arange(n, device="cuda") + pos0
    q, k, v = _rope(q.double(), at, nh, hd), _rope(k.double(), at, nkv, hd), v.double().reshape(n, nkv, hd)
    m = 0
    if old is not None:
        ok, ov = old
        m = ok.shape[0]
        k = torch.cat([_rope(ok.double(), torch.arange(m, device="cuda") + first, nkv, hd), k])
        v = torch.cat([ov.double().reshape(m, nkv, hd), v])
    return _attend(q, k, v, nkv, m)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _q8(x):
    """kore's Q8_K rounding of activations, as values: -127 at the first value of the largest magnitude."""
    b = x.reshape(-1, 256)
    i = b.abs().argmax(1, keepdim=True)
    top = b.gather(1, i)
    inv = torch.where(top == 0, torch.zeros_like(top), -127.0 / top)
    q = torch.clamp(torch.round(inv * b), max=127)
    return torch.where(inv == 0, torch.zeros_like(b), q / inv).reshape(x.shape)


def _exact_layer(x, mats, vecs, width, attend, rounded):
    """One layer in float64; attend(q, k, v) -> rows; rounded: the decode's Q8_K activations."""
    r = _q8 if rounded else (lambda t: t)
    w = [_deq(t, a) for t, _, _, a in mats]

    def mul(i, t):
        return t @ w[i].t()

    h = r(_rms(x, vecs["attn_norm"]))
    q, k, v = (mul(i, h) + vecs[b].double() for i, b in enumerate(("bq", "bk", "bv")))
    x = x + mul(3, r(attend(q, k, v)))
    h = r(_rms(x, vecs["ffn_norm"]))
    g, u = mul(4, h), mul(5, h)
    return x + mul(6, r(g * torch.sigmoid(g) * u))


def exact(case, seed):
    c, kind = case, case["kind"]
    first, n_old = _cache_rows(c) if kind in ("decode", "prefill", "host", "layers") else (0, 0)
    if kind in ("decode", "prefill", "host"):
        nh, nkv, hd = c["nh"], c["nkv"], c["hd"]
        outs = []
        for l, (q, k, v) in enumerate(_step_inputs(c, seed)):
            old = _cache(c, seed, l, nkv, hd) if n_old else None
            if c.get("window", 0) and n_old == c["window"]:
                old, f = (old[0][1:], old[1][1:]), first + 1     # the new row takes the oldest one's slot
                old = old if old[0].shape[0] else None
            else:
                f = first
            outs.append(_exact_attn(q, k, v, old, c["pos"] if kind == "decode" else c["pos0"], f, nh, nkv, hd))
        if kind == "host":
            return [o[0] if c["rows"] == 1 else o for o in outs]
        return torch.stack(outs)
    if kind == "matmul":
        g = _gen(seed)
        w = _blocks(g, c["type"], c["rows"], c["cols"])
        return _normal(g, c["nb"], c["cols"]).double() @ _deq(c["type"], w).t()
    if kind == "layers":
        E, FF, nh, nkv = WIDTHS[c["width"]]
        x, g = _normal(_gen(seed + 1), c["rows"], E).double(), _gen(seed)
        for l in range(c["layers"]):
            mats, vecs = _layer_weights(g, c["width"], l)
            old = _cache(c, seed, l, nkv, E // nh) if n_old else None
            x = _exact_layer(x, mats, vecs, c["width"],
                             lambda q, k, v: _exact_attn(q, k, v, old, c["pos0"], 0, nh, nkv, E // nh), c["rows"] == 1)
        return x
    # the engine
    E, FF, nh, nkv = WIDTHS[c["width"]]
    hd, g = E // nh, _gen(seed)
    emb, head = _blocks(g, Q4K, c["vocab"], E, 25.0), _blocks(g, Q6K, c["vocab"], E)
    norm = 1 + 0.1 * _normal(g, 1, E)[0]
    layers = [_layer_weights(g, c["width"], l) for l in range(c["layers"])]
    caches = [None] * c["layers"]

    def step(tokens, pos0, rounded):
        x = _deq(Q4K, emb[torch.as_tensor(np.asarray(tokens, np.int64), device="cuda")])
        for l, (mats, vecs) in enumerate(layers):
            def attend(q, k, v):
                n = q.shape[0]
                at = torch.arange(n, device="cuda") + pos0
                q, k, v = _rope(q, at, nh, hd), _rope(k, at, nkv, hd), v.reshape(n, nkv, hd)
                if caches[l] is not None:
                    k, v = torch.cat([caches[l][0], k]), torch.cat([caches[l][1], v])
                caches[l] = (k, v)
                return _attend(q, k, v, nkv, pos0)
            x = _exact_layer(x, mats, vecs, c["width"], attend, rounded)
        return x

    def logits(x):
        h = _q8(_rms(x, norm))
        return torch.cat([h @ _deq(Q6K, head[i:i + 16384]).t() for i in range(0, c["vocab"], 16384)], 1)[0]

    chunks, tokens = _tokens(c, seed)
    rows = torch.cat([step(t, p, False) for p, t in chunks])
    out = [logits(rows[-1:])]
    for i, t in enumerate(tokens):
        out.append(logits(step([t], c["prompt"] + i, True)))
    return {"rows": rows, "logits": torch.stack(out)}
