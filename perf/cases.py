"""The work this library is timed on: quantized projections from one decode row to a
long prompt, in the four weight formats, and the decoder model's two calls.

A "linear" case is one pass of m rows through `weights` projections of one shape
(the same projection of as many layers: their weights are read from memory, as in a
model, and not from a cache that the previous call filled).  With `graph` the pass
is recorded once into a HIP graph and replayed, as a serving loop does with steps of
a few rows, whose launches would cost more host time than the kernels take.

A "model" case is one call of the decoder model on a cache that holds `pos`
positions: `rows` > 1 a prompt (forward_cached, the logits of every row), `rows` = 1
a decode step (forward_decode).

Weights are normal and quantized to their format, activations normal with a gain per
channel, as the rows of a transformer's residual stream have.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mini-rust-inference_amd"))
import mri_llama as L  # noqa: E402
import mri_qmatmul as M  # noqa: E402

WEIGHT_BYTES = {"int8": 1.0, "q8_0": 34 / 32, "q4_0": 18 / 32, "w4a8": 18 / 32}


def linear(fmt, m, k, n, weights, graph, name=None):
    c = {"kind": "linear", "fmt": fmt, "m": m, "k": k, "n": n, "weights": weights, "graph": graph}
    return dict(c, name=name) if name else c


def model(fmt, dim, heads, kv_heads, ffn, vocab, layers, pos, rows, name=None):
    c = {"kind": "model", "fmt": fmt, "dim": dim, "heads": heads, "kv_heads": kv_heads,
         "ffn": ffn, "vocab": vocab, "layers": layers, "pos": pos, "rows": rows}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: three rows of odd length through one small projection,
        # launched by itself; what it costs is launches and latency
        linear("int8", 3, 1000, 777, 1, False, "few_rows_int8_odd"),
        # single-token decode: the up projection of a 4096-wide model in each of the
        # two GGUF formats, as the file holds them (Q4_0 with f32 activations)
        linear("q8_0", 1, 4096, 11008, 6, True, "decode_q8_0"),
        linear("q4_0", 1, 4096, 11008, 8, True, "decode_q4_0"),
        # a step of several sequences at once
        linear("int8", 24, 4096, 4096, 12, True, "batch24_int8"),
        linear("q8_0", 16, 4096, 11008, 6, True, "batch16_q8_0"),
        # a short prompt, or a chunk of one: an odd number of rows
        linear("q8_0", 100, 4096, 4096, 6, False, "chunk100_q8_0"),
        # prompts: fused q/k/v, down (K = 11008), up, and the longest prompt
        linear("q8_0", 512, 4096, 12288, 2, False, "prompt512_q8_0"),
        linear("w4a8", 333, 11008, 4096, 3, False, "prompt333_w4a8"),
        linear("q4_0", 256, 4096, 11008, 1, False, "prompt256_q4_0"),
        linear("int8", 2048, 4096, 11008, 2, False, "prompt2048_int8"),
        # the decoder layer: a 512-token prompt with the reference model's own
        # INT8 weights, and one decode step at 600 positions with Q8_0 weights
        model("int8", 4096, 32, 32, 11008, 32000, 1, 0, 512, "layer_prompt512_int8"),
        model("q8_0", 4096, 32, 32, 11008, 32000, 1, 600, 1, "layer_decode_q8_0"),
    ]


MOST_FLOPS = 2 * 2.0 * 2048 * 4096 * 11008     # of the largest listed case
MOST_FLOPS_Q4_0 = 2.0 * 256 * 4096 * 11008     # of the largest listed Q4_0 case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Projections of 1 to 2048 rows, K and N of 256 to 12288 (K in whole blocks of
    32 for the block formats, whole KiB half of the time, as models have it), and
    small to full-width decoder layers with and without grouped heads (up to three
    of them where the activations stay f32; see tolerance() for the others)."""
    while True:
        if rng.random() < 0.15:
            hd = rng.choice((64, 128))
            kv = rng.choice((1, 2, 4, 8))
            heads = kv * rng.choice((1, 2, 4))
            dim = heads * hd
            rows = 1 if rng.random() < 0.5 else _log(rng, 2, 512)
            fmt = rng.choice(("int8", "q8_0", "w4a8", "q4_0"))
            c = model(fmt, dim, heads, kv, 32 * rng.randint(2 * dim // 32, 3 * dim // 32),
                      16 * _log(rng, 64, 2000), rng.randint(1, 3) if fmt == "q4_0" else 1,
                      _log(rng, 1, 600), rows)
            if c["fmt"] == "q4_0" and work(c)["flops"] > MOST_FLOPS_Q4_0:
                continue
            return c
        fmt = rng.choice(("int8", "q8_0", "w4a8", "q4_0"))
        m = _log(rng, 1, 2048)
        k = _log(rng, 256, 12288)
        if rng.random() < 0.5:
            k = max(1, round(k / 1024)) * 1024
        elif fmt != "int8":
            k = max(8, round(k / 32)) * 32
        n = _log(rng, 256, 12288)
        if rng.random() < 0.5:
            n = max(1, round(n / 256)) * 256
        c = linear(fmt, m, k, n, rng.randint(1, 4), m <= 32)
        most = MOST_FLOPS_Q4_0 if fmt == "q4_0" else MOST_FLOPS
        if work(c)["flops"] <= most:
            return c


# ---------------------------------------------------------------- inputs
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + salt) % (1 << 62))
    return g


def _half_away(y):
    """Round half away from zero, of f32 values, exactly."""
    y = y.double()
    return torch.sign(y) * torch.floor(y.abs() + 0.5)


def _scale127(mx):
    """max|x| / 127 and its reciprocal, each rounded once to f32 (1 for zeros)."""
    s = torch.where(mx == 0, torch.ones_like(mx), (mx.double() / 127.0).float())
    return s, (1.0 / s.double()).float()


def _weight(fmt, n, k, seed, salt):
    """A projection's quantized weights as a program holds them: (int8 rows, scales)
    or raw GGUF blocks, on the GPU."""
    w = torch.randn(n, k, device="cuda", generator=_gen(seed, salt)) * 0.02
    if fmt == "int8":
        s, inv = _scale127(w.abs().amax(dim=1))
        return torch.clamp(_half_away(w * inv[:, None]), -127, 127).to(torch.int8), s
    b = w.view(n, k // 32, 32)
    d = (b.abs().amax(dim=2) / (127.0 if fmt == "q8_0" else 7.0)).half()
    q = torch.round(b / d.float()[:, :, None])
    if fmt == "q8_0":
        raw = torch.empty(n, k // 32, 34, dtype=torch.uint8, device="cuda")
        raw[:, :, 2:] = torch.clamp(q, -127, 127).to(torch.int8).view(torch.uint8)
    else:
        raw = torch.empty(n, k // 32, 18, dtype=torch.uint8, device="cuda")
        nib = (torch.clamp(q, -8, 7) + 8).to(torch.uint8)
        raw[:, :, 2:] = nib[:, :, 0::2] | (nib[:, :, 1::2] << 4)
    raw[:, :, :2] = d.view(torch.uint8).view(n, k // 32, 2)
    return raw.view(-1), None


def _handle(fmt, n, k, seed, salt):
    q, s = _weight(fmt, n, k, seed, salt)
    if fmt == "int8":
        h = M.QMatrix.from_device(q, s)
    elif fmt == "q8_0":
        h = M.Q8Matrix.from_raw_device(q, n, k)
    elif fmt == "w4a8":
        h = M.Q4Matrix.from_raw_device(q, n, k)
    else:
        return q, n, k
    torch.cuda.synchronize()  # the upload has read q
    return h


def _rows(m, k, seed, salt):
    g = _gen(seed, salt)
    x = torch.randn(m, k, device="cuda", generator=g)
    return x * torch.exp(0.5 * torch.randn(k, device="cuda", generator=g))


def _project(fmt, x, w, out):
    if fmt == "int8":
        M.matmul_int8_from_f32(x, w, out)
    elif fmt == "q8_0":
        M.matmul_q8_0_direct(x, w, out)
    elif fmt == "w4a8":
        M.matmul_q4_0_w4a8(x, w, out)
    else:
        M.matmul_q4_0_dequant(x, w[0], w[1], w[2], out)


_NAMES = ("wq", "wk", "wv", "wo", "wgate", "wup", "wdown")


def _shapes(c):
    hd = c["dim"] // c["heads"]
    kvd, d, f = c["kv_heads"] * hd, c["dim"], c["ffn"]
    return ((d, d), (kvd, d), (kvd, d), (d, d), (f, d), (f, d), (d, f))


def _model_host(c, seed):
    """Embedding table, norms and token ids of a model case."""
    g = _gen(seed, 7)
    emb = torch.randn(c["vocab"], c["dim"], device="cuda", generator=g)
    norms = 1.0 + 0.1 * torch.randn(2 * c["layers"] + 1, c["dim"], device="cuda", generator=g)
    toks = torch.randint(0, c["vocab"], (c["pos"] + c["rows"],), device="cuda", generator=g)
    return emb, norms, toks.cpu().numpy().astype(np.uint32)


_EPS, _BASE = 1e-5, 10000.0
_stream = None


def prepare(case, seed):
    global _stream
    c = case
    if c["kind"] == "linear":
        ws = [_handle(c["fmt"], c["n"], c["k"], seed, 100 + i) for i in range(c["weights"])]
        xs = [_rows(c["m"], c["k"], seed, 500 + i) for i in range(c["weights"])]
        outs = [torch.empty(c["m"], c["n"], device="cuda") for _ in ws]
        st = {"fmt": c["fmt"], "ws": ws, "xs": xs, "outs": outs, "graph": None}
        if c["graph"]:
            if _stream is None:
                _stream = torch.cuda.Stream()
            torch.cuda.synchronize()
            with torch.cuda.stream(_stream):  # the stream's staging exists before the recording
                for x, w, o in zip(xs, ws, outs):
                    _project(c["fmt"], x, w, o)
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=_stream):
                for x, w, o in zip(xs, ws, outs):
                    _project(c["fmt"], x, w, o)
            st["graph"] = g
        return st
    emb, norms, toks = _model_host(c, seed)
    layers = []
    for i in range(c["layers"]):
        lay = {nm: _handle(c["fmt"], n, k, seed, 1000 + 10 * i + j)
               for j, (nm, (n, k)) in enumerate(zip(_NAMES, _shapes(c)))}
        lay["attn_norm"], lay["ffn_norm"] = norms[2 * i].cpu().numpy(), norms[2 * i + 1].cpu().numpy()
        layers.append(lay)
    out = _handle(c["fmt"], c["vocab"], c["dim"], seed, 990)
    cfg = {"dim": c["dim"], "n_heads": c["heads"], "n_kv_heads": c["kv_heads"], "ffn": c["ffn"],
           "vocab": c["vocab"], "max_seq": c["pos"] + c["rows"] + 8, "eps": _EPS, "rope_base": _BASE}
    mod = L.Llama(cfg, emb.cpu().numpy(), norms[-1].cpu().numpy(), out, layers)
    cache = mod.kv_cache()
    if c["pos"]:
        mod.forward_cached(toks[:c["pos"]], 0, cache,
                           torch.empty(c["pos"], c["vocab"], device="cuda"))
        torch.cuda.synchronize()
    return {"model": mod, "cache": cache, "toks": toks[c["pos"]:], "pos": c["pos"],
            "logits": torch.empty(c["rows"], c["vocab"], device="cuda")}


def run(state):
    if "model" in state:
        if len(state["toks"]) == 1:
            state["model"].forward_decode(state["toks"][0], state["pos"], state["cache"],
                                          state["logits"])
        else:
            state["model"].forward_cached(state["toks"], state["pos"], state["cache"],
                                          state["logits"])
        return state["logits"]
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        for x, w, o in zip(state["xs"], state["ws"], state["outs"]):
            _project(state["fmt"], x, w, o)
    return state["outs"]


def work(case):
    c = case
    wb = WEIGHT_BYTES[c["fmt"]]
    if c["kind"] == "linear":
        m, k, n = c["m"], c["k"], c["n"]
        scales = 4 * n if c["fmt"] == "int8" else 0
        return {"bytes": c["weights"] * (wb * n * k + scales + 4.0 * m * (k + n)),
                "flops": c["weights"] * 2.0 * m * k * n}
    r, d, hd = c["rows"], c["dim"], c["dim"] // c["heads"]
    elems = c["layers"] * sum(n * k for n, k in _shapes(c)) + c["vocab"] * d
    keys = sum(c["pos"] + i + 1 for i in range(r))  # visible keys of all rows
    kvd = c["kv_heads"] * hd
    return {"bytes": wb * elems + 4.0 * (r * d + r * c["vocab"])
            + c["layers"] * 2 * 4.0 * kvd * (c["pos"] + 2 * r),
            "flops": 2.0 * r * elems + c["layers"] * 4.0 * keys * c["heads"] * hd}


def tolerance(case):
    """Projections: int8 products and their int32 sums are exact, and the f32 terms
    are added in 32 bits (up to 384 block terms, or 12288 products for Q4_0);
    measured against 64 bits 4e-8 to 4e-7.  A decoder layer with int8 activations
    quantizes them five times in turn: one last-bit difference moves a value by one
    of 127 steps, the next quantization sees that in many values, and from there on
    two correct evaluations differ by the quantization's own noise, 1e-2 of a layer's
    logits (measured against 64 bits 1.1e-2, 2.1e-2 after two layers)."""
    c = case
    if c["kind"] == "model":
        return {"rel": 1e-4 if c["fmt"] == "q4_0" else 3e-2}
    return {"rel": 2e-6, "max": 2e-5}


# ---------------------------------------------------------------- in 64 bits
def _dense(fmt, n, k, seed, salt):
    q, s = _weight(fmt, n, k, seed, salt)
    if fmt == "int8":
        return q.double() * s.double()[:, None]
    width = 34 if fmt == "q8_0" else 18
    raw = q.view(n, k // 32, width)
    d = raw[:, :, :2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        v = raw[:, :, 2:].contiguous().view(torch.int8).double()
    else:
        v = torch.stack((raw[:, :, 2:] & 15, raw[:, :, 2:] >> 4), dim=3).view(n, k // 32, 32)
        v = v.double() - 8.0
    return (v * d).view(n, k)


def _exact_project(fmt, x, w):
    """x [m, k] (f32 values) times w^T in f64, with the format's own quantization of
    the activations: none for Q4_0, one scale for all rows for INT8, else one a row."""
    if fmt != "q4_0":
        x = x.float()
        mx = x.abs().amax().expand(x.shape[0]) if fmt == "int8" else x.abs().amax(dim=1)
        s, inv = _scale127(mx)
        x = torch.clamp(_half_away(x * inv[:, None]), -127, 127) * s.double()[:, None]
    return x.double() @ w.t()


def _exact_model(c, seed):
    emb, norms, toks = _model_host(c, seed)
    fmt, hd, heads, kvh = c["fmt"], c["dim"] // c["heads"], c["heads"], c["kv_heads"]
    total = c["pos"] + c["rows"]
    e = (2 * np.arange(hd // 2, dtype=np.float32)) / np.float32(hd)
    theta = np.float32(1.0) / np.power(np.float32(_BASE), e)
    ang = torch.from_numpy(np.arange(total, dtype=np.float32)[:, None] * theta).cuda().double()
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]

    def norm(x, w):
        return w.double() * (x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + _EPS))

    def rope(t, p0):
        a, b = t[:, :, 0::2], t[:, :, 1::2]
        cc, ss = cos[p0:p0 + t.shape[0]], sin[p0:p0 + t.shape[0]]
        return torch.stack((a * cc - b * ss, b * cc + a * ss), dim=3).flatten(2)

    # the calls of the program: the prefix, then the timed rows (INT8 activations
    # take one scale a call)
    calls = [(0, c["pos"])] if c["pos"] else []
    calls.append((c["pos"], total))
    xs = [emb[torch.from_numpy(toks[a:b].astype(np.int64)).cuda()].double() for a, b in calls]
    for i in range(c["layers"]):
        w = {nm: _dense(fmt, n, k, seed, 1000 + 10 * i + j)
             for j, (nm, (n, k)) in enumerate(zip(_NAMES, _shapes(c)))}
        ks, vs = [], []
        for j, (a, b) in enumerate(calls):
            x, r = xs[j], b - a
            h = norm(x, norms[2 * i])
            q = rope(_exact_project(fmt, h, w["wq"]).view(r, heads, hd), a)
            ks.append(rope(_exact_project(fmt, h, w["wk"]).view(r, kvh, hd), a))
            vs.append(_exact_project(fmt, h, w["wv"]).view(r, kvh, hd))
            kk = torch.cat(ks).repeat_interleave(heads // kvh, dim=1)
            vv = torch.cat(vs).repeat_interleave(heads // kvh, dim=1)
            hidden = torch.arange(b, device="cuda")[None, :] > torch.arange(a, b, device="cuda")[:, None]
            att = torch.empty(r, heads, hd, dtype=torch.float64, device="cuda")
            for hh in range(heads):
                sc = (q[:, hh] @ kk[:, hh].t()) / math.sqrt(hd)
                att[:, hh] = torch.softmax(sc.masked_fill(hidden, -math.inf), dim=1) @ vv[:, hh]
            x = x + _exact_project(fmt, att.view(r, -1), w["wo"])
            h = norm(x, norms[2 * i + 1])
            gate = _exact_project(fmt, h, w["wgate"])
            up = _exact_project(fmt, h, w["wup"])
            xs[j] = x + _exact_project(fmt, gate / (1 + torch.exp(-gate)) * up, w["wdown"])
    return _exact_project(fmt, norm(xs[-1], norms[-1]), _dense(fmt, c["vocab"], c["dim"], seed, 990))


def exact(case, seed):
    c = case
    if c["kind"] == "model":
        return _exact_model(c, seed)
    return [_exact_project(c["fmt"], _rows(c["m"], c["k"], seed, 500 + i),
                           _dense(c["fmt"], c["n"], c["k"], seed, 100 + i))
            for i in range(c["weights"])]
