"""The work that a program using this library has it do, as cases that can be timed and checked:
the C ABI's two serving calls (julia_cuda_run, julia_hip_run_batched), an encoder layer and the
head as such a program chains the per-op calls on its own device memory and stream, and the fused
GEMMs and attention by themselves. Widths are the ModernBERT-base shapes (d = 768, 12 heads of 64,
GeGLU 1152, head feed-forward 1536, vocabulary 50368) and the narrower model of the tests (d = 384).
Lengths go from a request's few marker rows to 64 concatenated requests (about 18.7k rows), request
lengths are the benchmark's (72 to 1024 tokens, log-normal with a mean near 293).
"""

import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "julia-cuda_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import julia_hip as jh  # noqa: E402

EPS = 1e-5
VOCAB, INTER, LAYERS, QTYPES = 50368, 1152, 22, 3
MAX_LENGTH, BATCH_ROWS, MAX_POSITIONS = 1024, 20480, 8192
THETA_GLOBAL, THETA_LOCAL, WINDOW = 160000.0, 10000.0, 64
MODEL_SEED = 42
MARKERS = 6  # options a request scores
MOST_ROWS = 18752


def head_ff(d):
    return 2 * d


def lengths(case):
    """The request lengths of a case with `requests`: drawn from its `lens` number, so that every
    pass of the case has the same ones."""
    r = random.Random(case["lens"])
    out = []
    for _ in range(case["requests"]):
        n = math.exp(r.gauss(math.log(260.0 * case["mean"] / 293.0), 0.5))
        out.append(int(min(1024, max(72, round(n)))))
    return out


# ------------------------------------------------------------------------------ the cases
GEMMS = ("lnrope", "lngeglu", "lnbias", "lnbiasrelu", "lnbiasgelu")


def gemm_shape(epi, d):
    """(n, k) of the projection that has this epilogue in a model of width d."""
    return {"lnrope": (3 * d, d), "lngeglu": (2 * INTER, d), "lnbias": (3 * d, d),
            "lnbiasrelu": (head_ff(d), d), "lnbiasgelu": (d, d)}[epi]


def listed():
    return [
        # A full serving queue: 16 requests of ordinary lengths, one forward pass each.
        {"name": "run_16_requests", "kind": "run", "requests": 16, "mean": 293, "lens": 4},
        # Throughput serving: 64 requests packed into one forward pass over their rows.
        {"name": "run_batched_64", "kind": "batched", "requests": 64, "mean": 293, "lens": 44},
        # The smallest call of the head: the scorer's first linear on one request's markers.
        {"name": "lin1_6", "kind": "gemm", "epi": "lnbiasgelu", "d": 768, "m": 6},
        # The attention input projection of one request of mean length.
        {"name": "qkv_293", "kind": "gemm", "epi": "lnrope", "d": 768, "m": 293},
        # The MLP's first projection on a longer request.
        {"name": "wi_512", "kind": "gemm", "epi": "lngeglu", "d": 768, "m": 512},
        # The same projections on concatenated requests: a small batch and a full one.
        {"name": "qkv_4096", "kind": "gemm", "epi": "lnrope", "d": 768, "m": 4096},
        {"name": "wi_18752", "kind": "gemm", "epi": "lngeglu", "d": 768, "m": 18752},
        # Embedding and a global layer on one long request, through the per-op calls.
        {"name": "layer_1024", "kind": "layer", "d": 768, "window": 0, "rows": 1024},
        # Embedding and a windowed layer on 64 concatenated requests.
        {"name": "layer_batch_64", "kind": "layer", "d": 768, "window": WINDOW, "requests": 64, "mean": 293,
         "lens": 45},
        # Final norm, a head layer and the scorer at the narrow width, on a few requests' rows.
        {"name": "head_batch_10", "kind": "head", "d": 384, "requests": 10, "mean": 293, "lens": 46},
        # Attention alone: one document of an odd length, and a full batch of requests.
        {"name": "attention_2029", "kind": "attention", "d": 768, "window": 0, "rows": 2029},
        {"name": "attention_batch_64", "kind": "attention", "d": 768, "window": 0, "requests": 64, "mean": 293,
         "lens": 47},
    ]


def log_int(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    lens = rng.randrange(1 << 20)
    some = {"requests": log_int(rng, 2, 60), "mean": rng.randint(200, 293), "lens": lens}
    kind = rng.choice(("run", "batched", "gemm", "gemm", "gemm", "layer", "layer", "head", "attention", "attention"))
    if kind == "run":
        return {"kind": kind, "requests": rng.randint(10, 16), "mean": rng.randint(150, 293), "lens": lens}
    if kind == "batched":
        return {"kind": kind, **some, "requests": log_int(rng, 10, 60)}
    d = rng.choice((768, 768, 384))
    if kind == "gemm":
        return {"kind": kind, "epi": rng.choice(GEMMS), "d": d, "m": log_int(rng, 3, MOST_ROWS)}
    window = rng.choice((0, WINDOW))
    if rng.random() < 0.5:
        case = {"kind": kind, "d": d, **some}
    else:
        case = {"kind": kind, "d": d, "rows": log_int(rng, 24, 4096)}
    if kind != "head":
        case["window"] = window
    return case


# ------------------------------------------------------------------------------ inputs
def generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + stream) % (1 << 62))
    return g


def normal16(seed, stream, shape, std=1.0, mean=0.0):
    x = torch.randn(shape, generator=generator(seed, stream), device="cuda", dtype=torch.float32)
    return (x * std + mean).half()


def normal32(seed, stream, shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=generator(seed, stream), device="cuda", dtype=torch.float32) * std + mean


def bits(a):
    """numpy f16 bit patterns -> a device tensor."""
    return torch.from_numpy(a.view(np.float16)).cuda()


class Linear:
    """A projection's weights laid out for the GEMMs: W (f16, fragment order) and, where it has a
    LayerNorm folded in, its column sums; a bias where it has one. `plain` is W as [n][k]."""

    def __init__(self, seed, stream, n, k, ln, bias=False, geglu=False):
        w = normal32(seed, stream, (n, k), 0.02).cpu().numpy()
        if geglu:
            w = w[jh.geglu_rows(n // 2)]
        self.colsum = None
        if ln:
            gamma = normal32(seed, stream + 1, (k,), 0.1, 1.0).cpu().numpy()
            w16, cs = jh.fold_layernorm(w, gamma)
            self.colsum = torch.from_numpy(cs).cuda()
        else:
            w16 = jh.round_f16(w)
        self.n, self.k = n, k
        self.plain = bits(w16)
        self.w = bits(jh.pack_frag(w16))
        self.bias = normal32(seed, stream + 2, (n,), 0.02) if bias else None


def row_stats(x):
    """(sum, sum of squares) of each row's 64-column groups."""
    g = x.float().reshape(x.shape[0], -1, 64)
    return torch.stack((g.sum(2), (g * g).sum(2)), 2).contiguous()


def rows_of(case):
    return case["rows"] if "rows" in case else sum(lengths(case))


def sequences(case):
    """(per-row positions, per-row sequence bounds) of concatenated requests, or (None, None)."""
    if "requests" not in case:
        return None, None
    pos, seg, at = [], [], 0
    for n in lengths(case):
        pos.append(np.arange(n, dtype=np.int32))
        seg.append(np.tile(np.array([at, at + n], np.int32), (n, 1)))
        at += n
    return torch.from_numpy(np.concatenate(pos)).cuda(), torch.from_numpy(np.concatenate(seg)).cuda()


def gemm_positions(m):
    """Rows past the RoPE table are concatenated requests: positions that start over."""
    return None if m <= MAX_POSITIONS else (torch.arange(m, dtype=torch.int32) % 293).cuda()


_ENGINE = None


def engine():
    """The loaded model: one for the life of the program."""
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = jh.Engine(f"synthetic:seed={MODEL_SEED}", max_length=MAX_LENGTH, batch_rows=BATCH_ROWS)
    return _ENGINE


def requests(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n in lengths(case):
        ids = rng.integers(0, VOCAB, n).astype(np.uint32)
        markers = np.sort(rng.choice(n, MARKERS, replace=False)).astype(np.uint32)
        out.append((ids, markers, int(rng.integers(0, QTYPES))))
    return out


def rope(theta):
    return torch.from_numpy(jh.rope_table(theta, MAX_POSITIONS)).cuda()


def ptr(t):
    return t.data_ptr() if t is not None else 0


def gemm_inputs(case, seed):
    m, d, epi = case["m"], case["d"], case["epi"]
    n, k = gemm_shape(epi, d)
    a = normal16(seed, 1, (m, k), 1.0, 0.1)
    return a, Linear(seed, 10, n, k, True, "bias" in epi, "geglu" in epi), gemm_positions(m)


def layer_inputs(case, seed):
    d = case["d"]
    g = generator(seed, 1)
    return {
        "ids": torch.randint(0, VOCAB, (rows_of(case),), generator=g, device="cuda", dtype=torch.int32),
        "table": normal16(seed, 2, (VOCAB, d), 0.02),
        "gamma": normal32(seed, 3, (d,), 0.1, 1.0),
        "qkv": Linear(seed, 10, 3 * d, d, False),
        "wo": Linear(seed, 20, d, d, False),
        "wi": Linear(seed, 30, 2 * INTER, d, True, geglu=True),
        "wo_mlp": Linear(seed, 40, d, INTER, False),
    }


def head_inputs(case, seed):
    d, rows = case["d"], rows_of(case)
    r = np.random.default_rng(seed)
    at, marks = 0, []
    for n in lengths(case) if "requests" in case else [rows]:
        marks.append(at + np.sort(r.choice(n, min(MARKERS, n), replace=False)))
        at += n
    return {
        "x": normal16(seed, 1, (rows, d), 1.0, 0.1),
        "gamma": normal32(seed, 2, (d,), 0.1, 1.0),
        "type": normal32(seed, 3, (d,), 0.02),
        "markers": torch.from_numpy(np.concatenate(marks).astype(np.int32)).cuda(),
        "in_proj": Linear(seed, 10, 3 * d, d, True, True),
        "out_proj": Linear(seed, 20, d, d, False, True),
        "linear1": Linear(seed, 30, head_ff(d), d, True, True),
        "linear2": Linear(seed, 40, d, head_ff(d), False, True),
        "lin1": Linear(seed, 50, d, d, True, True),
        "lin2": normal16(seed, 60, (d,), 0.02),
        "lin2_b": 0.01,
    }


def half_buffer(*shape):
    return torch.zeros(shape, dtype=torch.float16, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("run", "batched"):
        return {"kind": kind, "engine": engine(), "requests": requests(case, seed)}
    # The caller's own stream, device buffers and the arguments of its calls, set up once.
    s = {"kind": kind, "stream": torch.cuda.current_stream().cuda_stream, "scratch": jh.Scratch()}
    if kind == "gemm":
        a, lin, pos = gemm_inputs(case, seed)
        m, n, k = case["m"], lin.n, lin.k
        stats = row_stats(a)
        c = half_buffer(m, n // 2 if "geglu" in case["epi"] else n)
        table = rope(THETA_GLOBAL) if "rope" in case["epi"] else None
        s["keep"] = (a, lin, pos, stats, table)
        s["out"] = c
        s["args"] = jh.gemm_args(case["epi"], ptr(a), ptr(lin.w), ptr(c), m, n, k, stats_in=ptr(stats),
                                 colsum=ptr(lin.colsum), eps=EPS, bias=ptr(lin.bias), rope=ptr(table),
                                 positions=ptr(pos), rope_rows=MAX_POSITIONS if table is not None else 0)
        return s
    pos, seg = sequences(case)
    rows, d = rows_of(case), case["d"]
    s["seg"], s["rows"], s["d"], s["window"] = seg, rows, d, case.get("window", 0)
    qkv, o = half_buffer(rows, 3 * d), half_buffer(rows, d)
    if kind == "attention":
        qkv = normal16(seed, 1, (rows, 3 * d))
        s.update(qkv=qkv, out=o)
        return s
    stats_a, stats_b = (torch.zeros((rows, d // 64, 2), device="cuda") for _ in range(2))
    x = half_buffer(rows, d)

    def call(epi, a, lin, c, stats_in=None, stats_out=None, **more):
        return jh.gemm_args(epi, ptr(a), ptr(lin.w), ptr(c), rows, lin.n, lin.k, stats_in=ptr(stats_in),
                            colsum=ptr(lin.colsum), eps=EPS, bias=ptr(lin.bias), stats_out=ptr(stats_out), **more)

    if kind == "layer":
        w = layer_inputs(case, seed)
        mid = half_buffer(rows, INTER)
        table = rope(THETA_LOCAL if case["window"] else THETA_GLOBAL)
        s.update(w=w, keep=(table, pos, stats_a), qkv=qkv, o=o)
        s["calls"] = [
            call("rope", x, w["qkv"], qkv, rope=ptr(table), positions=ptr(pos), rope_rows=MAX_POSITIONS),
            call("resstats", o, w["wo"], x, stats_out=stats_a),
            call("lngeglu", x, w["wi"], mid, stats_in=stats_a),
            call("resstats", mid, w["wo_mlp"], x, stats_out=stats_b)]
        s["x"] = x
        s["out"] = {"x": x, "stats": stats_b, "qkv": qkv, "o": o, "mid": mid}
        return s
    w = head_inputs(case, seed)
    mid, y = half_buffer(rows, head_ff(d)), half_buffer(rows, d)
    logits = torch.zeros(len(w["markers"]), device="cuda")
    s.update(w=w, keep=(stats_a, stats_b), qkv=qkv, o=o, x=x, stats=stats_a, y=y, logits=logits)
    s["calls"] = [
        call("lnbias", x, w["in_proj"], qkv, stats_in=stats_a),
        call("biasresstats", o, w["out_proj"], x, stats_out=stats_b),
        call("lnbiasrelu", x, w["linear1"], mid, stats_in=stats_b),
        call("biasresstats", mid, w["linear2"], x, stats_out=stats_a),
        call("lnbiasgelu", x, w["lin1"], y, stats_in=stats_a)]
    s["out"] = {"x": x, "stats": stats_a, "qkv": qkv, "o": o, "mid": mid, "y": y, "logits": logits}
    return s


def attend(s, qkv, o):
    if s["seg"] is None:
        jh.attention(qkv.data_ptr(), o.data_ptr(), s["rows"], s["d"], s["window"], 1, s["scratch"], s["stream"])
    else:
        jh.attention_seg(qkv.data_ptr(), o.data_ptr(), s["rows"], s["d"], s["window"], s["seg"].data_ptr(),
                         s["scratch"], s["stream"])


def run(s):
    kind, st = s["kind"], s["stream"] if "stream" in s else 0
    if kind in ("run", "batched"):
        return np.concatenate(s["engine"].run(s["requests"], batched=kind == "batched")[0])
    scratch = s["scratch"]
    if kind == "gemm":
        jh.gemm(s["args"], scratch=scratch, stream=st)
        return s["out"]
    if kind == "attention":
        attend(s, s["qkv"], s["out"])
        return s["out"]
    w, rows, d, x = s["w"], s["rows"], s["d"], s["x"]
    if kind == "layer":
        qkv, wo, wi, wo_mlp = s["calls"]
        jh.embed(w["ids"].data_ptr(), rows, w["table"].data_ptr(), VOCAB, d, w["gamma"].data_ptr(), EPS,
                 x.data_ptr(), st)
        jh.gemm(qkv, scratch=scratch, stream=st)
        attend(s, s["qkv"], s["o"])
        jh.gemm(wo, scratch=scratch, stream=st)
        jh.gemm(wi, scratch=scratch, stream=st)
        jh.gemm(wo_mlp, scratch=scratch, stream=st)
        return s["out"]
    in_proj, out_proj, linear1, linear2, lin1 = s["calls"]
    jh.norm_add(w["x"].data_ptr(), rows, d, w["gamma"].data_ptr(), w["type"].data_ptr(), EPS, x.data_ptr(),
                s["stats"].data_ptr(), st)
    jh.gemm(in_proj, scratch=scratch, stream=st)
    attend(s, s["qkv"], s["o"])
    jh.gemm(out_proj, scratch=scratch, stream=st)
    jh.gemm(linear1, scratch=scratch, stream=st)
    jh.gemm(linear2, scratch=scratch, stream=st)
    jh.gemm(lin1, scratch=scratch, stream=st)
    jh.score(s["y"].data_ptr(), rows, d, w["lin2"].data_ptr(), w["lin2_b"], w["markers"].data_ptr(),
             len(w["markers"]), s["logits"].data_ptr(), st)
    return s["out"]


# ------------------------------------------------------------------------------ what a pass needs
def pairs(case, window):
    """(query, key) pairs that attention computes."""
    total = 0
    for n in lengths(case) if "requests" in case else [case["rows"]]:
        if window == 0 or window >= n:
            total += n * n
        else:
            total += n * (2 * window + 1) - window * (window + 1)
    return total


def attention_work(case, window, d):
    rows = rows_of(case)
    return 8 * rows * d + (8 * rows if "requests" in case else 0), 4 * d * pairs(case, window)


def gemm_work(m, n, k, out, ln=False):
    return 2 * (m * k + n * k + m * out) + (4 * n + 8 * m * (k // 64) if ln else 0), 2 * m * n * k


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        n, k = gemm_shape(case["epi"], case["d"])
        b, f = gemm_work(case["m"], n, k, n // 2 if "geglu" in case["epi"] else n, True)
        if "rope" in case["epi"]:
            b += 256 * min(case["m"], MAX_POSITIONS)
        return {"bytes": b, "flops": f}
    rows = rows_of(case)
    if kind in ("run", "batched"):
        d = 768
        weights = LAYERS * (4 * d * d + 3 * INTER * d) + 2 * (4 * d * d + 2 * d * head_ff(d)) + d * d
        # Every row passes the encoder and the head's attention input; the marker rows the rest.
        flops = 2 * rows * (LAYERS * (4 * d * d + 3 * INTER * d) + 2 * 3 * d * d + d * d + 2 * d * head_ff(d))
        flops += 2 * case["requests"] * MARKERS * (2 * d * d + 2 * d * head_ff(d))
        n_global = (LAYERS + 2) // 3
        flops += 4 * d * (n_global * pairs(case, 0) + (LAYERS - n_global) * pairs(case, WINDOW) + 2 * pairs(case, 0))
        passes = case["requests"] if kind == "run" else 1
        return {"bytes": 2 * weights * passes + 2 * rows * d + 4 * rows, "flops": flops}
    d = case["d"]
    b, f = attention_work(case, case.get("window", 0), d)
    if kind == "attention":
        return {"bytes": b, "flops": f}
    # The blocks: the inputs and weights read once, the returned activations written once.
    if kind == "layer":
        b = 2 * rows * (d + d + 3 * d + d + INTER) + 8 * rows * (d // 64) + 2 * (4 * d * d + 3 * INTER * d)
        f += 2 * rows * (4 * d * d + 3 * INTER * d)
    else:
        ff = head_ff(d)
        b = 2 * rows * (d + d + 3 * d + d + ff + d) + 8 * rows * (d // 64) + 2 * (5 * d * d + 2 * d * ff)
        f += 2 * rows * (5 * d * d + 2 * d * ff)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times what the same path shows with its sums in another order, all f16 results:
    a GEMM over its tile heights and K splits 2.3e-5, attention over its key ranges 3.1e-4 (the
    weights are rounded to f16 under a running maximum), which a block's later steps carry on, and
    the whole model over its three ways through the kernels 1.4e-3 (a logit by up to 4.4e-3)."""
    if case["kind"] in ("run", "batched"):
        return {"rel": 6e-3, "max": 2e-2}
    return {"rel": 1e-4 if case["kind"] == "gemm" else 1.2e-3}


# ------------------------------------------------------------------------------ the same in 64 bits
def f64(t):
    return t.to(torch.float64)


def normalised(x, eps=EPS):
    mean = x.mean(1, keepdim=True)
    return (x - mean) / torch.sqrt(((x - mean) ** 2).mean(1, keepdim=True) + eps)


def gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def geglu(y):
    """Rows of W are interleaved in groups of 32: inputs, then their gates."""
    g = y.reshape(y.shape[0], -1, 2, 32)
    return (gelu(g[:, :, 0]) * g[:, :, 1]).reshape(y.shape[0], -1)


def rotated(qkv, d, table, pos):
    """The rotate-half of q and k (dimensions i and i + 32 of each head)."""
    t = f64(table)[pos.long()]
    co, sn = t[:, None, :, 0], t[:, None, :, 1]
    h = qkv[:, : 2 * d].reshape(len(qkv), -1, 2, 32)
    a, b = h[:, :, 0], h[:, :, 1]
    out = torch.stack((a * co - b * sn, b * co + a * sn), 2).reshape(len(qkv), 2 * d)
    return torch.cat((out, qkv[:, 2 * d:]), 1)


def attended(qkv, d, window, lens):
    out, at = torch.empty((len(qkv), d), dtype=torch.float64, device=qkv.device), 0
    for n in lens:
        for h in range(d // 64):
            q, k, v = (qkv[at:at + n, i * d + h * 64:i * d + h * 64 + 64] for i in range(3))
            sc = (q @ k.T) / 8.0
            if window:
                i = torch.arange(n, device=qkv.device)
                sc = sc.masked_fill((i[:, None] - i[None, :]).abs() > window, -math.inf)
            out[at:at + n, h * 64:h * 64 + 64] = torch.softmax(sc, 1) @ v
        at += n
    return out


def stats64(x):
    g = x.reshape(x.shape[0], -1, 64)
    return torch.stack((g.sum(2), (g * g).sum(2)), 2)


def fragments(e, name, index, n, k):
    """A weight matrix of the engine as [n][k], from its MFMA fragment order."""
    t = torch.from_numpy(e.tensor_host(name, index).view(np.float16)[: n * k].copy()).cuda()
    return f64(t.reshape(n // 64, k // 32, 4, 4, 16, 8).permute(0, 2, 4, 1, 3, 5).reshape(n, k))


def model64(e, reqs):
    """The model's logits for the requests, in 64 bits, from the engine's own (f16) weights."""
    d, ff = 768, head_ff(768)

    def vec(name, index=0):
        return f64(torch.from_numpy(e.tensor_host(name, index, np.float32)).cuda())

    lens = [len(r[0]) for r in reqs]
    pos = torch.cat([torch.arange(n) for n in lens]).cuda()
    ids = torch.from_numpy(np.concatenate([r[0] for r in reqs]).astype(np.int64)).cuda()
    emb = torch.from_numpy(e.tensor_host("tok_emb").view(np.float16)[: VOCAB * d].reshape(VOCAB, d)).cuda()
    x = normalised(f64(emb[ids])) * vec("emb_norm")[:d]
    tables = [vec(n)[: MAX_POSITIONS * 64].reshape(MAX_POSITIONS, 32, 2) for n in ("rope_global", "rope_local")]
    for i in range(LAYERS):
        local = i % 3 != 0
        w = fragments(e, "wqkv", i, 3 * d, d)
        qkv = rotated((x if i == 0 else normalised(x)) @ w.T, d, tables[local], pos)
        x = x + attended(qkv, d, WINDOW if local else 0, lens) @ fragments(e, "wo", i, d, d).T
        mid = geglu(normalised(x) @ fragments(e, "wi", i, 2 * INTER, d).T)
        x = x + mid @ fragments(e, "wo_mlp", i, d, INTER).T
    types = vec("type_emb")[: QTYPES * d].reshape(QTYPES, d)
    kind = torch.cat([torch.full((len(r[0]),), r[2]) for r in reqs]).cuda()
    x = normalised(x) * vec("final_norm")[:d] + types[kind]
    for i in range(2):
        qkv = normalised(x) @ fragments(e, "in_proj", i, 3 * d, d).T + vec("in_proj_b", i)[: 3 * d]
        x = x + attended(qkv, d, 0, lens) @ fragments(e, "out_proj", i, d, d).T + vec("out_proj_b", i)[:d]
        mid = torch.relu(normalised(x) @ fragments(e, "linear1", i, ff, d).T + vec("linear1_b", i)[:ff])
        x = x + mid @ fragments(e, "linear2", i, d, ff).T + vec("linear2_b", i)[:d]
    y = gelu(normalised(x) @ fragments(e, "lin1", 0, d, d).T + vec("lin1_b")[:d])
    w = f64(torch.from_numpy(e.tensor_host("lin2").view(np.float16)[:d].copy()).cuda())
    bias = float(jh.synth(MODEL_SEED, 2005, 1, 0.0, 0.02)[0])  # the synthetic scorer's last bias
    out, at = [], 0
    for r in reqs:
        out.append((y[at + torch.from_numpy(r[1].astype(np.int64)).cuda()] @ w + bias).cpu())
        at += len(r[0])
    return torch.cat(out).numpy()


def linear64(x, lin):
    y = x @ f64(lin.plain).T
    return y if lin.bias is None else y + f64(lin.bias)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("run", "batched"):
        return model64(engine(), requests(case, seed))
    if kind == "gemm":
        a, lin, pos = gemm_inputs(case, seed)
        y = linear64(normalised(f64(a)), lin)
        if case["epi"] == "lnrope":
            p = torch.arange(len(a), device="cuda") if pos is None else pos
            return rotated(y, case["d"], rope(THETA_GLOBAL), p)
        if case["epi"] == "lngeglu":
            return geglu(y)
        return torch.relu(y) if case["epi"] == "lnbiasrelu" else gelu(y) if case["epi"] == "lnbiasgelu" else y
    rows, d, window = rows_of(case), case["d"], case.get("window", 0)
    lens = lengths(case) if "requests" in case else [rows]
    if kind == "attention":
        return attended(f64(normal16(seed, 1, (rows, 3 * d))), d, window, lens)
    if kind == "layer":
        w = layer_inputs(case, seed)
        pos, _ = sequences(case)
        pos = torch.arange(rows, device="cuda") if pos is None else pos
        x = normalised(f64(w["table"][w["ids"].long()])) * f64(w["gamma"])
        qkv = rotated(linear64(x, w["qkv"]), d, rope(THETA_LOCAL if window else THETA_GLOBAL), pos)
        o = attended(qkv, d, window, lens)
        x = x + linear64(o, w["wo"])
        mid = geglu(linear64(normalised(x), w["wi"]))
        x = x + linear64(mid, w["wo_mlp"])
        return {"x": x, "stats": stats64(x), "qkv": qkv, "o": o, "mid": mid}
    w = head_inputs(case, seed)
    x = normalised(f64(w["x"])) * f64(w["gamma"]) + f64(w["type"])
    qkv = linear64(normalised(x), w["in_proj"])
    o = attended(qkv, d, 0, lens)
    x = x + linear64(o, w["out_proj"])
    mid = torch.relu(linear64(normalised(x), w["linear1"]))
    x = x + linear64(mid, w["linear2"])
    y = gelu(linear64(normalised(x), w["lin1"]))
    logits = y[w["markers"].long()] @ f64(w["lin2"]) + w["lin2_b"]
    return {"x": x, "stats": stats64(x), "qkv": qkv, "o": o, "mid": mid, "y": y, "logits": logits}
