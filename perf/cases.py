"""The work whose speed is measured: passes through the engine's public entry points.

Sizes are those of the 213M-parameter encoder (n_embd 1,024, FFN 2,304, 16 query and 8 KV
heads of 64, SnowLily rank 64, sliding window 256) at the lengths that the benchmark, the
tests and the published timings use: one linear of 128 rows up to a document of 65,536
tokens. Kinds of case:

  linear     quantize_rows and linear_i8: one projection of fp32 rows
  mlp        rmsnorm_quantize_rows and Builder.mlp: the MLP half of every block
  attention  attention() alone, full or banded
  attn       the mixer of an attention block: norm, fused QKV, DyT and RoPE, attention, gate,
             c_proj + residual (band > 0: the sliding-window block)
  lily       the mixer of a SnowLily block: norm and Builder.lily
  forward    Encoder.forward of the whole model on device tensors
  encode     Encoder.encode of the whole model on host arrays, as a request comes in

Every result is the reference's bit for bit (that is the engine's contract: the order of every
fp32 operation is the reference's), so the tolerance is exact everywhere.
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch

C, INTER, HEADS, KV_HEADS, HEAD_DIM, RANK = 1024, 2304, 16, 8, 64, 64
KV = KV_HEADS * HEAD_DIM
TAPS = 5
EPS = 1e-8
ROPE_BASE = {"full": 100000.0, "band": 10000.0}
# lengths of a mixed batch: 32 documents of 16 to 2,048 tokens (numpy's default_rng(1))
DOCS32 = " ".join(str(n) for n in np.random.default_rng(1).integers(16, 2048, 32, endpoint=True))

_CACHE = {}


def _nxg():
    """The engine package, whose directory name is not an identifier."""
    name = "nexterabert_cpp_amd"
    if name not in sys.modules:
        pkg = Path(__file__).resolve().parent.parent / "nexterabert.cpp_amd"
        spec = importlib.util.spec_from_file_location(name, pkg / "__init__.py", submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def listed():
    return [
        # one 1,024 x 1,024 projection of a short text: launches and latency
        {"name": "linear_128", "kind": "linear", "rows": 128, "n_in": C, "n_out": C, "residual": False},
        # the MLP of one 1,024-token sequence (the published latency) and of the largest batch
        {"name": "mlp_1024", "kind": "mlp", "lengths": "1024"},
        {"name": "mlp_65536", "kind": "mlp", "lengths": "65536"},
        # the mixers: full attention over one short document, the sliding window and SnowLily
        # over a mixed batch of 32 documents
        {"name": "attn_512", "kind": "attn", "lengths": "512", "band": 0},
        {"name": "swa_32docs", "kind": "attn", "lengths": DOCS32, "band": 256},
        {"name": "lily_32docs", "kind": "lily", "lengths": DOCS32},
        # attention alone: one sequence, the window over a batch of 8, a mixed batch, and the
        # longest document the published timings have
        {"name": "attention_1x1024", "kind": "attention", "lengths": "1024", "band": 0},
        {"name": "attention_band_8x1024", "kind": "attention", "lengths": " ".join(["1024"] * 8), "band": 256},
        {"name": "attention_32docs", "kind": "attention", "lengths": DOCS32, "band": 0},
        {"name": "attention_65536", "kind": "attention", "lengths": "65536", "band": 0},
        # whole calls: the published single-sequence latency, and a request of a few short texts
        {"name": "forward_1x1024", "kind": "forward", "lengths": "1024"},
        {"name": "encode_short", "kind": "encode", "lengths": "23 7 61 34"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_lengths(rng, most):
    """One document, several alike, or a mixed batch; at most `most` tokens in all."""
    shape = rng.choice(["one", "alike", "mixed", "mixed"])
    if shape == "one":
        return str(_log(rng, 5, most))
    if shape == "alike":
        n = rng.randint(2, 16)
        return " ".join([str(_log(rng, 16, min(2048, most // n)))] * n)
    out = []
    for _ in range(rng.randint(2, 32)):
        out.append(_log(rng, 5, 2048))
        if sum(out) > most:
            out[-1] = max(1, out[-1] - (sum(out) - most))
            break
    return " ".join(map(str, out))


def draw(rng):
    kind = rng.choice(["linear", "mlp", "attention", "attention", "attn", "attn", "lily", "forward", "encode"])
    if kind == "linear":
        n_in, n_out = rng.choice([(C, C), (C, 2048), (C, 3072), (C, INTER), (INTER, C), (C, RANK), (RANK, C), (320, 512)])
        return {"kind": kind, "rows": _log(rng, 1, 65536), "n_in": n_in, "n_out": n_out, "residual": rng.random() < 0.5}
    if kind in ("mlp", "lily"):
        return {"kind": kind, "lengths": _draw_lengths(rng, 65536)}
    if kind in ("attention", "attn"):
        band = rng.choice([0, 256])
        return {"kind": kind, "lengths": _draw_lengths(rng, 65536 if band else 32768), "band": band}
    return {"kind": kind, "lengths": _draw_lengths(rng, 16384 if kind == "forward" else 4096)}


# --- what a case needs -----------------------------------------------------------------------

def _lengths(case):
    return [int(n) for n in case["lengths"].split()]


def _half(case):
    return case["band"] // 2 if case["band"] else -1


def _key_pairs(case):
    """(query, key) pairs of one head."""
    half, pairs = _half(case), 0
    for n in _lengths(case):
        if half < 0 or 2 * half + 1 >= 2 * n:
            pairs += n * n
        else:
            w = min(half, n - 1)
            pairs += n * (2 * w + 1) - w * (w + 1)
    return pairs


def _gemm_work(rows, n_in, n_out):
    return 2 * rows * n_in * n_out, n_in * n_out + 4 * n_out * ((n_in + 255) // 256)


def work(case):
    """Multiplications and additions, and the bytes of inputs, weights and outputs."""
    kind = case["kind"]
    if kind == "linear":
        T = case["rows"]
        f, w = _gemm_work(T, case["n_in"], case["n_out"])
        return {"bytes": w + 4 * T * (case["n_in"] + case["n_out"] * (2 if case["residual"] else 1)), "flops": f}
    T = sum(_lengths(case))
    if kind == "attention":
        return {"bytes": 4 * T * (2 * C + 2 * KV), "flops": 4 * HEAD_DIM * HEADS * _key_pairs(case)}

    def linears(shapes):
        fs, ws = zip(*(_gemm_work(r, i, o) for r, i, o in shapes))
        return sum(fs), sum(ws)

    mlp = [(T, C, INTER), (T, INTER, C)]
    attn = [(T, C, C + 2 * KV), (T, C, C), (T, C, C)]
    lily = [(T, C, RANK), (T, C, RANK), (T, RANK, C), (T, C, C), (T, C, C), (T, C, C)]
    if kind in ("mlp", "lily", "attn"):
        f, w = linears({"mlp": mlp, "lily": lily, "attn": attn}[kind])
        if kind == "attn":
            f += 4 * HEAD_DIM * HEADS * _key_pairs(case)
        return {"bytes": 8 * T * C + w, "flops": f}
    # whole model: 8 lily, 5 sliding-window, 3 full attention, 2 hra blocks (block of 4)
    B = sum((n + 3) // 4 for n in _lengths(case))
    hra = [(T, C, 3 * C), (B, C, C + 2 * KV), (T, C, C), (T, C, C)]
    f, w = linears(mlp * 18 + lily * 8 + attn * 8 + hra * 2)
    quarter = " ".join(str((n + 3) // 4) for n in _lengths(case))
    for n, lens, band in ((5, case["lengths"], 256), (3, case["lengths"], 0), (2, quarter, 0)):
        f += n * 4 * HEAD_DIM * HEADS * _key_pairs({"lengths": lens, "band": band})
    return {"bytes": w + T * (4 + 8 * C) + 4 * C * len(_lengths(case)), "flops": f}


def tolerance(case):
    return "exact"


# --- inputs ----------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _unif(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, device="cuda", generator=g)


def _int8_weight(g, n_in, n_out):
    """N(0, 0.02) rows as load time leaves them: int8 and one scale per row and 256 inputs.
    Returns the device weight and the rows it stands for, in 64 bits."""
    nb = (n_in + 255) // 256
    w = torch.zeros(n_out, nb * 256, device="cuda")
    w[:, :n_in] = 0.02 * _randn(g, n_out, n_in)
    w = w.view(n_out, nb, 256)
    scale = w.abs().amax(2) / 127
    q = (w / scale[:, :, None]).round().clamp(-127, 127)
    rows = (q.double() * scale.double()[:, :, None]).reshape(n_out, nb * 256)[:, :n_in]
    q = q.to(torch.int8).reshape(n_out, nb * 256)[:, :n_in]
    nxg = _nxg()
    host = nxg.I8Weight(q.contiguous().cpu().numpy(), scale.t().contiguous().cpu().numpy(), np.zeros((nb, n_out), np.int32))
    return nxg.DeviceWeight(host), rows


def _rope(n_pos, base):
    """cos and sin of position * base^(-2i / head_dim), fp32 tables [n_pos][head_dim / 2]."""
    i = np.arange(HEAD_DIM // 2)
    a = np.arange(n_pos)[:, None] * (float(base) ** (-2.0 * i / HEAD_DIM))[None, :]
    return [torch.from_numpy(f(a).astype(np.float32)).cuda() for f in (np.cos, np.sin)]


def _scales(case):
    """Scalable-Softmax scales of full attention (1/8 (s ln n + b)), 1/8 for the window."""
    n = np.array(_lengths(case), np.float64)
    s = 0.125 * (0.3 * np.log(n) + 0.2) if case["band"] == 0 else np.full(n.size, 0.125)
    return s.astype(np.float32)


def _model():
    """The whole model (random weights, a Q4_K_M file), loaded once as a program loads it."""
    if "model" not in _CACHE:
        nxg = _nxg()
        from nexterabert_cpp_amd import synth
        with tempfile.TemporaryDirectory() as tmp:
            path = os.path.join(tmp, "model.gguf")
            synth.write_random_model(nxg, path, "Q4_K_M", seed=0)
            _CACHE["model"] = nxg.Encoder(path)
    return _CACHE["model"]


def prepare(case, seed):
    nxg, kind, g = _nxg(), case["kind"], _gen(seed)
    s = {"case": case, "nxg": nxg}
    if kind == "linear":
        T = case["rows"]
        s["w"], s["w64"] = _int8_weight(g, case["n_in"], case["n_out"])
        s["x"] = _randn(g, T, case["n_in"])
        s["res"] = _randn(g, T, case["n_out"]) if case["residual"] else None
        return s
    lens = _lengths(case)
    T, cu = sum(lens), nxg.cu_offsets_of(lens)
    s["cu"] = cu
    if kind in ("forward", "encode"):
        s["lengths"] = lens
        s["model"] = _model()
        ids = torch.randint(0, s["model"].n_vocab, (T,), device="cuda", generator=g, dtype=torch.int32)
        if kind == "encode":
            s["ids"] = ids.cpu().numpy()
        else:
            s["ids"] = ids
            s["hidden"] = torch.empty(T, C, device="cuda")
            s["pooled"] = torch.empty(len(lens), C, device="cuda")
        return s
    if kind == "attention":
        # after DyT: tanh within about +-1
        s["q"] = _unif(g, 0.8, 1.2, 1) * torch.tanh(0.7 * _randn(g, T, C))
        s["k"] = torch.tanh(0.7 * _randn(g, KV_HEADS, T, HEAD_DIM))
        s["v"] = 0.6 * _randn(g, KV_HEADS, T, HEAD_DIM)
        s["scale"] = _scales(case)
        return s
    s["x"] = _randn(g, T, C)
    s["gain"] = _unif(g, 0.8, 1.2, C)
    shapes = {"mlp": {"c_fc": (C, INTER), "c_proj": (INTER, C)},
              "attn": {"qkv": (C, C + 2 * KV), "c_gate": (C, C), "c_proj": (C, C)},
              "lily": {"ltc_conv.in_proj": (C, RANK), "ltc_conv.A": (C, RANK), "ltc_conv.out_proj": (RANK, C),
                       "x_proj": (C, C), "B_proj": (C, C), "c_proj": (C, C)}}[kind]
    made = {n + ".weight": _int8_weight(g, *io) for n, io in shapes.items()}
    s["w64"] = {n: m[1] for n, m in made.items()}
    s["builder"] = nxg.Builder({n: m[0] for n, m in made.items()})
    if kind == "attn":
        s["dyt"] = [_unif(g, lo, hi, HEAD_DIM) for lo, hi in ((0.3, 1.0), (0.8, 1.2)) * 2]
        s["rope"] = _rope(max(lens), ROPE_BASE["band" if case["band"] else "full"])
        s["scale"] = _scales(case)
    if kind == "lily":
        s["ltc"], s["taps"] = _unif(g, -0.5, 0.5, TAPS, RANK), _unif(g, -0.5, 0.5, TAPS, C)
    return s


def run(s):
    nxg, case = s["nxg"], s["case"]
    kind = case["kind"]
    if kind == "linear":
        return nxg.linear_i8(s["w"], nxg.quantize_rows(s["x"]), residual=s["res"])
    if kind == "attention":
        return nxg.attention(s["q"], s["k"], s["v"], s["cu"], s["scale"], HEADS, KV_HEADS, half=_half(case),
                             workspace="auto")
    if kind == "forward":
        s["model"].forward(s["ids"], s["lengths"], hidden=s["hidden"], pooled=s["pooled"], normalize=True)
        return s["hidden"], s["pooled"]
    if kind == "encode":
        return s["model"].encode(s["ids"], s["lengths"], pooled=True, normalize=True)
    b, cu = s["builder"], s["cu"]
    b.reset()
    h = b.rms_norm(s["x"], s["gain"], EPS)
    if kind == "mlp":
        return b.mlp("c_fc.weight", "c_proj.weight", h, s["x"], cu_offsets=cu)
    if kind == "lily":
        return b.lily("", h, s["x"], s["ltc"], s["taps"], cu)
    q, k, v = nxg.linear_i8_split(b.i8["qkv.weight"], h, [C, KV, KV])
    q, k, v = nxg.qkv_prep(q, k, v, *s["dyt"], *s["rope"], cu, HEADS, KV_HEADS)
    y = nxg.attention(q, k, v, cu, s["scale"], HEADS, KV_HEADS, half=_half(case), workspace="auto")
    return b.gated_out("", y, y, s["x"], cu_offsets=cu)


# --- the same in 64 bits ---------------------------------------------------------------------

def _quant64(x):
    """Rows on the int8 grid of their 256-value blocks, as values."""
    T, n = x.shape
    nb = (n + 255) // 256
    p = torch.zeros(T, nb * 256, dtype=torch.float64, device=x.device)
    p[:, :n] = x
    p = p.view(T, nb, 256)
    amax = p.abs().amax(2, keepdim=True)
    step = torch.where(amax > 0, amax / 127, torch.ones_like(amax))
    return ((p / step).round() * step).reshape(T, nb * 256)[:, :n]


def _lin64(x, w):
    out = torch.empty(x.shape[0], w.shape[0], dtype=torch.float64, device=x.device)
    wt = w.t().contiguous()
    for r in range(0, x.shape[0], 16384):
        torch.mm(_quant64(x[r:r + 16384]), wt, out=out[r:r + 16384])
    return out


def _rms64(x, gain):
    x = x.double()
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * gain.double()


def _attention64(q, k, v, case, scale):
    """q [T][HEADS * 64], k and v [KV_HEADS][T][64], all in 64 bits."""
    out, half, t0 = torch.empty_like(q), _half(case), 0
    for d, n in enumerate(_lengths(case)):
        step = 2048 if n <= 16384 else 4096
        for h in range(HEADS):
            kt = k[h * KV_HEADS // HEADS, t0:t0 + n].t().contiguous()
            vh = v[h * KV_HEADS // HEADS, t0:t0 + n].contiguous()
            for r in range(0, n, step):
                m = min(step, n - r)
                lo, hi = (0, n) if half < 0 else (max(0, r - half), min(n, r + m + half))
                s = torch.mm(q[t0 + r:t0 + r + m, 64 * h:64 * h + 64].contiguous(), kt[:, lo:hi].contiguous())
                s *= float(scale[d])
                if half >= 0:
                    off = torch.arange(lo, hi, device=q.device)[None, :] - torch.arange(r, r + m, device=q.device)[:, None]
                    s.masked_fill_(off.abs() > half, -math.inf)
                out[t0 + r:t0 + r + m, 64 * h:64 * h + 64] = torch.mm(torch.softmax(s, 1), vh[lo:hi])
        t0 += n
    return out


def _prep64(x, alpha, beta, rope, cu, heads):
    """DyT, then the rotation of each row's position in its document: [T][heads][64]."""
    T = x.shape[0]
    x = beta.double() * torch.tanh(alpha.double() * x.view(T, heads, HEAD_DIM))
    lens = np.diff(cu)
    pos = torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).cuda()
    c, s = (t.double()[pos][:, None, :] for t in rope)
    a, b = x[..., :HEAD_DIM // 2], x[..., HEAD_DIM // 2:]
    return torch.cat([a * c + b * s, b * c - a * s], 2)


def _dwconv64(x, taps, cu):
    """Depthwise convolution inside each document, zeros outside it."""
    out = torch.empty_like(x)
    p = taps.shape[0] // 2
    for a, b in zip(cu[:-1], cu[1:]):
        n = int(b - a)
        xp = torch.zeros(n + 2 * p, x.shape[1], dtype=x.dtype, device=x.device)
        xp[p:p + n] = x[int(a):int(b)]
        out[int(a):int(b)] = sum(taps[j].double() * xp[j:j + n] for j in range(taps.shape[0]))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "encode"):
        return None          # rounding to int8 in 18 blocks in turn: 64 bits take other steps
    s = prepare(case, seed)
    if kind == "linear":
        y = _lin64(s["x"].double(), s["w64"])
        return y if s["res"] is None else y + s["res"].double()
    if kind == "attention":
        return _attention64(s["q"].double(), s["k"].double(), s["v"].double(), case, s["scale"])
    w, x, cu = s["w64"], s["x"].double(), s["cu"]
    h = _rms64(s["x"], s["gain"])
    if kind == "mlp":
        u = torch.relu(_lin64(h, w["c_fc.weight"]))
        return x + _lin64(u * u, w["c_proj.weight"])
    if kind == "lily":
        z, r = _lin64(h, w["ltc_conv.in_proj.weight"]), _lin64(h, w["ltc_conv.A.weight"])
        a = _lin64(_dwconv64(z, s["ltc"], cu) + r, w["ltc_conv.out_proj.weight"])
        xp, b = _lin64(h, w["x_proj.weight"]), _lin64(h, w["B_proj.weight"])
        return x + _lin64(_dwconv64(a * xp, s["taps"], cu) * b, w["c_proj.weight"])
    qkv = _lin64(h, w["qkv.weight"])
    qa, qb, ka, kb = s["dyt"]
    q = _prep64(qkv[:, :C], qa, qb, s["rope"], cu, HEADS).reshape(-1, C)
    k = _prep64(qkv[:, C:C + KV], ka, kb, s["rope"], cu, KV_HEADS).transpose(0, 1).contiguous()
    v = qkv[:, C + KV:].reshape(-1, KV_HEADS, HEAD_DIM).transpose(0, 1).contiguous()
    y = _attention64(q, k, v, case, s["scale"])
    return x + _lin64(torch.sigmoid(_lin64(y, w["c_gate.weight"])) * y, w["c_proj.weight"])
