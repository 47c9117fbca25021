"""The work that a program gives this framework, as cases that can be timed.

Each case is one pass through the public entry points of the C ABI's Python
binding (rfp4), on device tensors that torch owns, or one call of an engine.
The sizes are those of the three models that the binding has presets for
(Llama-3-8B, TinyLlama-1.1B, Llama-3.2-1B) and of the GEMV, attention and GEMM
examples of tests/ and bench.py; draw() spreads them over the ranges between
and around these, odd and ragged sizes among them.

Kinds of case (the "op" of a case):
  gemv      one projection of one token, E8M0 or f32 block scales
  mlp       the feed-forward block of one token: norm, gate|up with SwiGLU, down
  head      the LM head of one token with its argmax
  attn      decode attention over a context (fp16 or f32 K/V)
  attnp     causal attention of prompt rows
  gemm      bf16 activation rows quantized to MXFP4, times a weight matrix
  prefill   an engine's batched prefill of a prompt through one layer and the head
  generate  an engine's prompt-then-greedy loop through the whole model
"""
import math
import os
import sys

import numpy as np
import torch  # before the library: both then use torch's HIP runtime

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rust-fp4-blackwell_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import rfp4  # noqa: E402

EPS = 1e-5
# one layer: in a second one, a row whose MXFP4 codes moved by one rounding in
# the first is up to a fifth off, and no two correct programs would agree
PREFILL_LAYERS = 1


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one projection of a 2048-wide model: the smallest call, a few MB of
        # weights, where the launch and the memory latency count
        {"name": "gemv-2048", "op": "gemv", "n": 2048, "k": 2048, "scale": "e8m0"},
        # the f32-scale drop-in of the reference's weights: gate or up of Llama-3.2-1B
        {"name": "gemv-f32-8192x2048", "op": "gemv", "n": 8192, "k": 2048, "scale": "f32"},
        # a token's feed-forward block at the Llama-3-8B widths
        {"name": "mlp-8b", "op": "mlp", "dim": 4096, "ffn": 14336},
        # a token's LM head and argmax at the Llama-3-8B widths: the widest matrix of a step
        {"name": "head-8b", "op": "head", "dim": 4096, "vocab": 128256},
        # decode attention, the reference's f32 cache layout and its harness's context
        {"name": "attn-f32-512", "op": "attn", "nh": 32, "nkv": 8, "hd": 64, "seq": 512, "kv": "f32", "layout": "token"},
        # decode attention of Llama-3-8B at the context of the headline benchmark
        {"name": "attn-8b-4096", "op": "attn", "nh": 32, "nkv": 8, "hd": 128, "seq": 4096, "kv": "f16", "layout": "head"},
        # a long prompt's second chunk: causal rows after a context, ragged
        {"name": "attnp-8b-1531+517", "op": "attnp", "nh": 32, "nkv": 8, "hd": 128, "rows": 1531, "pos0": 517},
        # a batch of 32 decode rows through the gate|up projection of Llama-3-8B
        {"name": "gemm-8b-32", "op": "gemm", "m": 32, "n": 28672, "k": 4096},
        # 512 prompt rows through the down projection of Llama-3-8B
        {"name": "gemm-8b-512", "op": "gemm", "m": 512, "n": 4096, "k": 14336},
        # a 700-token prompt through a layer and the head at the Llama-3-8B widths
        {"name": "prefill-8b-700", "op": "prefill", "model": "llama3-8b", "rows": 700, "pos0": 0},
        # a short chat turn with the whole of TinyLlama-1.1B: 4 prompt tokens, 13 new ones
        {"name": "generate-tiny-200", "op": "generate", "model": "tinyllama-1.1b", "ctx": 200, "prompt": 4, "new": 13},
        # the headline benchmark: the whole of Llama-3-8B decoding at context 4096
        {"name": "generate-8b-4096", "op": "generate", "model": "llama3-8b", "ctx": 4096, "prompt": 4, "new": 13},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gemv", "mlp", "head", "attn", "attn", "attnp", "gemm", "gemm", "prefill", "generate"])
    if op == "gemv":  # any row count; K any number of 32-value blocks
        return {"op": op, "n": _log(rng, 256, 32768), "k": 32 * _log(rng, 16, 448), "scale": rng.choice(["e8m0", "e8m0", "f32"])}
    if op == "mlp":
        return {"op": op, "dim": 64 * _log(rng, 12, 80), "ffn": 64 * _log(rng, 30, 256)}
    if op == "head":
        return {"op": op, "dim": 64 * _log(rng, 12, 80), "vocab": _log(rng, 8000, 128256)}
    if op == "attn":
        kv = rng.choice(["f16", "f16", "f32"])
        nkv, group = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 8])
        return {"op": op, "nh": nkv * group, "nkv": nkv, "hd": 64 if kv == "f32" else rng.choice([64, 128]),
                "seq": _log(rng, 1, 16384), "kv": kv, "layout": "token" if kv == "f32" else rng.choice(["head", "token"])}
    if op == "attnp":
        nkv, group = rng.choice([2, 4, 8]), rng.choice([1, 2, 4, 8])
        return {"op": op, "nh": nkv * group, "nkv": nkv, "hd": rng.choice([64, 128]), "rows": _log(rng, 1, 2048),
                "pos0": rng.choice([0, _log(rng, 1, 4096)])}
    if op == "gemm":  # K as the tiles take it, N any multiple of 4
        return {"op": op, "m": _log(rng, 1, 2048), "n": 4 * _log(rng, 128, 7168), "k": 256 * _log(rng, 4, 56)}
    if op == "prefill":
        return {"op": op, "model": rng.choice(sorted(rfp4.PRESETS)), "rows": _log(rng, 1, 1024), "pos0": rng.choice([0, _log(rng, 1, 1024)])}
    return {"op": op, "model": rng.choice(sorted(rfp4.PRESETS)), "ctx": _log(rng, 1, 4096), "prompt": rng.randint(1, 6), "new": rng.randint(1, 8)}


# ------------------------------------------------------------------ MXFP4 in torch
_LEVELS = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _quantize(x):
    """OCP MXFP4 rows of x [rows][k]: (codes u8 [rows][k/2], E8M0 scales u8 [rows][k/32])."""
    rows, k = x.shape
    b = x.reshape(rows, k // 32, 32)
    amax = b.abs().amax(-1)
    se = torch.where(amax > 0, torch.frexp(amax)[1].to(torch.int32) - 3, torch.zeros((), dtype=torch.int32, device=x.device))
    v = torch.ldexp(b, -se[..., None])
    a = v.abs()
    mid = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], dtype=x.dtype, device=x.device)
    # nearest level, a tie to the even code
    low, high = torch.bucketize(a, mid, right=False), torch.bucketize(a, mid, right=True)
    code = torch.where(low % 2 == 0, low, high)
    code = (code + 8 * (torch.signbit(v) & (code >= 0)).to(code.dtype)).to(torch.uint8).reshape(rows, k // 2, 2)
    sb = torch.where(amax > 0, se + 127, torch.zeros_like(se) + 0).to(torch.uint8)
    return code[..., 0] | (code[..., 1] << 4), sb


def _dequantize(codes, scales, k):
    """f64 values [rows][k] of codes (u8) with E8M0 (u8) or f32 scales per 32."""
    lut = torch.tensor(list(_LEVELS) + [-v for v in _LEVELS], dtype=torch.float64, device=codes.device)
    c = codes.reshape(-1, k // 2)
    w = torch.stack((lut[(c & 15).long()], lut[(c >> 4).long()]), -1).reshape(-1, k // 32, 32)
    s = scales.reshape(-1, k // 32)
    s = torch.ldexp(torch.ones((), dtype=torch.float64, device=codes.device), s.to(torch.int32) - 127) if s.dtype == torch.uint8 else s.double()
    return (w * s[..., None]).reshape(-1, k)


def _matvec(codes, scales, k, x, step=8192):
    """f64 W.x (x [k]) or x.W^T (x [rows][k]), W dequantized by parts."""
    codes, scales = codes.reshape(-1, k // 2), scales.reshape(-1, k // 32)
    parts = [x @ _dequantize(codes[i:i + step], scales[i:i + step], k).t() for i in range(0, codes.shape[0], step)]
    return torch.cat(parts, -1)


# ------------------------------------------------------------------ inputs
def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _weights(g, n, k, scale="e8m0"):
    """A weight matrix as checkpoints give them: N(0, 0.02^2) quantized (E8M0),
    or the reference harness's uniform codes and f32 scales."""
    if scale == "f32":
        codes = torch.randint(0, 256, (n, k // 2), generator=g, device="cuda", dtype=torch.uint8)
        return codes, 0.25 + torch.randint(0, 8, (n, k // 32), generator=g, device="cuda").float() * 0.03125
    parts = [_quantize(0.02 * _normal(g, min(8192, n - i), k)) for i in range(0, n, 8192)]
    return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])


class _View:
    """A device buffer of the engine as torch sees it; keeps the engine alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(owner, ptr, shape, typestr):
    return torch.as_tensor(_View(owner, ptr, shape, typestr), device="cuda")


def _engine(case, seed):
    """An engine with synthetic weights and, before the first position, a synthetic context."""
    dims = dict(rfp4.PRESETS[case["model"]])
    ctx = case["pos0"] if case["op"] == "prefill" else case["ctx"]
    steps = case["rows"] if case["op"] == "prefill" else case["prompt"] + case["new"] - 1
    if case["op"] == "prefill":
        dims["n_layers"] = PREFILL_LAYERS
    eng = rfp4.Engine(rfp4.model_config(max_seq=ctx + steps + 1, **dims), seed)
    eng.prefill_kv(seed + 1, ctx)
    n = case["rows"] if case["op"] == "prefill" else case["prompt"]
    prompt = np.random.default_rng(seed).integers(0, dims["vocab"], n).astype(np.uint32)
    k, v, count = rfp4.P(), rfp4.P(), rfp4.SZ()
    rfp4.check(rfp4.load().llama_engine_kv(eng.h, 0, rfp4.C.byref(k), rfp4.C.byref(v), rfp4.C.byref(count)))
    nkv, hd = dims["n_kv_heads"], dims["head_dim"]
    shape = (dims["n_layers"], nkv, count.value // (nkv * hd), hd)
    kc, vc = _view(eng, k.value, shape, "<f2"), _view(eng, v.value, shape, "<f2")
    return {"op": case["op"], "eng": eng, "dims": dims, "prompt": prompt, "ctx": ctx, "seed": seed, "new": case.get("new"), "all": (kc, vc),
            "written": (kc[:, :, ctx:ctx + steps], vc[:, :, ctx:ctx + steps])}


def prepare(case, seed):
    rfp4.init(0)
    op = case["op"]
    if op in ("prefill", "generate"):
        return _engine(case, seed)
    g = _rng(seed)
    s = {"op": op, "case": case}
    f32 = dict(dtype=torch.float32, device="cuda")
    if op == "gemv":
        n, k = case["n"], case["k"]
        s["w"], s["ws"] = _weights(g, n, k, case["scale"])
        s["x"], s["y"] = _normal(g, k), torch.empty(n, **f32)
    elif op == "mlp":
        d, f = case["dim"], case["ffn"]
        s["norm"] = (1 + 0.02 * _normal(g, d)).half()
        s["gu"], s["gus"] = _weights(g, 2 * f, d)
        s["dn"], s["dns"] = _weights(g, d, f)
        s["x"] = 3 * _normal(g, d)
        s["h"], s["a"], s["y"] = torch.empty(d, **f32), torch.empty(f, **f32), torch.empty(d, **f32)
    elif op == "head":
        n, k = case["vocab"], case["dim"]
        s["w"], s["ws"] = _weights(g, n, k)
        s["x"], s["y"] = _normal(g, k), torch.empty(n, **f32)
        s["work"] = torch.empty(rfp4.mx4_gemv_argmax_workspace(n), dtype=torch.uint8, device="cuda")
        s["best"] = torch.empty(1, dtype=torch.int32, device="cuda")
    elif op in ("attn", "attnp"):
        nh, nkv, hd = case["nh"], case["nkv"], case["hd"]
        seq = case["seq"] if op == "attn" else case["pos0"] + case["rows"]
        dt = torch.float16 if case.get("kv", "f16") == "f16" else torch.float32
        shape = (seq, nkv, hd) if case.get("layout") == "token" else (nkv, seq, hd)
        s["k"], s["v"] = _normal(g, *shape).to(dt), _normal(g, *shape).to(dt)
        s["ts"], s["hs"] = (nkv * hd, hd) if case.get("layout") == "token" else (hd, seq * hd)
        s["q"] = _normal(g, *((nh, hd) if op == "attn" else (case["rows"], nh, hd)))
        s["y"] = torch.empty_like(s["q"])
    else:
        m, n, k = case["m"], case["n"], case["k"]
        s["w"], s["ws"] = _weights(g, n, k)
        s["wst"] = torch.zeros(rfp4.mx4_scales_tiled_bytes(n, k), dtype=torch.uint8, device="cuda")  # laid out once, as an engine does
        rfp4.mx4_scales_tile(_stream(), n, k, s["ws"].data_ptr(), s["wst"].data_ptr())
        s["x"] = _normal(g, m, k).bfloat16()
        s["c"], s["cs"] = torch.empty(m, k // 2, dtype=torch.uint8, device="cuda"), torch.empty(m, k // 32, dtype=torch.uint8, device="cuda")
        s["cst"] = torch.zeros(rfp4.mx4_scales_tiled_bytes(m, k), dtype=torch.uint8, device="cuda")
        s["y"] = torch.empty(m, n, **f32)
    # the handles that a program holds: its stream and its buffers' addresses
    s["stream"], s["ptr"] = _stream(), {name: t.data_ptr() for name, t in s.items() if isinstance(t, torch.Tensor)}
    return s


def _stream():
    return torch.cuda.current_stream().cuda_stream


# ------------------------------------------------------------------ one pass
def run(s):
    op = s["op"]
    if op == "prefill":
        nxt = s["eng"].prefill(s["prompt"], s["ctx"])
        return {"next": nxt, "logits": s["eng"].logits(), "k": s["written"][0], "v": s["written"][1]}
    if op == "generate":
        ids = s["eng"].generate(s["prompt"], s["ctx"], s["new"])
        return {"ids": ids, "logits": s["eng"].logits(), "k": s["written"][0], "v": s["written"][1]}
    c, st, p = s["case"], s["stream"], s["ptr"]
    if op == "gemv":
        (rfp4.fp4_gemv if c["scale"] == "f32" else rfp4.mx4_gemv)(st, c["n"], c["k"], p["w"], p["ws"], p["x"], p["y"])
    elif op == "mlp":
        rfp4.rmsnorm_f16w(st, c["dim"], EPS, p["x"], p["norm"], p["h"])
        rfp4.mx4_gemv_swiglu(st, c["ffn"], c["dim"], c["ffn"], p["gu"], p["gus"], p["h"], p["a"])
        rfp4.mx4_gemv(st, c["dim"], c["ffn"], p["dn"], p["dns"], p["a"], p["y"])
    elif op == "head":
        rfp4.mx4_gemv_argmax(st, c["vocab"], c["dim"], p["w"], p["ws"], p["x"], p["y"], p["work"], p["best"])
        return {"logits": s["y"], "best": s["best"]}
    elif op == "attn" and c["kv"] == "f32":
        rfp4.attn_decode(st, c["nh"], c["nkv"], c["seq"], p["q"], p["k"], p["v"], p["y"])
    elif op == "attn":
        rfp4.attn_decode_f16(st, c["nh"], c["nkv"], c["hd"], c["seq"], p["q"], p["k"], p["v"], s["ts"], s["hs"], p["y"])
    elif op == "attnp":
        w = c["nh"] * c["hd"]
        rfp4.attn_prefill_f16(st, c["nh"], c["nkv"], c["hd"], c["pos0"], c["rows"], p["q"], w, p["k"], p["v"], s["ts"], s["hs"], p["y"], w)
    else:
        rfp4.mx4_quantize_tiled(st, c["m"], c["k"], p["x"], True, p["c"], p["cs"], p["cst"])
        rfp4.fp4_gemm_tiled(st, c["m"], c["n"], c["k"], p["c"], p["cs"], p["cst"], p["w"], p["ws"], p["wst"], p["y"])
        return {"c": s["y"], "codes": s["c"], "scales": s["cs"]}
    return s["y"]


# ------------------------------------------------------------------ what a pass cannot do without
def _mx(n, k, sb=1):
    return n * k // 2 + n * k // 32 * sb


def work(case):
    op = case["op"]
    if op == "gemv":
        n, k = case["n"], case["k"]
        return {"bytes": _mx(n, k, 4 if case["scale"] == "f32" else 1) + 4 * (n + k), "flops": 2 * n * k}
    if op == "mlp":
        d, f = case["dim"], case["ffn"]
        return {"bytes": _mx(2 * f, d) + _mx(d, f) + 10 * d, "flops": 6 * d * f}
    if op == "head":
        n, k = case["vocab"], case["dim"]
        return {"bytes": _mx(n, k) + 4 * (n + k), "flops": 2 * n * k}
    if op == "attn":
        nh, nkv, hd, seq = case["nh"], case["nkv"], case["hd"], case["seq"]
        return {"bytes": 2 * nkv * hd * seq * (2 if case["kv"] == "f16" else 4) + 8 * nh * hd, "flops": 4 * nh * hd * seq}
    if op == "attnp":
        nh, nkv, hd, n, p = case["nh"], case["nkv"], case["hd"], case["rows"], case["pos0"]
        return {"bytes": 4 * nkv * hd * (p + n) + 8 * n * nh * hd, "flops": 4 * nh * hd * (n * p + n * (n + 1) // 2)}
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _mx(n, k) + 2 * m * k + _mx(m, k) + 4 * m * n, "flops": 2 * m * n * k}
    d = dict(rfp4.PRESETS[case["model"]])
    dim, ffn, hd, nh, nkv, v = d["dim"], d["ffn"], d["head_dim"], d["n_heads"], d["n_kv_heads"], d["vocab"]
    layers = PREFILL_LAYERS if op == "prefill" else d["n_layers"]
    per = (nh + 2 * nkv) * hd * dim + nh * hd * dim + 3 * dim * ffn
    if op == "prefill":
        n, p = case["rows"], case["pos0"]
        att = n * p + n * (n + 1) // 2
        return {"bytes": layers * (_mx(per, 32) // 32 + 4 * nkv * hd * (p + n)) + _mx(v, dim) + 2 * n * dim + 4 * v,
                "flops": layers * (2 * n * per + 4 * nh * hd * att) + 2 * v * dim}
    steps, c = case["prompt"] + case["new"] - 1, case["ctx"]
    seqs = sum(c + i + 1 for i in range(steps))
    return {"bytes": steps * (layers * _mx(per, 32) // 32 + _mx(v, dim) + 4 * v + 2 * dim) + layers * 4 * nkv * hd * seqs,
            "flops": steps * 2 * (layers * per + v * dim) + layers * 4 * nh * hd * seqs}


def tolerance(case):
    # f32 arithmetic and f32 sums, in another order: measured against exact()
    # and stated with a factor of about four
    if case["op"] == "prefill":  # fp16 K and V rows (4e-6 from exact); the last row's logits, should an MXFP4 code of it move
        return {"rel": 1e-2, "max": 0.5}
    if case["op"] == "generate":  # new K and V rows are fp16: a rounding apart moves their last bit
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-5, "max": 1e-4}


# ------------------------------------------------------------------ the same in 64 bits
def _attend(q, k, v, pos0):
    """Causal attention in f64: q [rows][nh][hd], k and v [nkv][seq][hd]."""
    rows, nh, hd = q.shape
    nkv, seq = k.shape[0], k.shape[1]
    out = torch.empty_like(q)
    see = torch.arange(seq, device=q.device)[None] <= pos0 + torch.arange(rows, device=q.device)[:, None]
    for h in range(nh):
        kv = h * nkv // nh
        sc = (q[:, h] @ k[kv].t().contiguous()) / math.sqrt(hd)
        out[:, h] = torch.softmax(sc.masked_fill(~see, -math.inf), -1) @ v[kv]
    return out


def _silu(g):
    return g / (1 + torch.exp(-g))


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + float(np.float32(EPS))) * w.double()


def _rotate(x, pos, theta):
    """Rotate-half RoPE of x [rows][heads][hd] at positions pos [rows]."""
    hd = x.shape[-1]
    j = torch.arange(hd // 2, dtype=torch.float64, device=x.device)
    a = pos.double()[:, None] * (1.0 / torch.pow(torch.tensor(theta, dtype=torch.float64, device=x.device), 2 * j / hd))[None]
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    x0, x1 = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat((x0 * cos - x1 * sin, x1 * cos + x0 * sin), -1)


def _model(s):
    """The engine's weights as its prepare() made them: device views, and the norms and embeddings drawn again."""
    eng, d, seed = s["eng"], s["dims"], s["seed"]

    def proj(layer, i):
        c, sc, cb, sb = eng.weight(layer, i)
        return _view(eng, c, (cb,), "|u1"), _view(eng, sc, (sb,), "|u1")

    def half(stream, offset, n):
        t = torch.empty(n, dtype=torch.float16, device="cuda")
        torch.cuda.synchronize()
        rfp4.synth_f16(_stream(), seed, stream, 0.02, offset, n, t.data_ptr())
        torch.cuda.synchronize()
        return t

    return {"layers": [[proj(i, j) for j in range(7)] for i in range(d["n_layers"])], "head": proj(-1, 0),
            "norms": [(half(0xA0000 + 2 * i, 1.0, d["dim"]), half(0xA0000 + 2 * i + 1, 1.0, d["dim"])) for i in range(d["n_layers"])],
            "last": half(0xAFFFF, 1.0, d["dim"]), "embed": half(0xE0000, 0.0, d["vocab"] * d["dim"]).reshape(d["vocab"], d["dim"])}


def _layers(s, m, tokens, pos0, kc, vc, quantized):
    """The residual stream after every layer (f64), new K and V put into kc, vc as fp16.
    `quantized`: projection inputs as MXFP4 rows, as the batched prefill defines them."""
    d = s["dims"]
    nh, nkv, hd = d["n_heads"], d["n_kv_heads"], d["head_dim"]
    x = m["embed"][tokens].double()
    rows = x.shape[0]
    pos = pos0 + torch.arange(rows, device="cuda")
    inp = (lambda t: _dequantize(*_quantize(t), t.shape[-1])) if quantized else (lambda t: t)
    for i, w in enumerate(m["layers"]):
        h = inp(_norm(x, m["norms"][i][0]))
        q, k, v = (_matvec(*w[j], d["dim"], h).reshape(rows, -1, hd) for j in range(3))
        q, k = _rotate(q, pos, d["theta"]), _rotate(k, pos, d["theta"])
        kc[i, :, pos0:pos0 + rows] = k.transpose(0, 1).half()
        vc[i, :, pos0:pos0 + rows] = v.transpose(0, 1).half()
        a = _attend(q, kc[i, :, :pos0 + rows].double(), vc[i, :, :pos0 + rows].double(), pos0)
        x = x + _matvec(*w[3], nh * hd, inp(a.reshape(rows, nh * hd)))
        h = inp(_norm(x, m["norms"][i][1]))
        y = _silu(_matvec(*w[4], d["dim"], h)) * _matvec(*w[5], d["dim"], h)
        x = x + _matvec(*w[6], d["ffn"], inp(y))
    return x


def exact(case, seed):
    s = prepare(case, seed)
    torch.cuda.synchronize()
    op = case["op"]
    if op == "gemv":
        return _matvec(s["w"], s["ws"], case["k"], s["x"].double())
    if op == "mlp":
        d, f = case["dim"], case["ffn"]
        h = _norm(s["x"].double(), s["norm"])
        u = _matvec(s["gu"], s["gus"], d, h)
        return _matvec(s["dn"], s["dns"], f, _silu(u[:f]) * u[f:])
    if op == "head":
        return {"logits": _matvec(s["w"], s["ws"], case["dim"], s["x"].double()), "best": None}
    if op in ("attn", "attnp"):
        k, v = s["k"].double(), s["v"].double()
        if case.get("layout") == "token":
            k, v = k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous()
        q = s["q"].double()
        return _attend(q[None], k, v, case["seq"] - 1)[0] if op == "attn" else _attend(q, k, v, case["pos0"])
    if op == "gemm":
        x = _dequantize(*_quantize(s["x"].double()), case["k"])
        return {"c": _matvec(s["w"], s["ws"], case["k"], x), "codes": None, "scales": None}
    m, (kc, vc), ctx, d = _model(s), [t.clone() for t in s["all"]], s["ctx"], s["dims"]
    prompt = torch.from_numpy(s["prompt"].astype(np.int64)).cuda()
    if op == "prefill":
        _layers(s, m, prompt, ctx, kc, vc, True)
        steps = case["rows"]
        # logits: no such value. Where a rounding apart moves one MXFP4 code of
        # the last row (about one row in thirty) they are percents away
        logits, out = None, {"next": None}
    else:
        steps, tok = case["prompt"] + case["new"] - 1, None
        for i in range(steps):
            t = prompt[i:i + 1] if i < case["prompt"] else tok
            x = _layers(s, m, t, ctx + i, kc, vc, False)
            logits = _matvec(*m["head"], d["dim"], _norm(x[-1], m["last"]))
            tok = logits.argmax().reshape(1)
        out = {"ids": None}
    return {**out, "logits": logits, "k": kc[:, :, ctx:ctx + steps].double(), "v": vc[:, :, ctx:ctx + steps].double()}
