"""The work a user of this library has it do, as timed cases.

A case is a dict of plain values. `kind` says which entry points a pass goes through:

  gemv       one projection of one token: the int4-hier GEMV, or the f16 one of a lossless table
  attn       one token's attention layer: RoPE, the KV append and attention over the cache
  gemm       one projection of a chunk of tokens, int4-hier or f16
  attn_chunk a chunk's causal attention over the cache
  mlp        a chunk's MLP block: norm, gate|up with SwiGLU, down into the residual, next norm
  decode     the engine's captured decode step, the host choosing each token
  prefill    the engine's chunked prompt pass, up to the last token's logits

Shapes are those of the two models this repository is configured for (engine.QWEN05B and
engine.QWEN7B). `draw` spreads the same kinds over sizes between and around the listed ones.
"""
import ctypes as C
import math

import numpy as np
import torch

from whetstone_amd import engine as E
from whetstone_amd import ffi
from whetstone_amd import kernels as K

EPS = 1e-6
THETA = 1e6
MODELS = {"0.5B": E.QWEN05B, "7B": E.QWEN7B}


def listed():
    return [
        # The smallest call: one block's qkv projection of one token.
        dict(name="gemv_qkv_05b", kind="gemv", fmt="hier", inf=896, outf=1152, bias=True, accum=False),
        # The quantised head of one token, by itself.
        dict(name="gemv_head_05b", kind="gemv", fmt="hier", inf=896, outf=151936, bias=False,
             accum=False),
        # The head of a model converted with its f16 head kept (the converter's default).
        dict(name="gemv_head_fp16_05b", kind="gemv", fmt="fp16", inf=896, outf=151936, bias=False,
             accum=False),
        # One decode token's attention in a long conversation, at a position of no round number.
        dict(name="attn_7b", kind="attn", model="7B", pos=2177, max_seq=2312, qk_norm=False),
        # Verifying five speculated tokens: the widest projection of a small batch.
        dict(name="gemm_verify_7b", kind="gemm", fmt="hier", inf=3584, outf=37888, n=5, bias=False,
             accum=False),
        # One prefill chunk's down projection into the residual stream.
        dict(name="gemm_down_05b", kind="gemm", fmt="hier", inf=4864, outf=896, n=256, bias=False,
             accum=True),
        # A chunk of a long prompt attending to all that is before it; a ragged last chunk.
        dict(name="attn_chunk_7b", kind="attn_chunk", model="7B", n=243, pos0=1792, max_seq=2312),
        # The MLP of a whole prompt at once.
        dict(name="mlp_7b", kind="mlp", model="7B", n=1000),
        # Sixteen tokens of a conversation with the small model.
        dict(name="decode_05b", kind="decode", model="0.5B", ctx=600, steps=16, qk_norm=False,
             rescore=0),
        # Eight tokens of a long conversation with the large model.
        dict(name="decode_7b", kind="decode", model="7B", ctx=2080, steps=8, qk_norm=False, rescore=0),
        # A long prompt in full chunks (QK-norm, as its configuration has it).
        dict(name="prefill_05b", kind="prefill", model="0.5B", n=4096, qk_norm=True),
        # An ordinary prompt of no round length: three full chunks and a ragged one.
        dict(name="prefill_7b", kind="prefill", model="7B", n=1000, qk_norm=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """An in_features: a multiple of 64, as every width of the two models is."""
    return max(lo, min(hi, 64 * max(1, _log_int(rng, lo, hi) // 64)))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "attn", "gemm", "gemm", "attn_chunk", "mlp", "decode",
                       "prefill"])
    model = rng.choice(["0.5B", "7B"])
    if kind in ("gemv", "gemm"):
        fmt = "fp16" if rng.random() < 0.25 else "hier"
        inf = _width(rng, 896, 18944)
        outf = _log_int(rng, 512, min(152064, (1 << 28 if fmt == "hier" else 1 << 27) // inf))
        c = dict(kind=kind, fmt=fmt, inf=inf, outf=outf, bias=rng.random() < 0.5,
                 accum=rng.random() < 0.5)
        if kind == "gemm":
            c["n"] = _log_int(rng, 2, 256)
        return c
    if kind == "attn":
        max_seq = _log_int(rng, 256, 8192)
        return dict(kind=kind, model=model, pos=rng.randrange(max_seq), max_seq=max_seq,
                    qk_norm=rng.random() < 0.3)
    if kind == "attn_chunk":
        n, pos0 = _log_int(rng, 2, 256), rng.randrange(4096)
        return dict(kind=kind, model=model, n=n, pos0=pos0, max_seq=pos0 + n + rng.randrange(300))
    if kind == "mlp":
        return dict(kind=kind, model=model, n=_log_int(rng, 2, 1000))
    if kind == "decode":
        small = model == "0.5B"
        return dict(kind=kind, model=model, ctx=_log_int(rng, 32, 4000 if small else 2080),
                    steps=rng.randrange(1, 9), qk_norm=rng.random() < 0.5,
                    rescore=32 if small and rng.random() < 0.5 else 0)
    return dict(kind=kind, model=model, n=_log_int(rng, 2, 4096 if model == "0.5B" else 1000),
                qk_norm=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs


class Buffer(K.DeviceBuffer):
    """A torch tensor's memory as the library's device buffer; torch keeps it."""

    def __init__(self, t):
        self.t = t
        self.dtype = np.dtype(str(t.dtype).replace("torch.", ""))
        self.n = t.numel()
        self.ptr = C.c_void_p(t.data_ptr())

    def close(self):
        self.ptr = C.c_void_p()


def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(seed * 1009 + salt)


def _normal(g, shape, std=1.0, dtype=torch.float32, mean=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dtype)


def _hier(seed, salt, inf, outf):
    """N(0, 0.02) weights packed to int4-hier-g32, as (qw, si, sb)."""
    qw = torch.empty(outf * inf // 8, dtype=torch.int32, device="cuda")
    si = torch.empty(outf * inf // 32, dtype=torch.uint8, device="cuda")
    sb = torch.empty(outf, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ffi.call("wst_fixture_pack_hier", qw.data_ptr(), si.data_ptr(), sb.data_ptr(), inf, 0, outf,
             seed, 7000 + salt, 0.02)
    K.synchronize()
    return qw, si, sb


def _linear(qw, si, sb, inf, outf):
    bufs = [Buffer(qw), Buffer(si), Buffer(sb)]
    bufs[0].dtype = bufs[2].dtype = np.dtype(np.uint32)
    return K.QuantLinearHier(*bufs, inf, outf)


def _model(case, seed):
    cfg = dict(MODELS[case["model"]], qk_norm=int(case["qk_norm"]), rescore_k=case.get("rescore", 0))
    return E.Model(cfg, seed=seed)


def _ids(case, seed, n):
    return np.random.default_rng(seed + 17).integers(0, MODELS[case["model"]]["vocab"], n)


def _shape(case):
    m = MODELS[case["model"]]
    return m["n_q"], m["n_kv"], m["head_dim"]


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "seed": seed}
    if kind in ("gemv", "gemm"):
        inf, outf, n = case["inf"], case["outf"], case.get("n", 1)
        g = _gen(seed)
        if case["fmt"] == "hier":
            s["packed"] = _hier(seed, 0, inf, outf)
            s["lin"] = _linear(*s["packed"], inf, outf)
        else:
            s["w"] = _normal(g, (outf, inf), 0.02, torch.float16)
        s["x"] = _normal(g, (n * inf,), 1.0, torch.float16)
        s["bias"] = _normal(g, (outf,), 0.1, torch.float16) if case["bias"] else None
        s["y"] = (_normal(g, (n * outf,)) if case["accum"] else
                  torch.zeros(n * outf, device="cuda"))
        for k in ("w", "x", "bias", "y"):
            if s.get(k) is not None:
                s["b_" + k] = Buffer(s[k])
    elif kind in ("attn", "attn_chunk"):
        n_q, n_kv, hd = _shape(case)
        g = _gen(seed)
        n = case.get("n", 1)
        ms, seen = case["max_seq"], case["pos"] if kind == "attn" else case["pos0"] + n
        s["qkv"] = _normal(g, (n, (n_q + 2 * n_kv) * hd))
        for k in ("k", "v"):
            s[k] = torch.zeros(n_kv, ms, hd, dtype=torch.float16, device="cuda")
            s[k][:, :seen] = _normal(g, (n_kv, seen, hd), 1.0, torch.float16)
        s["out"] = torch.zeros(n, n_q * hd, dtype=torch.float16, device="cuda")
        if kind == "attn":
            s["rope"] = K.RopeTable(ms, hd, THETA)
            s["part"] = torch.zeros(max(1, ffi.lib().wst_attn_partial_floats(n_q, hd, ms)),
                                    device="cuda")
            s["pos"] = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
            s["qn"], s["kn"] = ((_normal(g, (hd,), 0.02, torch.float16, 1.0) for _ in range(2))
                                if case["qk_norm"] else (None, None))
    elif kind == "mlp":
        m = MODELS[case["model"]]
        H, I, n = m["hidden"], m["inter"], case["n"]
        g = _gen(seed)
        s["gu"], s["down"] = _hier(seed, 1, H, 2 * I), _hier(seed, 2, I, H)
        s["x"] = _normal(g, (n, H))
        s["n1"], s["n2"] = (_normal(g, (H,), 0.02, torch.float16, 1.0) for _ in range(2))
        s["h"] = torch.zeros(n, H, dtype=torch.float16, device="cuda")
        s["act"] = torch.zeros(n, I, dtype=torch.float16, device="cuda")
    elif kind == "decode":
        s["ids"] = _ids(case, seed, case["ctx"] + case["steps"])
        s["model"] = _model(case, seed)
        s["eng"] = E.Engine(s["model"], case["ctx"] + 256)
        s["eng"].prefill(s["ids"][:case["ctx"]])
        s["eng"].capture_graph()
    else:
        s["ids"] = _ids(case, seed, case["n"])
        s["model"] = _model(case, seed)
        s["eng"] = E.Engine(s["model"], case["n"] + 64)
    return s


# -------------------------------------------------------------------- a pass


def _ptr(t):
    return None if t is None else t.data_ptr()


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemv":
        if case["fmt"] == "hier":
            s["lin"].gemv_ex(s["b_x"], s.get("b_bias"), s["b_y"], case["accum"])
        else:
            K.gemv_fp16(s["b_w"], s["b_x"], s.get("b_bias"), s["b_y"], case["inf"], case["outf"],
                        case["accum"])
        return s["y"]
    if kind == "gemm":
        if case["fmt"] == "hier":
            s["lin"].gemm(s["b_x"], s.get("b_bias"), s["b_y"], case["n"], case["accum"])
        else:
            ffi.call("wst_gemm_fp16", _ptr(s["w"]), _ptr(s["x"]), _ptr(s["bias"]), _ptr(s["y"]),
                     case["inf"], case["outf"], case["n"], int(case["accum"]))
        return s["y"]
    if kind == "attn":
        n_q, n_kv, hd = _shape(case)
        ffi.call("wst_attn_decode_fused", _ptr(s["qkv"]), _ptr(s["k"]), _ptr(s["v"]),
                 s["rope"].cos.ptr, s["rope"].sin.ptr, _ptr(s["part"]), _ptr(s["out"]), n_q, n_kv,
                 hd, _ptr(s["pos"]), case["max_seq"], 1.0 / math.sqrt(hd), _ptr(s["qn"]),
                 _ptr(s["kn"]), EPS)
        return s["out"], s["k"], s["v"]
    if kind == "attn_chunk":
        n_q, n_kv, hd = _shape(case)
        ffi.call("wst_attn_chunk", _ptr(s["qkv"]), _ptr(s["k"]), _ptr(s["v"]), _ptr(s["out"]), n_q,
                 n_kv, hd, case["pos0"], case["n"], case["max_seq"], 1.0 / math.sqrt(hd))
        return s["out"]
    if kind == "mlp":
        m = MODELS[case["model"]]
        H, I, n = m["hidden"], m["inter"], case["n"]
        ffi.call("wst_rmsnorm_chunk", _ptr(s["x"]), _ptr(s["n1"]), _ptr(s["h"]), H, n, EPS)
        ffi.call("wst_gemm_hier_swiglu_chunk", *map(_ptr, s["gu"]), _ptr(s["h"]), _ptr(s["act"]), H,
                 I, n)
        ffi.call("wst_gemm_hier_norm_chunk", *map(_ptr, s["down"]), _ptr(s["act"]), None,
                 _ptr(s["x"]), I, H, n, 1, _ptr(s["n2"]), EPS, _ptr(s["h"]))
        return s["x"], s["h"], s["act"]
    eng = s["eng"]
    if kind == "decode":
        eng.rewind(case["ctx"])
        for t in s["ids"][case["ctx"]:]:
            eng.forward(int(t))
            eng.token()
        return eng.logits()
    eng.reset()
    eng.prefill(s["ids"])
    return eng.logits()


# ---------------------------------------------------------------- its cost


def _packed_bytes(inf, outf):
    return outf * (inf // 2 + inf // 32 + 4)


def _model_matrices(m):
    H, I, hd = m["hidden"], m["inter"], m["head_dim"]
    return [(H, (m["n_q"] + 2 * m["n_kv"]) * hd), (m["n_q"] * hd, H), (H, 2 * I), (I, H)]


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        inf, outf, n = case["inf"], case["outf"], case.get("n", 1)
        w = _packed_bytes(inf, outf) if case["fmt"] == "hier" else 2 * inf * outf
        return {"bytes": w + 2 * n * inf + (8 if case["accum"] else 4) * n * outf +
                (2 * outf if case["bias"] else 0), "flops": 2 * n * inf * outf}
    if kind in ("attn", "attn_chunk"):
        n_q, n_kv, hd = _shape(case)
        n, pos0 = (1, case["pos"]) if kind == "attn" else (case["n"], case["pos0"])
        kv = 4 * n_kv * hd * (pos0 + (n if kind == "attn_chunk" else 1))
        return {"bytes": kv + 4 * n * (n_q + (2 * n_kv if kind == "attn" else 0)) * hd +
                2 * n * n_q * hd,
                "flops": 4 * n_q * hd * (n * pos0 + n * (n + 1) // 2)}
    m = MODELS[case["model"]]
    H, I, hd = m["hidden"], m["inter"], m["head_dim"]
    if kind == "mlp":
        n = case["n"]
        return {"bytes": _packed_bytes(H, 2 * I) + _packed_bytes(I, H) + 10 * n * H + 2 * n * I,
                "flops": 6 * n * H * I}
    layers, head = _model_matrices(m), (H, m["vocab"])
    weights = m["n_layers"] * sum(_packed_bytes(*x) for x in layers) + _packed_bytes(*head)
    macs = m["n_layers"] * sum(a * b for a, b in layers)
    row = 4 * m["n_layers"] * m["n_kv"] * hd  # a cached position's bytes
    if kind == "decode":
        k, ctx = case["steps"], case["ctx"]
        seen = k * ctx + k * (k + 1) // 2
        return {"bytes": k * weights + seen * row,
                "flops": 2 * k * (macs + head[0] * head[1]) + 4 * seen * m["n_layers"] * m["n_q"] * hd}
    n = case["n"]
    # the head: the last token's logits
    return {"bytes": weights + n * row,
            "flops": 2 * (n * macs + head[0] * head[1]) +
            4 * m["n_layers"] * m["n_q"] * hd * (n * (n + 1) // 2)}


def tolerance(case):
    """About four times the error that the path measures against 64 bits."""
    kind = case["kind"]
    if kind == "gemv":
        # f32 sums of f16 activations; the int4 form holds them in 14 bits a group (measured 2.7e-5)
        return {"rel": 1e-4 if case["fmt"] == "hier" else 2e-6}
    if kind == "gemm":
        # the int4 form multiplies weights rounded to f16 (measured 2.1e-4)
        return {"rel": 8e-4 if case["fmt"] == "hier" else 4e-6}
    if kind in ("attn", "attn_chunk"):
        return {"rel": 1.2e-3}  # an f16 output; a chunk's f16 softmax weights (measured 2.9e-4)
    if kind == "mlp":
        return {"rel": 2e-3}  # f16 activations between the products (measured 5.2e-4)
    return {"rel": 2e-2}  # f16 activations through all the layers (measured 1.5e-3 to 5.7e-3)


# -------------------------------------------------------- the same in 64 bits


def _dequant(packed, inf, rows=None):
    """Rows r0..r1 of a packed matrix in f64: q * (d * ls) - dmin * lm."""
    qw, si, sb = packed
    r0, r1 = rows or (0, sb.numel())
    n = r1 - r0
    q = qw.view(-1, inf // 8)[r0:r1]
    sh = torch.arange(0, 32, 4, device=q.device, dtype=torch.int32)
    nib = ((q.unsqueeze(-1) >> sh) & 15).reshape(n, inf // 32, 32).double()
    idx = si.view(-1, inf // 32)[r0:r1].int()
    dd = sb[r0:r1].view(torch.float16).view(n, 2).double()
    d, dmin = dd[:, 0], dd[:, 1]
    s = d[:, None] * (idx & 15).double()
    m = dmin[:, None] * (idx >> 4).double()
    return (nib * s[..., None] - m[..., None]).reshape(n, inf)


def _product(x, packed, inf, outf):
    """x [n][inf] f64 times the packed matrix's transpose."""
    step = max(1, (1 << 27) // inf)
    return torch.cat([x @ _dequant(packed, inf, (r, min(r + step, outf))).T
                      for r in range(0, outf, step)], 1)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rotate(x, pos):
    """x [n][heads][hd] at positions pos [n]: the half rotation."""
    half = x.shape[-1] // 2
    f = THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    a = pos.double()[:, None] * f
    c, s = a.cos()[:, None], a.sin()[:, None]
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)


def _attend(q, k, v, pos0):
    """q [n][n_q][hd] at pos0 .. over k, v [n_kv][seq][hd]: causal softmax attention."""
    n, n_q, hd = q.shape
    n_kv, seq = k.shape[0], k.shape[1]
    mask = (torch.arange(seq, device=q.device)[None, :] >
            pos0 + torch.arange(n, device=q.device)[:, None])
    out = torch.empty_like(q)
    for h in range(n_q):
        kv = h // (n_q // n_kv)
        p = (q[:, h] @ k[kv].T / math.sqrt(hd)).masked_fill(mask, -math.inf).softmax(-1)
        out[:, h] = p @ v[kv]
    return out


def _fetch(model, name):
    """A packed matrix of the model as torch tensors, with its in and out features."""
    qw, si, sb, inf, outf = model.tensor(name)
    got = [torch.empty(n, dtype=t, device="cuda")
           for n, t in ((inf * outf // 8, torch.int32), (inf * outf // 32, torch.uint8),
                        (outf, torch.int32))]
    torch.cuda.synchronize()
    for t, p in zip(got, (qw, si, sb)):
        ffi.call("wst_memcpy_d2d", t.data_ptr(), p, t.numel() * t.element_size())
    K.synchronize()
    return got, inf, outf


def _vector(model, name):
    return torch.from_numpy(model.vector_host(name).view(np.float16)).cuda().double()


def _forward(model, ids, rescore):
    """The last token's logits of the whole sequence."""
    c = model.cfg
    n_q, n_kv, hd, I = c["n_q"], c["n_kv"], c["head_dim"], c["inter"]
    ids = torch.from_numpy(np.asarray(ids)).cuda()
    n = ids.numel()
    pos = torch.arange(n, device="cuda")
    table, H, V = _fetch(model, "embed")
    rows = ids.unique()
    x = _dequant([table[0].view(V, -1)[rows].reshape(-1), table[1].view(V, -1)[rows].reshape(-1),
                  table[2][rows]], H)[torch.searchsorted(rows, ids)]
    for l in range(c["n_layers"]):
        qkv = _product(_norm(x, _vector(model, f"L{l}.in_norm")), *_fetch(model, f"L{l}.qkv"))
        if c["qkv_bias"]:
            qkv = qkv + _vector(model, f"L{l}.qkv_bias")
        qkv = qkv.view(n, n_q + 2 * n_kv, hd)
        q, k, v = qkv[:, :n_q], qkv[:, n_q:n_q + n_kv], qkv[:, n_q + n_kv:]
        if c["qk_norm"]:
            q, k = _norm(q, _vector(model, f"L{l}.q_norm")), _norm(k, _vector(model, f"L{l}.k_norm"))
        a = _attend(_rotate(q, pos), _rotate(k, pos).transpose(0, 1), v.transpose(0, 1), 0)
        x = x + _product(a.reshape(n, n_q * hd), *_fetch(model, f"L{l}.o"))
        gu = _product(_norm(x, _vector(model, f"L{l}.post_norm")), *_fetch(model, f"L{l}.gate_up"))
        x = x + _product(torch.nn.functional.silu(gu[:, :I]) * gu[:, I:],
                         *_fetch(model, f"L{l}.down"))
    h = _norm(x[-1:], _vector(model, "final_norm"))
    logits = _product(h, *_fetch(model, "lm_head"))[0]
    if rescore:
        # the f16 copy of the head recomputes the logits within the smallest 2^c / 64 nats of the
        # maximum that holds the k largest
        gaps = [2.0 ** r / 64 for r in range(12)]
        counts = [int((logits >= logits.max() - g).sum()) for g in gaps]
        r = next((i for i, k in enumerate(counts) if k >= rescore), 11)
        while r > 0 and counts[r] > 16 * rescore:
            r -= 1
        full = torch.from_numpy(model.vector_host("rescore").view(np.float16)).cuda().view(V, H)
        pick = logits >= logits.max() - gaps[r]
        logits[pick] = full[pick].double() @ h[0]
    return logits


def exact(case, seed):
    s = prepare(case, seed)
    torch.cuda.synchronize()
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        x = s["x"].double().view(-1, case["inf"])
        y = (_product(x, s["packed"], case["inf"], case["outf"]) if case["fmt"] == "hier" else
             torch.cat([x @ w.double().T for w in s["w"].split((1 << 27) // case["inf"])], 1))
        if case["bias"]:
            y = y + s["bias"].double()
        return y.reshape(-1) + s["y"].double() if case["accum"] else y.reshape(-1)
    if kind == "attn":
        n_q, n_kv, hd = _shape(case)
        p = case["pos"]
        rows = s["qkv"].double().view(1, -1, hd)
        q, kn, vn = rows[:, :n_q], rows[:, n_q:n_q + n_kv], rows[:, n_q + n_kv:]
        if case["qk_norm"]:
            q, kn = _norm(q, s["qn"].double()), _norm(kn, s["kn"].double())
        at = torch.tensor([p], device="cuda")
        k, v = s["k"].double(), s["v"].double()
        k[:, p], v[:, p] = _rotate(kn, at)[0], vn[0]
        out = _attend(_rotate(q, at), k[:, :p + 1], v[:, :p + 1], p)
        return out.view(1, -1), k, v
    if kind == "attn_chunk":
        n_q, n_kv, hd = _shape(case)
        seen = case["pos0"] + case["n"]
        q = s["qkv"].double().view(case["n"], -1, hd)[:, :n_q]
        return _attend(q, s["k"][:, :seen].double(), s["v"][:, :seen].double(),
                       case["pos0"]).reshape(case["n"], -1)
    if kind == "mlp":
        m = MODELS[case["model"]]
        H, I = m["hidden"], m["inter"]
        x = s["x"].double()
        gu = _product(_norm(x, s["n1"].double()), s["gu"], H, 2 * I)
        act = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
        x = x + _product(act, s["down"], I, H)
        return x, _norm(x, s["n2"].double()), act
    return _forward(s["model"], s["ids"], case.get("rescore", 0)).cpu().numpy()
