"""The chunk GEMMs over the shapes where their tiles end: int4-hier products
against float64 products of the dequantised weights.

Tolerance: the kernels multiply weights rounded to f16 (relative 2^-11) in
f32, so the error of an output is at most 2^-11 sum|w x| plus the f32 sums'
own error, far below it; twice that is allowed, and 1e-5 of the result for the
bias and the accumulate.
"""
import numpy as np
import pytest

from conftest import dev_f16, f16
from whetstone_amd import ffi

pytestmark = pytest.mark.gpu


def _operands(orc, wk, in_f, out_f, n, seed):
    p, _ = orc.quantize(orc.fixture_normal(seed, 1, in_f * out_f), in_f, out_f)
    lin = wk.QuantLinearHier.from_packed(p)
    xb = f16(orc, orc.fixture_normal(seed, 2, n * in_f, 1.0))
    bias = f16(orc, orc.fixture_normal(seed, 3, out_f, 0.3))
    w = orc.dequantize(p).astype(np.float64).reshape(out_f, in_f)
    x = xb.view(np.float16).astype(np.float64).reshape(n, in_f)
    return lin, w, x, dev_f16(wk, xb), bias.view(np.float16).astype(np.float64), dev_f16(wk, bias)


def _check(got, x, w, ref):
    bound = 2.0 * 2.0 ** -11 * (np.abs(x) @ np.abs(w).T) + 1e-5 * (1 + np.abs(ref))
    worst = float(np.max(np.abs(got - ref) / bound))
    assert worst <= 1.0, worst


# rows of an odd number of groups: the last 64-column step is half empty
@pytest.mark.parametrize("in_f,out_f,n,accum", [(1248, 4200, 32, False), (2080, 70, 5, True),
                                                (2144, 300, 130, False)])
def test_gemm_odd_group_counts(orc, wk, in_f, out_f, n, accum):
    print(f"gemm {in_f} -> {out_f}, {n} tokens", flush=True)
    lin, w, x, xd, bias, bd = _operands(orc, wk, in_f, out_f, n, 61)
    y0 = orc.fixture_normal(61, 4, n * out_f, 1.0)
    y = wk.DeviceBuffer.from_array(y0.copy())
    ffi.call("wst_gemm_int4_hier", lin.qw.ptr, lin.si.ptr, lin.sb.ptr, xd.ptr, bd.ptr, y.ptr, in_f,
             out_f, n, int(accum))
    ref = x @ w.T + bias
    if accum:
        ref = ref + y0.reshape(n, out_f)
    _check(y.numpy().astype(np.float64).reshape(n, out_f), x, w, ref)


# rows of 128-column steps: one step, an odd and an even count of them; one
# row, a row tile's edge and one past it; one token, a token tile's edge and one
# past it; K split (long rows) with and without the accumulate
@pytest.mark.parametrize("in_f,out_f,n,accum", [(128, 1, 1, False), (256, 256, 128, True),
                                                (384, 257, 129, False), (896, 127, 127, True),
                                                (1152, 130, 70, False), (4864, 896, 256, True),
                                                (3584, 1056, 1000, False), (9216, 33, 200, True),
                                                # rows that end in half a step: a step and a half, split
                                                # and unsplit, each token tile
                                                (192, 1, 1, False), (192, 300, 33, True),
                                                (960, 257, 65, False), (4928, 96, 7, True),
                                                (1216, 9000, 600, False)])
def test_gemm_step_rows(orc, wk, in_f, out_f, n, accum):
    print(f"gemm {in_f} -> {out_f}, {n} tokens", flush=True)
    lin, w, x, xd, bias, bd = _operands(orc, wk, in_f, out_f, n, 62)
    y0 = orc.fixture_normal(62, 4, (n + 1) * out_f, 1.0)
    y = wk.DeviceBuffer.from_array(y0.copy())
    ffi.call("wst_gemm_int4_hier", lin.qw.ptr, lin.si.ptr, lin.sb.ptr, xd.ptr, bd.ptr, y.ptr, in_f,
             out_f, n, int(accum))
    got = y.numpy().astype(np.float64).reshape(n + 1, out_f)
    ref = x @ w.T + bias
    if accum:
        ref = ref + y0.reshape(n + 1, out_f)[:n]
    _check(got[:n], x, w, ref)
    assert np.array_equal(got[n], y0.reshape(n + 1, out_f)[n])  # nothing past the last token


def _off_a_word(wk, lin):
    """The index bytes at an odd address: the register tiles refuse them."""
    si = lin.si.numpy()
    return wk.DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.uint8), si]))


# the wide LDS tiles, which take what the register tiles refuse: index bytes off
# a word (off 1) and rows of one 64-column step (off 0). 256-token tiles split and
# not, 128-token tiles split and not, the last tile ragged in both directions,
# fewer steps than the kernel's four in flight
@pytest.mark.parametrize("in_f,out_f,n,accum,off", [(2112, 130, 37, True, 1), (1536, 8260, 100, False, 1),
                                                    (2048, 300, 300, False, 1), (2048, 2100, 520, True, 1),
                                                    (128, 4100, 300, False, 1), (64, 4100, 70, True, 0)])
def test_gemm_wide_tiles(orc, wk, in_f, out_f, n, accum, off):
    print(f"wide tiles {in_f} -> {out_f}, {n} tokens", flush=True)
    lin, w, x, xd, bias, bd = _operands(orc, wk, in_f, out_f, n, 69)
    si = _off_a_word(wk, lin)
    y0 = orc.fixture_normal(69, 4, (n + 1) * out_f, 1.0)
    y = wk.DeviceBuffer.from_array(y0.copy())
    ffi.call("wst_gemm_int4_hier", lin.qw.ptr, si.at(1) if off else lin.si.ptr, lin.sb.ptr, xd.ptr,
             bd.ptr, y.ptr, in_f, out_f, n, int(accum))
    got = y.numpy().astype(np.float64).reshape(n + 1, out_f)
    y0 = y0.reshape(n + 1, out_f)
    ref = x @ w.T + bias + (y0[:n] if accum else 0.0)
    _check(got[:n], x, w, ref)
    assert np.array_equal(got[n], y0[n])  # nothing past the last token


@pytest.mark.parametrize("in_f,inter,n,off", [(2048, 70, 300, 1), (896, 4099, 40, 1), (64, 2050, 257, 0)])
def test_gemm_swiglu_wide_tiles(orc, wk, in_f, inter, n, off):
    print(f"wide gate|up {in_f} -> {inter}, {n} tokens", flush=True)
    lin, w, x, xd, _, _ = _operands(orc, wk, in_f, 2 * inter, n, 70)
    si = _off_a_word(wk, lin)
    act = wk.DeviceBuffer.from_array(np.full((n + 1) * inter, 7.0, np.float16))
    ffi.call("wst_gemm_hier_swiglu_chunk", lin.qw.ptr, si.at(1) if off else lin.si.ptr, lin.sb.ptr,
             xd.ptr, act.ptr, in_f, inter, n)
    _check_swiglu(act.numpy().astype(np.float64).reshape(n + 1, inter), x, w, inter, n)


@pytest.mark.parametrize("in_f,inter,n", [(128, 1, 1), (256, 128, 128), (896, 161, 129),
                                          (384, 700, 300), (192, 100, 40), (320, 4000, 300)])
def test_gemm_swiglu_step_rows(orc, wk, in_f, inter, n):
    print(f"gate|up {in_f} -> {inter}, {n} tokens", flush=True)
    lin, w, x, xd, _, _ = _operands(orc, wk, in_f, 2 * inter, n, 63)
    act = wk.DeviceBuffer.from_array(np.full((n + 1) * inter, 7.0, np.float16))
    ffi.call("wst_gemm_hier_swiglu_chunk", lin.qw.ptr, lin.si.ptr, lin.sb.ptr, xd.ptr, act.ptr,
             in_f, inter, n)
    _check_swiglu(act.numpy().astype(np.float64).reshape(n + 1, inter), x, w, inter, n)


def _check_swiglu(got, x, w, inter, n):
    gu = x @ w.T
    err = 2.0 * 2.0 ** -11 * (np.abs(x) @ np.abs(w).T) + 1e-5
    g, u = gu[:, :inter], gu[:, inter:]
    silu = g / (1 + np.exp(-g))
    # silu' <= 1.1: the products' errors through silu(g) * u, and the f16 store
    bound = 1.1 * err[:, :inter] * np.abs(u) + np.abs(silu) * err[:, inter:]
    bound = 1.1 * bound + 2.0 ** -10 * np.abs(silu * u) + 1e-4
    worst = float(np.max(np.abs(got[:n] - silu * u) / bound))
    assert worst <= 1.0, worst
    assert np.all(got[n] == 7.0)


@pytest.mark.parametrize("in_f,n_q,n_kv,hd,pos0,n,qk", [(3584, 28, 4, 128, 5, 2049, False),
                                                        (896, 14, 2, 64, 3, 4000, True),
                                                        (192, 14, 2, 64, 0, 20, True),
                                                        (192, 14, 2, 64, 7, 130, False),
                                                        (256, 8, 2, 128, 0, 20, False),
                                                        (256, 28, 4, 128, 1, 700, False)])
def test_gemm_rope_epilogue_equals_gemm_then_rope_cache(orc, wk, in_f, n_q, n_kv, hd, pos0, n, qk):
    """Shapes whose projection runs unsplit, so that the tiles' epilogue rotates
    and appends: against the GEMM then wst_rope_cache_chunk, bit for bit, at
    both head sizes and each token tile (the last one ragged, the cache ending
    at the last token)."""
    print(f"rope epilogue hd {hd}, {n} tokens", flush=True)
    out_f, max_seq = (n_q + 2 * n_kv) * hd, pos0 + n
    lin = wk.QuantLinearHier(*(wk.DeviceBuffer(k, t) for k, t in (
        (out_f * in_f // 8, np.uint32), (out_f * in_f // 32, np.uint8), (out_f, np.uint32))),
        in_f, out_f)
    ffi.call("wst_fixture_pack_hier", lin.qw.ptr, lin.si.ptr, lin.sb.ptr, in_f, 0, out_f, 64, 1, 0.02)
    x = dev_f16(wk, f16(orc, orc.fixture_normal(64, 2, n * in_f, 1.0)))
    b = dev_f16(wk, f16(orc, orc.fixture_normal(64, 3, out_f, 0.3)))
    norms = [dev_f16(wk, f16(orc, 1.0 + orc.fixture_normal(64, 4 + i, hd, 0.1))) if qk else None
             for i in range(2)]
    qn, kn = (v.ptr if v is not None else None for v in norms)
    c, s = orc.rope_table(max_seq, hd, 1e6)
    cd, sd = wk.DeviceBuffer.from_array(c), wk.DeviceBuffer.from_array(s)
    out = []
    for fused in (False, True):
        qkv = wk.DeviceBuffer(n * out_f, np.float32)
        k, v = (wk.DeviceBuffer(n_kv * max_seq * hd, np.float16) for _ in range(2))
        if fused:
            ffi.call("wst_gemm_hier_rope_chunk", lin.qw.ptr, lin.si.ptr, lin.sb.ptr, x.ptr, b.ptr,
                     qkv.ptr, in_f, k.ptr, v.ptr, cd.ptr, sd.ptr, n_q, n_kv, hd, pos0, n, max_seq,
                     qn, kn, 1e-6)
        else:
            ffi.call("wst_gemm_int4_hier", lin.qw.ptr, lin.si.ptr, lin.sb.ptr, x.ptr, b.ptr,
                     qkv.ptr, in_f, out_f, n, 0)
            ffi.call("wst_rope_cache_chunk", qkv.ptr, k.ptr, v.ptr, cd.ptr, sd.ptr, n_q, n_kv, hd,
                     pos0, n, max_seq, qn, kn, 1e-6)
        out.append([t.numpy() for t in (qkv, k, v)])
    for a, e in zip(*out):
        assert np.array_equal(a.view(np.uint8), e.view(np.uint8))


@pytest.mark.parametrize("in_f,out_f,n,accum", [(128, 1, 1, False), (192, 130, 33, True),
                                                (896, 257, 65, False), (960, 1000, 256, True),
                                                (4864, 96, 7, True), (256, 9000, 600, False),
                                                # on the register tiles
                                                (960, 9000, 600, True), (192, 9001, 1100, False),
                                                (3136, 4100, 40, True)])
def test_gemm_fp16_step_rows(orc, wk, in_f, out_f, n, accum):
    """f16 weights over the same edges: the operands are exact, so only the f32
    sums differ from float64 (at most in_f + 16 additions of relative 2^-24)."""
    print(f"f16 gemm {in_f} -> {out_f}, {n} tokens", flush=True)
    wb = f16(orc, orc.fixture_normal(65, 1, in_f * out_f, 0.05))
    xb = f16(orc, orc.fixture_normal(65, 2, n * in_f, 1.0))
    bb = f16(orc, orc.fixture_normal(65, 3, out_f, 0.3))
    y0 = orc.fixture_normal(65, 4, (n + 1) * out_f, 1.0)
    y = wk.DeviceBuffer.from_array(y0.copy())
    wd, xd, bd = dev_f16(wk, wb), dev_f16(wk, xb), dev_f16(wk, bb)
    ffi.call("wst_gemm_fp16", wd.ptr, xd.ptr, bd.ptr, y.ptr, in_f, out_f, n, int(accum))
    w = wb.view(np.float16).astype(np.float64).reshape(out_f, in_f)
    x = xb.view(np.float16).astype(np.float64).reshape(n, in_f)
    ref = x @ w.T + bb.view(np.float16).astype(np.float64)
    if accum:
        ref = ref + y0.reshape(n + 1, out_f)[:n]
    got = y.numpy().astype(np.float64).reshape(n + 1, out_f)
    bound = (in_f + 16) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + np.abs(ref) + 1)
    assert float(np.max(np.abs(got[:n] - ref) / bound)) <= 1.0
    assert np.array_equal(got[n], y0.reshape(n + 1, out_f)[n])


# rows that end in half a step: each column meets its own weight once, so an
# infinite x gives the sign's infinity and leaves the other tokens alone
@pytest.mark.parametrize("kind,in_f,out_f,n", [("hier", 192, 40, 70), ("hier", 960, 257, 130),
                                               ("fp16", 960, 9000, 600),
                                               ("fp16", 3136, 4100, 40)])
def test_gemm_half_step_rows_infinite_x(orc, wk, kind, in_f, out_f, n):
    print(f"{kind} gemm {in_f} -> {out_f}, {n} tokens, Inf in x", flush=True)
    rng = np.random.default_rng(66)
    x = rng.standard_normal((n, in_f)).astype(np.float16)
    y = wk.DeviceBuffer(n * out_f, np.float32)
    if kind == "hier":
        p, _ = orc.quantize(orc.fixture_normal(66, 1, in_f * out_f), in_f, out_f)
        lin = wk.QuantLinearHier.from_packed(p)
        w = orc.dequantize(p).astype(np.float16).astype(np.float64).reshape(out_f, in_f)
    else:
        wb = f16(orc, orc.fixture_normal(66, 1, in_f * out_f, 0.05))
        wd = dev_f16(wk, wb)
        w = wb.view(np.float16).astype(np.float64).reshape(out_f, in_f)
    tok, col = n // 2, in_f - 1 - n % 64
    x[tok, col] = np.inf
    xd = dev_f16(wk, x.view(np.uint16).reshape(-1))
    if kind == "hier":
        ffi.call("wst_gemm_int4_hier", lin.qw.ptr, lin.si.ptr, lin.sb.ptr, xd.ptr, None, y.ptr,
                 in_f, out_f, n, 0)
    else:
        ffi.call("wst_gemm_fp16", wd.ptr, xd.ptr, None, y.ptr, in_f, out_f, n, 0)
    got = y.numpy().reshape(n, out_f)
    clear = np.abs(w[:, col]) > 1e-4  # (a weight that rounds to zero times Inf is NaN)
    assert clear.sum() > out_f // 2
    assert np.array_equal(got[tok][clear], np.sign(w[clear, col]).astype(np.float32) * np.inf)
    assert np.all(np.isfinite(np.delete(got, tok, axis=0)))


# a row whose scale is infinite stays infinite: the columns past its end add no
# 0 * Inf (rows of half a step, of a whole number of steps, of odd group counts)
@pytest.mark.parametrize("in_f,n", [(192, 5), (960, 70), (896, 70), (1248, 70)])
def test_gemm_infinite_scale_stays_infinite(wk, in_f, n):
    print(f"gemm {in_f} columns, an infinite scale, {n} tokens", flush=True)
    out_f, bad = 130, 129
    qw = wk.DeviceBuffer.from_array(np.full(out_f * in_f // 8, 0x77777777, np.uint32))
    si = wk.DeviceBuffer.from_array(np.full(out_f * in_f // 32, 0x11, np.uint8))
    d = np.full(out_f, 0x2000, np.uint32)  # d 2^-7, dmin 0
    d[bad] = 0x7C00
    sb = wk.DeviceBuffer.from_array(d)
    x = dev_f16(wk, np.full(n * in_f, 0x3C00, np.uint16))
    y = wk.DeviceBuffer(n * out_f, np.float32)
    ffi.call("wst_gemm_int4_hier", qw.ptr, si.ptr, sb.ptr, x.ptr, None, y.ptr, in_f, out_f, n, 0)
    got = y.numpy().reshape(n, out_f)
    assert np.all(got[:, bad] == np.inf)
    assert np.all(np.delete(got, bad, axis=1) == 7 * in_f / 128)  # (exact in f32)


@pytest.mark.parametrize("hd,n_q,n_kv,pos0,n", [(64, 14, 2, 1702, 37), (128, 28, 4, 900, 37),
                                                (128, 28, 4, 5, 37)])
def test_attn_chunk_output_between_words(orc, wk, hd, n_q, n_kv, pos0, n):
    """An output that starts on an odd f16: the same values as an aligned one,
    and nothing beside them."""
    qkv = wk.DeviceBuffer.from_array(orc.fixture_normal(67, 1, n * (n_q + 2 * n_kv) * hd, 1.0))
    k, v = (dev_f16(wk, f16(orc, orc.fixture_normal(67, i, n_kv * 1800 * hd, 1.0))) for i in (2, 3))
    res = []
    for shift in (0, 1):
        out = wk.DeviceBuffer.from_array(np.full(n * n_q * hd + 2, 7.0, np.float16))
        ffi.call("wst_attn_chunk", qkv.ptr, k.ptr, v.ptr, out.at(shift), n_q, n_kv, hd, pos0,
                 n, 1800, hd ** -0.5)
        o = out.numpy()
        assert np.all(o[:shift] == 7.0) and np.all(o[n * n_q * hd + shift:] == 7.0)
        res.append(o[shift:n * n_q * hd + shift].view(np.uint16))
    assert np.array_equal(*res)


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("hd,n_q,n_kv,pos0,n", [(128, 28, 4, 645, 7), (128, 28, 4, 652, 7),
                                                (128, 8, 8, 1001, 256), (128, 4, 2, 0, 131),
                                                (128, 4, 4, 0, 1), (64, 14, 2, 300, 33),
                                                (64, 8, 8, 1687, 6), (64, 8, 8, 1688, 6),
                                                (64, 14, 2, 677, 511), (64, 14, 2, 0, 512)])
def test_attn_chunk_positions(orc, wk, hd, n_q, n_kv, pos0, n, planned):
    """Both kernels on both sides of the rule that picks one (planned calls stay
    on the shared-tile kernel), a wave's last tiles empty or partly attended,
    NaN past the attended end, against float64.

    Bound: P is rounded to f16 (2^-11 of each weight), the scores keep 22 bits
    of |q||k| (scores of order 1: 2^-13 allowed), the output is rounded to f16."""
    print(f"chunk attention hd {hd}, {n} tokens at {pos0}", flush=True)
    max_seq, g = pos0 + n + 40, n_q // n_kv
    rng = np.random.default_rng(68)
    qkv = rng.standard_normal((n, n_q + 2 * n_kv, hd)).astype(np.float32)
    k, v = (rng.standard_normal((n_kv, max_seq, hd)).astype(np.float16) for _ in range(2))
    k[:, pos0 + n:] = np.nan
    v[:, pos0 + n:] = np.nan
    kd, vd = (dev_f16(wk, t.view(np.uint16).reshape(-1)) for t in (k, v))
    qd = wk.DeviceBuffer.from_array(qkv.reshape(-1))
    out = wk.DeviceBuffer(n * n_q * hd, np.float16)
    ffi.call("wst_attn_chunks", qd.ptr, kd.ptr, vd.ptr, out.ptr, n_q, n_kv, hd, pos0, n, max_seq,
             hd ** -0.5, n if planned else 0)
    got = out.numpy().astype(np.float64).reshape(n, n_q, hd)
    for h in range(n_q):
        kh, vh = (t[h // g, :pos0 + n].astype(np.float64) for t in (k, v))
        s = qkv[:, h].astype(np.float64) @ kh.T * hd ** -0.5
        s[np.arange(pos0 + n)[None] > pos0 + np.arange(n)[:, None]] = -np.inf
        p = np.exp(s - s.max(axis=1, keepdims=True))
        p /= p.sum(axis=1, keepdims=True)
        ref, mag = p @ vh, p @ np.abs(vh)
        bound = (2.0 ** -11 + 2.0 ** -13) * mag + 2.0 ** -11 * np.abs(ref) + 2.0 ** -24
        worst = float(np.max(np.abs(got[:, h] - ref) / bound))
        assert worst <= 1.0, (h, worst)
