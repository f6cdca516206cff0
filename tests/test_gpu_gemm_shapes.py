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
