"""Weights that a route may not round to 16 bits: beyond the 16-bit copy's size limit, and under f32 results of the f32 GEMV."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers

pytestmark = pytest.mark.gpu

# One rounding of the result, 2^-11 over sqrt(3) in the 2-norm; a rounding of the weights would add as much again (factor 1.41)
TOL_F16 = 2.0 ** -11 / 3 ** 0.5 * 1.1


@pytest.mark.parametrize("m,n,bs", [(33, 2100, 64), (70, 2100, 64), (100, 2100, 64), (17, 2100, 32), (24, 2100, 128), (32, 2100, 64), (24, 15000, 32), (100, 15000, 32)])
def test_eight_bit_weights_beyond_the_limit_stream_in_row_blocks(port, m, n, bs):
    ep = E.RocmExecutionProvider(0, {"dense_gemm_max_mb": "1"})
    k = 1024
    b, s, zp = synth.make_weights_bits(n, k, bs, 8, m, zero_points=True, scale_lo=0.002, scale_hi=0.004, scale_dtype=E.F16)
    a = synth.make_activation(m, k, m, E.F16)
    bias = np.random.default_rng(m).standard_normal((m, n)).astype(np.float16)
    want = port.matmul_f64_bits(synth.to_f32(a, E.F16), b, synth.to_f32(s, E.F16), zp, n, k, bs, 8)
    y, variant = E.matmul_nbits(ep, a, E.F16, b, s, E.F16, zp, n, k, bs, bias=bias, bias_dtype=E.F16, bits=8)
    assert variant == "decode_mfma_packed8"
    assert helpers.rel_l2(synth.to_f32(y, E.F16), want + bias.astype(np.float64)) <= TOL_F16
    y, variant = E.matmul_nbits(ep, a, E.F16, b, s, E.F16, zp, n, k, bs, bits=8, y_dtype=E.F32)
    assert variant == "gemv_nbits_f32" and helpers.rel_l2(y, want) <= 2e-6
    ep.shutdown()


@pytest.mark.parametrize("limit_mb,m,y_dt,expect", [
    ("1024", 2, E.F32, "gemv_nbits_f32"), ("1", 40, E.F32, "gemv_nbits_f32"), ("1", 100, E.F16, "act_order+decode_mfma_packed"), ("1024", 100, E.F16, "act_order+prefill_mfma_lds")])
def test_act_order(port, limit_mb, m, y_dt, expect):
    ep = E.RocmExecutionProvider(0, {"dense_gemm_max_mb": limit_mb})
    n, k, bs = 1100, 1024, 128
    b, s, zp = synth.make_weights(n, k, bs, m, zero_points=True, scale_lo=0.005, scale_hi=0.02, scale_dtype=E.F16)
    g = (np.arange(k) // bs).astype(np.int32)
    np.random.default_rng(m).shuffle(g)
    a = synth.make_activation(m, k, m, E.F16)
    y, variant = E.matmul_nbits(ep, a, E.F16, b, s, E.F16, zp, n, k, bs, g_idx=g, y_dtype=y_dt)
    assert variant == expect
    want = synth.to_f32(a, E.F16).astype(np.float64) @ port.dequantize_nk_gidx(b, synth.to_f32(s, E.F16), zp, g, n, k, bs, 4).astype(np.float64).T
    tol = 2e-6 if y_dt == E.F32 else TOL_F16 if limit_mb == "1" else TOL_F16 * 2 ** 0.5
    assert helpers.rel_l2(synth.to_f32(y, y_dt), want) <= tol
    ep.shutdown()


@pytest.mark.parametrize("bs,m", [(32, 40), (32, 100), (256, 40), (256, 100), (128, 24)])
def test_act_order_beyond_the_limit_keeps_its_weights(port, bs, m):
    """Whatever the block size: no route that rounds the weights takes the call."""
    ep = E.RocmExecutionProvider(0, {"dense_gemm_max_mb": "1"})
    n, k = 1100, 1024
    b, s, zp = synth.make_weights(n, k, bs, m, zero_points=True, scale_lo=0.005, scale_hi=0.02, scale_dtype=E.F16)
    g = (np.arange(k) // bs).astype(np.int32)
    np.random.default_rng(m).shuffle(g)
    a = synth.make_activation(m, k, m, E.F16)
    y, variant = E.matmul_nbits(ep, a, E.F16, b, s, E.F16, zp, n, k, bs, g_idx=g)
    want = synth.to_f32(a, E.F16).astype(np.float64) @ port.dequantize_nk_gidx(b, synth.to_f32(s, E.F16), zp, g, n, k, bs, 4).astype(np.float64).T
    # f32 sums round to another f16 value than the 64-bit ones only where these lie next to a boundary, weights rounded to f16 move every second result
    assert (np.asarray(y) != want.astype(np.float16)).mean() <= 0.02, variant
    ep.shutdown()


@pytest.mark.parametrize("bits,bs,m", [(4, 128, 24), (4, 128, 100), (4, 256, 40), (8, 64, 24), (8, 64, 100), (2, 64, 40)])
def test_act_order_with_unaligned_activations_keeps_its_weights(ep, port, bits, bs, m):
    """The 16-bit copy's kernel wants A on 16 bytes: calls whose A is not, which keep their weights, keep them sorted too (the gathered rows are aligned)."""
    n, k, dt = 1100, 1024, E.F16
    make = synth.make_weights if bits == 4 else lambda *args, **kw: synth.make_weights_bits(args[0], args[1], args[2], bits, args[3], **kw)
    b, s, zp = make(n, k, bs, m, zero_points=True, scale_lo=0.002, scale_hi=0.004, scale_dtype=dt)
    g = (np.arange(k) // bs).astype(np.int32)
    np.random.default_rng(m).shuffle(g)
    a = synth.make_activation(m, k, m, dt)
    ops = E.DeviceOperands(ep, b, s, dt, zp, n, k, bs, bits=bits, g_idx=g)
    ab, yb = ep.upload(np.concatenate([np.zeros(1, np.float16), a.ravel()])), ep.allocate(m * n * 2)
    try:
        views = ops.views(ab, dt, m)
        views[0] = E.TensorView(ab.ptr, dt, (m, k), byte_offset=2)
        ops.kernel.execute(views, [E.TensorView(yb.ptr, dt, (m, n))])
        got, variant = ep.download(yb, (m, n), np.float16), ops.kernel.last_variant()
    finally:
        ep.deallocate(ab)
        ep.deallocate(yb)
        ops.free()
    want = synth.to_f32(a, dt).astype(np.float64) @ port.dequantize_nk_gidx(b, synth.to_f32(s, dt), zp, g, n, k, bs, bits).astype(np.float64).T
    assert (got != want.astype(np.float16)).mean() <= 0.02, variant


@pytest.mark.parametrize("bits,m,first", [(8, 40, False), (8, 100, True), (4, 100, True), (4, 100, False)])
def test_calls_that_may_not_allocate_keep_their_weights(ep, port, bits, m, first):
    """execute_static has no 16-bit copy of 8-bit or act-order weights to multiply by: they stay in 32 bits there, also behind an execute of the node."""
    n, k, bs, dt = 1100, 1024, 128, E.F16
    make = synth.make_weights if bits == 4 else lambda *args, **kw: synth.make_weights_bits(args[0], args[1], args[2], 8, args[3], **kw)
    b, s, zp = make(n, k, bs, m, zero_points=True, scale_lo=0.002, scale_hi=0.004, scale_dtype=dt)
    g = (np.arange(k) // bs).astype(np.int32)
    if bits == 4:
        np.random.default_rng(m).shuffle(g)
    a = synth.make_activation(m, k, m, dt)
    ops = E.DeviceOperands(ep, b, s, dt, zp, n, k, bs, bits=bits, g_idx=g if bits == 4 else None)
    ab, yb = ep.upload(a), ep.allocate(m * n * 4)
    try:
        # (g_idx is range-checked once, by an execute)
        if first or bits == 4:
            ops.kernel.execute(ops.views(ab, dt, m if first else 1), [E.TensorView(yb.ptr, dt, (m if first else 1, n))])
        ops.kernel.execute_static(ops.views(ab, dt, m), [E.TensorView(yb.ptr, E.F32, (m, n))])
        got, variant = ep.download(yb, (m, n), np.float32), ops.kernel.last_variant()
    finally:
        ep.deallocate(ab)
        ep.deallocate(yb)
        ops.free()
    want = synth.to_f32(a, dt).astype(np.float64) @ port.dequantize_nk_gidx(b, synth.to_f32(s, dt), zp, g, n, k, bs, bits).astype(np.float64).T
    assert helpers.rel_l2(got, want) <= 2e-6, variant
