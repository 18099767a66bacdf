"""8-bit and act-order weights with 16-bit activations: sums as good as plain f32 sums of activation times (q - zp), and infinities, NaN and values
near the end of the range that come out as those sums give them."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers

pytestmark = pytest.mark.gpu

ONE_ROUNDING = {E.F16: 2.0 ** -11 / 3 ** 0.5 * 1.1, E.BF16: 2.0 ** -8 / 3 ** 0.5 * 1.1}      # of the result, in the 2-norm

# bits, type, block size, m, n, k - the row counts of every build, then the wide ones; n * k at least what streams a repacked copy
CASES = [
    (4, E.F16, 128, 1, 1200, 3584),
    (4, E.BF16, 32, 1, 700, 904),
    (4, E.BF16, 128, 4, 1200, 3584),
    (4, E.F16, 64, 7, 640, 2048),
    (4, E.BF16, 128, 16, 1200, 3584),
    (4, E.F16, 32, 16, 23000, 256),
    (4, E.BF16, 128, 12, 18448, 640),
    (4, E.F16, 64, 29, 14400, 448),
    (4, E.F16, 128, 16, 36890, 256),                    # grids that workgroups of more than eight waves spread over the CUs
    (4, E.BF16, 64, 5, 40010, 192),
    (4, E.BF16, 32, 9, 40010, 128),
    (8, E.BF16, 128, 4, 36890, 256),
    (8, E.F16, 32, 16, 40010, 128),
    (8, E.BF16, 64, 12, 60010, 192),                    # more columns than that
    (8, E.F16, 128, 1, 1200, 3584),
    (8, E.BF16, 32, 1, 4700, 904),
    (8, E.BF16, 128, 4, 1200, 3584),
    (8, E.F16, 64, 7, 640, 2048),
    (8, E.BF16, 128, 16, 1200, 3584),
    (8, E.F16, 32, 16, 23000, 256),
    (8, E.BF16, 128, 12, 18448, 640),
    (8, E.F16, 64, 29, 14400, 448),
]


def node(bits, dt, bs, m, n, k, scale, s_dt=None):
    """(b, scales, zp, g_idx or None, the groups in any case, a sample of the columns)"""
    make = synth.make_weights if bits == 4 else lambda *args, **kw: synth.make_weights_bits(args[0], args[1], args[2], 8, args[3], **kw)
    b, s, zp = make(n, k, bs, n + m, zero_points=True, scale_lo=scale, scale_hi=2 * scale, scale_dtype=s_dt or dt)
    g = (np.arange(k) // bs).astype(np.int32)
    if bits == 4:                                        # act-order: the groups' elements scattered over K
        np.random.default_rng(m).shuffle(g)
    cols = np.arange(n) if n <= 1200 else np.unique(np.concatenate([np.random.default_rng(n).integers(0, n, 1200), np.arange(n - 40, n)]))
    return b, s, zp, g if bits == 4 else None, g, cols


def weights64(port, b, s, zp, g, cols, k, bs, bits, dt):
    part = [np.ascontiguousarray(np.asarray(x).reshape(np.asarray(b).shape[0], -1)[cols]) for x in (b, synth.to_f32(s, dt), zp)]
    return port.dequantize_nk_gidx(part[0], part[1], part[2], g, len(cols), k, bs, bits).astype(np.float64)


@pytest.mark.parametrize("bits,dt,bs,m,n,k", CASES)
def test_results_round_like_plain_f32_sums(ep, port, bits, dt, bs, m, n, k):
    """Of K terms' f32 sum, sqrt(K) roundings of 2^-25 are left: 1.8e-6 of the terms' norm at K = 3584, which is the output's here. A result of
    size y rounds another way than the 64-bit sum where that lies so close to a boundary: 2 * 1.8e-6 / (unit / y), below 0.7 % of results with units of at
    least 2^-11 y (f16), of normal size, and an eighth of that in bf16. Sums that carry an offset of 2^10 with the weights show in 3 to 4 %."""
    b, s, zp, g, order, cols = node(bits, dt, bs, m, n, k, 0.004 if bits == 4 else 0.0004)
    a = synth.make_activation(m, k, m, dt)
    y, variant = E.matmul_nbits(ep, a, dt, b, s, dt, zp, n, k, bs, bits=bits, g_idx=g)
    got = np.asarray(y).view(np.uint16).reshape(m, n)[:, cols]
    want = synth.to_f32(a, dt).astype(np.float64) @ weights64(port, b, s, zp, order, cols, k, bs, bits, dt).T
    rounded = np.asarray(synth.to_dtype(want.astype(np.float32), dt)).view(np.uint16)
    size = np.abs(want) > 0.1 * np.sqrt((want ** 2).mean())
    assert (got != rounded)[size].mean() <= (7e-3 if dt == E.F16 else 9e-4), variant
    assert helpers.rel_l2(synth.to_f32(y, dt)[:, cols], want) <= ONE_ROUNDING[dt]


@pytest.mark.parametrize("bits,dt,bs,m,n,k", CASES)
def test_infinities_nan_and_the_largest_values(ep, port, bits, dt, bs, m, n, k):
    b, s, zp, g, order, cols = node(bits, dt, bs, m, n, k, 0.004 if bits == 4 else 0.0004)
    top = 65504.0 if dt == E.F16 else 3.3895313892515355e38
    w = weights64(port, b, s, zp, order, cols, k, bs, bits, dt)
    kinds = ["plus", "minus", "nan", "both", "top", "plus and top"]
    for first in range(0, len(kinds), m):                  # a kind a row, over as many calls as that takes
        a = synth.to_f32(synth.make_activation(m, k, first, dt), dt)
        row_kind = dict(enumerate(kinds[first:first + m]))
        for row, kind in row_kind.items():
            if kind.startswith("plus"):
                a[row, 5] = np.inf
            elif kind == "minus":
                a[row, k - 1] = -np.inf
            elif kind == "nan":
                a[row, 70] = np.nan
            elif kind == "both":
                a[row, 3], a[row, k - 60] = np.inf, -np.inf
            if kind.endswith("top"):
                a[row, 64:68] = top * np.array([1, -1, 1, 1])
        y, variant = E.matmul_nbits(ep, synth.to_dtype(a, dt), dt, b, s, dt, zp, n, k, bs, bits=bits, g_idx=g)
        got = synth.to_f32(y, dt).reshape(m, n)[:, cols].astype(np.float64)
        for row in range(m):
            kind = row_kind.get(row)
            with np.errstate(invalid="ignore", over="ignore"):
                want = (a[row].astype(np.float64) * w).sum(axis=1)
                if kind in (None, "top"):
                    fits = np.abs(want) < 0.99 * top       # what the result's type holds
                    assert fits.any() and helpers.rel_l2(got[row][fits] / (top if kind else 1.0), want[fits] / (top if kind else 1.0)) <= ONE_ROUNDING[dt], (row, kind, variant)
                else:
                    assert np.array_equal(got[row], want, equal_nan=True), (row, kind, variant)


@pytest.mark.parametrize("dt,bs,m,n,k", [(E.F16, 32, 1, 300, 904), (E.BF16, 128, 4, 300, 1024), (E.F16, 64, 16, 300, 1024), (E.BF16, 64, 8, 23000, 256), (E.BF16, 128, 31, 14400, 256)])
def test_act_order_with_f32_scales(ep, port, dt, bs, m, n, k):
    b, s, zp, g, order, cols = node(4, dt, bs, m, n, k, 0.004, E.F32)
    a = synth.to_f32(synth.make_activation(m, k, m, dt), dt)
    a[0, 5] = np.inf
    if m > 1 and dt == E.BF16:
        a[1, 64:68] = 3.3895313892515355e38 * np.array([1, -1, 1, 1])
    y, variant = E.matmul_nbits(ep, synth.to_dtype(a, dt), dt, b, s, E.F32, zp, n, k, bs, g_idx=g)
    assert variant == "act_order+decode_mfma_packed"
    got = synth.to_f32(y, dt).reshape(m, n)[:, cols].astype(np.float64)
    w = weights64(port, b, s, zp, order, cols, k, bs, 4, E.F32)
    for row in range(m):
        with np.errstate(invalid="ignore"):
            want = (a[row].astype(np.float64) * w).sum(axis=1)
        if row == 0:
            assert np.array_equal(got[row], want, equal_nan=True)
        else:
            assert helpers.rel_l2(got[row] / np.abs(a[row]).max(), want / np.abs(a[row]).max()) <= ONE_ROUNDING[dt], row
