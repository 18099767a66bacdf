"""f32 activations on the matrix cores (csrc/kernels/gemm_f32.hip): edges of its tiles, its split of K and its dispatch, against the oracle in double precision."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers

pytestmark = pytest.mark.gpu

# Products are exact (three bf16 parts of an activation times an integer of four bits and a sign) and every sum is an f32 sum: at most
# K + K / 32 roundings of 2^-24 on the way to an output. As independent errors they add up to sqrt(4864 * 33 / 32) * 2^-24 = 4.2e-6 of the
# terms' norm, which for these zero-mean operands is the output's norm.
TOL = 4.2e-6

CASES = [
    # s_dt, bs, zero points, m, n, k, bias, y type
    (E.F32, 32, False, 5, 128, 32, "none", E.F32),          # one run of K, one wave
    (E.F32, 32, True, 5, 129, 896, "column", E.F32),        # 16 x 16 tiles, a ragged last column tile
    (E.F32, 64, True, 17, 130, 900, "none", E.F32),         # ... a ragged last row tile and a partial last block
    (E.F16, 128, True, 63, 140, 4100, "row", E.F32),
    (E.F32, 256, False, 64, 128, 4864, "column", E.F16),
    (E.F32, 32, True, 65, 1100, 68, "none", E.F32),         # 32 x 32 tiles, fewer runs than waves
    (E.BF16, 32, True, 200, 900, 896, "row", E.BF16),
    (E.F32, 64, False, 300, 1000, 516, "column", E.F32),    # two column tiles per wave, the second one beyond N in the last workgroup
    (E.F16, 32, True, 513, 2017, 160, "none", E.F32),       # more workgroups than CUs: four waves
    (E.F32, 128, True, 8, 16416, 256, "none", E.F32),       # five to eight rows on a wide call: the streaming kernel keeps it
]


@pytest.mark.parametrize("s_dt,bs,zero_points,m,n,k,bias_kind,y_dt", CASES)
def test_matches_double_precision(ep, port, s_dt, bs, zero_points, m, n, k, bias_kind, y_dt):
    b, s, zp = synth.make_weights(n, k, bs, n + k, zero_points=zero_points, scale_lo=0.002, scale_hi=0.01, scale_dtype=s_dt)
    rng = np.random.default_rng(m)
    # magnitudes over 24 binary orders: all three parts of a value matter
    a = (synth.make_activation(m, k, n, E.F32).astype(np.float64) * np.exp2(rng.integers(-12, 12, (m, 1)))).astype(np.float32)
    bias = None if bias_kind == "none" else rng.standard_normal((m, n) if bias_kind == "row" else n).astype(np.float32)
    y, variant = E.matmul_nbits(ep, a, E.F32, b, s, s_dt, zp, n, k, bs, bias=bias, y_dtype=y_dt)
    assert variant == ("gemv_f32_valu" if (m, n) == (8, 16416) else "gemm_f32_mfma")
    want = port.matmul_f64(a, b, synth.to_f32(s, s_dt), zp, n, k, bs)
    if bias is not None:
        want = want + bias.astype(np.float64)
    got = synth.to_f32(y, y_dt).astype(np.float64)
    # a narrow result adds its own rounding, half a unit of 2^-10 (f16) or 2^-7 (bf16), to each value
    tol = TOL + {E.F32: 0.0, E.F16: 2.0 ** -11, E.BF16: 2.0 ** -8}[y_dt]
    for row in range(m):                                    # by row: the rows differ in magnitude
        assert helpers.rel_l2(got[row], want[row]) <= tol, row


# the three tile shapes; K a whole number of blocks in one wave, K that ends inside a block, and both split over the waves of a workgroup
SPECIAL = [(20, 128, 96), (70, 1100, 96), (600, 1100, 96), (20, 128, 100), (70, 1100, 100), (600, 1100, 100), (20, 128, 896), (70, 1100, 896), (600, 1100, 900)]


@pytest.mark.parametrize("m,n,k", SPECIAL)
def test_infinities_nan_and_the_largest_values(ep, port, m, n, k):
    """An infinite activation gives what its products give (NaN only over a weight of zero or against the other infinity), one near the
    end of the range a finite result, and no other row notices."""
    b, s, zp = synth.make_weights(n, k, 32, n, zero_points=True, scale_lo=0.002, scale_hi=0.01, scale_dtype=E.F32)
    a = synth.make_activation(m, k, n, E.F32)
    a[1, 5], a[2, 40], a[3, 70], a[4, 3], a[4, 64] = np.inf, -np.inf, np.nan, np.inf, -np.inf
    a[5, 32:64] = np.finfo(np.float32).max * np.where(np.arange(32) % 3 == 0, -1, 1)
    y, variant = E.matmul_nbits(ep, a, E.F32, b, s, E.F32, zp, n, k, 32, y_dtype=E.F32)
    assert variant == "gemm_f32_mfma"
    w = port.dequantize_nk_bits(b, s, zp, n, k, 32, 4).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        want = np.stack([(a[r].astype(np.float64) * w).sum(axis=1) for r in range(m)])
    for row in range(m):
        if row in (1, 2, 3, 4):
            assert np.array_equal(y[row].astype(np.float64), want[row], equal_nan=True), row
        elif row == 5:                                      # outputs beyond the range of f32 are infinities
            inside = np.abs(want[row]) < 0.99 * np.finfo(np.float32).max
            assert inside.any() and helpers.rel_l2(y[row][inside].astype(np.float64) * 2.0 ** -100, want[row][inside] * 2.0 ** -100) <= TOL
        else:
            assert helpers.rel_l2(y[row].astype(np.float64), want[row]) <= TOL, row


def test_activations_of_more_than_two_gib(ep, port):
    """Elements beyond K read as zeros wherever the row lies: weights in the padding of a last, partial block meet nothing."""
    m, n, k, bs, rows = 140000, 128, 4100, 32, 1000
    b, s, zp = synth.make_weights(n, k, bs, 1, zero_points=True, scale_lo=0.002, scale_hi=0.01, scale_dtype=E.F32)
    a = synth.make_activation(rows, k, 1, E.F32)
    y, variant = E.matmul_nbits(ep, np.tile(a, (m // rows, 1)), E.F32, b, s, E.F32, zp, n, k, bs)
    assert variant == "gemm_f32_mfma"
    blocks = y.reshape(m // rows, rows, n)
    assert helpers.rel_l2(blocks[0], port.matmul_f64(a, b, s, zp, n, k, bs)) <= TOL
    assert all(np.array_equal(block, blocks[0]) for block in blocks[1:])


@pytest.mark.parametrize("m,n,k", SPECIAL)
def test_the_smallest_values(ep, port, m, n, k):
    """Rows of tiny activations, down to subnormal ones, keep their 24 bits - alone, and beside rows whose infinities or largest values send a wave round again."""
    b, s, zp = synth.make_weights(n, k, 32, n, zero_points=True, scale_lo=8.0, scale_hi=16.0, scale_dtype=E.F32)
    a = synth.make_activation(m, k, n, E.F32)
    tiny = {1: -112, 3: -118, 5: -126, 7: -130, 9: -100, 19: -122}
    for row, e in tiny.items():
        a[row] = (a[row].astype(np.float64) * 2.0 ** e).astype(np.float32)
    w = port.dequantize_nk_bits(b, s, zp, n, k, 32, 4).astype(np.float64)
    for beside in ("ordinary", "infinite", "largest"):
        if beside == "infinite":
            a[0, 5], a[4, 40] = np.inf, -np.inf
        elif beside == "largest":
            a[0, 5], a[4, 40] = 1.0, 1.0
            a[2, 0:32] = np.finfo(np.float32).max * np.where(np.arange(32) % 3 == 0, -1, 1)
        y, variant = E.matmul_nbits(ep, a, E.F32, b, s, E.F32, zp, n, k, 32, y_dtype=E.F32)
        assert variant == "gemm_f32_mfma"
        for row in [*tiny, 6, m - 1]:
            assert helpers.rel_l2(y[row].astype(np.float64) * 2.0 ** 120, (a[row].astype(np.float64) * w).sum(axis=1) * 2.0 ** 120) <= TOL, (beside, row)


@pytest.mark.parametrize("s_dt,bs,zero_points,m,n,k", [
    (E.F16, 64, True, 15, 130, 896),       # 16 x 16 tiles: a row short of one, and one row more
    (E.F32, 32, False, 17, 128, 96),       # ... fewer runs than waves
    (E.F32, 256, True, 33, 1100, 4864),
    (E.F32, 32, True, 95, 1100, 704),      # 32 x 32 tiles: 22 runs over eight waves, the last one has one
    (E.BF16, 32, False, 97, 1100, 800),    # ... 25 runs: four a wave, the last wave has none
    (E.F32, 32, True, 545, 1100, 288),     # two column tiles a wave, nine runs
])
def test_whole_blocks(ep, port, s_dt, bs, zero_points, m, n, k):
    """K a whole number of blocks: rows pass through LDS. Rows and shares of K at the edges of tiles."""
    test_matches_double_precision(ep, port, s_dt, bs, zero_points, m, n, k, "none", E.F32)


@pytest.mark.parametrize("s_dt,bs,zero_points,m,n,k", [
    (E.BF16, 32, True, 200, 900, 900),     # 32 x 32 tiles
    (E.F16, 64, False, 100, 1100, 836),    # ... fewer runs in the last block than in the others
    (E.F16, 32, True, 513, 2017, 164),     # two column tiles a wave
    (E.BF16, 128, False, 545, 1100, 1028),
])
def test_partial_last_blocks_under_16_bit_scales(ep, port, s_dt, bs, zero_points, m, n, k):
    test_matches_double_precision(ep, port, s_dt, bs, zero_points, m, n, k, "none", E.F32)


@pytest.mark.parametrize("k", [896, 900])
@pytest.mark.parametrize("m,n", [(20, 128), (70, 1100), (600, 1100)])
def test_one_waves_share_is_walked_again(ep, port, m, n, k):
    """Infinities and tiny rows in one wave's share of K: that wave goes round again while the others wait for its sums."""
    b, s, zp = synth.make_weights(n, k, 32, n, zero_points=True, scale_lo=8.0, scale_hi=16.0, scale_dtype=E.F32)
    a = synth.make_activation(m, k, n, E.F32)
    w = port.dequantize_nk_bits(b, s, zp, n, k, 32, 4).astype(np.float64)
    for start in (0, 448, k - 36):                          # the first wave's share, one in the middle, the last one's
        x = a.copy()
        x[1] = x[3] = 0.0
        x[1, start:start + 32] = (a[1, :32].astype(np.float64) * 2.0 ** -118).astype(np.float32)
        x[3, start + 4:start + 36] = (a[3, :32].astype(np.float64) * 2.0 ** -126).astype(np.float32)
        for infinite in (False, True):
            if infinite:
                x[2, start + 9] = np.inf
            y, variant = E.matmul_nbits(ep, x, E.F32, b, s, E.F32, zp, n, k, 32, y_dtype=E.F32)
            assert variant == "gemm_f32_mfma"
            for row in (0, 1, 3, 4, m - 1):
                assert helpers.rel_l2(y[row].astype(np.float64) * 2.0 ** 120, (x[row].astype(np.float64) * w).sum(axis=1) * 2.0 ** 120) <= TOL, (start, infinite, row)
        with np.errstate(invalid="ignore"):
            assert np.array_equal(y[2].astype(np.float64), (x[2].astype(np.float64) * w).sum(axis=1), equal_nan=True), start
