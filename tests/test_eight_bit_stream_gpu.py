"""8-bit weights over the repacked stream: row counts of every build, ragged edges, block sizes, against the oracle."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers

pytestmark = pytest.mark.gpu

# The result's own rounding: half a unit of 2^-10 (f16) or 2^-7 (bf16), relative to a value at least half the unit's binade, uniform in it:
# 2^-11 / sqrt(3) and 2^-8 / sqrt(3) in the 2-norm, and 1e-4 of room (test_plain_sums_gpu.py holds the sums to less).
TOL = {E.F16: 2.0 ** -11 / 3 ** 0.5 + 1e-4, E.BF16: 2.0 ** -8 / 3 ** 0.5 + 1e-4}

CASES = [
    # type, block size, zero points, m, n, k
    (E.BF16, 128, True, 1, 4099, 1024),         # one row; a ragged last column group
    (E.F16, 32, False, 1, 4672, 904),           # K ends inside a tile and inside a block
    (E.F16, 64, True, 1, 256, 18944),           # more tile groups than waves
    (E.BF16, 128, True, 3, 2050, 2048 + 128),   # an odd number of tiles: the last group is half empty
    (E.BF16, 32, True, 4, 4690, 896),
    (E.F16, 128, False, 7, 1200, 3584),
    (E.BF16, 64, True, 8, 4600, 1000),
    (E.F16, 128, True, 16, 1300, 3584),
    (E.BF16, 32, True, 16, 23000, 256),         # wide calls: the kernel that shares the activations
    (E.F16, 64, True, 9, 21000, 320),
    (E.BF16, 128, True, 16, 18448, 384),
    (E.F16, 128, True, 5, 40000, 256),
    (E.BF16, 128, False, 12, 100000, 128),
    (E.BF16, 64, True, 31, 16400, 448),
    (E.F16, 128, True, 32, 16385, 512),
]


@pytest.mark.parametrize("dt,bs,zero_points,m,n,k", CASES)
def test_matches_oracle(ep, port, dt, bs, zero_points, m, n, k):
    b, s, zp = synth.make_weights_bits(n, k, bs, 8, n + m, zero_points=zero_points, scale_lo=0.002, scale_hi=0.004, scale_dtype=dt)
    a = synth.make_activation(m, k, m, dt)
    bias = synth.to_dtype(np.linspace(-1, 1, n).astype(np.float32), dt)
    y, variant = E.matmul_nbits(ep, a, dt, b, s, dt, zp, n, k, bs, bias=bias, bias_dtype=dt, bits=8)
    assert variant == "decode_mfma_packed8"
    cols = np.arange(n) if n < 6000 else np.unique(np.concatenate([np.arange(64), np.random.default_rng(n).integers(0, n, 400), np.arange(n - 64, n)]))
    kb = -(-k // bs)
    want = port.matmul_f64_bits(synth.to_f32(a, dt), np.ascontiguousarray(np.asarray(b).reshape(n, -1)[cols]), np.ascontiguousarray(synth.to_f32(s, dt).reshape(n, kb)[cols]),
                                None if zp is None else np.ascontiguousarray(np.asarray(zp).reshape(n, -1)[cols]), len(cols), k, bs, 8, bias=synth.to_f32(bias, dt)[cols])
    assert helpers.rel_l2(synth.to_f32(y, dt)[:, cols], want) <= TOL[dt]


def test_f32_results_keep_their_route(ep, port):
    """An f32 result of a 16-bit row stays on the plain GEMV."""
    m, n, k, bs = 2, 4100, 1024, 128
    b, s, zp = synth.make_weights_bits(n, k, bs, 8, 3, zero_points=True, scale_lo=0.002, scale_hi=0.004, scale_dtype=E.F16)
    a = synth.make_activation(m, k, 3, E.F16)
    y, variant = E.matmul_nbits(ep, a, E.F16, b, s, E.F16, zp, n, k, bs, bits=8, y_dtype=E.F32)
    assert variant == "gemv_nbits_f32"
    assert helpers.rel_l2(y, port.matmul_f64_bits(synth.to_f32(a, E.F16), b, synth.to_f32(s, E.F16), zp, n, k, bs, 8)) <= 1e-5
