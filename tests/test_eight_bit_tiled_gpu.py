"""The tiled kernel over packed 8-bit weights: its tiles, slices of K and edges, against the oracle."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers

pytestmark = pytest.mark.gpu

# One rounding of a weight and one of the result to the 16-bit type, each 2^-11 (f16) or 2^-8 (bf16) over sqrt(3) in the 2-norm
TOL = {E.F16: 2 ** 0.5 * 2.0 ** -11 / 3 ** 0.5 * 1.1, E.BF16: 2 ** 0.5 * 2.0 ** -8 / 3 ** 0.5 * 1.1}

CASES = [
    # type, block size, zero points, m, n, k, tile (0: the planner's)
    (E.BF16, 128, True, 65, 1100, 1024, 0),
    (E.F16, 32, True, 129, 2050, 576, 1),        # 128 x 128
    (E.BF16, 64, False, 300, 1000, 1088, 2),     # 256 x 128
    (E.F16, 128, True, 257, 4100, 320, 3),       # 256 x 256
    (E.BF16, 32, True, 513, 2100, 512, 3),
    (E.F16, 256, False, 70, 2000, 768, 4),       # 128 x 64
    (E.BF16, 128, True, 128, 520, 8192, 0),      # slices of K
    (E.F16, 32, False, 18, 560, 2048, 0),        # narrow calls above 16 rows
    (E.F16, 128, True, 33, 16385, 512, 0),       # wide ones above 32
]


@pytest.mark.parametrize("dt,bs,zero_points,m,n,k,tile", CASES)
def test_matches_oracle(port, dt, bs, zero_points, m, n, k, tile):
    ep = E.RocmExecutionProvider(0, {"prefill_tile": str(tile)} if tile else None)
    b, s, zp = synth.make_weights_bits(n, k, bs, 8, n + m, zero_points=zero_points, scale_lo=0.002, scale_hi=0.004, scale_dtype=dt)
    a = synth.make_activation(m, k, m, dt)
    bias = synth.to_dtype(np.linspace(-1, 1, n).astype(np.float32), dt)
    y, variant = E.matmul_nbits(ep, a, dt, b, s, dt, zp, n, k, bs, bias=bias, bias_dtype=dt, bits=8)
    assert variant == "prefill_mfma_lds8"
    want = port.matmul_f64_bits(synth.to_f32(a, dt), b, synth.to_f32(s, dt), zp, n, k, bs, 8, bias=synth.to_f32(bias, dt))
    assert helpers.rel_l2(synth.to_f32(y, dt), want) <= TOL[dt]
    ep.shutdown()


@pytest.mark.parametrize("dt", [E.F16, E.BF16])
def test_weight_tiles_are_the_product_rounded_once(ep, port, dt):
    """One-hot rows read the kernel's weights back: (q - zp) * scale rounded once to the 16-bit type, for every q and zero point."""
    n, k, bs, m = 4096, 256, 128, 256
    rng = np.random.default_rng(1)
    b = rng.integers(0, 256, (n, k // bs, bs)).astype(np.uint8)
    zp = rng.integers(0, 256, (n, k // bs)).astype(np.uint8)
    s = synth.to_dtype((rng.random((n, k // bs)) * 0.01 + 0.001).astype(np.float32), dt)
    a = synth.to_dtype(np.eye(m, k, dtype=np.float32), dt)
    y, variant = E.matmul_nbits(ep, a, dt, b, s, dt, zp, n, k, bs, bits=8)
    assert variant == "prefill_mfma_lds8"
    want = port.narrow(np.ascontiguousarray(port.dequantize_nk_bits(b, synth.to_f32(s, dt), zp, n, k, bs, 8)[:, :m].T), dt)
    assert np.array_equal(np.asarray(y).view(np.uint16).reshape(m, n), np.asarray(want).view(np.uint16).reshape(m, n))
