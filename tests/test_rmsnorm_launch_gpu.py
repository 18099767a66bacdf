"""The normalization launch at the edges of its forms: pieces held in registers, rows staged in LDS, rows beyond LDS."""
import numpy as np
import pytest

import oracle
from onnx_genai_amd import ep as E
from onnx_genai_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a_dt,g_dt", [(E.F16, E.F32), (E.BF16, E.BF16)])
@pytest.mark.parametrize("k", [128, 2048, 4096, 4224, 32768, 32896])
def test_bits_equal_the_oracles(ep, port, a_dt, g_dt, k):
    """Five rows take the launch of its own; the product over normalized rows is the plain node's over the oracle's rows, bit for bit."""
    m, n, bs, eps = 5, 33, 128, 1e-6
    b, s, zp = synth.make_weights(n, k, bs, k, zero_points=True, scale_lo=0.002, scale_hi=0.01, scale_dtype=a_dt)
    a = synth.make_activation(m, k, k, a_dt)
    gamma = synth.to_dtype((1.0 + 0.25 * np.random.default_rng(k).standard_normal(k)).astype(np.float32), g_dt)
    o_dt = oracle.F16 if a_dt == E.F16 else oracle.BF16
    rows = port.rmsnorm16(np.asarray(a).reshape(m, k), gamma, oracle.F32 if g_dt == E.F32 else o_dt, eps, o_dt)
    y, variant = E.matmul_nbits(ep, a, a_dt, b, s, a_dt, zp, n, k, bs, gamma=gamma, gamma_dtype=g_dt, rmsnorm_epsilon=eps)
    want, _ = E.matmul_nbits(ep, rows, a_dt, b, s, a_dt, zp, n, k, bs)
    assert variant.startswith("rmsnorm+")
    assert np.array_equal(np.asarray(y).view(np.uint16), np.asarray(want).view(np.uint16))
