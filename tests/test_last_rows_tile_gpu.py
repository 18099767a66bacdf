"""Last row blocks of the 256 x 256 tiled kernel of at most 64 rows are narrower tiles: the bits of the same rows in a whole tile."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,sdt,bits,bs,n,k,bias", [
    (E.F16, E.F16, 4, 32, 520, 576, "columns"),
    (E.F16, E.F32, 4, 64, 257, 320, None),               # no 16-byte stores
    (E.BF16, E.BF16, 4, 128, 1000, 256, "rows"),
    (E.BF16, E.F32, 4, 32, 512, 128, "columns"),
    (E.BF16, E.BF16, 8, 128, 513, 4096, None),           # slices of K
    (E.F16, E.F16, 8, 32, 2056, 576, "rows"),
])
def test_the_bits_of_a_whole_tile(dt, sdt, bits, bs, n, k, bias):
    ep = E.RocmExecutionProvider(0, {"prefill_tile": "3"})
    whole = 512
    b, s, zp = synth.make_weights_bits(n, k, bs, bits, n, zero_points=True, scale_lo=0.002, scale_hi=0.004, scale_dtype=sdt)
    a = synth.make_activation(whole, k, n, dt)
    add = {"columns": np.linspace(-1, 1, n), "rows": np.linspace(-1, 1, whole * n).reshape(whole, n)}.get(bias)

    def run(rows):
        part = None if add is None else synth.to_dtype((add[:rows] if bias == "rows" else add).astype(np.float32), dt)
        y, variant = E.matmul_nbits(ep, a[:rows], dt, b, s, sdt, zp, n, k, bs, bias=part, bias_dtype=dt, bits=bits)
        assert variant.startswith("prefill_mfma")
        return np.asarray(y).view(np.uint16).reshape(rows, n)

    want = run(whole)
    for rows in (257, 265, 288, 289, 320, 321):
        assert np.array_equal(run(rows), want[:rows]), rows
    ep.shutdown()
