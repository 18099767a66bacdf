"""accuracy_level = 4 calls tall and wide enough for 256 x 128 tiles: against the oracle on a sample of columns, and bit for bit what 128 x 128 tiles give."""
import ctypes as C

import numpy as np
import pytest

import oracle
from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers
from tests.golden.make_dispatch_table import ffi_args

pytestmark = pytest.mark.gpu


def tile_rows(ep, m, n, k, bs):
    rows = C.c_int()
    assert ep.lib.rocm_acc4_mfma_plan(C.byref(ffi_args(E.F16, bs, True, m, n, k)), ep.device_info()["compute_units"], C.byref(rows), None) == 0
    return rows.value


@pytest.mark.parametrize("s_dt,bs,zero_points,m,n,k,bias_kind", [
    (E.F16, 64, True, 500, 16370, 192, "column"),      # ragged last tiles both ways, an odd count of steps
    (E.F32, 64, False, 385, 16384, 64, "none"),        # one step; one row in the last 32 x 32 tiles
    (E.BF16, 64, True, 512, 16257, 576, "row"),        # nine steps: whole rounds of loads and a rest
    (E.F16, 64, True, 1200, 12763, 192, "column"),     # 5 x 100 tiles: a band of four whole row blocks, and one of 176 rows
    (E.BF16, 64, True, 2304, 7040, 192, "none"),       # 9 x 55: bands of four, four and one row block, a count that eight XCDs do not divide
    (E.F16, 128, True, 500, 16370, 8192, "row"),       # a block over two steps
    (E.F32, 256, False, 511, 16300, 8448, "column"),   # ... over four
])
def test_matches_oracle_and_smaller_tiles(ep, port, s_dt, bs, zero_points, m, n, k, bias_kind):
    a_dt = E.BF16 if s_dt == E.BF16 else E.F16
    b, s, zp = synth.make_weights(n, k, bs, n + k, zero_points=zero_points, scale_lo=0.002, scale_hi=0.01, scale_dtype=s_dt)
    a = synth.make_activation(m, k, m, a_dt)
    rng = np.random.default_rng(k)
    bias = None if bias_kind == "none" else rng.standard_normal((m, n) if bias_kind == "row" else n).astype(np.float32)
    run = lambda rows, extra: E.matmul_nbits(ep, a[rows], a_dt, b, s, s_dt, zp, n, k, bs, bias=extra, accuracy_level=4, y_dtype=E.F32)  # noqa: E731
    y, variant = run(slice(0, m), bias)
    assert variant == "acc4_mfma_i8" and tile_rows(ep, m, n, k, bs) == 256
    cols = np.unique(np.concatenate([np.arange(0, n, n // 40), [31, 32, 63, 64, 127, 128, n - 2, n - 1]]))
    want = port.matmul_acc4_f32(synth.to_f32(a, a_dt), b[cols], synth.to_f32(s, s_dt)[cols], None if zp is None else zp[cols], cols.size, k, bs, oracle.ROUND_HALF_EVEN)
    if bias is not None:
        want = want + (bias[:, cols] if bias_kind == "row" else bias[cols])
    assert helpers.rel_l2(y[:, cols], want) <= 1e-5        # the bar of the parity contract
    for rows in (slice(0, 200), slice(m - 201, m)):        # too few tiles for the taller ones, too many for slices of K
        assert tile_rows(ep, rows.stop - rows.start, n, k, bs) == 128
        short, _ = run(rows, bias[rows] if bias_kind == "row" else bias)
        assert np.array_equal(y[rows], short)
