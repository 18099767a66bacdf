"""accuracy_level = 4 calls whose grids of tiles are ragged where tiles are handed out: counts that eight XCDs do not divide, bands of fewer than four row
blocks, one tile, one row or column of tiles, slices of K. Every tile has to be taken once."""
import ctypes as C

import numpy as np
import pytest

import oracle
from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers
from tests.golden.make_dispatch_table import ffi_args

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,bs,slices", [
    (17, 100, 128, 64, 1),          # one tile
    (640, 896, 256, 64, 1),         # 7 x 5: a band of four row blocks and one of one
    (1100, 300, 192, 32, 1),        # 3 x 9, fewer tiles in a band than two an XCD
    (130, 1920, 128, 128, 1),       # 15 x 2
    (100, 1200, 2048, 64, 4),       # 10 x 1 over slices of K
    (400, 700, 4096, 128, 8),       # 6 x 4
    (520, 8200, 192, 64, 1),        # 65 x 5: two workgroups on a CU, padded rows in LDS
])
def test_every_tile_once(ep, port, m, n, k, bs, slices):
    got = C.c_int()
    assert ep.lib.rocm_acc4_mfma_plan(C.byref(ffi_args(E.F16, bs, True, m, n, k)), ep.device_info()["compute_units"], None, C.byref(got)) == 0
    assert got.value == slices
    b, s, zp = synth.make_weights(n, k, bs, n + k, zero_points=True, scale_lo=0.002, scale_hi=0.01, scale_dtype=E.F16)
    a = synth.make_activation(m, k, m, E.F16)
    y, variant = E.matmul_nbits(ep, a, E.F16, b, s, E.F16, zp, n, k, bs, accuracy_level=4, y_dtype=E.F32)
    assert variant == "acc4_mfma_i8"
    want = port.matmul_acc4_f32(synth.to_f32(a, E.F16), b, synth.to_f32(s, E.F16), zp, n, k, bs, oracle.ROUND_HALF_EVEN)
    assert helpers.rel_l2(y, want) <= 1e-5        # the bar of the parity contract
    worst = np.abs(y - want).max()
    assert worst <= 1e-4 * np.sqrt(np.mean(np.square(want.astype(np.float64)))), worst      # no tile stands out


@pytest.mark.parametrize("s_dt,m,n,k,bs", [
    (E.F16, 777, 4864, 96, 32),          # block size 32: 7 x 38, nine rows in the last row block
    (E.F32, 1153, 3500, 160, 32),        # ... 10 x 28: bands of four, four and one whole row block, and one of one row
    (E.BF16, 60, 33000, 64, 32),         # ... one row block, not whole
    (E.F16, 300, 16300, 8192, 64),       # rows of B 4096 bytes apart: 3 x 128, over no slices
    (E.F16, 17, 16384, 8192, 128),       # ... 1 x 128 over slices of K
])
def test_runs_of_tiles(ep, port, s_dt, m, n, k, bs):
    """Grids whose tiles go out in runs instead of launch order: a column of every column block, over all rows."""
    a_dt = E.BF16 if s_dt == E.BF16 else E.F16
    args, tile = ffi_args(E.F16, bs, True, m, n, k), [C.c_int64(), C.c_int64()]
    assert ep.lib.rocm_acc4_mfma_tile(C.byref(args), ep.device_info()["compute_units"], C.c_int64(8), C.byref(tile[0]), C.byref(tile[1])) == 0
    assert (tile[0].value, tile[1].value) != (0, 8)
    b, s, zp = synth.make_weights(n, k, bs, n + k, zero_points=True, scale_lo=0.002, scale_hi=0.01, scale_dtype=s_dt)
    a = synth.make_activation(m, k, m, a_dt)
    y, variant = E.matmul_nbits(ep, a, a_dt, b, s, s_dt, zp, n, k, bs, accuracy_level=4, y_dtype=E.F32)
    assert variant == "acc4_mfma_i8"
    cols = np.append(np.arange(0, n, 128) + np.arange(-(-n // 128)) * 37 % (n - (n - 1) // 128 * 128), n - 1)
    want = port.matmul_acc4_f32(synth.to_f32(a, a_dt), b[cols], synth.to_f32(s, s_dt)[cols], zp[cols], cols.size, k, bs, oracle.ROUND_HALF_EVEN)
    assert helpers.rel_l2(y[:, cols], want) <= 1e-5        # the bar of the parity contract
    worst = np.abs(y[:, cols] - want).max()
    assert worst <= 1e-4 * np.sqrt(np.mean(np.square(want.astype(np.float64)))), worst
