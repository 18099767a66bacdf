"""Columns beyond the last whole round of 256 x 256 tiles go to smaller tiles in a launch of their own: the same bits, and only where they fit one to a CU."""
import ctypes as C

import numpy as np
import pytest

from onnx_genai_amd import build
from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests.test_abi_cpu import _FfiArgs


def rest(m, n, k, dt=E.BF16, bs=128):
    lib = C.CDLL(build.LIB)
    lib.rocm_prefill_mfma_rest.restype = C.c_int64
    lib.rocm_prefill_mfma_rest.argtypes = [C.c_void_p, C.c_int, C.c_uint64, C.POINTER(C.c_int), C.POINTER(C.c_int)]
    args = _FfiArgs()
    args.a, args.b, args.scales, args.y = 0x10000, 0x20000, 0x30000, 0x40000         # never dereferenced: alignment only
    args.a_dtype = args.scale_dtype = args.y_dtype = dt
    args.m, args.n, args.k, args.block_size = m, n, k, bs
    rows, cols = C.c_int(), C.c_int()
    count = lib.rocm_prefill_mfma_rest(C.byref(args), 0, C.c_uint64(0), C.byref(rows), C.byref(cols))
    for choice in (1, 2, 3, 4):                              # one tile for all columns, as asked for
        assert lib.rocm_prefill_mfma_rest(C.byref(args), choice, C.c_uint64(0), None, None) == 0
    return count, rows.value, cols.value


# rows, columns, K, what of it is left for smaller tiles (columns, tile)
PLANS = [
    (300, 37888, 3584, (5120, 128, 64)),
    (512, 37888, 3584, (5120, 128, 128)),
    (1024, 37888, 3584, (5120, 256, 128)),
    (4352, 4096, 14336, (256, 128, 64)),
    (768, 37888, 3584, (0, 0, 0)),                # two workgroups of any smaller tile to a CU
    (2048, 37888, 3584, (0, 0, 0)),
    (8192, 14336, 4096, (0, 0, 0)),               # whole rounds
    (4352, 28672, 4096, (0, 0, 0)),               # seven rounds before it
    (4096, 37888, 3584, (1024, 128, 128)),
]


@pytest.mark.parametrize("m,n,k,want", PLANS)
def test_the_rule(m, n, k, want):
    assert rest(m, n, k) == want


@pytest.mark.gpu
@pytest.mark.parametrize("dt,sdt,bits,bs,m,n,k,tile,bias", [
    (E.F16, E.F16, 4, 32, 1200, 14336, 256, (128, 64), "columns"),
    (E.BF16, E.F32, 4, 128, 500, 37888, 256, (128, 128), None),
    (E.BF16, E.BF16, 4, 64, 1024, 21241, 128, (256, 128), "columns"),    # ragged columns, no 16-byte stores
    (E.BF16, E.BF16, 8, 128, 300, 33030, 128, (128, 64), "rows"),
])
def test_the_bits_of_whole_tiles(dt, sdt, bits, bs, m, n, k, tile, bias):
    count, rows, cols = rest(m, n, k, dt, bs)
    assert count > 0 and (rows, cols) == tile
    b, s, zp = synth.make_weights_bits(n, k, bs, bits, n, zero_points=True, scale_lo=0.002, scale_hi=0.004, scale_dtype=sdt)
    a = synth.make_activation(m, k, n, dt)
    add = {"columns": np.linspace(-1, 1, n), "rows": np.linspace(-1, 1, m * n).reshape(m, n)}.get(bias)
    add = None if add is None else synth.to_dtype(add.astype(np.float32), dt)
    got = []
    for config in (None, {"prefill_tile": "3"}):
        ep = E.RocmExecutionProvider(0, config)
        y, variant = E.matmul_nbits(ep, a, dt, b, s, sdt, zp, n, k, bs, bias=add, bias_dtype=dt, bits=bits)
        assert variant.startswith("prefill_mfma")
        got.append(np.asarray(y).view(np.uint16))
        ep.shutdown()
    assert np.array_equal(got[0], got[1])
