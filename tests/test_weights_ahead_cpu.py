"""What a normalization launch reads ahead lies within the repacked copies of the launch behind it, workgroup by workgroup. No GPU work."""
import ctypes as C

import pytest

from onnx_genai_amd import build
from tests.test_abi_cpu import _FfiArgs


class _Ahead(C.Structure):
    _fields_ = [("first", C.c_void_p), ("second", C.c_void_p), ("bytes", C.c_uint64), ("workgroups", C.c_uint32)]


class _Plan(C.Structure):
    _fields_ = [("shared_activations", C.c_int), ("rows_build", C.c_int), ("waves", C.c_int), ("groups_per_wave", C.c_int), ("register_sets", C.c_int),
                ("activation_sums", C.c_int), ("workgroups", C.c_int64)]


@pytest.mark.parametrize("bs", [32, 64, 128])
@pytest.mark.parametrize("m", [1, 4, 5, 16, 24, 64])
def test_ranges_lie_within_the_copies(m, bs):
    lib = C.CDLL(build.LIB)
    lib.rocm_decode_packed_bytes.restype = C.c_uint64
    seen = 0
    for n, k in [(16, 128), (100, 896), (3584, 3584), (4608, 3584), (9472, 3584), (18944, 3584), (14336, 4096), (18945, 3584), (152064, 3584), (3584, 18944)]:
        for pair in (0, 2):
            args = _FfiArgs()
            args.a, args.b, args.scales, args.y = 0x10000, 0x20000, 0x30000, 0x40000           # never dereferenced: alignment only
            args.a_dtype = args.scale_dtype = args.y_dtype = 16
            args.m, args.n, args.k, args.block_size = m, n, k, bs
            ahead, plan = _Ahead(), _Plan()
            ok = lib.rocm_decode_packed_ahead(C.byref(args), C.c_void_p(0x100000), C.c_void_p(0x200000 if pair else 0), 0, C.byref(ahead))
            assert ok == (lib.rocm_decode_packed_plan(C.byref(args), 0, pair, 256, C.byref(plan)) == 0)
            if not ok:
                continue
            seen += 1
            assert ahead.first == 0x100000 and ahead.second == (0x200000 if pair else None) and ahead.bytes % 16 == 0
            assert 0 < ahead.workgroups <= plan.workgroups or ahead.workgroups == 0
            assert ahead.workgroups * ahead.bytes <= lib.rocm_decode_packed_bytes(C.byref(args)) < (ahead.workgroups + 1) * ahead.bytes
    assert seen > 0 or m > 16
