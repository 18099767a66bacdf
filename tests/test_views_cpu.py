"""The packed view arrays that execute hands to the C ABI: field for field what a CTensorView array holds."""
import ctypes as C

import numpy as np

from onnx_genai_amd import ep as E


def test_packed_views_read_back_as_ctensorviews():
    views = [E.TensorView(0x1000, E.F32, (2, 3, 896)), E.TensorView.absent(E.U8), E.TensorView(0x2000, E.BF16, (4, 8), strides=(-16, 2), byte_offset=32, device_type=5, device_index=7),
             E.TensorView(0x3000, E.U8, (np.int64(5),)), E.TensorView(0x4000, E.F16, ())]
    for given in (views, [*views, E.TensorView(0x5000, E.F32, (-1, 2.0))]):         # (the last one takes the converting path)
        buf, at = E._packed_views(given)
        got = (E.CTensorView * len(given)).from_address(at)
        for g, v in zip(got, given):
            assert (g.data or 0, g.dtype, g.ndim, g.byte_offset, g.device_type, g.device_index) == (v.data or 0, v.dtype, len(v.shape), v.byte_offset, v.device_type, v.device_index)
            assert [g.shape[i] for i in range(g.ndim)] == [int(d) % 2**64 for d in v.shape]
            assert bool(g.strides) == (v.strides is not None)
            if v.strides is not None:
                assert [g.strides[i] for i in range(g.ndim)] == list(v.strides)


def test_addresses_as_ctypes_pointers():
    """What a ctypes field takes as an address is an address here too."""
    for given, address in ((C.c_void_p(0x6000), 0x6000), (C.c_void_p(), 0)):
        buf, at = E._packed_views((E.TensorView(given, E.F32, (4,)),))
        assert (E.CTensorView.from_address(at).data or 0) == address
