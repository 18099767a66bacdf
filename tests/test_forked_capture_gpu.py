"""A second stream that is forked from a capture and joins it again: what is recorded behind the join waits for both, and shares no launch."""
import ctypes as C

import numpy as np
import pytest

from onnx_genai_amd import build
from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests.test_abi_cpu import _FfiArgs

pytestmark = pytest.mark.gpu
TO_DEVICE_FROM_DEVICE = 3


@pytest.mark.parametrize("overwrites", [False, True])
def test_a_fork_that_joins(ep, overwrites):
    lib = C.CDLL(build.LIB)

    def hip(name, *args):                                    # of the runtime that the library is linked with
        assert getattr(lib, name)(*args) == 0, name

    lib.rocm_decode_packed_bytes.restype = C.c_uint64
    lib.rocm_step_tail_create.restype = C.c_void_p
    m, k, n, bs, dt = 2, 896, 304, 32, E.F16
    size = m * n * 2
    x = ep.upload(synth.make_activation(m, k, 1, dt))
    y = [ep.allocate(size) for _ in range(3)]
    copy = ep.allocate(size)
    outs = [*y[:2], copy if overwrites else y[2], copy]      # (the third node's result: its own, or what the other stream has written before)
    args, packed, keep = [], [], []
    for i in range(3):
        b, s, zp = synth.make_weights(n, k, bs, i, zero_points=True, scale_lo=0.002, scale_hi=0.01, scale_dtype=dt)
        keep += [ep.upload(t) for t in (b, s, zp)]
        a = _FfiArgs()
        a.a, a.y = x.ptr, outs[i].ptr
        a.b, a.scales, a.zp = (t.ptr for t in keep[-3:])
        a.a_dtype = a.scale_dtype = a.y_dtype = dt
        a.bias_dtype = E.F32
        a.m, a.n, a.k, a.block_size = m, n, k, bs
        args.append(a)
        packed.append(ep.allocate(lib.rocm_decode_packed_bytes(C.byref(a))))
    ep.sync()
    first, second, forked, joins = (C.c_void_p() for _ in range(4))
    for stream in (first, second):
        hip("hipStreamCreate", C.byref(stream))
    for event in (forked, joins):
        hip("hipEventCreate", C.byref(event))
    for a, p in zip(args, packed):
        assert lib.rocm_launch_pack_decode(C.byref(a), C.c_void_p(p.ptr), first) == 0
    tail = C.c_void_p(lib.rocm_step_tail_create())

    def step(tail):
        node = lambda i: lib.rocm_launch_decode_packed(C.byref(args[i]), C.c_void_p(packed[i].ptr), 0, first, tail)  # noqa: E731
        assert node(0) == 0
        hip("hipEventRecord", forked, first)
        hip("hipStreamWaitEvent", second, forked, 0)
        hip("hipMemcpyAsync", C.c_void_p(copy.ptr), C.c_void_p(y[0].ptr), C.c_size_t(size), TO_DEVICE_FROM_DEVICE, second)
        assert node(1) == 0                                  # may share the first one's launch: nothing between them on their stream
        hip("hipEventRecord", joins, second)
        hip("hipStreamWaitEvent", first, joins, 0)
        assert node(2) == 0                                  # behind the copy

    def read():
        got = [np.empty(size, np.uint8) for _ in outs]
        for to, buf in zip(got, outs):
            ep.copy_to_host(to, buf)
        return got

    def clear():
        for buf in outs:
            ep.copy_from_host(buf, np.full(size, 0x55, np.uint8))

    clear()
    step(None)
    hip("hipStreamSynchronize", first)
    want = read()
    assert np.array_equal(want[0], want[3]) != overwrites
    assert lib.rocm_ffi_capture_begin(first) == 0
    step(tail)
    graph, nodes = C.c_void_p(), C.c_size_t()
    assert lib.rocm_ffi_capture_end(first, C.byref(graph), C.byref(nodes)) == 0
    assert nodes.value == 3                                  # the first two nodes, the copy, the third node
    for _ in range(3):
        clear()
        assert lib.rocm_ffi_graph_launch(graph, first) == 0
        hip("hipStreamSynchronize", first)
        for w, g in zip(want, read()):
            assert np.array_equal(w, g)
    assert lib.rocm_ffi_graph_destroy(graph) == 0
    lib.rocm_step_tail_destroy(tail)
    for event in (forked, joins):
        hip("hipEventDestroy", event)
    for stream in (first, second):
        hip("hipStreamDestroy", stream)
