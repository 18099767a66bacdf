"""The fused gate/up node over 8-bit weights: every call of a node gives what its first one gave, and that is the oracle's."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,bs,m,n,k", [
    (E.BF16, 128, 1, 4608, 1024),       # large enough for a repacked copy of 8-bit weights: up to four rows, and beyond
    (E.F16, 32, 4, 4608, 1024),
    (E.BF16, 64, 9, 2100, 512),
    (E.F16, 128, 2, 320, 256),          # too small for one
])
def test_calls_after_the_first(ep, port, dt, bs, m, n, k):
    kb = k // bs
    halves = [synth.make_weights_bits(n, k, bs, 8, seed, zero_points=True, scale_lo=0.0002, scale_hi=0.0004, scale_dtype=dt) for seed in (n, n + 1)]
    a = synth.make_activation(m, k, m, dt)
    bufs = [ep.upload(x) for half in halves for x in half] + [ep.upload(a), ep.allocate(m * n * 2)]
    bg, sg, zg, bu, su, zu, ab, yb = bufs
    kernel = ep.get_kernel({"K": k, "N": n, "bits": 8, "block_size": bs, "gate_up_swiglu": 1})
    kernel.set_constant_inputs([False] + [True] * 7)
    w = lambda b: E.TensorView(b.ptr, E.U8, (n, kb, bs))  # noqa: E731
    s = lambda b: E.TensorView(b.ptr, dt, (n, kb))  # noqa: E731
    z = lambda b: E.TensorView(b.ptr, E.U8, (n, kb))  # noqa: E731
    views = [E.TensorView(ab.ptr, dt, (m, k)), w(bg), s(sg), w(bu), s(su), E.TensorView.absent(E.F32), z(zg), z(zu)]
    try:
        got = []
        for _ in range(3):
            ep.copy_from_host(yb, np.full(m * n * 2, 0xEE, np.uint8))
            kernel.execute(views, [E.TensorView(yb.ptr, dt, (m, n))])
            got.append(ep.download(yb, (m, n), np.uint16))
    finally:
        kernel.release()
        for buf in bufs:
            ep.deallocate(buf)
    gate, up = (port.matmul_f64_bits(synth.to_f32(a, dt), b, synth.to_f32(sc, dt), zp, n, k, bs, 8).astype(np.float32) for b, sc, zp in halves)
    want = port.swiglu(port.narrow(gate, dt), port.narrow(up, dt), dt)
    # three roundings to 16 bits (gate, up, result), each half a unit: 2^-11 (f16) or 2^-8 (bf16); silu passes a relative error on by a factor below 1.3 + |x|
    assert helpers.rel_l2(synth.to_f32(got[0].view(np.float16) if dt == E.F16 else got[0], dt), synth.to_f32(np.asarray(want), dt)) <= 4 * (2.0 ** -11 if dt == E.F16 else 2.0 ** -8)
    assert np.array_equal(got[1], got[0]) and np.array_equal(got[2], got[0])
