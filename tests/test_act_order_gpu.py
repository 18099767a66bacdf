"""Act-order weights whose groups are whole blocks in another order: sorted once, then served by the kernels for contiguous blocks."""
import numpy as np
import pytest

from onnx_genai_amd import ep as E
from onnx_genai_amd import synth
from tests import helpers

pytestmark = pytest.mark.gpu

TOL = {E.F32: 1e-5, E.F16: 5e-3, E.BF16: 5e-3}      # the bars of the parity contract


def weights(n, k, bs, bits, dt, seed):
    if bits == 4:
        return synth.make_weights(n, k, bs, seed, zero_points=True, scale_lo=0.005, scale_hi=0.02, scale_dtype=dt)
    return synth.make_weights_bits(n, k, bs, bits, seed, zero_points=True, scale_lo=0.001, scale_hi=0.003, scale_dtype=dt)


def shuffled_groups(k, bs, seed):
    g = (np.arange(k) // bs).astype(np.int32)
    np.random.default_rng(seed).shuffle(g)
    return g


def expected(port, a, a_dt, b, s, zp, g, n, k, bs, bits):
    return synth.to_f32(a, a_dt).astype(np.float64) @ port.dequantize_nk_gidx(b, synth.to_f32(s, a_dt), zp, g, n, k, bs, bits).astype(np.float64).T


@pytest.mark.parametrize("a_dt,bits,bs,m,n,k", [
    (E.F16, 4, 128, 1, 300, 3584),
    (E.BF16, 4, 32, 4, 129, 896),
    (E.BF16, 4, 64, 16, 72, 1024),
    (E.F16, 4, 128, 100, 264, 512),
    (E.F32, 4, 32, 3, 64, 260),             # K % block_size != 0: the last group is the short one
    (E.F32, 4, 32, 70, 160, 256),
    (E.F16, 4, 16, 2, 40, 208),
    (E.F16, 8, 32, 1, 100, 320),
    (E.BF16, 8, 128, 9, 136, 512),
    (E.F16, 2, 64, 3, 72, 512),
])
def test_matches_oracle(ep, port, a_dt, bits, bs, m, n, k):
    b, s, zp = weights(n, k, bs, bits, a_dt, n)
    g = shuffled_groups(k, bs, m)
    a = synth.make_activation(m, k, 5, a_dt)
    y, variant = E.matmul_nbits(ep, a, a_dt, b, s, a_dt, zp, n, k, bs, bits=bits, g_idx=g)
    assert variant.startswith("act_order+")
    assert helpers.rel_l2(synth.to_f32(y, a_dt), expected(port, a, a_dt, b, s, zp, g, n, k, bs, bits)) <= TOL[a_dt]


def test_weights_that_change_and_groups_that_do_not_sort(ep, port):
    """A node that moves to other tensors sorts those (a freed copy's address may come back), and one group longer than a block is served unsorted."""
    a_dt, bs, bits, m, n, k = E.F16, 32, 4, 2, 64, 256
    a = synth.make_activation(m, k, 5, a_dt)
    ab, yb = ep.upload(a), ep.allocate(m * n * 2)
    kernel = ep.get_kernel({"K": k, "N": n, "bits": bits, "block_size": bs})
    kernel.set_constant_inputs([False, True, True, True, True])
    out = [E.TensorView(yb.ptr, a_dt, (m, n))]
    held = []
    try:
        for seed, regular in ((1, True), (2, True), (3, False), (4, True)):
            b, s, zp = weights(n, k, bs, bits, a_dt, seed)
            g = shuffled_groups(k, bs, seed)
            if not regular:
                g[g == 1] = 0
            bufs = [ep.upload(x) for x in (b, s, zp, g)]
            held += bufs
            views = [E.TensorView(ab.ptr, a_dt, (m, k)), E.TensorView(bufs[0].ptr, E.U8, (n, k // bs, bs // 2)), E.TensorView(bufs[1].ptr, a_dt, (n, k // bs)),
                     E.TensorView(bufs[2].ptr, E.U8, (n, k // bs // 2)), E.TensorView(bufs[3].ptr, E.I32, (k,))]
            for _ in range(2):
                kernel.execute(views, out)
                assert kernel.last_variant().startswith("act_order+") == regular
                got = ep.download(yb, (m, n), np.float16)
                assert helpers.rel_l2(got.astype(np.float64), expected(port, a, a_dt, b, s, zp, g, n, k, bs, bits)) <= TOL[a_dt]
    finally:
        kernel.release()
        for buf in held + [ab, yb]:
            ep.deallocate(buf)


def test_graph_replays_sort_the_rows_of_their_own_time(ep, port):
    """A recorded call gathers the activations that lie in its input buffer when it is replayed."""
    a_dt, bs, m, n, k = E.BF16, 64, 3, 96, 512
    b, s, zp = weights(n, k, bs, 4, a_dt, 9)
    g = shuffled_groups(k, bs, 9)
    ops = E.DeviceOperands(ep, b, s, a_dt, zp, n, k, bs, g_idx=g)
    ab, yb = ep.upload(synth.make_activation(m, k, 1, a_dt)), ep.allocate(m * n * 2)
    try:
        ops.run(ab, a_dt, m, yb)
        ep.capture_begin()
        ops.run(ab, a_dt, m, yb)
        graph = ep.capture_end()
        for seed in (2, 3, 4):
            a = synth.make_activation(m, k, seed, a_dt)
            ep.copy_from_host(ab, a)
            graph.replay()
            got = synth.to_f32(ep.download(yb, (m, n), np.uint16), a_dt)
            assert helpers.rel_l2(got, expected(port, a, a_dt, b, s, zp, g, n, k, bs, 4)) <= TOL[a_dt]
            ops.run(ab, a_dt, m, yb)
            assert np.array_equal(got, synth.to_f32(ep.download(yb, (m, n), np.uint16), a_dt))
        graph.release()
    finally:
        ep.deallocate(ab)
        ep.deallocate(yb)
        ops.free()


@pytest.mark.parametrize("bs,m", [(128, 8), (128, 1), (256, 5)])
def test_a_height_recorded_without_a_repacked_copy(ep, port, bs, m):
    """A prompt sorts the weights but makes no repacked copy; a few rows first seen inside a capture take the tiled kernel from five rows, and the
    f32 GEMV below."""
    a_dt, n, k, tall = E.F16, 300, 512, 40
    b, s, zp = weights(n, k, bs, 4, a_dt, 9)
    g = shuffled_groups(k, bs, 9)
    ops = E.DeviceOperands(ep, b, s, a_dt, zp, n, k, bs, g_idx=g)
    ab, yb = ep.upload(synth.make_activation(tall, k, 1, a_dt)), ep.allocate(tall * n * 2)
    try:
        ops.run(ab, a_dt, tall, yb)
        assert ops.kernel.last_variant() == "act_order+prefill_mfma_lds"
        ep.capture_begin()
        ops.run(ab, a_dt, m, yb)
        variant = ops.kernel.last_variant()
        graph = ep.capture_end()
        assert variant == ("act_order+prefill_mfma_lds" if m >= 5 else "act_order+gemv_generic_f32")
        for seed in (2, 3, 4):
            a = synth.make_activation(m, k, seed, a_dt)
            ep.copy_from_host(ab, a)
            graph.replay()
            got = synth.to_f32(ep.download(yb, (m, n), np.float16), a_dt)
            assert helpers.rel_l2(got, expected(port, a, a_dt, b, s, zp, g, n, k, bs, 4)) <= TOL[a_dt]
        graph.release()
    finally:
        ep.deallocate(ab)
        ep.deallocate(yb)
        ops.free()


@pytest.mark.parametrize("first", [0.0, np.inf])
@pytest.mark.parametrize("a_dt,bs,s_dt,k", [(E.F16, 128, E.F16, 1000), (E.BF16, 128, E.BF16, 3584), (E.BF16, 32, E.F32, 1000), (E.F16, 64, E.F32, 520), (E.F16, 32, E.F16, 8),
                                            (E.F16, 128, E.F16, 18944), (E.BF16, 128, E.BF16, 26624), (E.BF16, 128, E.BF16, 26632), (E.F16, 32, E.F16, 16384), (E.F16, 32, E.F16, 16392)])
def test_one_row_gathered_inside_the_kernel(ep, a_dt, bs, s_dt, k, first):
    """The bits of a row gathered by a launch of its own, which a row off a 16-byte boundary takes: ragged K, the longest rows the kernel takes and the first that it
    does not, and a row whose first element, which the places beyond K point at, is infinite."""
    n = 72
    b, s, zp = synth.make_weights(n, k, bs, k, zero_points=True, scale_lo=0.005, scale_hi=0.02, scale_dtype=s_dt)
    ops = E.DeviceOperands(ep, b, s, s_dt, zp, n, k, bs, g_idx=shuffled_groups(k, bs, k))
    a = np.asarray(synth.to_f32(synth.make_activation(1, k, 7, a_dt), a_dt)).copy().reshape(1, k)
    if first != 0.0:
        a[0, 0] = first
    a = np.asarray(synth.to_dtype(a, a_dt)).view(np.uint16).ravel()
    ab, yb = ep.upload(np.concatenate([a, np.zeros(4, np.uint16), a])), ep.allocate(n * 2)
    got = []
    try:
        for start in (0, k * 2 + 8):                       # (K is a multiple of 8: the second row is off by half of 16 bytes)
            ops.run(E.DeviceBuffer(ab.ptr + start, k * 2), a_dt, 1, yb)
            assert ops.kernel.last_variant() == "act_order+decode_mfma_packed"
            got.append(ep.download(yb, (n,), np.uint16))
        assert np.array_equal(got[0], got[1])
    finally:
        ep.deallocate(ab)
        ep.deallocate(yb)
        ops.free()
