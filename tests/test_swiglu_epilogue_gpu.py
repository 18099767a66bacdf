"""The SwiGLU epilogue's launch against the oracle over every 16-bit gate value, and at the edges of its 16-byte pieces."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from onnx_genai_amd import ep as E

pytestmark = pytest.mark.gpu


def _launch(ep, gate, up, dtype, decomposed, offset=0):
    """offset: elements by which all three matrices lie beyond a 16-byte boundary."""
    pad = lambda x: torch.from_numpy(np.concatenate([np.zeros(offset, np.uint16), x]).view(np.int16)).cuda()  # noqa: E731
    g, u = pad(gate), pad(up)
    y = torch.full((offset + gate.size + 8,), 0x5555, dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    lib = E.load_library()
    at = lambda t: C.c_void_p(t.data_ptr() + 2 * offset)  # noqa: E731
    assert lib.rocm_launch_swiglu(at(g), at(u), C.c_int64(gate.size), dtype, int(decomposed), at(y), None) == 0
    torch.cuda.synchronize()
    out = y.cpu().numpy().view(np.uint16)
    assert (out[:offset] == 0x5555).all() and (out[offset + gate.size:] == 0x5555).all()
    return out[offset:offset + gate.size]


def _same(got, want, dtype):
    exponent, magnitude = (0x7C00, 0x7FFF) if dtype == E.F16 else (0x7F80, 0x7FFF)
    nan = (want & magnitude) > exponent
    assert np.array_equal((got & magnitude) > exponent, nan)
    assert np.array_equal(got[~nan], want[~nan])


@pytest.mark.parametrize("decomposed", [False, True])
@pytest.mark.parametrize("dtype", [E.F16, E.BF16])
def test_every_gate_value(ep, port, dtype, decomposed):
    """Bit-equal for all 65536 gate values (signed zeros, denormals, infinities; a NaN stays one) under several up values."""
    o_dt = oracle.F16 if dtype == E.F16 else oracle.BF16
    gate = np.arange(65536, dtype=np.uint16)
    for value in (1.0, -0.37109375, 3000.0, 2.0 ** -20):
        up = port.narrow(np.full(65536, value, np.float32), o_dt).view(np.uint16)
        want = np.asarray(port.swiglu(gate, up, o_dt, decomposed)).view(np.uint16)
        _same(_launch(ep, gate, up, dtype, decomposed), want, dtype)


@pytest.mark.parametrize("count,offset", [(1, 0), (7, 0), (8, 0), (2055, 0), (2055, 1), (64, 4)])
def test_pieces_and_remainders(ep, port, count, offset):
    rng = np.random.default_rng(count + offset)
    gate, up = (rng.standard_normal(count).astype(np.float16).view(np.uint16) for _ in range(2))
    want = np.asarray(port.swiglu(gate, up, oracle.F16, False)).view(np.uint16)
    _same(_launch(ep, gate, up, E.F16, False, offset), want, E.F16)
