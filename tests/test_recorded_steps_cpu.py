"""What the workgroups of a recorded launch read of repacked weights lies within their node's copy, and is all of it. No GPU work."""
import ctypes as C
import itertools

import pytest

from onnx_genai_amd import build


class _Nodes(C.Structure):
    _fields_ = [("nodes", C.c_int), ("columns", C.c_int * 4), ("packed", C.c_void_p * 4), ("stream", C.c_uint32)]


class _Reads(C.Structure):
    _fields_ = [("grid", C.c_uint32), ("rows", C.c_uint32), ("first", C.c_uint64), ("bytes", C.c_uint64)]


def launch_of(widths, stream):
    """A launch's nodes with their copies far apart, and (begin, end) of each copy."""
    copies = [((i + 1) << 40, ((i + 1) << 40) + (n + 15) // 16 * stream) for i, n in enumerate(widths)]
    return _Nodes(len(widths), (*widths,), (*(begin for begin, _ in copies),), stream), copies


def orders():
    for widths in [(16, 33, 896), (128, 128, 896), (15, 16), (17, 4864), (256, 8192), (16, 48, 17, 128), (1, 1, 1, 1), (2048, 151936), (896, 896, 4864, 4864)]:
        yield from sorted(set(itertools.permutations(widths)))


@pytest.mark.parametrize("widths", orders(), ids=str)
def test_a_shared_launch_reads_within_the_copies(widths):
    lib = C.CDLL(build.LIB)
    stream = 9216
    nodes, copies = launch_of(widths, stream)
    out = _Reads()
    if lib.rocm_step_reads(C.byref(nodes), 0, 0, C.byref(out)) != 0:
        assert max(widths) * len(widths) > 2 * sum(widths)                          # (too many workgroups without columns: launches of their own)
        return
    grid, rows = out.grid, out.rows
    assert rows == len(widths) and grid == (max(widths) + 15) // 16
    for y, (begin, end) in enumerate(copies):
        at = begin
        for x in range(grid):
            assert lib.rocm_step_reads(C.byref(nodes), x, y, C.byref(out)) == 0
            if out.bytes:
                assert out.first == at and out.bytes == stream and at + stream <= end
                at += stream
        assert at == end
