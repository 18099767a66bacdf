"""What the workgroups of a recorded launch read of repacked weights lies within their node's copy, and is all of it. No GPU work."""
import ctypes as C
import itertools

import pytest

from onnx_genai_amd import build
from tests.test_weights_ahead_cpu import _Ahead


class _Nodes(C.Structure):
    _fields_ = [("nodes", C.c_int), ("columns", C.c_int * 4), ("packed", C.c_void_p * 4), ("stream", C.c_uint32), ("threads", C.c_uint32)]


class _Reads(C.Structure):
    _fields_ = [("grid", C.c_uint32), ("rows", C.c_uint32), ("ahead", C.c_uint32), ("first", C.c_uint64), ("bytes", C.c_uint64)]


def launch_of(widths, stream, threads=256, base=1):
    """A launch's nodes with their copies far apart, and (begin, end) of each copy."""
    copies = [((i + base) << 40, ((i + base) << 40) + (n + 15) // 16 * stream) for i, n in enumerate(widths)]
    return _Nodes(len(widths), (*widths,), (*(begin for begin, _ in copies),), stream, threads), copies


def orders():
    for widths in [(16, 33, 896), (128, 128, 896), (15, 16), (17, 4864), (256, 8192), (16, 48, 17, 128), (1, 1, 1, 1), (2048, 151936), (896, 896, 4864, 4864)]:
        yield from sorted(set(itertools.permutations(widths)))


@pytest.mark.parametrize("widths", orders(), ids=str)
def test_a_shared_launch_reads_within_the_copies(widths):
    lib = C.CDLL(build.LIB)
    stream = 9216
    nodes, copies = launch_of(widths, stream)
    out = _Reads()
    if lib.rocm_step_reads(C.byref(nodes), None, 0, 0, C.byref(out)) != 0:
        assert max(widths) * len(widths) > 2 * sum(widths)                          # (too many workgroups without columns: launches of their own)
        return
    grid, rows = out.grid, out.rows
    assert rows == len(widths) and grid == (max(widths) + 15) // 16
    for y, (begin, end) in enumerate(copies):
        at = begin
        for x in range(grid):
            assert lib.rocm_step_reads(C.byref(nodes), None, x, y, C.byref(out)) == 0
            if out.bytes:
                assert out.first == at and out.bytes == stream and at + stream <= end
                at += stream
        assert at == end


def check_ahead(blocks, copies, stream, workgroups):
    """[(block, first, bytes)] that are read ahead: the shares of the first `workgroups` of each copy, whole, each byte once, by blocks of the XCD of the workgroup they are for."""
    read = {}
    for block, first, count in blocks:
        copy = next((begin, end) for begin, end in copies if begin <= first < end)
        assert first % 16 == 0 and first + count <= copy[1]
        workgroup = (first - copy[0]) // stream
        assert first + count <= copy[0] + (workgroup + 1) * stream and block % 8 == workgroup % 8 and workgroup < workgroups
        read.setdefault(copy, []).append((first, first + count))
    for copy, ranges in read.items():
        ranges.sort()
        assert ranges[0][0] == copy[0] and ranges[-1][1] == copy[0] + workgroups * stream
        assert all(a[1] == b[0] for a, b in zip(ranges, ranges[1:]))
    return len(read)


# the launch's widths, the next one's, its bytes to 16 columns, threads of a workgroup, copies that are read ahead
CHAINS = [
    ((896,), (4864,), 9216, 320, 1),
    ((896, 128, 128), (896,), 9216, 128, 1),
    ((16,), (4864, 4864), 9216, 320, 2),                     # two streams
    ((72,), (4864, 896), 9216, 64, 2),                       # the second one narrower: as many of each
    ((304,), (896, 4864), 18432, 1024, 2),                   # the first one narrower
    ((72,), (130, 4864, 17), 9216, 256, 2),                  # nine workgroups of the first, and the third is not read
    ((72,), (100, 4864, 17), 9216, 256, 0),                  # fewer than eight of the first
    ((33,), (1000, 1000), 4224, 448, 1),                     # a grid that is no multiple of eight: the second one lies on other XCDs
    ((16, 48, 17, 128), (152064,), 145920, 896, 1),          # more than fits the budget
    ((3584,), (37888,), 145920, 1024, 1),
    ((896,), (16,), 145920, 64, 0),                          # too narrow
    ((152064,), (3584,), 145920, 1024, 0),                   # not a short launch
]


@pytest.mark.parametrize("widths,next_widths,stream,threads,streams", CHAINS, ids=str)
def test_a_short_launch_reads_the_next_ones_copies(widths, next_widths, stream, threads, streams):
    lib = C.CDLL(build.LIB)
    nodes, copies = launch_of(widths, 2304 if streams else stream, threads)
    behind, next_copies = launch_of(next_widths, stream, threads, base=9)
    out = _Reads()
    assert lib.rocm_step_reads(C.byref(nodes), C.byref(behind), 0, 0, C.byref(out)) == 0
    grid, rows, ahead = out.grid, out.rows, out.ahead
    seen = []
    for y in range(rows):
        for x in range(grid):
            assert lib.rocm_step_reads(C.byref(nodes), C.byref(behind), x, y, C.byref(out)) == 0
            if y < len(widths):                              # its own columns, as with nothing behind it
                assert out.bytes == 0 or copies[y][0] <= out.first and out.first + out.bytes <= copies[y][1]
            elif out.bytes:
                seen.append((y * grid + x, out.first, out.bytes))
    assert check_ahead(seen, next_copies, stream, ahead) == streams
    assert (ahead > 0) == (streams > 0) and (rows > len(widths)) == (streams > 0)


@pytest.mark.parametrize("columns,stream,pair,rows,budget", [
    (4608, 8640, False, 1, 8000000), (4608, 69120, False, 16, 8000000), (37888, 69120, False, 1, 8000000), (18944, 69120, True, 4, 8000000), (18944, 276480, True, 16, 8000000),
    (100, 8640, True, 7, 8000000), (112, 8640, False, 64, 8000000), (2000, 16, False, 3, 8000000), (2000, 16, True, 9, 1000), (4096, 304 * 1024, False, 8, 8000000)])
def test_a_normalization_reads_the_next_launchs_copies(columns, stream, pair, rows, budget):
    lib = C.CDLL(build.LIB)
    lib.rocm_weights_ahead_reads.restype = C.c_uint64
    workgroups = columns // 16
    copies = [((i + 1) << 40, ((i + 1) << 40) + workgroups * stream) for i in range(2 if pair else 1)]
    description = _Ahead(copies[0][0], copies[1][0] if pair else None, stream, workgroups)
    out = _Reads()
    each = lambda block: lib.rocm_weights_ahead_reads(C.byref(description), C.c_uint64(budget), 256, rows, block, C.byref(out))  # noqa: E731
    blocks, ahead, seen = each(0), out.ahead, []
    for block in range(blocks):
        each(block)
        assert block >= rows or out.bytes == 0               # (the rows' own blocks)
        if out.bytes:
            seen.append((block, out.first, out.bytes))
    assert ahead == min(workgroups, budget // (stream * len(copies))) // 8 * 8
    assert check_ahead(seen, copies, stream, ahead) == (len(copies) if ahead else 0)
    assert sum(count for _, _, count in seen) <= budget
