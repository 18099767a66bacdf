"""Which build, wave count and register sets the launchers pick for the benchmark configurations' shapes, held against the
committed table tests/golden/dispatch_table.json (no GPU work: the planning entry points only do arithmetic on shapes).

The launch rules hold dozens of measured thresholds; correctness of whatever they pick is covered by the GPU tests, but
nothing else would notice a rule tuned for one shape quietly moving a benchmark shape to another build.
"""
import ctypes as C
import json
import os

import pytest

from onnx_genai_amd import build
from tests.golden import make_dispatch_table as T

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(build.LIB):
        pytest.skip("library not built")
    return T.load()


def test_benchmark_shapes_keep_their_launch_plans(lib):
    with open(os.path.join(HERE, "golden", "dispatch_table.json")) as f:
        want = json.load(f)
    got = T.table(lib)
    assert len(got) == len(want) == 4 * 10 + 6 + 3
    for g, w in zip(got, want):
        assert g == w, f"launch plan moved:\n  now  {g}\n  was  {w}\n(if intended: python tests/golden/make_dispatch_table.py, and review the diff)"


def test_headline_decode_step_plans(lib):
    """The five calls of the Qwen2.5-7B decode step at one row, spelled out: one tile group of 512 k per wave (three on the
    long K), one register set, the activation-sums form, sixteen columns per workgroup."""
    rows = {(r["shape"], r["m"]): r for r in T.table(lib) if r["config"] == "configs[2]"}
    for shape, waves, groups, workgroups in [("qkv", 7, 1, 288), ("o", 7, 1, 224), ("gate_up", 7, 1, 2368), ("down", 13, 3, 224), ("lm_head", 7, 1, 9504)]:
        r = rows[(shape, 1)]
        assert (r["shared_activations"], r["rows_build"], r["waves"], r["groups_per_wave"], r["register_sets"], r["activation_sums"], r["workgroups"]) == \
            (0, 1, waves, groups, 1, 1, workgroups), r
    # 16 rows: the wide shapes share one LDS copy of the activations; gate/up spreads its 2368 column groups over one workgroup per CU
    r = rows[("gate_up", 16)]
    assert r["shared_activations"] == 1 and r["waves"] == 10 and r["workgroups"] == 237
    assert rows[("lm_head", 16)]["shared_activations"] == 1 and rows[("down", 16)]["shared_activations"] == 0


def test_plans_follow_the_compute_unit_count(lib):
    """The CU count is an input of the plan, not a literal: on a chip of 304 CUs the gate/up grid at 16 rows is no longer
    'between one and one and a half workgroups per CU' and keeps eight waves a workgroup."""
    a = T.ffi_args(T.BF16, 128, True, 16, 37888, 3584)
    p256, p304 = T.DecodePlan(), T.DecodePlan()
    assert lib.rocm_decode_packed_plan(C.byref(a), 0, 0, 256, C.byref(p256)) == 0
    assert lib.rocm_decode_packed_plan(C.byref(a), 0, 0, 304, C.byref(p304)) == 0
    assert (p256.waves, p256.workgroups) == (10, 237)
    assert (p304.waves, p304.workgroups) == (8, 296)
    # a mid-size split-K grid fits more waves on more CUs
    b = T.ffi_args(T.BF16, 128, True, 16, 13824, 5120)
    q128, q256 = T.DecodePlan(), T.DecodePlan()
    assert lib.rocm_decode_packed_plan(C.byref(b), 0, 0, 128, C.byref(q128)) == 0
    assert lib.rocm_decode_packed_plan(C.byref(b), 0, 0, 256, C.byref(q256)) == 0
    assert q128.waves <= q256.waves and q128.waves * q128.groups_per_wave >= 10 and q256.waves * q256.groups_per_wave >= 10
    assert lib.rocm_decode_packed_plan(C.byref(a), 0, 0, 0, C.byref(p256)) == -1


def test_acc4_calls_that_take_the_taller_tiles(lib):
    """accuracy_level 4: 256 x 128 tiles where their grid fills its rounds, from K = 8192 at block 128 and never at block 32; the same shares of a smaller chip."""
    def rows(m, n, k, bs, cus=256):
        out = C.c_int()
        assert lib.rocm_acc4_mfma_plan(C.byref(T.ffi_args(T.F16, bs, True, m, n, k)), cus, C.byref(out), None) == 0
        return out.value
    assert rows(4096, 57344, 8192, 64) == rows(2048, 10240, 8192, 64) == rows(512, 28672, 4096, 64) == rows(512, 57344, 8192, 128) == 256
    assert rows(768, 37888, 3584, 64) == rows(600, 57344, 8192, 64) == rows(2048, 10240, 8192, 128) == rows(4096, 37888, 3584, 128) == rows(4096, 57344, 8192, 32) == 128
    assert rows(512, 14336, 4096, 64, cus=128) == 256 and rows(512, 14336, 4096, 64) == 128


@pytest.mark.parametrize("m,n,k,bs,height,runs", [
    # block size 32 and 256 x 128 tiles: runs of tiles
    (777, 4864, 896, 32, 128, True),             # 266 tiles of 128 x 128, nine rows in the last row block
    (130, 37888, 3584, 32, 128, True),           # two rows in the last of two row blocks
    (1200, 12763, 4096, 64, 256, True),          # 5 x 100: a band of four whole row blocks, and one of 176 rows
    (2304, 7040, 4096, 64, 256, True),           # 9 x 55: bands of four, four and one row block
    (385, 16384, 64, 64, 256, True),             # one whole row block and one of 129 rows
    (60, 37888, 3584, 32, 128, True),            # one row block, not whole
    # wide grids whose rows of B are a multiple of 4096 (2048) bytes apart
    (300, 57300, 8192, 64, 128, True), (17, 16384, 16384, 128, 128, True), (100, 45056, 4096, 64, 128, True),
    # the others keep launch order
    (777, 4864, 896, 64, 128, False), (1300, 6144, 4096, 64, 128, False), (600, 10240, 8192, 64, 128, False), (300, 32768, 4096, 64, 128, False),
    (300, 32768, 8448, 64, 128, False), (130, 4608, 3584, 128, 128, False),
])
def test_acc4_tiles_are_handed_out_once_and_partial_rows_last(lib, m, n, k, bs, height, runs):
    """accuracy_level 4, tall calls: workgroups to tiles is one-to-one, and the tiles of a last row block that is not whole come behind all others."""
    args = T.ffi_args(T.F16, bs, True, m, n, k)
    planned, row, col = C.c_int(), C.c_int64(), C.c_int64()
    assert lib.rocm_acc4_mfma_plan(C.byref(args), 256, C.byref(planned), None) == 0 and planned.value == height
    rows, cols = -(-m // height), -(-n // 128)
    tiles = []
    for w in range(rows * cols):
        assert lib.rocm_acc4_mfma_tile(C.byref(args), 256, C.c_int64(w), C.byref(row), C.byref(col)) == 0
        tiles.append((row.value, col.value))
    assert sorted(tiles) == [(r, c) for r in range(rows) for c in range(cols)]
    assert (tiles == sorted(tiles)) == (not runs)
    if m % height:
        assert {r for r, _ in tiles[(rows - 1) * cols:]} == {rows - 1}
    if runs:                                  # an XCD's first tiles are neighbours
        mine = tiles[0::8]
        assert mine[1] in ((mine[0][0] + 1, mine[0][1]), (mine[0][0], mine[0][1] + 1))
    assert lib.rocm_acc4_mfma_tile(C.byref(args), 256, C.c_int64(rows * cols), C.byref(row), C.byref(col)) == -1
