"""The native call path of ep.py: the records that reach the C ABI are those of the packed views, and what is not plain is left alone."""
import ctypes as C
import os
import shutil
import subprocess
import sys
import sysconfig

import numpy as np
import pytest

from onnx_genai_amd import build
from onnx_genai_amd import ep as E

SOURCE = r"""
#include <stdint.h>
#include <string.h>
typedef struct { void* data; uint32_t dtype, ndim; const uint64_t* shape; const int64_t* strides; uint64_t byte_offset; uint32_t device_type, device_index; } View;
typedef struct { uint32_t code, message_len; uint8_t message[256]; } Status;
int64_t seen[4096]; int used = 0; uint32_t code = 0;
static void put(const View* v, uint32_t n)
{
    for (uint32_t i = 0; i < n; ++i) {
        const int64_t head[7] = {(int64_t)(uintptr_t)v[i].data, v[i].dtype, v[i].ndim, (int64_t)v[i].byte_offset, v[i].device_type, v[i].device_index, v[i].strides != 0};
        memcpy(seen + used, head, sizeof(head));
        used += 7;
        for (uint32_t d = 0; d < v[i].ndim; ++d) seen[used++] = (int64_t)v[i].shape[d];
        if (v[i].strides) for (uint32_t d = 0; d < v[i].ndim; ++d) seen[used++] = v[i].strides[d];
    }
}
Status record(void* kernel, const View* in, uint32_t n_in, View* out, uint32_t n_out, void* workspace, uint64_t bytes)
{
    Status s = {code, 5, "wrong"};
    used = 0;
    seen[used++] = (int64_t)(uintptr_t)kernel; seen[used++] = n_in; seen[used++] = n_out; seen[used++] = (int64_t)(uintptr_t)workspace; seen[used++] = (int64_t)bytes;
    put(in, n_in);
    put(out, n_out);
    return s;
}
"""


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    where = tmp_path_factory.mktemp("calls")
    (where / "record.c").write_text(SOURCE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(where / "record.c"), "-o", str(where / "record.so")], check=True)
    return C.CDLL(str(where / "record.so"))


def call(lib, inputs, outputs):
    return E._calls.execute(C.cast(lib.record, C.c_void_p).value, 0x77, inputs, outputs, 0x88, 99)


def test_records_are_those_of_the_views(recorder):
    inputs = [E.TensorView(0x7FFF_FFFF_F000, E.F32, (2, 3, 896)), E.TensorView.absent(E.U8),
              E.TensorView(0x2000, E.BF16, (4, 8), strides=(-16, 2), byte_offset=2**40, device_type=5, device_index=7), E.TensorView(0x4000, E.F16, ())]
    outputs = (E.TensorView(0x5000, E.F16, (1, 2**33)),)
    want = [0x77, len(inputs), 1, 0x88, 99]
    for v in (*inputs, *outputs):
        want += [v.data or 0, v.dtype, len(v.shape), v.byte_offset, v.device_type, v.device_index, int(v.strides is not None), *v.shape, *(v.strides or ())]
    assert call(recorder, inputs, outputs) is None
    assert list((C.c_int64 * len(want)).in_dll(recorder, "seen")) == want
    assert C.c_int.in_dll(recorder, "used").value == len(want)


def test_a_status_comes_back_with_its_message(recorder):
    code = C.c_uint32.in_dll(recorder, "code")
    code.value = 3
    try:
        assert call(recorder, [], []) == (3, b"wrong")
    finally:
        code.value = 0


@pytest.mark.parametrize("view", [
    E.TensorView(C.c_void_p(0x6000), E.F32, (4,)), E.TensorView(0x10, E.F32, (np.int64(4),)), E.TensorView(0x10, E.F32, (-1,)), E.TensorView(0x10, E.F32, [4]),
    E.TensorView(0x10, 2**32, (4,)), E.TensorView(0x10, E.F32, (4,), byte_offset=-1), E.TensorView(-16, E.F32, (4,)), E.TensorView(0x10, E.F32, (4, 4), strides=(1,)),
    E.TensorView(0x10, E.F32, (1,) * 9), E.TensorView(0x10, True, (4,)), object()])
def test_what_is_not_plain_is_left_alone(recorder, view):
    C.c_int.in_dll(recorder, "used").value = -1
    assert call(recorder, [view], []) is False
    assert call(recorder, [], [view]) is False
    assert call(recorder, iter([]), []) is False
    assert call(recorder, [E.TensorView.absent()] * 17, []) is False
    assert C.c_int.in_dll(recorder, "used").value == -1


def execute(lib, inputs, outputs, workspace=None):
    """The public execute of a kernel whose library is the recorder; -> what the recorder saw."""
    kernel = E.MatMulNBitsKernel.__new__(E.MatMulNBitsKernel)
    lib.execute_at = C.cast(lib.record, C.c_void_p).value
    lib.nxrt_rocm_matmul_nbits_execute = lib.record
    lib.record.restype = E.NxrtStatus
    lib.record.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p, C.c_uint32, C.c_void_p, C.c_uint64]
    kernel.lib, kernel.handle = lib, C.c_void_p(0x77)
    kernel.execute(inputs, outputs, workspace)
    return list((C.c_int64 * C.c_int.in_dll(lib, "used").value).in_dll(lib, "seen"))


def test_calls_without_the_native_path_are_the_same(recorder, monkeypatch):
    inputs = [E.TensorView(0x1000, E.F32, (2, 3, 896)), E.TensorView.absent(E.U8), E.TensorView(0x2000, E.BF16, (4, 8), strides=(-16, 2), byte_offset=32)]
    outputs, workspace = [E.TensorView(0x5000, E.F16, (1, 4))], E.DeviceBuffer(0x9000, 512)
    want = execute(recorder, inputs, outputs, workspace)
    code = C.c_uint32.in_dll(recorder, "code")
    messages = []
    for native in (E._calls, None):
        monkeypatch.setattr(E, "_calls", native)
        assert execute(recorder, inputs, outputs, workspace) == want
        code.value = 3
        try:
            with pytest.raises(E.EpError) as failed:
                execute(recorder, inputs, outputs)
        finally:
            code.value = 0
        messages.append((failed.value.code, failed.value.message))
    assert messages == [(3, "wrong")] * 2


def test_the_package_imports_in_a_tree_that_is_not_built(tmp_path):
    """Only loading the library asks for a build; a module of another interpreter's name is not taken."""
    package = tmp_path / "onnx_genai_amd"
    shutil.copytree(build.HERE, package, ignore=lambda where, names: [n for n in names if n in ("build", "lib", "csrc", "__pycache__") or n.endswith(".so")])
    (package / "_calls.cpython-399-x86_64-linux-gnu.so").write_bytes(b"of another interpreter")
    code = "from onnx_genai_amd import ep\nassert ep._calls is None and ep.__file__.startswith({!r}), ep.__file__\ntry:\n    ep.load_library()\nexcept (OSError, RuntimeError) as e:\n    print('refused', e)"
    env = {k: v for k, v in os.environ.items() if k not in ("NXRT_ROCM_LIBRARY", "PYTHONPATH")}
    out = subprocess.run([sys.executable, "-c", code.format(str(tmp_path))], cwd=tmp_path, env=env, capture_output=True, text=True)
    assert out.returncode == 0 and "refused" in out.stdout, out.stdout + out.stderr


def test_the_module_carries_its_interpreter():
    assert E._calls.__file__ == build.CALLS and build.CALLS.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
