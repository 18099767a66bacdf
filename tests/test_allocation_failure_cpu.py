"""Calls whose device allocations fail, on the host side alone: the provider's sources linked against functions that stand for the GPU's."""
import os
import subprocess

import numpy as np
import pytest

from onnx_genai_amd import build
from onnx_genai_amd import ep as E

# What the GPU side answers where a zero would not do: one device, memory from the host's heap, groups that are whole blocks.
ANSWERS = {
    "rocm_ffi_error_string": "const char* rocm_ffi_error_string(int) { return \"out of memory\"; }",
    "rocm_ffi_device_count": "int rocm_ffi_device_count(int* n) { *n = 1; return 0; }",
    "rocm_ffi_malloc": "int rocm_ffi_malloc(void** p, size_t n) { if (failures_due > 0) { --failures_due; return 2; } *p = std::calloc(1, n); return 0; }",
    "rocm_ffi_free": "int rocm_ffi_free(void* p) { std::free(p); return 0; }",
    "rocm_g_idx_first_bad": "int rocm_g_idx_first_bad(const int32_t*, int64_t, int64_t, int64_t* bad, void*) { *bad = -1; return 0; }",
    "rocm_gidx_order": "int rocm_gidx_order(const int32_t*, int64_t, int, int32_t*, int* regular, void*) { *regular = 1; return 0; }",
}


@pytest.fixture(scope="module")
def host_only(tmp_path_factory):
    """The library's host sources with every other function of the GPU side answering zero; `failures_due`: allocations that are to fail."""
    where = tmp_path_factory.mktemp("host")
    objects = []
    for source in build.HOST_SOURCES:
        objects.append(str(where / (os.path.basename(source) + ".o")))
        subprocess.run(["g++", "-std=c++17", "-O0", "-fPIC", "-c", os.path.join(build.CSRC, source), "-o", objects[-1]], check=True)
    undefined = subprocess.run(["nm", "-u", *objects], check=True, capture_output=True, text=True).stdout.split()
    names = sorted({n for n in undefined if n.startswith("rocm_")})
    with open(where / "gpu.cpp", "w") as f:
        f.write("#include <cstdint>\n#include <cstdlib>\nextern \"C\" {\nint failures_due = 0;\n")
        f.writelines(ANSWERS.get(n, f"long {n}() {{ return 0; }}") + "\n" for n in names)
        f.write("}\n")
    library = str(where / "host_only.so")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-o", library, *objects, str(where / "gpu.cpp"), "-ldl"], check=True)
    with pytest.MonkeyPatch.context() as patch:
        patch.setattr(E, "LIB_PATH", library)
        patch.setattr(E, "_lib", None)
        yield E.load_library()


def test_act_order_weights_are_sorted_once_there_is_memory(host_only):
    """Without memory for the sorted copy a call is served unsorted; the next one asks again."""
    n, k, bs = 8, 64, 32
    provider = E.RocmExecutionProvider(0)
    failures = E.C.c_int.in_dll(host_only, "failures_due")
    arrays = [np.zeros(k, np.float16), np.zeros((n, k // bs, bs // 2), np.uint8), np.zeros((n, k // bs), np.float16), np.zeros((n, 1), np.uint8), np.zeros(k, np.int32), np.zeros(n, np.float16)]
    a, b, s, z, g, y = (E.TensorView(x.ctypes.data, dt, shape) for x, dt, shape in zip(
        arrays, (E.F16, E.U8, E.F16, E.U8, E.I32, E.F16), ((1, k), (n, k // bs, bs // 2), (n, k // bs), (n, 1), (k,), (1, n))))
    kernel = provider.get_kernel({"K": k, "N": n, "bits": 4, "block_size": bs})
    kernel.set_constant_inputs([False, True, True, True, True])
    try:
        variants = []
        for due in (1, 0):
            failures.value = due
            kernel.execute([a, b, s, z, g], [y])
            assert failures.value == 0
            variants.append(kernel.last_variant())
        assert not variants[0].startswith("act_order+") and variants[1].startswith("act_order+"), variants
    finally:
        kernel.release()
        provider.shutdown()
