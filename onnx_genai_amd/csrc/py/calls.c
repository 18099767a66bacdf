/* execute for the Python mirror of the provider's interface: reads the tensor views of a call, hands them to the library as the C ABI's records and calls it,
 * in one step. A short node (one row, 896 -> 4864) takes 4 us on the GPU, and packing its views in Python and passing them through ctypes took about as
 * long again. Views whose fields are not plain integers are left to the caller, which packs those itself. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

typedef struct {
    void* data;
    uint32_t dtype, ndim;
    const uint64_t* shape;
    const int64_t* strides;
    uint64_t byte_offset;
    uint32_t device_type, device_index;
} View;

typedef struct {
    uint32_t code, message_len;
    uint8_t message[256];
} Status;

typedef Status (*execute_fn)(void*, const View*, uint32_t, View*, uint32_t, void*, uint64_t);

enum { kMaxViews = 16, kMaxDims = 8 };

static PyObject *s_data, *s_dtype, *s_shape, *s_strides, *s_byte_offset, *s_device_type, *s_device_index;

/* 1: *out is the integer's value; 0: not a plain integer of that range */
static int plain(PyObject* o, uint64_t max, uint64_t* out)
{
    if (!o || !PyLong_CheckExact(o)) return 0;
    const unsigned long long v = PyLong_AsUnsignedLongLong(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) {
        PyErr_Clear();
        return 0;
    }
    *out = v;
    return v <= max;
}

static int read_view(PyObject* view, View* to, uint64_t* shape, int64_t* strides)
{
    PyObject* fields = PyObject_GenericGetDict(view, NULL);
    if (!fields) {
        PyErr_Clear();
        return 0;
    }
    int ok = 0;
    uint64_t dtype, offset, type, index, at = 0;
    PyObject* const data = PyDict_GetItemWithError(fields, s_data);
    PyObject* const dims = PyDict_GetItemWithError(fields, s_shape);
    PyObject* const steps = PyDict_GetItemWithError(fields, s_strides);
    if (!data || !dims || !steps || !PyTuple_CheckExact(dims) || PyTuple_GET_SIZE(dims) > kMaxDims) goto done;
    if (data != Py_None && !plain(data, UINT64_MAX, &at)) goto done;
    if (!plain(PyDict_GetItemWithError(fields, s_dtype), UINT32_MAX, &dtype) || !plain(PyDict_GetItemWithError(fields, s_byte_offset), UINT64_MAX, &offset) ||
        !plain(PyDict_GetItemWithError(fields, s_device_type), UINT32_MAX, &type) || !plain(PyDict_GetItemWithError(fields, s_device_index), UINT32_MAX, &index))
        goto done;
    const Py_ssize_t ndim = PyTuple_GET_SIZE(dims);
    for (Py_ssize_t i = 0; i < ndim; ++i)
        if (!plain(PyTuple_GET_ITEM(dims, i), UINT64_MAX, &shape[i])) goto done;
    to->strides = NULL;
    if (steps != Py_None) {
        if (!PyTuple_CheckExact(steps) || PyTuple_GET_SIZE(steps) != ndim) goto done;
        for (Py_ssize_t i = 0; i < ndim; ++i) {
            PyObject* const o = PyTuple_GET_ITEM(steps, i);
            if (!PyLong_CheckExact(o)) goto done;
            strides[i] = PyLong_AsLongLong(o);
            if (strides[i] == -1 && PyErr_Occurred()) goto done;
        }
        to->strides = strides;
    }
    to->data = (void*)(uintptr_t)at;
    to->dtype = (uint32_t)dtype;
    to->ndim = (uint32_t)ndim;
    to->shape = shape;
    to->byte_offset = offset;
    to->device_type = (uint32_t)type;
    to->device_index = (uint32_t)index;
    ok = 1;
done:
    PyErr_Clear();
    Py_DECREF(fields);
    return ok;
}

/* execute(function address, kernel address, inputs, outputs, workspace address, workspace bytes) -> None; (code, message) of a call that failed; False where
 * the views are not plain (nothing was called) */
static PyObject* execute(PyObject* self, PyObject* const* args, Py_ssize_t n)
{
    (void)self;
    if (n != 6) {
        PyErr_SetString(PyExc_TypeError, "execute takes six arguments");
        return NULL;
    }
    uint64_t function, kernel, workspace, bytes;
    if (!plain(args[0], UINT64_MAX, &function) || !plain(args[1], UINT64_MAX, &kernel) || !plain(args[4], UINT64_MAX, &workspace) || !plain(args[5], UINT64_MAX, &bytes)) Py_RETURN_FALSE;
    View views[kMaxViews];
    uint64_t shapes[kMaxViews][kMaxDims];
    int64_t strides[kMaxViews][kMaxDims];
    uint32_t count[2] = {0, 0}, used = 0;
    for (int side = 0; side < 2; ++side) {
        PyObject* const list = args[2 + side];
        const int is_list = PyList_CheckExact(list);
        if (!is_list && !PyTuple_CheckExact(list)) Py_RETURN_FALSE;
        const Py_ssize_t size = is_list ? PyList_GET_SIZE(list) : PyTuple_GET_SIZE(list);
        if (size > kMaxViews - (Py_ssize_t)used) Py_RETURN_FALSE;
        count[side] = (uint32_t)size;
        for (Py_ssize_t i = 0; i < size; ++i, ++used)
            if (!read_view(is_list ? PyList_GET_ITEM(list, i) : PyTuple_GET_ITEM(list, i), &views[used], shapes[used], strides[used])) Py_RETURN_FALSE;
    }
    Status status;
    Py_BEGIN_ALLOW_THREADS
    status = ((execute_fn)(uintptr_t)function)((void*)(uintptr_t)kernel, views, count[0], views + count[0], count[1], (void*)(uintptr_t)workspace, bytes);
    Py_END_ALLOW_THREADS
    if (status.code == 0) Py_RETURN_NONE;
    const uint32_t len = status.message_len < sizeof(status.message) ? status.message_len : (uint32_t)sizeof(status.message);
    return Py_BuildValue("(Iy#)", status.code, (const char*)status.message, (Py_ssize_t)len);
}

static PyMethodDef methods[] = {{"execute", (PyCFunction)(void (*)(void))execute, METH_FASTCALL, "One call of a kernel's execute."}, {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__calls(void)
{
    struct { PyObject** to; const char* name; } names[] = {{&s_data, "data"}, {&s_dtype, "dtype"}, {&s_shape, "shape"}, {&s_strides, "strides"},
                                                           {&s_byte_offset, "byte_offset"}, {&s_device_type, "device_type"}, {&s_device_index, "device_index"}};
    for (size_t i = 0; i < sizeof(names) / sizeof(names[0]); ++i)
        if (!(*names[i].to = PyUnicode_InternFromString(names[i].name))) return NULL;
    return PyModule_Create(&module);
}
