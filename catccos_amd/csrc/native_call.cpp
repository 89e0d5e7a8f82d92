// What the Python front end does for every call, in native code: output tensors, pointers out of tensors, the call itself.
// A call of ops.py launches one to five kernels and returns; a small one costs the host more than the GPU (quantizer of 16 rows 9.2 us, of which
// the launch 3.0, two torch.empty 3.4 and ctypes 0.5, where the kernel runs 3.3).  Here a tensor is 0.7 us and a call of 15 arguments 0.1:
// quantizer 9.2 -> 5.8 us, dense matmul 7.8 -> 5.3; the two in turn at 16 x 4096 x 7168 17.0 -> 12.2, which is what their kernels take.
//
//   run(address, *args)              int(*)(...) at `address`: tensors by their data pointer, None as null, integers (anything with __index__); ValueError for a tensor
//                                    that is not on the GPU.  Without the GIL, like a ctypes call.
//   empty(like, dtype, size, ...)    torch.empty on the device of `like`, which is a GPU (ValueError)
//
// Every entry point of the C ABI takes integers and pointers only, each of which has a register or an 8-byte slot of its own in
// the x86-64 System V convention, so one function type of kMaxArgs such arguments calls them all.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#if !defined(__x86_64__) || defined(_WIN32)
#error "x86-64 System V calling convention"
#endif

namespace {

constexpr Py_ssize_t kMaxArgs = 24;

PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 1 || n > 1 + kMaxArgs) {
        PyErr_SetString(PyExc_TypeError, "run(address, up to 24 arguments)");
        return nullptr;
    }
    const uint64_t address = PyLong_AsUnsignedLongLong(args[0]);
    if (address == 0 || PyErr_Occurred()) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
        return nullptr;
    }
    uint64_t v[kMaxArgs] = {};
    for (Py_ssize_t i = 1; i < n; ++i) {
        PyObject* const o = args[i];
        if (PyLong_Check(o)) {
            v[i - 1] = PyLong_AsUnsignedLongLongMask(o);
            if (v[i - 1] == (uint64_t)-1 && PyErr_Occurred()) return nullptr;
        } else if (THPVariable_Check(o)) {
            const at::Tensor& t = THPVariable_Unpack(o);
            if (!t.is_cuda()) {
                PyErr_SetString(PyExc_ValueError, "expected a GPU tensor");
                return nullptr;
            }
            v[i - 1] = reinterpret_cast<uint64_t>(t.data_ptr());
        } else if (PyIndex_Check(o)) {                                   // numpy's integers
            v[i - 1] = PyLong_AsUnsignedLongLongMask(o);
            if (v[i - 1] == (uint64_t)-1 && PyErr_Occurred()) return nullptr;
        } else if (o != Py_None) {
            PyErr_Format(PyExc_TypeError, "argument %zd: a tensor, an integer or None, not %s", i, Py_TYPE(o)->tp_name);
            return nullptr;
        }
    }
    using u = uint64_t;
    using Fn = int (*)(u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u);
    const Fn fn = reinterpret_cast<Fn>(address);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11], v[12], v[13], v[14], v[15], v[16], v[17], v[18], v[19],
            v[20], v[21], v[22], v[23]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
    END_HANDLE_TH_ERRORS
}

PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 3 || n > 6 || !THPVariable_Check(args[0]) || !THPDtype_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "empty(tensor, dtype, one to four sizes)");
        return nullptr;
    }
    int64_t size[4];
    for (Py_ssize_t i = 2; i < n; ++i) {
        size[i - 2] = PyLong_AsLongLong(args[i]);
        if (size[i - 2] == -1 && PyErr_Occurred()) return nullptr;
    }
    const at::Tensor& like = THPVariable_Unpack(args[0]);
    if (!like.is_cuda()) {
        PyErr_SetString(PyExc_ValueError, "expected a GPU tensor");
        return nullptr;
    }
    const at::ScalarType dtype = reinterpret_cast<THPDtype*>(args[1])->scalar_type;
    at::Tensor out;
    {
        pybind11::gil_scoped_release without_gil;
        out = at::empty(at::IntArrayRef(size, n - 2), at::TensorOptions().dtype(dtype).device(like.device()));
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(run)), METH_FASTCALL, "run(address, *args) -> int"},
    {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(empty)), METH_FASTCALL, "empty(like, dtype, *size) -> Tensor"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native_call", nullptr, -1, methods};

}  // namespace

// torch_version: the torch whose structures this reads
PyMODINIT_FUNC PyInit__native_call() {
    PyObject* const m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", CMX_TORCH_VERSION) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
