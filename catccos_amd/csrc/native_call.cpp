// What the Python front end does for every call, in native code: output tensors, pointers out of tensors, the call itself.
// A call of ops.py launches one to five kernels and returns; a small one costs the host more than the GPU (quantizer of 16 rows 5.0 us, of
// which the launch takes 3.1, where the kernel runs 3.0; with a call into here for each tensor and torch.empty behind it 5.9; quantizer and
// matmul of 16 x 4096 x 7168 9.6, so 11.3).
//
//   run(address, *args)              int(*)(...) at `address`: tensors by their data pointer, None as null, integers (anything with __index__); ValueError for a tensor
//                                    that is not on the GPU.  A tuple (dtype, one to four sizes) stands for a new tensor on the device of the first
//                                    tensor among the arguments, an Ellipsis for torch's current stream.  Without the GIL, like a ctypes call.
//                                    Returns what the entry point returned, or, where that is zero, the new tensors if there are any (one, or a
//                                    tuple of them).
//   empty(like, dtype, size, ...)    torch.empty on the device of `like`, which is a GPU (ValueError)
//
// Every entry point of the C ABI takes integers and pointers only, each of which has a register or an 8-byte slot of its own in
// the x86-64 System V convention, so one function type of kMaxArgs such arguments calls them all.
#include <Python.h>

#include <ATen/Context.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <cstdint>

#if !defined(__x86_64__) || defined(_WIN32)
#error "x86-64 System V calling convention"
#endif

namespace {

constexpr Py_ssize_t kMaxArgs = 24, kMaxOutputs = 4;

// Whether torch.empty would do no more than allocate: no mode, tracer or transform sees the calls of this thread, and new memory need not be
// filled (torch.use_deterministic_algorithms).
bool plain_allocation() {
    const c10::DispatchKeySet seen_by = c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set;
    return seen_by.empty() && !at::globalContext().deterministicAlgorithms();
}

// A tensor to be made: torch.empty's, without its way through the dispatcher (0.3 us of 0.8) where that leads nowhere else
struct NewTensor {
    int64_t size[4];
    size_t dims;
    at::ScalarType dtype;
    at::Tensor made;

    // spec: dtype, one to four sizes; false with an error set
    bool read(PyObject* const* spec, Py_ssize_t n) {
        if (n < 2 || n > 5 || !THPDtype_Check(spec[0])) {
            PyErr_SetString(PyExc_TypeError, "a new tensor: dtype, one to four sizes");
            return false;
        }
        dims = n - 1;
        for (size_t i = 0; i < dims; ++i) {
            size[i] = PyLong_AsLongLong(spec[i + 1]);
            if (size[i] == -1 && PyErr_Occurred()) return false;
        }
        dtype = reinterpret_cast<THPDtype*>(spec[0])->scalar_type;
        return true;
    }
    void make(const at::Tensor& like) {
        const at::IntArrayRef sizes(size, dims);
        if (plain_allocation()) {
            made = at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt);
            return;
        }
        made = at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
        TORCH_CHECK_VALUE(made.is_cuda(), "expected a GPU tensor");          // (a mode may give any)
    }
};

using u = uint64_t;
using Fn = int (*)(u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u);

// args[0], an entry point; null with an error set
Fn entry_point(PyObject* address) {
    const uint64_t v = PyLong_AsUnsignedLongLong(address);
    if (v == 0 && !PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
    return PyErr_Occurred() ? nullptr : reinterpret_cast<Fn>(v);
}

// a tensor, an integer or None as the 64 bits that an entry point gets; false with an error set
bool to_word(PyObject* o, Py_ssize_t i, uint64_t& v) {
    v = 0;
    if (PyLong_Check(o) || (!THPVariable_Check(o) && PyIndex_Check(o))) {              // (numpy's integers)
        v = PyLong_AsUnsignedLongLongMask(o);
        return !(v == (uint64_t)-1 && PyErr_Occurred());
    }
    if (THPVariable_Check(o)) {
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.is_cuda()) {
            PyErr_SetString(PyExc_ValueError, "expected a GPU tensor");
            return false;
        }
        v = reinterpret_cast<uint64_t>(t.data_ptr());
        return true;
    }
    if (o == Py_None) return true;
    PyErr_Format(PyExc_TypeError, "argument %zd: a tensor, an integer or None, not %s", i, Py_TYPE(o)->tp_name);
    return false;
}

PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 1 || n > 1 + kMaxArgs) {
        PyErr_SetString(PyExc_TypeError, "run(address, up to 24 arguments)");
        return nullptr;
    }
    const Fn fn = entry_point(args[0]);
    if (fn == nullptr) return nullptr;
    uint64_t v[kMaxArgs] = {};
    NewTensor outputs[kMaxOutputs];
    Py_ssize_t made = 0, at[kMaxOutputs];
    const at::Tensor* like = nullptr;
    Py_ssize_t stream = -1;
    for (Py_ssize_t i = 1; i < n; ++i) {
        if (PyTuple_CheckExact(args[i])) {
            if (made == kMaxOutputs) {
                PyErr_SetString(PyExc_TypeError, "at most four new tensors");
                return nullptr;
            }
            if (!outputs[made].read(PySequence_Fast_ITEMS(args[i]), PyTuple_GET_SIZE(args[i]))) return nullptr;
            at[made++] = i - 1;
            continue;
        }
        if (args[i] == Py_Ellipsis) {
            if (stream >= 0) {
                PyErr_SetString(PyExc_TypeError, "an Ellipsis stands for the stream, once");
                return nullptr;
            }
            stream = i - 1;
            continue;
        }
        if (!to_word(args[i], i, v[i - 1])) return nullptr;
        if (like == nullptr && THPVariable_Check(args[i])) like = &THPVariable_Unpack(args[i]);
    }
    if (made != 0 && like == nullptr) {
        PyErr_SetString(PyExc_ValueError, "expected a GPU tensor");
        return nullptr;
    }
    int rc;
    {
        pybind11::gil_scoped_release without_gil;
        if (stream >= 0) v[stream] = reinterpret_cast<uint64_t>(c10::hip::getCurrentHIPStream().stream());
        for (Py_ssize_t i = 0; i < made; ++i) {
            outputs[i].make(*like);
            v[at[i]] = reinterpret_cast<uint64_t>(outputs[i].made.data_ptr());
        }
        rc = fn(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11], v[12], v[13], v[14], v[15], v[16], v[17], v[18], v[19],
                v[20], v[21], v[22], v[23]);
    }
    if (rc != 0 || made == 0) return PyLong_FromLong(rc);
    if (made == 1) return THPVariable_Wrap(std::move(outputs[0].made));
    THPObjectPtr all(PyTuple_New(made));
    if (!all) return nullptr;
    for (Py_ssize_t i = 0; i < made; ++i) {
        PyObject* const t = THPVariable_Wrap(std::move(outputs[i].made));
        if (t == nullptr) return nullptr;
        PyTuple_SET_ITEM(all.get(), i, t);
    }
    return all.release();
    END_HANDLE_TH_ERRORS
}

PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 3 || n > 6 || !THPVariable_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "empty(tensor, dtype, one to four sizes)");
        return nullptr;
    }
    const at::Tensor& like = THPVariable_Unpack(args[0]);
    NewTensor out;
    if (!out.read(args + 1, n - 1)) return nullptr;
    if (!like.is_cuda()) {
        PyErr_SetString(PyExc_ValueError, "expected a GPU tensor");
        return nullptr;
    }
    {
        pybind11::gil_scoped_release without_gil;
        out.make(like);
    }
    return THPVariable_Wrap(std::move(out.made));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(run)), METH_FASTCALL, "run(address, *args) -> int, or the new tensors"},
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
