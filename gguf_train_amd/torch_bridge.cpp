// CPython module _gt_bridge: lends PyTorch tensors to libgt_attn and adopts its results, the two
// steps that every Python call of the library makes for each operand.  In Python, reading a tensor's
// pointer, shape and strides into ctypes arrays took 3 to 4 us per operand, most of the 22 us of a
// small call (fp32 B1 H4 L=S=128 D64, whose kernel runs 8 us); with these the call takes 9.9 us, and a
// session of B4 H32/8 D128 over a Q8_0 cache (500 prompt tokens, 8 steps of 3 calls) 306 us instead of
// 430.
//
// The C ABI stays free of PyTorch types: this module is its client, as the ctypes loader is.

#include <Python.h>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <exception>

#include "../include/gt_attn.h"

#ifndef GT_BRIDGE_HASH
#define GT_BRIDGE_HASH ""
#endif
#ifndef GT_BRIDGE_TARGET
#define GT_BRIDGE_TARGET ""
#endif

namespace {

int gt_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return GT_F32;
        case at::kHalf: return GT_F16;
        case at::kBFloat16: return GT_BF16;
        case at::kDouble: return GT_F64;
        case at::kChar: return GT_I8;
        case at::kByte: return GT_U8;
        case at::kShort: return GT_I16;
        case at::kInt: return GT_I32;
        case at::kLong: return GT_I64;
        case at::kBool: return GT_BOOL;
        default: return -1;
    }
}

// Borrowed memory stays pinned by its handle, so the release tokens the library queues carry no
// information here; they are dropped now and then so that the queue does not grow.
std::atomic<uint64_t> g_token{1};
uint64_t next_token() {
    const uint64_t t = g_token.fetch_add(1, std::memory_order_relaxed);
    if (t % 512 == 0) {
        uint64_t buf[1024];
        while (gt_external_released(buf, 1024) == 1024) {
        }
    }
    return t;
}

PyObject *raise_native() {
    const char *e = gt_last_error();
    PyErr_Format(PyExc_RuntimeError, "borrow: %s", e && *e ? e : "Native operation returned NULL");
    return nullptr;
}

// A gt_tensor* on a tensor's memory, which `keep` pins; freed with the object.
struct Handle {
    PyObject_HEAD
    gt_tensor *ptr;
    PyObject *keep;
};

void handle_dealloc(PyObject *self) {
    Handle *h = (Handle *)self;
    gt_tensor_free(h->ptr);
    Py_XDECREF(h->keep);
    Py_TYPE(self)->tp_free(self);
}

PyObject *handle_ptr(PyObject *self, void *) { return PyLong_FromVoidPtr(((Handle *)self)->ptr); }

PyObject *handle_keep(PyObject *self, void *) {
    PyObject *k = ((Handle *)self)->keep ? ((Handle *)self)->keep : Py_None;
    Py_INCREF(k);
    return k;
}

PyObject *handle_release(PyObject *self, PyObject *) {
    Handle *h = (Handle *)self;
    PyObject *p = PyLong_FromVoidPtr(h->ptr);
    if (p) h->ptr = nullptr;
    return p;
}

PyGetSetDef handle_getset[] = {{"ptr", handle_ptr, nullptr, "address of the gt_tensor", nullptr},
                               {"keep", handle_keep, nullptr, "what pins the memory", nullptr},
                               {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMethodDef handle_methods[] = {{"release", handle_release, METH_NOARGS, "gives the gt_tensor up to the caller"},
                                {nullptr, nullptr, 0, nullptr}};
PyTypeObject HandleType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject *wrap_handle(gt_tensor *p, PyObject *keep) {
    Handle *h = (Handle *)HandleType.tp_alloc(&HandleType, 0);
    if (!h) {
        gt_tensor_free(p);
        return nullptr;
    }
    h->ptr = p;
    h->keep = keep;
    Py_XINCREF(keep);
    return (PyObject *)h;
}

// borrow(tensor) -> Handle
PyObject *borrow(PyObject *, PyObject *arg) {
    if (!THPVariable_Check(arg)) {
        PyErr_SetString(PyExc_TypeError, "borrow: expected a torch.Tensor");
        return nullptr;
    }
    try {
        const at::Tensor &t = THPVariable_Unpack(arg);
        const int code = gt_code(t.scalar_type());
        if (code < 0) {
            const std::string name = c10::toString(t.scalar_type());
            PyErr_Format(PyExc_TypeError, "dtype %s is not supported by libgt_attn", name.c_str());
            return nullptr;
        }
        const bool cuda = t.is_cuda();
        const int index = cuda ? (int)t.get_device() : 0, ndim = (int)t.dim();
        const int64_t *shape = t.sizes().data();
        gt_tensor *p;
        if (t.numel() == 0) {
            // nothing to lend: an empty library tensor of the same shape and device
            p = gt_tensor_empty(ndim, shape, code, cuda ? GT_DEV_CUDA : GT_DEV_CPU, index);
            return p ? wrap_handle(p, nullptr) : raise_native();
        }
        const int64_t *strides = t.strides().data();
        void *data = t.data_ptr();
        p = cuda ? gt_tensor_from_device_ptr(ndim, shape, strides, code, index, data, next_token())
                 : gt_tensor_from_external(ndim, shape, strides, code, data, next_token());
        return p ? wrap_handle(p, arg) : raise_native();
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "borrow: unknown error");
    }
    return nullptr;
}

// borrow_q8(data, shape) -> Handle on the Q8_0 blocks in the contiguous uint8 device tensor `data`, a
// dense tensor of the logical shape; None when data is another kind of tensor or the shape holds other
// than integers.
PyObject *borrow_q8(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 2 || !THPVariable_Check(args[0]) || !PyTuple_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "borrow_q8: expected (tensor, tuple)");
        return nullptr;
    }
    const Py_ssize_t ndim = PyTuple_GET_SIZE(args[1]);
    if (ndim > GT_MAX_DIMS) Py_RETURN_NONE;
    int64_t shape[GT_MAX_DIMS + 1], strides[GT_MAX_DIMS + 1];
    for (Py_ssize_t i = 0; i < ndim; ++i) {
        shape[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(args[1], i));
        if (shape[i] == -1 && PyErr_Occurred()) {  // a float, say: the caller's path takes what int() takes
            PyErr_Clear();
            Py_RETURN_NONE;
        }
    }
    int64_t acc = 1;
    for (Py_ssize_t i = ndim - 1; i >= 0; --i) {
        strides[i] = acc;
        if (__builtin_mul_overflow(acc, shape[i], &acc)) Py_RETURN_NONE;
    }
    try {
        const at::Tensor &t = THPVariable_Unpack(args[0]);
        if (!t.is_cuda() || t.scalar_type() != at::kByte || !t.is_contiguous()) Py_RETURN_NONE;
        gt_tensor *p = gt_tensor_from_device_ptr((int)ndim, shape, strides, GT_Q8_0, (int)t.get_device(), t.data_ptr(), next_token());
        return p ? wrap_handle(p, args[0]) : raise_native();
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "borrow_q8: unknown error");
    }
    return nullptr;
}

// Handle(ptr, keep=None): owns an existing gt_tensor
PyObject *handle_new(PyTypeObject *, PyObject *args, PyObject *kwargs) {
    static const char *names[] = {"ptr", "keep", nullptr};
    PyObject *address = nullptr, *keep = nullptr;
    if (!PyArg_ParseTupleAndKeywords(args, kwargs, "O|O:Handle", const_cast<char **>(names), &address, &keep)) return nullptr;
    void *p = PyLong_AsVoidPtr(address);
    if (!p && PyErr_Occurred()) return nullptr;
    return wrap_handle((gt_tensor *)p, keep == Py_None ? nullptr : keep);
}

PyObject *g_from_dlpack = nullptr;  // torch._C._from_dlpack

// adopt(address) -> tensor owning the result's memory; the gt_tensor is freed.  None when the library
// refuses (gt_last_error says why).
PyObject *adopt(PyObject *, PyObject *arg) {
    gt_tensor *t = (gt_tensor *)PyLong_AsVoidPtr(arg);
    if (!t) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "adopt: NULL");
        return nullptr;
    }
    void *dl = gt_tensor_to_dlpack(t);
    gt_tensor_free(t);
    if (!dl) Py_RETURN_NONE;
    PyObject *capsule = PyCapsule_New(dl, "dltensor", nullptr);
    if (!capsule) return nullptr;
    PyObject *out = PyObject_CallFunctionObjArgs(g_from_dlpack, capsule, nullptr);
    Py_DECREF(capsule);
    return out;
}

// set_stream(address): the calling thread's stream
PyObject *set_stream(PyObject *, PyObject *arg) {
    void *s = PyLong_AsVoidPtr(arg);
    if (!s && PyErr_Occurred()) return nullptr;
    gt_set_stream(s);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"borrow", borrow, METH_O, "a Handle on a tensor's memory, without a copy"},
                         {"borrow_q8", (PyCFunction)(void (*)(void))borrow_q8, METH_FASTCALL, "a Handle on Q8_0 blocks"},
                         {"adopt", adopt, METH_O, "a tensor on a result's memory, without a copy"},
                         {"set_stream", set_stream, METH_O, "gt_set_stream"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_gt_bridge", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__gt_bridge(void) {
    HandleType.tp_name = "gguf_train_amd._gt_bridge.Handle";
    HandleType.tp_basicsize = sizeof(Handle);
    HandleType.tp_flags = Py_TPFLAGS_DEFAULT;
    HandleType.tp_new = handle_new;
    HandleType.tp_dealloc = handle_dealloc;
    HandleType.tp_getset = handle_getset;
    HandleType.tp_methods = handle_methods;
    HandleType.tp_doc = "Owns one gt_tensor* and frees it when dropped; `keep` pins borrowed memory.";
    if (PyType_Ready(&HandleType) < 0) return nullptr;
    if (!g_from_dlpack) {
        PyObject *c = PyImport_ImportModule("torch._C");
        g_from_dlpack = c ? PyObject_GetAttrString(c, "_from_dlpack") : nullptr;
        Py_XDECREF(c);
        if (!g_from_dlpack) return nullptr;
    }
    PyObject *m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&HandleType);
    if (PyModule_AddObject(m, "Handle", (PyObject *)&HandleType) < 0 ||
        PyModule_AddStringConstant(m, "SOURCE_HASH", GT_BRIDGE_HASH) < 0 ||
        PyModule_AddStringConstant(m, "BUILT_FOR", GT_BRIDGE_TARGET) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
