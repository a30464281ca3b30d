// The host side of a launch in native code: checks the operands of a call, puts their addresses into a copy of the call's argument struct and
// enters the library (libpsgemm.so), which is reached through the function addresses that the Python package passes in.
//
// In Python a launch with nine operands spends 3 to 4 us on these checks (four attributes a tensor) and on filling the struct field by field,
// next to 2.5 us of the launch itself, and decode-sized kernels run 2 to 10 us: MXFP4 32 x 7168 x 2048 with its quantiser took 10.5 us a pass,
// all of it host time, a MX MoE layer of 6 tokens 41 us where its kernels need 22.
//
// What is not accepted here (a tensor subclass, a wrong size, another device, ...) is not refused here either: the call returns
// DECLINED and the Python code, which runs the same checks one by one, says what is wrong or goes on.  Nothing is kept from one call for the
// next: sizes, types, devices and addresses are read anew every time.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

namespace {

constexpr long DECLINED = -1000;  // (the library's own codes are small negative numbers and HIP's errors)

// One operand of a launch.  Packed by flydsl_amd/_lib.py.
struct Operand {
    int32_t arg;     // which of the call's argument structs
    int32_t offset;  // of the address in it
    int32_t item;    // bytes of an element, 0 = any
    int32_t type;    // TYPE_*, plus OPTIONAL where None may stand in the operand's place
    int64_t need;    // least bytes
};
enum { TYPE_ANY = 0, TYPE_INT32 = 1, TYPE_FP32 = 2, TYPE_BF16 = 3, TYPE_FP16 = 4, OPTIONAL = 256 };

bool type_is(const at::Tensor& t, int type) {
    switch (type) {
        case TYPE_INT32: return t.scalar_type() == at::kInt;
        case TYPE_FP32: return t.scalar_type() == at::kFloat;
        case TYPE_BF16: return t.scalar_type() == at::kBFloat16;
        case TYPE_FP16: return t.scalar_type() == at::kHalf;
    }
    return true;
}

// a plain, contiguous device tensor on `device` (-1: on any, which becomes `device`)
const at::Tensor* operand(PyObject* o, int64_t& device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || !t.is_contiguous()) return nullptr;
    const int64_t d = t.get_device();
    if (device < 0) device = d;
    return d == device ? &t : nullptr;
}

// raw stream handle of an int or of an object with `cuda_stream`
bool stream_of(PyObject* o, void** out) {
    static PyObject* const name = PyUnicode_InternFromString("cuda_stream");
    PyObject* v = o;
    if (PyLong_CheckExact(o)) {
        Py_INCREF(v);
    } else {
        v = PyObject_GetAttr(o, name);
        if (!v || !PyLong_CheckExact(v)) {
            Py_XDECREF(v);
            PyErr_Clear();
            return false;
        }
    }
    *out = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

template <class F>
PyObject* guarded(F&& f) {
    long rc = DECLINED;
    try {
        rc = f();
    } catch (...) {  // (whatever torch throws about a tensor, the Python checks meet it again)
        rc = DECLINED;
    }
    return PyLong_FromLong(rc);
}

// f() without the interpreter's lock: the queue may be full.  f is the call into the library and nothing else, its arguments read before: asking a
// tensor for anything may throw or change it, and another thread may resize it meanwhile.
template <class F>
int released(F&& f) {
    struct Unlocked {
        PyThreadState* const state = PyEval_SaveThread();
        ~Unlocked() { PyEval_RestoreThread(state); }
    } unlocked;
    return f();
}

// launch(function address, (struct, ...), operands, stream, tensor or None, ...) -> return code of the library, or DECLINED.
// `struct`: bytes of the argument struct with everything but addresses; one or two of them.
PyObject* launch(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> long {
        if (n < 4 || !PyTuple_CheckExact(a[1]) || !PyBytes_CheckExact(a[2])) return DECLINED;
        const Py_ssize_t structs = PyTuple_GET_SIZE(a[1]), ops = n - 4;
        if (structs < 1 || structs > 2 || PyBytes_GET_SIZE(a[2]) != ops * (Py_ssize_t)sizeof(Operand)) return DECLINED;
        alignas(16) unsigned char arg[2][256];
        Py_ssize_t size[2] = {0, 0};
        for (Py_ssize_t i = 0; i < structs; i++) {
            PyObject* b = PyTuple_GET_ITEM(a[1], i);
            if (!PyBytes_CheckExact(b) || PyBytes_GET_SIZE(b) > (Py_ssize_t)sizeof(arg[0])) return DECLINED;
            size[i] = PyBytes_GET_SIZE(b);
            memcpy(arg[i], PyBytes_AS_STRING(b), (size_t)size[i]);
        }
        int64_t device = -1;
        for (Py_ssize_t i = 0; i < ops; i++) {
            Operand op;
            memcpy(&op, PyBytes_AS_STRING(a[2]) + i * (Py_ssize_t)sizeof(op), sizeof(op));
            if (a[4 + i] == Py_None && (op.type & OPTIONAL)) continue;
            if (op.arg < 0 || op.arg >= structs || op.offset < 0 || op.offset + (Py_ssize_t)sizeof(void*) > size[op.arg]) return DECLINED;
            const at::Tensor* t = operand(a[4 + i], device);
            if (!t || (op.item && (int64_t)t->element_size() != op.item) || !type_is(*t, op.type & ~OPTIONAL) || t->numel() * (int64_t)t->element_size() < op.need) return DECLINED;
            void* p = t->data_ptr();
            memcpy(arg[op.arg] + op.offset, &p, sizeof(p));
        }
        void* stream;
        if (!stream_of(a[3], &stream)) return DECLINED;
        void* fn = PyLong_AsVoidPtr(a[0]);
        if (!fn) {
            PyErr_Clear();
            return DECLINED;
        }
        return released([&] {
            return structs == 1 ? reinterpret_cast<int (*)(const void*, void*)>(fn)(arg[0], stream)
                                : reinterpret_cast<int (*)(const void*, const void*, void*)>(fn)(arg[0], arg[1], stream);
        });
    });
}

int x_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return 0;
        case at::kBFloat16: return 1;
        case at::kHalf: return 2;
        default: return -1;
    }
}

// quant_pertoken(function address, x, y, scale, output code, stream): x [M, K], y one byte an element, scale fp32 [M]
PyObject* quant_pertoken(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> long {
        int64_t device = -1;
        if (n != 6 || !PyLong_CheckExact(a[4])) return DECLINED;
        const at::Tensor *x = operand(a[1], device), *y = x ? operand(a[2], device) : nullptr, *s = y ? operand(a[3], device) : nullptr;
        void* stream;
        if (!s || x->dim() != 2 || x_code(*x) < 0 || y->element_size() != 1 || y->numel() != x->numel() || s->scalar_type() != at::kFloat || s->numel() != x->size(0) ||
            x->size(0) > INT32_MAX || x->size(1) > INT32_MAX || !stream_of(a[5], &stream))
            return DECLINED;
        const int code = (int)PyLong_AsLong(a[4]), from = x_code(*x), rows = (int)x->size(0), cols = (int)x->size(1);
        void *xp = x->data_ptr(), *yp = y->data_ptr(), *sp = s->data_ptr();
        auto fn = reinterpret_cast<int (*)(const void*, int32_t, void*, void*, int32_t, int32_t, int32_t, void*)>(PyLong_AsVoidPtr(a[0]));
        return released([&] { return fn(xp, from, yp, sp, rows, cols, code, stream); });
    });
}

// quant_mxfp4(function address, x, packed, scales, shuffle, stream): x [M, K], packed M * (K / 2) bytes, scales ceil(M / 32) * 32 * (K / 32) bytes
PyObject* quant_mxfp4(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> long {
        int64_t device = -1;
        if (n != 6 || !PyLong_CheckExact(a[4])) return DECLINED;
        const at::Tensor *x = operand(a[1], device), *y = x ? operand(a[2], device) : nullptr, *s = y ? operand(a[3], device) : nullptr;
        void* stream;
        if (!s || x->dim() != 2 || x_code(*x) < 0 || y->element_size() != 1 || s->element_size() != 1 || x->size(0) > INT32_MAX || x->size(1) > INT32_MAX ||
            y->numel() != x->size(0) * (x->size(1) / 2) || s->numel() != (x->size(0) + 31) / 32 * 32 * (x->size(1) / 32) || !stream_of(a[5], &stream))
            return DECLINED;
        const int shuffle = (int)PyLong_AsLong(a[4]), from = x_code(*x), rows = (int)x->size(0), cols = (int)x->size(1);
        void *xp = x->data_ptr(), *yp = y->data_ptr(), *sp = s->data_ptr();
        auto fn = reinterpret_cast<int (*)(const void*, int32_t, void*, void*, int32_t, int32_t, int32_t, void*)>(PyLong_AsVoidPtr(a[0]));
        return released([&] { return fn(xp, from, yp, sp, rows, cols, shuffle, stream); });
    });
}

// moe_reduce(function address, x, y, item, tokens, topk, dim, dtype code, stream): x [tokens, topk, dim], y [tokens, dim]
PyObject* moe_reduce(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> long {
        int64_t device = -1;
        if (n != 9) return DECLINED;
        int64_t v[5];
        for (int i = 0; i < 5; i++) {
            if (!PyLong_CheckExact(a[3 + i])) return DECLINED;
            v[i] = PyLong_AsLongLong(a[3 + i]);
        }
        const int64_t item = v[0], tokens = v[1], topk = v[2], dim = v[3];
        const at::Tensor *x = operand(a[1], device), *y = x ? operand(a[2], device) : nullptr;
        void* stream;
        if (!y || PyErr_Occurred() || tokens < 1 || tokens > INT32_MAX || topk < 1 || topk > INT32_MAX || dim < 1 || dim > INT32_MAX || (int64_t)x->element_size() != item || (int64_t)y->element_size() != item ||
            x->numel() / topk / dim < tokens || y->numel() / dim < tokens || !stream_of(a[8], &stream)) {
            PyErr_Clear();
            return DECLINED;
        }
        auto fn = reinterpret_cast<int (*)(const void*, void*, int32_t, int32_t, int32_t, int32_t, void*)>(PyLong_AsVoidPtr(a[0]));
        void *xp = x->data_ptr(), *yp = y->data_ptr();
        return released([&] { return fn(xp, yp, (int32_t)tokens, (int32_t)topk, (int32_t)dim, (int32_t)v[4], stream); });
    });
}

// moe_scale_sort(function address, scale, ids, num_valid, out, tokens, stream): scale [>= tokens, C] bytes, C % 8 == 0; out ceil(len(ids) / 32) * 32 rows of C
PyObject* moe_scale_sort(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> long {
        int64_t device = -1;
        if (n != 7 || !PyLong_CheckExact(a[5])) return DECLINED;
        const at::Tensor *s = operand(a[1], device), *ids = s ? operand(a[2], device) : nullptr, *nv = ids ? operand(a[3], device) : nullptr, *out = nv ? operand(a[4], device) : nullptr;
        if (!out) return DECLINED;
        const int64_t tokens = PyLong_AsLongLong(a[5]);
        void* stream;
        if (PyErr_Occurred() || tokens < 1 || tokens > INT32_MAX || s->dim() != 2 || s->element_size() != 1 || s->size(0) < tokens || s->size(1) % 8 || s->size(1) > INT32_MAX ||
            ids->scalar_type() != at::kInt || nv->scalar_type() != at::kInt || ids->numel() > INT32_MAX ||
            out->numel() * (int64_t)out->element_size() < (ids->numel() + 31) / 32 * 32 * s->size(1) || !stream_of(a[6], &stream)) {
            PyErr_Clear();
            return DECLINED;
        }
        auto fn = reinterpret_cast<int (*)(const void*, const void*, const void*, void*, int32_t, int32_t, int32_t, int32_t, void*)>(PyLong_AsVoidPtr(a[0]));
        const int cols = (int)s->size(1), size = (int)ids->numel();
        void *sp = s->data_ptr(), *ip = ids->data_ptr(), *np = nv->data_ptr(), *op = out->data_ptr();
        return released([&] { return fn(sp, ip, np, op, (int32_t)tokens, 1, cols, size, stream); });
    });
}

#define PSG_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {PSG_METHOD(launch),     PSG_METHOD(quant_pertoken), PSG_METHOD(quant_mxfp4),
                         PSG_METHOD(moe_reduce), PSG_METHOD(moe_scale_sort), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddIntConstant(m, "DECLINED", DECLINED) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
