// The extension module ferric_amd._host: DeviceBuffer as a C type, and the mat-vec call with the output it allocates.
//
// Every operator of the Python mirror allocates its output, so the cost of that object is part of the shortest calls: as a Python
// class around ctypes (c_void_p, byref, __init__, __del__) it took 3.4 us of a 7.1 us Q4_K 1024 x 5120 mat-vec, whose kernel takes
// 4.4 us. A C type over the library's fhip_malloc / fhip_free does the same in a few hundred nanoseconds. A launch itself costs
// the host 3 us on this runtime (0.9 us without arguments: the argument block is written to device memory and read back), which is
// most of what is left of such a call, so matmul_q does all of its conversions here instead of in ctypes, and the three calls of routed experts do: through ctypes
// they took the host 21.5 us where their kernels take 11 - 14, now 16 (1024 x 2048, 2 of 128 experts, one token 22.0 -> 15.8).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <stddef.h>
#include <structmember.h>

namespace {

int (*p_malloc)(void**, size_t) = nullptr;
int (*p_free)(void*) = nullptr;
int (*p_matmul_q)(const void*, const void*, size_t, void*, void*) = nullptr;
int (*p_moe_topk)(const void*, const void*, size_t, size_t, size_t, int, float, int, void*, void*) = nullptr;
int (*p_swiglu_id)(const void*, const void*, size_t, const void*, size_t, size_t, void*, void*) = nullptr;
int (*p_id_wsum)(const void*, const void*, size_t, const void*, size_t, size_t, void*, void*, void*) = nullptr;
PyTypeObject* g_buffer_type = nullptr;
PyObject* g_value = nullptr;         // "value"
PyObject* g_c_void_p = nullptr;      // ctypes.c_void_p
PyObject* g_first_use = nullptr;     // called before the first allocation: initialises the device, calls bind()
PyObject* g_check = nullptr;         // raises for a return code

struct Buffer {
    PyObject_HEAD
    void* mem;
    PyObject* nbytes;                // as it was given
    PyObject* ptr;                   // c_void_p of mem, made when it is first asked for
    PyObject* dict;                  // attributes a user hangs on the object, made when there are some
    PyObject* weak;
};

// the exception for a return code of the library
int raise_rc(int rc) {
    PyObject* r = PyObject_CallFunction(g_check, "i", rc);
    if (r) { Py_DECREF(r); PyErr_Format(PyExc_RuntimeError, "libferric_hip returned %d", rc); }
    return -1;
}

int ready() {
    if (p_malloc) return 0;
    if (!g_first_use) { PyErr_SetString(PyExc_RuntimeError, "ferric_amd._host: setup() has not been called"); return -1; }
    PyObject* r = PyObject_CallNoArgs(g_first_use);
    if (!r) return -1;
    Py_DECREF(r);
    if (!p_malloc) { PyErr_SetString(PyExc_RuntimeError, "ferric_amd._host: bind() has not been called"); return -1; }
    return 0;
}
void buffer_holds(Buffer* self, void* mem, PyObject* n) {
    self->mem = mem;
    Py_INCREF(n);
    Py_XSETREF(self->nbytes, n);
}
int buffer_allocate(Buffer* self, size_t bytes, PyObject* n) {
    if (ready()) return -1;
    int rc;
    void* mem = nullptr;
    Py_BEGIN_ALLOW_THREADS           // may wait for the device
    rc = p_malloc(&mem, bytes);
    Py_END_ALLOW_THREADS
    if (rc) return raise_rc(rc);
    buffer_holds(self, mem, n);
    return 0;
}

int buffer_init(Buffer* self, PyObject* args, PyObject* kw) {
    static const char* names[] = {"nbytes", nullptr};
    PyObject* n = nullptr;
    if (!PyArg_ParseTupleAndKeywords(args, kw, "O:DeviceBuffer", (char**)names, &n)) return -1;
    if (self->mem) { PyErr_SetString(PyExc_TypeError, "DeviceBuffer: already allocated"); return -1; }
    PyObject* whole = PyNumber_Index(n);
    if (!whole) return -1;
    const size_t bytes = PyLong_AsSize_t(whole);
    const bool bad = bytes == (size_t)-1 && PyErr_Occurred();
    const int rc = bad ? -1 : buffer_allocate(self, bytes, whole);
    Py_DECREF(whole);
    return rc;
}

int buffer_traverse(Buffer* self, visitproc visit, void* arg) {
    Py_VISIT(Py_TYPE(self));
    Py_VISIT(self->dict);
    return 0;
}
int buffer_clear(Buffer* self) {
    Py_CLEAR(self->dict);
    return 0;
}

void buffer_dealloc(Buffer* self) {
    PyTypeObject* type = Py_TYPE(self);
    PyObject_GC_UnTrack(self);
    if (self->weak) PyObject_ClearWeakRefs((PyObject*)self);
    if (self->mem) {
        void* mem = self->mem;
        self->mem = nullptr;
        Py_BEGIN_ALLOW_THREADS       // a block the pool does not keep goes to hipFree, which waits for the device
        (void)p_free(mem);
        Py_END_ALLOW_THREADS
    }
    Py_CLEAR(self->nbytes);
    Py_CLEAR(self->ptr);
    Py_CLEAR(self->dict);
    type->tp_free((PyObject*)self);
    Py_DECREF(type);
}

PyObject* buffer_ptr(Buffer* self, void*) {
    if (!self->ptr && !(self->ptr = PyObject_CallFunction(g_c_void_p, "n", (Py_ssize_t)self->mem))) return nullptr;
    Py_INCREF(self->ptr);
    return self->ptr;
}
PyObject* buffer_nbytes(Buffer* self, void*) {
    PyObject* n = self->nbytes ? self->nbytes : Py_None;
    Py_INCREF(n);
    return n;
}

PyGetSetDef buffer_getset[] = {
    {"ptr", (getter)buffer_ptr, nullptr, "device address (ctypes.c_void_p)", nullptr},
    {"nbytes", (getter)buffer_nbytes, nullptr, "bytes asked for", nullptr},
    {"__dict__", PyObject_GenericGetDict, PyObject_GenericSetDict, nullptr, nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr},
};
PyMemberDef buffer_members[] = {
    {"__dictoffset__", T_PYSSIZET, offsetof(Buffer, dict), READONLY, nullptr},
    {"__weaklistoffset__", T_PYSSIZET, offsetof(Buffer, weak), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr},
};
PyType_Slot buffer_slots[] = {
    {Py_tp_init, (void*)buffer_init},
    {Py_tp_new, (void*)PyType_GenericNew},
    {Py_tp_dealloc, (void*)buffer_dealloc},
    {Py_tp_traverse, (void*)buffer_traverse},
    {Py_tp_clear, (void*)buffer_clear},
    {Py_tp_getset, (void*)buffer_getset},
    {Py_tp_members, (void*)buffer_members},
    {Py_tp_doc, (void*)"DeviceBuffer(nbytes)\n\nnbytes of device memory, freed with the object. Work enqueued on any stream may still use it "
                       "then: the library does not hand\nthe memory out again before the device has been idle once (fhip_free), so scratch can be "
                       "dropped without a synchronisation."},
    {0, nullptr},
};
PyType_Spec buffer_spec = {"ferric_amd._host.DeviceBuffer", sizeof(Buffer), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC, buffer_slots};

// what a ctypes pointer, an address or None stands for
bool address(PyObject* h, void** out) {
    *out = nullptr;
    if (h == Py_None) return true;
    if (PyLong_Check(h)) {
        *out = PyLong_AsVoidPtr(h);
        return !PyErr_Occurred();
    }
    PyObject* v = PyObject_GetAttr(h, g_value);
    if (!v) return false;
    if (v != Py_None) *out = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    return !PyErr_Occurred();
}

// matmul_q(x buffer, weight handle, rows, output columns, stream) -> buffer of rows x columns f32: fhip_malloc and fhip_matmul_q.
// The handle and the stream are ctypes pointers or addresses; the stream may be None. NotImplemented for a buffer of another type: the caller goes through
// ctypes, which takes whatever `ptr` such an object has.
PyObject* matmul_q(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 5) { PyErr_SetString(PyExc_TypeError, "matmul_q(DeviceBuffer, handle, rows, columns, stream)"); return nullptr; }
    if (!PyObject_TypeCheck(a[0], g_buffer_type)) Py_RETURN_NOTIMPLEMENTED;
    const size_t rows = PyLong_AsSize_t(a[2]), cols = PyLong_AsSize_t(a[3]);
    if (PyErr_Occurred()) return nullptr;
    void *handle[2];
    if (!address(a[1], &handle[0]) || !address(a[4], &handle[1])) return nullptr;
    PyObject* nbytes = PyLong_FromSize_t(rows * cols * sizeof(float));
    if (!nbytes) return nullptr;
    Buffer* out = ready() ? nullptr : (Buffer*)g_buffer_type->tp_alloc(g_buffer_type, 0);
    if (!out) { Py_DECREF(nbytes); return nullptr; }
    void *x = ((Buffer*)a[0])->mem, *y = nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS           // once for both: giving the interpreter away and taking it back is 0.1 us
    rc = p_malloc(&y, rows * cols * sizeof(float));
    if (!rc) rc = p_matmul_q(handle[0], x, rows, y, handle[1]);
    Py_END_ALLOW_THREADS
    if (y) buffer_holds(out, y, nbytes);
    Py_DECREF(nbytes);
    if (rc) { raise_rc(rc); Py_DECREF(out); return nullptr; }
    return (PyObject*)out;
}

bool sizes(PyObject* const* a, int n, size_t* out) {
    for (int i = 0; i < n; i++) {
        PyObject* whole = PyNumber_Index(a[i]);
        if (!whole) return false;
        out[i] = PyLong_AsSize_t(whole);
        Py_DECREF(whole);
        if (out[i] == (size_t)-1 && PyErr_Occurred()) return false;
    }
    return true;
}
// bytes of a x b x c floats; a size that wraps is refused as the allocation of a Python int that large is
bool float_bytes(size_t a, size_t b, size_t c, size_t* out) {
    size_t n;
    if (!__builtin_mul_overflow(a, b, &n) && !__builtin_mul_overflow(n, c, &n) && !__builtin_mul_overflow(n, sizeof(float), out)) return true;
    PyErr_SetString(PyExc_OverflowError, "the result's size does not fit a size_t");
    return false;
}
// a DeviceBuffer of `bytes` that launch(its memory, `scratch` bytes more or null) has been enqueued into
template <class Launch>
PyObject* result(size_t bytes, size_t scratch, Launch launch) {
    PyObject* nbytes = PyLong_FromSize_t(bytes);
    if (!nbytes) return nullptr;
    Buffer* out = ready() ? nullptr : (Buffer*)g_buffer_type->tp_alloc(g_buffer_type, 0);
    if (!out) { Py_DECREF(nbytes); return nullptr; }
    void *y = nullptr, *ws = nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_malloc(&y, bytes);
    if (!rc && scratch) rc = p_malloc(&ws, scratch);
    if (!rc) rc = launch(y, ws);
    if (ws) (void)p_free(ws);        // (not handed out again before the device has been idle)
    Py_END_ALLOW_THREADS
    if (y) buffer_holds(out, y, nbytes);
    Py_DECREF(nbytes);
    if (rc) { raise_rc(rc); Py_DECREF(out); return nullptr; }
    return (PyObject*)out;
}
bool is_buffer(PyObject* o) { return PyObject_TypeCheck(o, g_buffer_type); }

// moe_topk(logits buffer, bias buffer or None, tokens, experts, k, sigmoid, scale, norm, stream) -> buffer of tokens x 2 k; NotImplemented as matmul_q
PyObject* moe_topk(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 9) { PyErr_SetString(PyExc_TypeError, "moe_topk(logits, bias, tokens, experts, k, sigmoid, scale, norm, stream)"); return nullptr; }
    if (!is_buffer(a[0]) || (a[1] != Py_None && !is_buffer(a[1]))) Py_RETURN_NOTIMPLEMENTED;
    size_t d[3], bytes;
    void* stream;
    const int sigmoid = PyObject_IsTrue(a[5]), norm = PyObject_IsTrue(a[7]);
    const float scale = (float)PyFloat_AsDouble(a[6]);
    if (PyErr_Occurred() || !sizes(a + 2, 3, d) || !address(a[8], &stream) || !float_bytes(d[0], 2, d[2], &bytes)) return nullptr;
    const void *x = ((Buffer*)a[0])->mem, *bias = a[1] == Py_None ? nullptr : ((Buffer*)a[1])->mem;
    return result(bytes, 0, [&](void* y, void*) { return p_moe_topk(x, bias, d[0], d[1], d[2], sigmoid, scale, norm, y, stream); });
}
// swiglu_id(x buffer, weight handle, tokens, selection buffer, k, outputs, stream) -> buffer of tokens x k x outputs
PyObject* swiglu_id(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 7) { PyErr_SetString(PyExc_TypeError, "swiglu_id(x, handle, tokens, selection, k, outputs, stream)"); return nullptr; }
    if (!is_buffer(a[0]) || !is_buffer(a[3])) Py_RETURN_NOTIMPLEMENTED;
    size_t t, d[2], bytes;
    void *w, *stream;
    if (!sizes(a + 2, 1, &t) || !sizes(a + 4, 2, d) || !address(a[1], &w) || !address(a[6], &stream) || !float_bytes(t, d[0], d[1], &bytes)) return nullptr;
    const void *x = ((Buffer*)a[0])->mem, *sel = ((Buffer*)a[3])->mem;
    return result(bytes, 0, [&](void* y, void*) { return p_swiglu_id(w, x, t, sel, d[0], d[1], y, stream); });
}
// id_wsum(x buffer, weight handle, tokens, selection buffer, k, outputs, stream) -> buffer of tokens x outputs
PyObject* id_wsum(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 7) { PyErr_SetString(PyExc_TypeError, "id_wsum(x, handle, tokens, selection, k, outputs, stream)"); return nullptr; }
    if (!is_buffer(a[0]) || !is_buffer(a[3])) Py_RETURN_NOTIMPLEMENTED;
    size_t t, d[2], bytes, scratch;
    void *w, *stream;
    if (!sizes(a + 2, 1, &t) || !sizes(a + 4, 2, d) || !address(a[1], &w) || !address(a[6], &stream) || !float_bytes(t, 1, d[1], &bytes) || !float_bytes(t, d[0], d[1], &scratch)) return nullptr;
    const void *x = ((Buffer*)a[0])->mem, *sel = ((Buffer*)a[3])->mem;
    return result(bytes, scratch, [&](void* y, void* ws) { return p_id_wsum(w, x, t, sel, d[0], d[1], y, ws, stream); });
}

PyObject* setup(PyObject*, PyObject* args) {
    PyObject *first_use, *check;
    if (!PyArg_ParseTuple(args, "OO", &first_use, &check)) return nullptr;
    Py_INCREF(first_use);
    Py_XSETREF(g_first_use, first_use);
    Py_INCREF(check);
    Py_XSETREF(g_check, check);
    Py_RETURN_NONE;
}
// resolves the functions used here in the library that is loaded from `path`
PyObject* bind(PyObject*, PyObject* args) {
    const char* path;
    if (!PyArg_ParseTuple(args, "s", &path)) return nullptr;
    void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!lib) { PyErr_Format(PyExc_ImportError, "%s", dlerror()); return nullptr; }
    p_free = (int (*)(void*))dlsym(lib, "fhip_free");
    p_matmul_q = (int (*)(const void*, const void*, size_t, void*, void*))dlsym(lib, "fhip_matmul_q");
    p_moe_topk = (decltype(p_moe_topk))dlsym(lib, "fhip_moe_topk");
    p_swiglu_id = (decltype(p_swiglu_id))dlsym(lib, "fhip_matmul_q_swiglu_id");
    p_id_wsum = (decltype(p_id_wsum))dlsym(lib, "fhip_matmul_q_id_wsum");
    p_malloc = (int (*)(void**, size_t))dlsym(lib, "fhip_malloc");
    if (!p_malloc || !p_free || !p_matmul_q || !p_moe_topk || !p_swiglu_id || !p_id_wsum) { p_malloc = nullptr; PyErr_Format(PyExc_ImportError, "%s does not export what it should", path); return nullptr; }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"setup", setup, METH_VARARGS, "setup(first_use, check)"},
                         {"matmul_q", (PyCFunction)(void*)matmul_q, METH_FASTCALL, "matmul_q(x buffer, weight handle, rows, columns, stream)"},
                         {"moe_topk", (PyCFunction)(void*)moe_topk, METH_FASTCALL, "moe_topk(logits, bias, tokens, experts, k, sigmoid, scale, norm, stream)"},
                         {"swiglu_id", (PyCFunction)(void*)swiglu_id, METH_FASTCALL, "swiglu_id(x, handle, tokens, selection, k, outputs, stream)"},
                         {"id_wsum", (PyCFunction)(void*)id_wsum, METH_FASTCALL, "id_wsum(x, handle, tokens, selection, k, outputs, stream)"},
                         {"bind", bind, METH_VARARGS, "bind(library path)"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Device memory objects of ferric_amd.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* ctypes = PyImport_ImportModule("ctypes");
    if (!ctypes) return nullptr;
    g_c_void_p = PyObject_GetAttrString(ctypes, "c_void_p");
    Py_DECREF(ctypes);
    if (!g_c_void_p || !(g_value = PyUnicode_InternFromString("value"))) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    PyObject* type = PyType_FromSpec(&buffer_spec);
    if (!type || PyModule_AddObject(m, "DeviceBuffer", type) < 0) { Py_XDECREF(type); Py_DECREF(m); return nullptr; }
    g_buffer_type = (PyTypeObject*)type;
    return m;
}
