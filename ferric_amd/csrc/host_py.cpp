// The extension module ferric_amd._host: DeviceBuffer as a C type, and the mat-vec call with the output it allocates.
//
// Every operator of the Python mirror allocates its output, so the cost of that object is part of the shortest calls: as a Python
// class around ctypes (c_void_p, byref, __init__, __del__) it took 3.4 us of a 7.1 us Q4_K 1024 x 5120 mat-vec, whose kernel takes
// 4.4 us. A C type over the library's fhip_malloc / fhip_free does the same in a few hundred nanoseconds. A launch itself costs
// the host 3 us on this runtime (0.9 us without arguments: the argument block is written to device memory and read back), which is
// most of what is left of such a call, so matmul_q does all of its conversions here instead of in ctypes.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <stddef.h>
#include <structmember.h>

namespace {

int (*p_malloc)(void**, size_t) = nullptr;
int (*p_free)(void*) = nullptr;
int (*p_matmul_q)(const void*, const void*, size_t, void*, void*) = nullptr;
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

// matmul_q(x buffer, weight handle, rows, output columns, stream) -> buffer of rows x columns f32: fhip_malloc and fhip_matmul_q.
// The handle and the stream are ctypes pointers or addresses; the stream may be None. NotImplemented for a buffer of another type: the caller goes through
// ctypes, which takes whatever `ptr` such an object has.
PyObject* matmul_q(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 5) { PyErr_SetString(PyExc_TypeError, "matmul_q(DeviceBuffer, handle, rows, columns, stream)"); return nullptr; }
    if (!PyObject_TypeCheck(a[0], g_buffer_type)) Py_RETURN_NOTIMPLEMENTED;
    const size_t rows = PyLong_AsSize_t(a[2]), cols = PyLong_AsSize_t(a[3]);
    if (PyErr_Occurred()) return nullptr;
    void* handle[2] = {nullptr, nullptr};
    for (int i = 0; i < 2; i++) {
        PyObject* h = a[i ? 4 : 1];
        if (h == Py_None) continue;
        if (PyLong_Check(h)) {
            handle[i] = PyLong_AsVoidPtr(h);
            if (PyErr_Occurred()) return nullptr;
            continue;
        }
        PyObject* v = PyObject_GetAttr(h, g_value);
        if (!v) return nullptr;
        if (v != Py_None) handle[i] = PyLong_AsVoidPtr(v);
        Py_DECREF(v);
        if (PyErr_Occurred()) return nullptr;
    }
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
    p_malloc = (int (*)(void**, size_t))dlsym(lib, "fhip_malloc");
    if (!p_malloc || !p_free || !p_matmul_q) { p_malloc = nullptr; PyErr_Format(PyExc_ImportError, "%s does not export what it should", path); return nullptr; }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"setup", setup, METH_VARARGS, "setup(first_use, check)"},
                         {"matmul_q", (PyCFunction)(void*)matmul_q, METH_FASTCALL, "matmul_q(x buffer, weight handle, rows, columns, stream)"},
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
