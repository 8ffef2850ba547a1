// CPython side of Executor.enqueue: from the method call to nceClusterTaskEnqueue without interpreted code in between.
//
// A small task's enqueue is host time: 2.2 us of hipLaunchKernel, and as much again for everything around it when the
// descriptor is found in Python and handed over through ctypes (0.85 us: two Python frames, tuple and integer objects per
// argument, the foreign-function call). Here the method is a vectorcall that looks the task's wired descriptor up (four dict
// reads with interned keys) and calls the library by address: 3.07 -> 2.6 us per enqueue of a 32 x 32 x 16 convolution.
//
// What the task's finalize() would do is only decided here, never done: anything but "one variant, descriptor already wired to
// these very objects" goes to the Python method _enqueue_slow(). As in a ctypes call, the interpreter lock is released while the
// library runs.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/nce_hip.h"

namespace {

typedef nce_result_t (*enqueue_fn)(nce_executor_handle_t, const nce_cluster_task_desc_t*, void*);

struct EnqueueBase {
    PyObject_HEAD
    enqueue_fn fn;
    nce_executor_handle_t handle;
};

PyObject *s_variants, *s_desc, *s_ppe, *s_wired, *s_slow, *s_check, *s_task, *s_stream;

// The descriptor of a task that finalize() would return unchanged; nullptr: ask finalize(). No reference is kept: the caller's
// arguments hold the task, the task its descriptor.
const nce_cluster_task_desc_t* wired_descriptor(PyObject* task) {
    PyObject** const dp = _PyObject_GetDictPtr(task);
    if (dp == nullptr || *dp == nullptr) return nullptr;
    PyObject* const variants = PyDict_GetItemWithError(*dp, s_variants);
    PyObject* const desc = PyDict_GetItemWithError(*dp, s_desc);
    PyObject* const ppe = PyDict_GetItemWithError(*dp, s_ppe);
    PyObject* const wired = PyDict_GetItemWithError(*dp, s_wired);
    if (variants == nullptr || desc == nullptr || ppe == nullptr || wired == nullptr) {
        PyErr_Clear();
        return nullptr;
    }
    if (!PyList_CheckExact(variants) || PyList_GET_SIZE(variants) != 1 || !PyTuple_CheckExact(wired) || PyTuple_GET_SIZE(wired) != 4) return nullptr;
    if (PyTuple_GET_ITEM(wired, 0) != desc || PyTuple_GET_ITEM(wired, 1) != PyList_GET_ITEM(variants, 0) || PyTuple_GET_ITEM(wired, 2) != ppe) return nullptr;
    PyObject* const address = PyTuple_GET_ITEM(wired, 3);
    if (!PyLong_CheckExact(address)) return nullptr;
    const auto* const d = static_cast<const nce_cluster_task_desc_t*>(PyLong_AsVoidPtr(address));
    return d != nullptr && d->num_variants == 1 ? d : nullptr;
}

PyObject* enqueue(PyObject* self, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    PyObject* task = nargs > 0 ? args[0] : nullptr;
    PyObject* stream = nargs > 1 ? args[1] : nullptr;
    bool bad = nargs > 2;
    const Py_ssize_t nkw = kwnames != nullptr ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t i = 0; i < nkw; ++i) {
        PyObject* const name = PyTuple_GET_ITEM(kwnames, i);
        PyObject** const slot = PyUnicode_Compare(name, s_task) == 0 ? &task : PyUnicode_Compare(name, s_stream) == 0 ? &stream : nullptr;
        if (slot == nullptr || *slot != nullptr) bad = true;
        else *slot = args[nargs + i];
    }
    if (bad || task == nullptr) {
        PyErr_SetString(PyExc_TypeError, "enqueue(task, stream=None)");
        return nullptr;
    }
    if (stream == nullptr) stream = Py_None;
    EnqueueBase* const e = reinterpret_cast<EnqueueBase*>(self);
    const nce_cluster_task_desc_t* const d = e->fn != nullptr ? wired_descriptor(task) : nullptr;
    void* s = nullptr;
    if (d == nullptr || (stream != Py_None && !PyLong_Check(stream))) return PyObject_CallMethodObjArgs(self, s_slow, task, stream, nullptr);
    if (stream != Py_None) {
        s = PyLong_AsVoidPtr(stream);
        if (s == nullptr && PyErr_Occurred()) return nullptr;
    }
    nce_result_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = e->fn(e->handle, d, s);
    Py_END_ALLOW_THREADS
    if (rc == NCE_RESULT_SUCCESS) Py_RETURN_NONE;
    PyObject* const code = PyLong_FromLong((long)rc);
    if (code == nullptr) return nullptr;
    PyObject* const r = PyObject_CallMethodObjArgs(self, s_check, code, nullptr);
    Py_DECREF(code);
    return r;
}

// _bind(function address, executor handle): what enqueue() calls, and with what.
PyObject* bind(PyObject* self, PyObject* args) {
    PyObject *fn, *handle;
    if (!PyArg_ParseTuple(args, "O!O!", &PyLong_Type, &fn, &PyLong_Type, &handle)) return nullptr;
    EnqueueBase* const e = reinterpret_cast<EnqueueBase*>(self);
    e->fn = reinterpret_cast<enqueue_fn>(PyLong_AsVoidPtr(fn));
    e->handle = static_cast<nce_executor_handle_t>(PyLong_AsVoidPtr(handle));
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"enqueue", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(enqueue)), METH_FASTCALL | METH_KEYWORDS,
     "enqueue(task, stream=None)\n--\n\nnceClusterTaskEnqueue of the task on a HIP stream (its handle as an int; None: the default stream)."},
    {"_bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyType_Slot slots[] = {{Py_tp_methods, methods}, {Py_tp_new, reinterpret_cast<void*>(PyType_GenericNew)}, {0, nullptr}};
PyType_Spec spec = {"npu_plugin_amd._native.EnqueueBase", sizeof(EnqueueBase), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE, slots};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    const struct {
        PyObject** at;
        const char* name;
    } names[] = {{&s_variants, "_variants"}, {&s_desc, "desc"}, {&s_ppe, "_ppe"}, {&s_wired, "_wired"},
                 {&s_slow, "_enqueue_slow"}, {&s_check, "_check"}, {&s_task, "task"}, {&s_stream, "stream"}};
    for (const auto& n : names)
        if ((*n.at = PyUnicode_InternFromString(n.name)) == nullptr) return nullptr;
    PyObject* const m = PyModule_Create(&module_def);
    if (m == nullptr) return nullptr;
    PyObject* const t = PyType_FromSpec(&spec);
    if (t == nullptr || PyModule_AddObject(m, "EnqueueBase", t) < 0) {
        Py_XDECREF(t);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
