// The launch path of orinfer_amd/lib.py in native code: named arguments -> void** -> orx_enqueue.
//
// A decode projection takes 6 us on the GPU; the same marshalling in Python (geometry query, one ctypes object and one
// cast per argument, the validating launch) took 14 us per launch and bounded every eager call below about 30 us.
// Here it is one pass over the keyword dictionary: names are interned, so an argument is found by comparing
// pointers, a tensor's address is one method call, and the HIP launch runs with the interpreter lock given back.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stdint.h>

#include "../../include/orx.h"

namespace {

constexpr int kMaxArgs = 64;
PyObject* g_data_ptr = nullptr;  // interned "data_ptr"

struct Launcher {
    PyObject_HEAD
    orx_fn function;
    int count;
    PyObject* names[kMaxArgs];  // interned, owned
    int kinds[kMaxArgs];
};

// None -> 0, a tensor -> its data_ptr(), anything else through int()
bool address_of(PyObject* value, uint64_t* out) {
    if (value == Py_None) {
        *out = 0;
        return true;
    }
    PyObject* number;
    if (PyLong_CheckExact(value)) {
        number = Py_NewRef(value);
    } else {
        number = PyObject_CallMethodNoArgs(value, g_data_ptr);
        if (number == nullptr && PyErr_ExceptionMatches(PyExc_AttributeError)) {
            PyErr_Clear();
            number = PyNumber_Long(value);
        }
        if (number == nullptr) return false;
    }
    *out = PyLong_AsUnsignedLongLongMask(number);
    Py_DECREF(number);
    return !PyErr_Occurred();
}

int launcher_init(Launcher* self, PyObject* args, PyObject*) {
    unsigned long long handle = 0;
    PyObject *names = nullptr, *kinds = nullptr;
    if (!PyArg_ParseTuple(args, "KO!O!", &handle, &PyTuple_Type, &names, &PyTuple_Type, &kinds)) return -1;
    const Py_ssize_t count = PyTuple_GET_SIZE(names);
    if (handle == 0 || count > kMaxArgs || PyTuple_GET_SIZE(kinds) != count || self->count != 0) {
        PyErr_SetString(PyExc_ValueError, "Launcher takes a handle, up to 64 names and as many kinds, once");
        return -1;
    }
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* name = PyTuple_GET_ITEM(names, i);
        if (!PyUnicode_CheckExact(name)) {
            PyErr_SetString(PyExc_TypeError, "argument names are strings");
            return -1;
        }
        Py_INCREF(name);
        PyUnicode_InternInPlace(&name);
        self->names[i] = name;
        self->count = (int)i + 1;
        const long kind = PyLong_AsLong(PyTuple_GET_ITEM(kinds, i));
        if (kind == -1 && PyErr_Occurred()) return -1;
        self->kinds[i] = (int)kind;
    }
    self->function = reinterpret_cast<orx_fn>(static_cast<uintptr_t>(handle));
    return 0;
}

void launcher_dealloc(Launcher* self) {
    for (int i = 0; i < self->count; ++i) Py_XDECREF(self->names[i]);
    PyTypeObject* type = Py_TYPE(self);
    type->tp_free(reinterpret_cast<PyObject*>(self));
    Py_DECREF(type);
}

// enqueue(stream, named) -> the library's code, or None where the names are not exactly the kernel's
PyObject* launcher_enqueue(Launcher* self, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 2 || !PyDict_CheckExact(args[1])) {
        PyErr_SetString(PyExc_TypeError, "enqueue(stream, named arguments)");
        return nullptr;
    }
    uint64_t stream = 0;
    if (!address_of(args[0], &stream)) return nullptr;
    if (self->function == nullptr || PyDict_GET_SIZE(args[1]) != self->count) Py_RETURN_NONE;
    uint64_t storage[kMaxArgs];
    void* pointers[kMaxArgs];
    PyObject *key = nullptr, *value = nullptr;
    Py_ssize_t at = 0;
    int found = 0;
    while (PyDict_Next(args[1], &at, &key, &value)) {
        int index = 0;
        while (index < self->count && self->names[index] != key) ++index;
        if (index == self->count) {  // not the interned object: compare the text
            for (index = 0; index < self->count; ++index)
                if (PyUnicode_Check(key) && PyUnicode_Compare(self->names[index], key) == 0) break;
            if (index == self->count) Py_RETURN_NONE;
        }
        if (self->kinds[index] == 0) {
            if (!address_of(value, &storage[index])) return nullptr;
        } else {
            PyObject* number = PyNumber_Long(value);
            if (number == nullptr) return nullptr;
            // wraps, as ctypes.c_int32 does; the library checks the range of a row count
            const int32_t narrow = (int32_t)PyLong_AsUnsignedLongLongMask(number);
            Py_DECREF(number);
            storage[index] = (uint32_t)narrow;
        }
        ++found;
    }
    if (found != self->count) Py_RETURN_NONE;
    for (int i = 0; i < self->count; ++i) pointers[i] = &storage[i];
    int code;
    Py_BEGIN_ALLOW_THREADS
    code = orx_enqueue(self->function, reinterpret_cast<void*>(static_cast<uintptr_t>(stream)), pointers);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(code);
}

PyMethodDef launcher_methods[] = {
    {"enqueue", (PyCFunction)(void (*)(void))launcher_enqueue, METH_FASTCALL,
     "enqueue(stream, named): launch with a dictionary of arguments; the library's code, None if the names do not match"},
    {nullptr, nullptr, 0, nullptr}};

PyType_Slot launcher_slots[] = {{Py_tp_doc, (void*)"One resolved kernel's launch: Launcher(handle, names, kinds)"},
                                {Py_tp_new, (void*)PyType_GenericNew},
                                {Py_tp_init, (void*)launcher_init},
                                {Py_tp_dealloc, (void*)launcher_dealloc},
                                {Py_tp_methods, (void*)launcher_methods},
                                {0, nullptr}};
PyType_Spec launcher_spec = {"orinfer_amd._launcher.Launcher", (int)sizeof(Launcher), 0, Py_TPFLAGS_DEFAULT, launcher_slots};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launcher", "Native launch path over liborx.so", -1, nullptr,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launcher(void) {
    g_data_ptr = PyUnicode_InternFromString("data_ptr");
    PyObject* m = PyModule_Create(&module);
    PyObject* type = PyType_FromSpec(&launcher_spec);
    if (g_data_ptr == nullptr || m == nullptr || type == nullptr || PyModule_AddObject(m, "Launcher", type) != 0) {
        Py_XDECREF(type);
        Py_XDECREF(m);
        return nullptr;
    }
    return m;
}
