// _ptr.ptr(tensor, dtype=None, numel=None, name="tensor"): the device pointer of a tensor after the checks of ops._p, which
// every operation makes of every argument.  Asked through Python they are five calls a tensor, 0.34 us, here 0.07; an update in a caller's own step
// loop has nine tensors, and such a loop (30,011 neurons) waits for the host: 23.5 -> 19.3 us a step.  Whatever is not a plain device tensor that passes, errors
// included, goes to the function given to set_general (ops' own).  built_for: the torch whose headers it was compiled with.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {

PyObject *general = nullptr;

// the pointer, or nullptr: for the general way
void *plain(PyObject *obj, PyObject *dtype, PyObject *numel)
{
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(obj);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
    const c10::DispatchKeySet others({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                      c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor,
                                      c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
    if (t.key_set().has_any(others) || !t.is_contiguous()) return nullptr;
    if (dtype != Py_None) {
        if (!THPDtype_Check(dtype) || reinterpret_cast<THPDtype *>(dtype)->scalar_type != t.scalar_type()) return nullptr;
    }
    if (numel != Py_None) {
        if (!PyLong_CheckExact(numel)) return nullptr;
        int overflow = 0;
        const long long least = PyLong_AsLongLongAndOverflow(numel, &overflow);
        if (overflow != 0 || t.numel() < least) return nullptr;
    }
    return t.mutable_data_ptr();
}

PyObject *ptr(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames)
{
    if (kwnames == nullptr && nargs >= 1 && nargs <= 4) {
        if (args[0] == Py_None) Py_RETURN_NONE;
        try {
            void *p = plain(args[0], nargs > 1 ? args[1] : Py_None, nargs > 2 ? args[2] : Py_None);
            if (p != nullptr) return PyLong_FromVoidPtr(p);
        } catch (const std::exception &) {
            // (the general way raises it)
        }
    }
    if (general == nullptr) {
        PyErr_SetString(PyExc_RuntimeError, "_ptr.set_general has not been called");
        return nullptr;
    }
    return PyObject_Vectorcall(general, args, (size_t)nargs, kwnames);
}

PyObject *set_general(PyObject *, PyObject *f)
{
    Py_INCREF(f);
    Py_XDECREF(general);
    general = f;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"ptr", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(ptr)), METH_FASTCALL | METH_KEYWORDS, "device pointer of a checked tensor"},
    {"set_general", set_general, METH_O, "what takes the calls that ptr does not"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ptr", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ptr()
{
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "built_for", BMTK_AMD_TORCH) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
