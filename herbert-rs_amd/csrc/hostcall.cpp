// The host's side of a launch, natively: the check that every operand of every kernel passes, and the call of a module's C
// entry point. A step that is not a graph's replay makes one call a kernel with 15 to 30 arguments and checks five operands for
// each; in Python (attribute after attribute, a generator over a shape) and through ctypes (an object an argument) that took 9 of the 16
// microseconds that a launch costs the host, longer than most kernels of a short prompt run. A check takes 0.09 us here instead of 0.66,
// a call of 24 arguments that its entry point refuses 0.9 instead of 1.8.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <stdint.h>

#include <exception>

#if !defined(__x86_64__) || !defined(__linux__)
#error "entry points are called as the x86-64 System V calling convention passes their arguments"
#endif

namespace {

// What is called. Every entry point takes pointers, integers and up to FLOATS floats and returns int. The calling convention passes
// integers and pointers in one sequence (six registers, then the stack, eight bytes each) and floats in another
// (eight registers), so any such function can be called as one that takes all floats first and more integers than it has:
// it finds its own where it looks, and the caller takes the rest off the stack again.
constexpr int FLOATS = 8, WORDS = 40;
#define W8 uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t
typedef int (*Function)(float, float, float, float, float, float, float, float, W8, W8, W8, W8, W8);

struct Entry {
    Function function;
    int count;
    bool is_float[WORDS + FLOATS];
};
const char ENTRY[] = "herbert_rs_amd.entry";

void free_entry(PyObject* capsule) { delete (Entry*)PyCapsule_GetPointer(capsule, ENTRY); }

// entry(address, kinds): kinds has a letter an argument, 'f' for a float and 'i' for anything else.
PyObject* make_entry(PyObject*, PyObject* args) {
    unsigned long long address;
    const char* kinds;
    if (!PyArg_ParseTuple(args, "Ks", &address, &kinds)) return nullptr;
    int words = 0, floats = 0;
    Entry e;
    e.function = (Function)address;
    e.count = 0;
    for (; kinds[e.count]; ++e.count) {
        const bool f = kinds[e.count] == 'f';
        if ((f ? ++floats : ++words) > (f ? FLOATS : WORDS)) {
            PyErr_SetString(PyExc_ValueError, "an entry point with more arguments than are passed on");
            return nullptr;
        }
        e.is_float[e.count] = f;
    }
    return PyCapsule_New(new Entry(e), ENTRY, free_entry);
}

// invoke(entry, arguments...): what the function returns. None is a null pointer; the interpreter is free meanwhile.
PyObject* invoke(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Entry* e = n > 0 ? (Entry*)PyCapsule_GetPointer(args[0], ENTRY) : nullptr;
    if (!e) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "an entry point is needed");
        return nullptr;
    }
    if (n - 1 != e->count) return PyErr_Format(PyExc_TypeError, "the entry point takes %d arguments, not %zd", e->count, n - 1);
    float f[FLOATS] = {};
    uint64_t w[WORDS] = {};
    int nf = 0, nw = 0;
    for (int i = 0; i < e->count; ++i) {
        PyObject* a = args[1 + i];
        if (e->is_float[i]) {
            f[nf++] = (float)PyFloat_AsDouble(a);
        } else {
            w[nw++] = a == Py_None ? 0 : PyLong_AsUnsignedLongLongMask(a);
        }
    }
    if (PyErr_Occurred()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = e->function(f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], w[9],
                     w[10], w[11], w[12], w[13], w[14], w[15], w[16], w[17], w[18], w[19], w[20], w[21], w[22], w[23], w[24],
                     w[25], w[26], w[27], w[28], w[29], w[30], w[31], w[32], w[33], w[34], w[35], w[36], w[37], w[38], w[39]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

bool has_form(const at::Tensor& t, PyObject* dtype, PyObject* shape) {
    if (!t.is_cuda() || !t.is_contiguous()) return false;
    if (dtype != Py_None && (!THPDtype_Check(dtype) || ((THPDtype*)dtype)->scalar_type != t.scalar_type())) return false;
    if (shape == Py_None) return true;
    if (!PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != t.dim()) return false;
    for (int64_t i = 0; i < t.dim(); ++i) {
        PyObject* want = PyTuple_GET_ITEM(shape, i);
        if (want == Py_None) continue;
        const long long size = PyLong_AsLongLong(want);
        if ((size == -1 && PyErr_Occurred()) || size != t.size(i)) return false;
    }
    return true;
}

// fits(tensor, dtype or None, shape or None): True for a contiguous tensor on the GPU of that type and shape (None within the
// shape: any size). Anything else is False, and the caller says what is wrong; also a tensor that throws where it is asked (a sparse one
// or a subclass has no strides to look at): an exception of C++ must not leave a function that the interpreter called.
PyObject* fits(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "a tensor, a type and a shape are needed");
        return nullptr;
    }
    bool is = false;
    try {
        is = THPVariable_Check(args[0]) && has_form(THPVariable_Unpack(args[0]), args[1], args[2]);
    } catch (const std::exception&) {
    }
    PyErr_Clear();
    return PyBool_FromLong(is);
}

PyMethodDef methods[] = {{"entry", make_entry, METH_VARARGS, nullptr},
                         {"invoke", (PyCFunction)(void*)invoke, METH_FASTCALL, nullptr},
                         {"fits", (PyCFunction)(void*)fits, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "hostcall", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_hostcall() { return PyModule_Create(&module); }
