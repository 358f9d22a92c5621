// The Python calls' way into the library without ctypes: operands are looked at through the tensor's own C++ object, and the
// variant is launched from the same call.  What takes no part here (another operand type, a tensor that fails a check, integers
// that are none, an active torch function mode) is handed back, and cuda_hgemm_amd/binding.py says what is wrong with it or runs it.
//
// Bound by HIP's own launch, 2.4 ... 4.5 us by the host's speed: a loop of calls takes what the same loop in C does.  Through ctypes the
// operand checks, the conversion of seven arguments and the allocation of a result added 1.2 us (call: 256^3 5.2 -> 3.95 us) and
// 2.8 (hgemm: 7.5 -> 4.65), more than the kernel of every product up to about 768^3.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <stddef.h>

namespace {

typedef int (*run_fn)(int, const void *, const void *, void *, size_t, size_t, size_t);  // hgemm_variant_run

PyTypeObject *g_parameter_type;  // torch.nn.Parameter

const at::Tensor *tensor_of(PyObject *o) {
    if (!THPVariable_CheckExact(o) && Py_TYPE(o) != g_parameter_type) return nullptr;
    return &THPVariable_Unpack(o);
}

// The operand's address, or null if it is not a contiguous fp16 matrix of that shape on the GPU that starts on a 16-byte boundary.
void *operand(const at::Tensor &t, size_t rows, size_t cols) {
    if (t.scalar_type() != at::kHalf || !t.is_cuda() || t.layout() != at::kStrided || t.dim() != 2 || !t.unsafeGetTensorImpl()->has_storage())
        return nullptr;
    if ((size_t)t.size(0) != rows || (size_t)t.size(1) != cols || !t.is_contiguous()) return nullptr;
    void *ptr = t.data_ptr();
    return (reinterpret_cast<size_t>(ptr) & 15) ? nullptr : ptr;
}

bool size_of(PyObject *o, size_t *out) {
    if (!PyLong_CheckExact(o)) return false;
    *out = PyLong_AsSize_t(o);
    if (*out == (size_t)-1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

// Wrapped for transforms (vmap, forward-mode levels, functionalization): not a plain tensor's memory.
bool plain(const at::Tensor &t) {
    return !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                     c10::DispatchKey::Batched, c10::DispatchKey::Functionalize, c10::DispatchKey::Python}));
}

int launch(run_fn run, int index, const void *a, const void *b, void *c, size_t M, size_t N, size_t K) {
    int ran;
    Py_BEGIN_ALLOW_THREADS;
    ran = run(index, a, b, c, M, N, K);
    Py_END_ALLOW_THREADS;
    return ran;
}

// True: operands in order, launched.  False: not handled here, or the variant cannot run the shape.
bool try_call(run_fn run, int index, PyObject *const *args) {  // A, B, C, M, N, K
    size_t M, N, K;
    if (!size_of(args[3], &M) || !size_of(args[4], &N) || !size_of(args[5], &K)) return false;
    const at::Tensor *A = tensor_of(args[0]), *B = tensor_of(args[1]), *C = tensor_of(args[2]);
    if (!A || !B || !C || !plain(*A) || !plain(*B) || !plain(*C)) return false;
    void *a, *b, *c;
    try {
        a = operand(*A, M, K), b = operand(*B, N, K), c = operand(*C, M, N);
    } catch (...) {
        return false;
    }
    return a && b && c && launch(run, index, a, b, c, M, N, K) != 0;
}

// What HgemmLibrary.call is where this module is there: Caller(address of hgemm_variant_run, {variant name: index}, the method in
// Python).  A call with seven positional arguments and a name that the method has looked up before is tried here first.
struct Caller {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    PyObject *indices, *method;
    run_fn run;
};

PyObject *caller_call(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
    Caller *c = reinterpret_cast<Caller *>(self);
    if (!kwnames && PyVectorcall_NARGS(nargsf) == 7 && PyUnicode_CheckExact(args[0])) {
        PyObject *index = PyDict_GetItemWithError(c->indices, args[0]);  // borrowed
        if (!index && PyErr_Occurred()) return nullptr;
        if (index && try_call(c->run, (int)PyLong_AsLong(index), args + 1)) Py_RETURN_NONE;
    }
    return PyObject_Vectorcall(c->method, args, nargsf, kwnames);
}

PyObject *caller_new(PyTypeObject *type, PyObject *args, PyObject *) {
    unsigned long long run;
    PyObject *indices, *method;
    if (!PyArg_ParseTuple(args, "KO!O", &run, &PyDict_Type, &indices, &method)) return nullptr;
    Caller *c = reinterpret_cast<Caller *>(type->tp_alloc(type, 0));
    if (!c) return nullptr;
    c->vectorcall = caller_call;
    c->run = reinterpret_cast<run_fn>((size_t)run);
    Py_INCREF(indices), Py_INCREF(method);
    c->indices = indices, c->method = method;
    return reinterpret_cast<PyObject *>(c);
}
int caller_traverse(PyObject *self, visitproc visit, void *arg) {
    Py_VISIT(reinterpret_cast<Caller *>(self)->indices);
    Py_VISIT(reinterpret_cast<Caller *>(self)->method);
    return 0;
}
int caller_clear(PyObject *self) {
    Py_CLEAR(reinterpret_cast<Caller *>(self)->indices);
    Py_CLEAR(reinterpret_cast<Caller *>(self)->method);
    return 0;
}
void caller_dealloc(PyObject *self) {
    PyObject_GC_UnTrack(self);
    caller_clear(self);
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject make_caller_type() {
    PyTypeObject t = {PyVarObject_HEAD_INIT(nullptr, 0)};
    t.tp_name = "_call.Caller";
    t.tp_basicsize = sizeof(Caller);
    t.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_HAVE_VECTORCALL;
    t.tp_vectorcall_offset = offsetof(Caller, vectorcall);
    t.tp_call = PyVectorcall_Call;
    t.tp_new = caller_new;
    t.tp_traverse = caller_traverse;
    t.tp_clear = caller_clear;
    t.tp_dealloc = caller_dealloc;
    return t;
}
PyTypeObject g_caller_type = make_caller_type();

// product(run, index, A, B) -> a new tensor A . B^T; None: not handled here, or the variant cannot run the shape
PyObject *py_product(PyObject *, PyObject *const *args, Py_ssize_t n) {
    size_t run, index;
    if (n != 4 || !size_of(args[0], &run) || !size_of(args[1], &index) || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
    const at::Tensor *A = tensor_of(args[2]), *B = tensor_of(args[3]);
    if (!A || !B || !plain(*A) || !plain(*B) || A->dim() != 2 || B->dim() != 2) Py_RETURN_NONE;
    at::Tensor out;
    void *a, *b, *c;
    size_t M, N, K;
    try {
        M = (size_t)A->size(0), K = (size_t)A->size(1), N = (size_t)B->size(0);
        if (M == 0 || N == 0 || K == 0) Py_RETURN_NONE;
        a = operand(*A, M, K), b = operand(*B, N, K);
        if (!a || !b) Py_RETURN_NONE;
        out = at::empty({(int64_t)M, (int64_t)N}, at::TensorOptions().dtype(at::kHalf).device(A->device()));
        c = operand(out, M, N);
    } catch (...) {
        Py_RETURN_NONE;  // the caller's own way says what is wrong, out of memory among it
    }
    if (!c) Py_RETURN_NONE;
    if (!launch(reinterpret_cast<run_fn>(run), (int)index, a, b, c, M, N, K)) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
}

PyMethodDef kMethods[] = {
    {"product", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_product)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_call", "Launches libhgemm.so's variants on torch tensors.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call(void) {
    PyObject *nn = PyImport_ImportModule("torch.nn");
    if (!nn) return nullptr;
    PyObject *parameter = PyObject_GetAttrString(nn, "Parameter");
    Py_DECREF(nn);
    if (!parameter) return nullptr;
    g_parameter_type = reinterpret_cast<PyTypeObject *>(parameter);  // kept for the life of the process
    if (PyType_Ready(&g_caller_type) < 0) return nullptr;
    PyObject *module = PyModule_Create(&kModule);
    Py_INCREF(&g_caller_type);
    if (module && (PyModule_AddObject(module, "Caller", reinterpret_cast<PyObject *>(&g_caller_type)) < 0 ||
                   PyModule_AddStringConstant(module, "torch_version", TORCH_VERSION) < 0))
        Py_CLEAR(module);
    return module;
}
