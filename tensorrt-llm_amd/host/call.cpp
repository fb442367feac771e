// The ordinary matmul call of functional.py in native code: look the tensors over, allocate output and workspace, call
// woq_matmul on torch's current stream.  A call outside a graph is bound by the host (one row of 4096 x 4096 keeps the GPU
// busy for 4 us), and in Python the checks, the two allocations, the argument block and the three calls through ctypes
// took 9.5 ... 10.8 us on the host; here the same takes 5.4 (a call of a stream of calls).
//
// Only the plain case is taken: operands that are torch.Tensor or Parameter objects (no other subclass, no functorch wrapper), on a GPU,
// contiguous and of the expected types, no __torch_function__ mode, no output or workspace of the caller's, the
// library's own choice of kernels.  For everything else - wrong types and shapes included - the function returns None
// and the Python path in functional.py does the call, or says what is wrong with it: errors are worded in one place.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPStream.h>

#include "../../include/woq.h"

namespace
{
int (*g_matmul)(woq_matmul_args const*, void*) = nullptr;
size_t (*g_workspace_bytes)(int32_t, int32_t, int32_t, int32_t, int32_t) = nullptr;

// An operand: None (nullptr stays) or a plain, contiguous GPU tensor.  False: not for this path.
bool operand(PyObject* o, at::Tensor const*& t)
{
    t = nullptr;
    if (o == Py_None)
        return true;
    if (!THPVariable_CheckExact(o))
        return false;
    t = &THPVariable_Unpack(o);
    // (a functorch or functional wrapper is a torch.Tensor object too)
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
        c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
        c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    return !t->key_set().has_any(wrapped) && t->has_storage() && t->layout() == at::kStrided && t->is_cuda() && t->is_contiguous();
}

int dtype_of(at::ScalarType t)
{
    return t == at::kHalf ? WOQ_FP16 : t == at::kBFloat16 ? WOQ_BF16 : t == at::kFloat8_e4m3fn ? WOQ_FP8_E4M3 : -1;
}

// matmul(act, pre_quant_scale, weight, scales, zeros, bias, n, k, group_size, quant_algo, alpha, out_dtype)
// out_dtype: WOQ_FP16 / WOQ_BF16.  Returns the output, a non-zero woq_status, or None: not for this path.
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    if (!g_matmul || nargs != 12 || at::impl::torch_function_mode_enabled())
        Py_RETURN_NONE;
    at::Tensor const* t[6];
    for (int i = 0; i < 6; ++i)
        if (!operand(args[i], t[i]))
            Py_RETURN_NONE;
    at::Tensor const *act = t[0], *weight = t[2], *scales = t[3];
    if (!act || !weight || !scales || act->dim() < 1)
        Py_RETURN_NONE;
    long v[4];
    for (int i = 0; i < 4; ++i)
    {
        v[i] = PyLong_AsLong(args[6 + i]);
        if (v[i] == -1 && PyErr_Occurred())
        {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        if (v[i] < 0 || v[i] > INT32_MAX)
            Py_RETURN_NONE;
    }
    double const alpha = PyFloat_AsDouble(args[10]);
    long const out_dtype = PyLong_AsLong(args[11]);
    if (PyErr_Occurred())
    {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    if (out_dtype != WOQ_FP16 && out_dtype != WOQ_BF16)
        Py_RETURN_NONE;
    long const n = v[0], k = v[1], algo = v[3];
    at::ScalarType const out_type = out_dtype == WOQ_FP16 ? at::kHalf : at::kBFloat16;
    bool const w4a8 = algo & WOQ_ALGO_FP8_ALPHA;
    if (k == 0 || act->size(-1) != k || act->numel() / k > INT32_MAX)
        Py_RETURN_NONE;
    if (act->scalar_type() != out_type && act->scalar_type() != at::kFloat8_e4m3fn)
        Py_RETURN_NONE;
    for (int i : {1, 3, 4, 5}) // smoothing vector, scales, zeros, bias: the output's type (W4A8 tables: float16 too)
        if (t[i] && t[i]->scalar_type() != out_type && !(w4a8 && (i == 3 || i == 4) && t[i]->scalar_type() == at::kHalf))
            Py_RETURN_NONE;
    woq_matmul_args a = {};
    auto ptr = [](at::Tensor const* x) -> void const* { return x ? x->const_data_ptr() : nullptr; };
    a.act = ptr(act);
    a.pre_quant_scale = ptr(t[1]);
    a.weight = ptr(weight);
    a.scales = ptr(scales);
    a.zeros = ptr(t[4]);
    a.bias = ptr(t[5]);
    a.alpha = (float) alpha;
    a.m = (int32_t) (act->numel() / k);
    a.n = (int32_t) n;
    a.k = (int32_t) k;
    a.group_size = (int32_t) v[2];
    a.quant_algo = (int32_t) algo;
    a.act_dtype = dtype_of(act->scalar_type());
    a.out_dtype = (int32_t) out_dtype;
    a.regime = 0;
    auto size = act->sizes().vec();
    size.back() = n;
    int rc = 0;
    at::Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = at::empty(size, act->options().dtype(out_type).requires_grad(false));
        a.out = out.mutable_data_ptr();
        at::Tensor workspace;
        if (size_t const need = g_workspace_bytes(a.m, a.n, a.k, a.quant_algo, a.act_dtype))
        {
            workspace = at::empty({(int64_t) need}, out.options().dtype(at::kByte));
            a.workspace = workspace.mutable_data_ptr();
            a.workspace_bytes = need;
        }
        rc = g_matmul(&a, c10::hip::getCurrentHIPStream(act->device().index()).stream());
    }
    if (rc != 0)
        return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// What this file was compiled against: the torch whose tensors it looks into, the argument block of include/woq.h, Python.
// A torch or a library of another build may load all the same and be laid out differently; the caller compares.
PyObject* built_for(PyObject*, PyObject*)
{
    return Py_BuildValue("(siii)", WOQ_CALL_TORCH, WOQ_ABI_VERSION, PY_MAJOR_VERSION, PY_MINOR_VERSION);
}

// bind(address of woq_matmul, address of woq_workspace_bytes): the library that _lib.py loaded
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 2)
    {
        PyErr_SetString(PyExc_TypeError, "bind takes two addresses");
        return nullptr;
    }
    void* const f = PyLong_AsVoidPtr(args[0]);
    void* const g = PyLong_AsVoidPtr(args[1]);
    if (PyErr_Occurred())
        return nullptr;
    g_matmul = reinterpret_cast<decltype(g_matmul)>(f);
    g_workspace_bytes = reinterpret_cast<decltype(g_workspace_bytes)>(g);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"matmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(matmul)), METH_FASTCALL, nullptr},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(bind)), METH_FASTCALL, nullptr},
    {"built_for", built_for, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "woq_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
} // namespace

PyMODINIT_FUNC PyInit_woq_call(void)
{
    return PyModule_Create(&module);
}
