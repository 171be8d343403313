// The host side of a fused matmul on fp32 statistics in one native step: the checks, the output and the call into
// libnf4hip.so, which functional._matmul_nf4_on otherwise makes one attribute and one conversion at a time.
//
// A decode call on a small weight is as long as its host side: [4096, 4096], one row of x, a 4.6 us kernel: matmul_nf4 9.5 us through the
// interpreter, 5.3 this way, of which the launch is 2.9; a module around it 12.9 and 8.8.
//
// Only what can be handed over as it lies is taken: plain contiguous 16-byte aligned tensors of the expected types and
// sizes on x's device, no transform, mode or capture of dispatch around them.  Anything else returns None and goes through the
// interpreter, which converts, copies or raises as ever.
#define PY_SSIZE_T_CLEAN
#include <ATen/ATen.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cstdint>

namespace {

typedef size_t (*need_fn)(int64_t M, int64_t N, int64_t K);
typedef int (*matmul_fn)(const void* x, int x_dtype, int64_t M, const uint8_t* packed, const float* absmax, const float* lut16,
                         const void* bias, int64_t N, int64_t K, int blocksize, void* out, void* workspace,
                         size_t workspace_bytes, void* stream);
constexpr int BF16 = 0, F16 = 1;

// A tensor on the GPU whose memory can be used as it lies, or NULL.
const at::Tensor* plain(PyObject* o, at::ScalarType type) {
    if (!THPVariable_CheckExact(o)) {  // torch.Tensor and torch.nn.Parameter; subclasses have code of their own
        return nullptr;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    static constexpr c10::DispatchKeySet wrapped =
        c10::python_ks | c10::functorch_transforms_ks |
        c10::DispatchKeySet({c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Negative,
                             c10::DispatchKey::Conjugate});
    if (!t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(wrapped) || !t.has_storage() || t.scalar_type() != type ||
        !t.is_contiguous() || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) != 0)
        return nullptr;
    return &t;
}

// matmul(fn, need, x, qweight, absmax, quant_map, bias or None, N, K, blocksize, workspace or None, stream): the output, None
// where the call is not taken, or the library's status where it refused it.  fn serves x's type; x's device is current and
// `stream` its current stream.
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 12) {
        PyErr_SetString(PyExc_TypeError, "matmul takes 12 arguments");
        return nullptr;
    }
    const auto fn = reinterpret_cast<matmul_fn>(PyLong_AsVoidPtr(args[0]));
    const auto need = reinterpret_cast<need_fn>(PyLong_AsVoidPtr(args[1]));
    const int64_t N = PyLong_AsLongLong(args[7]), K = PyLong_AsLongLong(args[8]);
    const int blocksize = (int)PyLong_AsLong(args[9]);
    void* const stream = PyLong_AsVoidPtr(args[11]);
    if (PyErr_Occurred()) return nullptr;
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        Py_RETURN_NONE;
    if (!fn || !need || N <= 0 || K <= 0 || blocksize <= 0 || !THPVariable_Check(args[2])) Py_RETURN_NONE;
    const at::ScalarType type = THPVariable_Unpack(args[2]).scalar_type();
    if (type != at::kBFloat16 && type != at::kHalf) Py_RETURN_NONE;
    const at::Tensor *x = plain(args[2], type), *qweight = plain(args[3], at::kByte), *absmax = plain(args[4], at::kFloat);
    const at::Tensor* quant_map = plain(args[5], at::kFloat);
    const at::Tensor* bias = args[6] == Py_None ? nullptr : plain(args[6], type);
    if (!x || !qweight || !absmax || !quant_map || (!bias && args[6] != Py_None)) Py_RETURN_NONE;
    if (x->dim() < 1 || x->size(-1) != K || x->numel() == 0) Py_RETURN_NONE;
    const int64_t M = x->numel() / K;
    if (qweight->numel() < N * K / 2 || absmax->numel() < (N * K + blocksize - 1) / blocksize || quant_map->numel() < 16) Py_RETURN_NONE;
    if (bias && bias->numel() != N) Py_RETURN_NONE;
    for (const at::Tensor* t : {qweight, absmax, quant_map, bias})
        if (t && t->get_device() != x->get_device()) Py_RETURN_NONE;
    const at::Tensor* ws = nullptr;
    if (const size_t bytes = need(M, N, K)) {
        ws = args[10] == Py_None ? nullptr : plain(args[10], at::kByte);
        if (!ws || (size_t)ws->numel() < bytes || ws->get_device() != x->get_device()) Py_RETURN_NONE;
    }

    c10::SmallVector<int64_t, 5> sizes(x->sizes().begin(), x->sizes().end());
    sizes.back() = N;
    at::Tensor out = at::empty(sizes, x->options());
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        rc = fn(x->const_data_ptr(), type == at::kHalf ? F16 : BF16, M, static_cast<const uint8_t*>(qweight->const_data_ptr()),
                static_cast<const float*>(absmax->const_data_ptr()), static_cast<const float*>(quant_map->const_data_ptr()),
                bias ? bias->const_data_ptr() : nullptr, N, K, blocksize, out.mutable_data_ptr(), ws ? ws->mutable_data_ptr() : nullptr,
                ws ? (size_t)ws->numel() : 0, stream);
    }
    if (rc != 0) return PyLong_FromLong(rc);
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"matmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(matmul)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "nf4hip_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_nf4hip_host() {
    PyObject* const m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
