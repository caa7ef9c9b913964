// Host side of the two calls an FP8 linear makes (quantisation and GEMM), as a
// CPython extension: argument checks, output allocation and the C ABI call in
// one crossing.  Through Python checks, torch.empty and ctypes a call costs
// the host 10-13 us, more than a kernel on a few hundred rows takes; here 5.3
// (GEMM) and 5.6 us (quantisation), of which the launch is about half.  An
// FP8Linear of 512 tokens: 24.6 -> 14.9 us a call, of 2079 tokens per tensor
// 29.5 -> 20.2.
//
// Each function serves the plain case (exact tensors on one GPU, types and
// layouts the kernels take as they are) and returns None for everything else,
// including a call the library refuses: the Python caller then runs its general
// path, which converts, checks and raises as documented there.  A HIP error is
// raised here: the library's status has taken it from the runtime, so a second
// attempt would look clean, on work that may have failed.
//
// The C ABI functions are those of the library the Python side has loaded,
// passed to bind() by address.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/fvsr.h"

namespace {

struct Abi {
  decltype(&fvsr_quant_workspace_floats) quant_workspace_floats;
  decltype(&fvsr_quant_fp8_dt) quant_fp8_dt;
  decltype(&fvsr_fp8_gemm) fp8_gemm;
  decltype(&fvsr_gemm_amax_parts) gemm_amax_parts;
} abi{};

// The tensor behind a Python argument, or nullptr if it is not a plain tensor
// (or parameter) on a GPU.
const at::Tensor* plain_gpu(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

// Modes that intercept torch calls see the Python path's calls instead.
bool modes_active() {
  return at::impl::torch_function_mode_enabled() ||
         c10::impl::TorchDispatchModeTLS::any_modes_set();
}

void* stream_of(const at::Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return FVSR_DT_BF16;
    case at::kHalf: return FVSR_DT_F16;
    case at::kFloat: return FVSR_DT_F32;
    default: return -1;
  }
}

// What a call returns for a status other than FVSR_OK: None for one decided
// before any launch, an exception for a HIP error (worded as the Python path's).
PyObject* not_done(int rc, const char* what) {
  if (rc != FVSR_EHIP) Py_RETURN_NONE;
  PyErr_Format(PyExc_RuntimeError, "%s failed: HIP launch error (status %d)", what, rc);
  return nullptr;
}

// quantize(x2, per_token, gelu) -> (codes, scale) or None
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !abi.quant_fp8_dt) Py_RETURN_NONE;
  const at::Tensor* x = plain_gpu(args[0]);
  if (!x || x->dim() != 2 || x->numel() == 0 || x->stride(1) != 1 || modes_active())
    Py_RETURN_NONE;
  const int dt = dtype_code(*x);
  if (dt < 0) Py_RETURN_NONE;
  const int per_token = PyObject_IsTrue(args[1]), gelu = PyObject_IsTrue(args[2]);
  if (per_token < 0 || gelu < 0) return nullptr;  // no truth value: its exception
  const int64_t M = x->size(0), K = x->size(1);
  const int mode = per_token ? FVSR_SCALE_ROW : FVSR_SCALE_TENSOR;
  at::Tensor q = at::empty({M, K}, x->options().dtype(at::kFloat8_e4m3fn));
  const auto f32 = x->options().dtype(at::kFloat);
  at::Tensor s = per_token ? at::empty({M, 1}, f32) : at::empty({1}, f32);
  const int64_t wn = abi.quant_workspace_floats(M, K, mode);
  at::Tensor ws;
  if (wn > 0) ws = at::empty({wn}, f32);
  void* st = stream_of(*x);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = abi.quant_fp8_dt(x->data_ptr(), dt, M, K, x->stride(0), mode, gelu, q.data_ptr(),
                        (float*)s.data_ptr(), wn > 0 ? (float*)ws.data_ptr() : nullptr, wn, st);
  Py_END_ALLOW_THREADS
  if (rc != FVSR_OK) return not_done(rc, gelu ? "fused_gelu_quant_fp8" : "quantize_fp8");
  PyObject* qo = THPVariable_Wrap(std::move(q));
  PyObject* so = qo ? THPVariable_Wrap(std::move(s)) : nullptr;
  PyObject* r = so ? PyTuple_Pack(2, qo, so) : nullptr;
  Py_XDECREF(qo);
  Py_XDECREF(so);
  return r;
  END_HANDLE_TH_ERRORS
}

// gemm(x8, s, w8, w_scale, bias | None, amax_part | None) -> out or None; with
// amax_part the row-max epilogue.
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6 || !abi.fp8_gemm) Py_RETURN_NONE;
  const at::Tensor* t[6] = {};
  for (int i = 0; i < 6; ++i) {
    if (args[i] == Py_None) {
      if (i < 4) Py_RETURN_NONE;
      continue;
    }
    t[i] = plain_gpu(args[i]);
    if (!t[i] || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  }
  const at::Tensor &x = *t[0], &s = *t[1], &w = *t[2], &wsc = *t[3];
  if (x.scalar_type() != at::kFloat8_e4m3fn || w.scalar_type() != at::kFloat8_e4m3fn ||
      x.dim() != 2 || w.dim() != 2 || x.size(1) != w.size(1) || x.stride(1) != 1 ||
      w.stride(1) != 1 || s.scalar_type() != at::kFloat || wsc.scalar_type() != at::kFloat ||
      !s.is_contiguous() || !wsc.is_contiguous())
    Py_RETURN_NONE;
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0), ns = s.numel(), nw = wsc.numel();
  if ((ns != 1 && ns != M) || (nw != 1 && nw != N)) Py_RETURN_NONE;
  if (t[4] && (t[4]->scalar_type() != at::kBFloat16 || t[4]->dim() != 1 || t[4]->numel() != N ||
               !t[4]->is_contiguous()))
    Py_RETURN_NONE;
  if (t[5] && (t[5]->scalar_type() != at::kFloat || !t[5]->is_contiguous() ||
               t[5]->numel() < M * abi.gemm_amax_parts(N)))
    Py_RETURN_NONE;
  if (modes_active()) Py_RETURN_NONE;
  at::Tensor out = at::empty({M, N}, x.options().dtype(at::kBFloat16));
  void* st = stream_of(x);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = abi.fp8_gemm(x.data_ptr(), x.stride(0), (const float*)s.data_ptr(),
                    ns == M && M != 1 ? FVSR_SCALE_ROW : FVSR_SCALE_TENSOR, w.data_ptr(),
                    w.stride(0), (const float*)wsc.data_ptr(),
                    nw == N && N != 1 ? FVSR_SCALE_ROW : FVSR_SCALE_TENSOR,
                    t[4] ? t[4]->data_ptr() : nullptr, out.data_ptr(), N, M, N, K,
                    t[5] ? FVSR_EPI_ROWMAX : FVSR_EPI_BIAS,
                    t[5] ? (float*)t[5]->data_ptr() : nullptr, nullptr, nullptr, st);
  Py_END_ALLOW_THREADS
  if (rc != FVSR_OK) return not_done(rc, "fp8_gemm");
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// bind(quant_workspace_floats, quant_fp8_dt, fp8_gemm, gemm_amax_parts): the
// addresses of the C ABI functions.
PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long p[4];
  if (!PyArg_ParseTuple(args, "KKKK", &p[0], &p[1], &p[2], &p[3])) return nullptr;
  abi.quant_workspace_floats = (decltype(abi.quant_workspace_floats))(uintptr_t)p[0];
  abi.quant_fp8_dt = (decltype(abi.quant_fp8_dt))(uintptr_t)p[1];
  abi.fp8_gemm = (decltype(abi.fp8_gemm))(uintptr_t)p[2];
  abi.gemm_amax_parts = (decltype(abi.gemm_amax_parts))(uintptr_t)p[3];
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"bind", bind, METH_VARARGS, "addresses of the C ABI functions"},
    {"quantize", (PyCFunction)(void*)quantize, METH_FASTCALL, "quantize(x2, per_token, gelu)"},
    {"gemm", (PyCFunction)(void*)gemm, METH_FASTCALL, "gemm(x8, s, w8, w_scale, bias, amax_part)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fvsr_host", nullptr, -1, kMethods};

}  // namespace

// torch_version: the torch whose headers this was compiled against.
PyMODINIT_FUNC PyInit__fvsr_host() {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "torch_version", FVSR_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
