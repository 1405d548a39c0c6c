// The module calls of mflux_amd.nn as Python C functions: one crossing from
// Python per quantized linear, without the dispatcher.
//
// A modulation call is a 3 to 11 us kernel.  Through core.py's checks, the
// boxed call of a torch.ops operator with ten arguments and the reshapes around
// it, issuing one took 13.5 us of host time, so a chain of them ran at the
// host's pace (3072 -> 18432 at 8 bits: 13.6 us a call, the kernel 11.0; 256 ->
// 15360: 13.5 us, the kernel 4.7).  These functions take the ordinary case --
// plain contiguous HIP tensors of one 16-bit type that need no gradient, with
// nothing intercepting torch calls -- straight to the C ABI of include/mfq.h,
// and return None for every other case, malformed calls included: the caller
// then goes through core.py, which handles it or words the error.  Whatever can
// throw (allocations, looking up a pointer or the stream) happens with the
// interpreter's lock held; without it there is only the C call.  A profiler sees
// the operator that the call stands for.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/mfq.h"

namespace {

using at::Tensor;

// A tensor these functions may read by pointer: an ordinary torch.Tensor (or Parameter) on a HIP device,
// contiguous, no subclass, no lazily negated or conjugated view, nothing wrapped around it.
bool plain(const Tensor& t) {
  static const c10::DispatchKeySet kWrapped({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                             c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                             c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor,
                                             c10::DispatchKey::Negative, c10::DispatchKey::Conjugate});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kWrapped) && t.is_contiguous();
}

// None -> an undefined tensor; false: not a tensor at all
bool tensor_arg(PyObject* o, Tensor* out) {
  if (o == Py_None) return true;
  if (!THPVariable_CheckExact(o)) return false;  // torch.Tensor and Parameter, no other subclass
  *out = THPVariable_Unpack(o);
  return true;
}

bool int_arg(PyObject* o, int64_t* out) {
  if (!PyLong_Check(o)) return false;
  *out = PyLong_AsLongLong(o);
  if (*out == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// The operands of one call, checked; `ok` is false where core.py has to take it.
struct Linear {
  Tensor x, wq, scales, biases, bias;
  int64_t gs = 0, bits = 0, M = 0, K = 0, N = 0;
  int dtype = 0;
  bool float32 = false;  // x is float32, and so is y

  bool parse(PyObject* const* args) {
    return tensor_arg(args[0], &x) && tensor_arg(args[1], &wq) && tensor_arg(args[2], &scales) &&
           tensor_arg(args[3], &biases) && tensor_arg(args[4], &bias) && int_arg(args[5], &gs) &&
           int_arg(args[6], &bits) && check();
  }

  bool check() {
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled()) return false;
    if (torch::jit::tracer::isTracing()) return false;  // a trace would keep this call's result as a constant
    if (!plain(x) || !plain(wq) || !plain(scales) || !plain(biases) || (bias.defined() && !plain(bias))) return false;
    if (c10::GradMode::is_enabled() && (x.requires_grad() || (bias.defined() && bias.requires_grad()))) return false;
    const at::ScalarType t = scales.scalar_type();
    if (t == at::kBFloat16) dtype = MFQ_BF16;
    else if (t == at::kHalf) dtype = MFQ_F16;
    else return false;
    if (wq.scalar_type() != at::kUInt32 || biases.scalar_type() != t || x.scalar_type() != (float32 ? at::kFloat : t))
      return false;
    if (wq.dim() != 2 || scales.dim() != 2 || biases.sizes() != scales.sizes() || x.dim() < 1) return false;
    if ((gs != 32 && gs != 64 && gs != 128) || (bits != 3 && bits != 4 && bits != 5 && bits != 6 && bits != 8)) return false;
    N = wq.size(0);
    K = wq.size(1) * 32 / bits;
    if (scales.size(0) != N || K * bits != wq.size(1) * 32 || scales.size(1) * gs != K) return false;
    if (x.size(-1) != K || K == 0 || N == 0) return false;
    M = x.numel() / K;
    if (M == 0) return false;
    if (bias.defined() && (bias.scalar_type() != t || bias.dim() != 1 || bias.size(0) != N)) return false;
    const auto dev = x.device();
    return wq.device() == dev && scales.device() == dev && biases.device() == dev &&
           (!bias.defined() || bias.device() == dev);
  }

  // the output: x's leading dimensions and n columns
  Tensor out(int64_t n) const {
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = n;
    return at::empty(shape, x.options().requires_grad(false));
  }
  size_t workspace_bytes(int epilogue) const {
    size_t bytes = 0;
    mfq_qmm_t_plan(M, K, N, (int)gs, (int)bits, epilogue, nullptr, nullptr, nullptr, &bytes);
    return bytes;
  }
  Tensor workspace(size_t bytes) const { return at::empty({(int64_t)bytes}, x.options().dtype(at::kByte).requires_grad(false)); }
  std::vector<c10::IValue> inputs() const { return {x, wq, scales, biases, bias, gs, bits}; }  // for a profiler

  // where the operands are, for reading only (a copy-on-write tensor stays one)
  struct Pointers {
    const void *x, *scales, *biases, *bias;
    const uint32_t* wq;
    void* stream;
  };
  Pointers pointers() const {
    return {x.const_data_ptr(), scales.const_data_ptr(), biases.const_data_ptr(),
            bias.defined() ? bias.const_data_ptr() : nullptr, static_cast<const uint32_t*>(wq.const_data_ptr()),
            c10::hip::getCurrentHIPStream(x.get_device()).stream()};
  }
};

// y, or None where another route may take the call; a launch that failed is not issued a second time
PyObject* result(const char* fn, int rc, const Tensor& y) {
  TORCH_CHECK(rc != MFQ_ELAUNCH, fn, " failed: ", mfq_strerror(rc), " (status ", rc, ")");
  if (rc != MFQ_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(y);
}

// linear(x, weight, scales, biases, bias or None, group_size, bits) -> y or None
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Linear p;
  if (n != 7 || !p.parse(args)) Py_RETURN_NONE;
  RECORD_FUNCTION("mfq::qmm_t", p.inputs());
  const c10::hip::HIPGuardMasqueradingAsCUDA on_device(p.x.device());
  Tensor y = p.out(p.N), ws;
  const size_t ws_bytes = p.workspace_bytes(0);
  if (ws_bytes) ws = p.workspace(ws_bytes);
  const Linear::Pointers in = p.pointers();
  void *y_p = y.data_ptr(), *ws_p = ws_bytes ? ws.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = mfq_qmm_t_ws(in.x, p.dtype, p.M, p.K, in.wq, in.scales, in.biases, p.dtype, in.bias, p.N, (int)p.gs, (int)p.bits,
                    y_p, p.dtype, ws_p, ws_bytes, in.stream);
  Py_END_ALLOW_THREADS
  return result("mfq_qmm_t_ws", rc, y);
  END_HANDLE_TH_ERRORS
}

// linear_float32(x, weight, scales, biases, bias or None, group_size, bits) -> y or None: float32 x, rounded to the scales' type
// for the product, whose sums and bias are the float32 result
PyObject* linear_float32(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Linear p;
  p.float32 = true;
  if (n != 7 || !p.parse(args)) Py_RETURN_NONE;
  RECORD_FUNCTION("mfq::qmm_t", p.inputs());
  const c10::hip::HIPGuardMasqueradingAsCUDA on_device(p.x.device());
  Tensor y = p.out(p.N), rounded = at::empty({p.M, p.K}, p.scales.options().requires_grad(false)), ws;
  const size_t ws_bytes = p.workspace_bytes(0);
  if (ws_bytes) ws = p.workspace(ws_bytes);
  const Linear::Pointers in = p.pointers();
  void *y_p = y.data_ptr(), *r_p = rounded.data_ptr(), *ws_p = ws_bytes ? ws.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = mfq_round(static_cast<const float*>(in.x), p.M * p.K, p.dtype, r_p, in.stream);
  if (rc == MFQ_OK)
    rc = mfq_qmm_t_ws(r_p, p.dtype, p.M, p.K, in.wq, in.scales, in.biases, p.dtype, in.bias, p.N, (int)p.gs, (int)p.bits, y_p,
                      MFQ_F32, ws_p, ws_bytes, in.stream);
  Py_END_ALLOW_THREADS
  return result("mfq_round, mfq_qmm_t_ws", rc, y);
  END_HANDLE_TH_ERRORS
}

// silu_linear(x, weight, scales, biases, bias or None, group_size, bits) -> linear(silu(x)) or None
PyObject* silu_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Linear p;
  if (n != 7 || !p.parse(args)) Py_RETURN_NONE;
  if (p.M > 16 || (p.bits != 4 && p.bits != 8)) Py_RETURN_NONE;
  RECORD_FUNCTION(p.M > 4 ? "mfq::qmm_t" : "mfq::qmv_silu", p.inputs());
  const c10::hip::HIPGuardMasqueradingAsCUDA on_device(p.x.device());
  Tensor y = p.out(p.N), s;
  if (p.M > 4) s = p.out(p.K);  // five rows and more: the activation in a launch of its own
  const Linear::Pointers in = p.pointers();
  void *y_p = y.data_ptr(), *s_p = p.M > 4 ? s.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (p.M > 4) {
    rc = mfq_silu(in.x, p.dtype, p.M * p.K, s_p, in.stream);
    if (rc == MFQ_OK)
      rc = mfq_qmm_t(s_p, p.dtype, p.M, p.K, in.wq, in.scales, in.biases, p.dtype, in.bias, p.N, (int)p.gs, (int)p.bits,
                     y_p, p.dtype, in.stream);
  } else {
    rc = mfq_qmv_silu(in.x, p.dtype, p.M, p.K, in.wq, in.scales, in.biases, p.dtype, in.bias, p.N, (int)p.gs,
                      (int)p.bits, y_p, p.dtype, in.stream);
  }
  Py_END_ALLOW_THREADS
  return result(p.M > 4 ? "mfq_silu, mfq_qmm_t" : "mfq_qmv_silu", rc, y);
  END_HANDLE_TH_ERRORS
}

// epilogue_linear(x, weight, scales, biases, bias or None, group_size, bits, epilogue, gate or None, residual or
// None, act_from) -> y or None; the epilogues of mfq_qmm_t_epilogue
PyObject* epilogue_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Linear p;
  int64_t epilogue = 0, act_from = 0;
  Tensor gate, residual;
  if (n != 11 || !p.parse(args) || !int_arg(args[7], &epilogue) || !tensor_arg(args[8], &gate) ||
      !tensor_arg(args[9], &residual) || !int_arg(args[10], &act_from))
    Py_RETURN_NONE;
  if (p.M <= 16) Py_RETURN_NONE;  // the matvec kernels have no epilogue
  const void *gate_p = nullptr, *residual_p = nullptr;
  if (epilogue == MFQ_EPILOGUE_GATE_RESIDUAL) {
    const auto same = [&](const Tensor& t) {
      return plain(t) && t.scalar_type() == p.x.scalar_type() && t.device() == p.x.device() &&
             !(c10::GradMode::is_enabled() && t.requires_grad());
    };
    if (!same(gate) || !same(residual) || gate.numel() != p.N || residual.dim() != p.x.dim() ||
        residual.numel() != p.M * p.N || residual.size(-1) != p.N ||
        !residual.sizes().slice(0, residual.dim() - 1).equals(p.x.sizes().slice(0, p.x.dim() - 1)))
      Py_RETURN_NONE;
    gate_p = gate.const_data_ptr();
    residual_p = residual.const_data_ptr();
  } else if (epilogue == MFQ_EPILOGUE_SWIGLU) {
    if (p.N % 64) Py_RETURN_NONE;
  } else if (epilogue != MFQ_EPILOGUE_GELU || act_from < 0 || act_from > p.N || act_from % 8) {
    Py_RETURN_NONE;
  }
  RECORD_FUNCTION("mfq::qmm_t_epilogue", p.inputs());
  const c10::hip::HIPGuardMasqueradingAsCUDA on_device(p.x.device());
  Tensor y = p.out(epilogue == MFQ_EPILOGUE_SWIGLU ? p.N / 2 : p.N), ws;
  const size_t ws_bytes = p.workspace_bytes((int)epilogue);
  if (ws_bytes) ws = p.workspace(ws_bytes);
  const Linear::Pointers in = p.pointers();
  void *y_p = y.data_ptr(), *ws_p = ws_bytes ? ws.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = mfq_qmm_t_epilogue(in.x, p.dtype, p.M, p.K, in.wq, in.scales, in.biases, p.dtype, in.bias, p.N, (int)p.gs,
                          (int)p.bits, (int)epilogue, gate_p, residual_p, act_from, y_p, p.dtype, ws_p, ws_bytes,
                          in.stream);
  Py_END_ALLOW_THREADS
  return result("mfq_qmm_t_epilogue", rc, y);
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"linear", (PyCFunction)(void*)linear, METH_FASTCALL, "x @ dequantize(w).T (+ bias), or None"},
    {"linear_float32", (PyCFunction)(void*)linear_float32, METH_FASTCALL, "the same of a float32 x, or None"},
    {"silu_linear", (PyCFunction)(void*)silu_linear, METH_FASTCALL, "silu(x) @ dequantize(w).T (+ bias), or None"},
    {"epilogue_linear", (PyCFunction)(void*)epilogue_linear, METH_FASTCALL, "a linear with its epilogue, or None"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "libmfq_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_libmfq_torch(void) { return PyModule_Create(&kModule); }
