// torch.ops.mfq.*: the PyTorch-ROCm face of libmfq.  Each op checks its tensors,
// allocates the outputs from torch's caching allocator on the inputs' device,
// and calls the C ABI of include/mfq.h on torch's current HIP stream: no device
// synchronisation, no state of its own.  (PyTorch-ROCm presents its HIP devices
// under the "cuda" device type, hence the ...MasqueradingAsCUDA guard and the
// CUDA dispatch key.)  Only the HIP dispatch key is
// registered, so a CPU tensor is refused by the dispatcher (there is no CPU
// implementation to fall back to).  mflux_amd.core calls these ops; the error
// texts a user sees for bad arguments are produced there, in MLX's wording.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <tuple>

#include "../../include/mfq.h"

namespace {

using at::Tensor;

int dtype_code(at::ScalarType t, const char* what) {
  switch (t) {
    case at::kFloat: return MFQ_F32;
    case at::kHalf: return MFQ_F16;
    case at::kBFloat16: return MFQ_BF16;
    default: TORCH_CHECK(false, "mfq: ", what, " must be float32, float16 or bfloat16, got ", t);
  }
}

void check_status(const char* fn, int rc) {
  TORCH_CHECK(rc == MFQ_OK, fn, " failed: ", mfq_strerror(rc), " (status ", rc, ")");
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

void check_packed(const Tensor& wq, const Tensor& scales, const Tensor& biases) {
  TORCH_CHECK(wq.scalar_type() == at::kUInt32, "mfq: the packed weight must be uint32, got ", wq.scalar_type());
  TORCH_CHECK(wq.dim() == 2 && scales.dim() == 2 && biases.dim() == 2, "mfq: packed weight, scales and biases are 2-D");
  TORCH_CHECK(scales.scalar_type() == biases.scalar_type() && scales.sizes() == biases.sizes(),
              "mfq: scales and biases must agree in dtype and shape");
  TORCH_CHECK(wq.is_contiguous() && scales.is_contiguous() && biases.is_contiguous(), "mfq: operands must be contiguous");
  TORCH_CHECK(scales.device() == wq.device() && biases.device() == wq.device(), "mfq: operands on different devices");
}

std::tuple<Tensor, Tensor, Tensor> quantize_affine(const Tensor& w, int64_t group_size, int64_t bits) {
  TORCH_CHECK(w.dim() == 2 && w.is_contiguous(), "mfq::quantize_affine: w must be a contiguous matrix");
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(w.device());
  const int64_t rows = w.size(0), K = w.size(1);
  TORCH_CHECK(group_size > 0 && K % group_size == 0 && (K * bits) % 32 == 0, "mfq::quantize_affine: bad K");
  Tensor wq = at::empty({rows, K * bits / 32}, w.options().dtype(at::kUInt32));
  Tensor scales = at::empty({rows, K / group_size}, w.options());
  Tensor biases = at::empty_like(scales);
  if (rows == 0) return {wq, scales, biases};
  check_status("mfq_quantize_affine",
               mfq_quantize_affine(w.data_ptr(), dtype_code(w.scalar_type(), "w"), rows, K, (int)group_size, (int)bits,
                                   static_cast<uint32_t*>(wq.data_ptr()), scales.data_ptr(), biases.data_ptr(),
                                   stream_of(w)));
  return {wq, scales, biases};
}

Tensor dequantize_affine(const Tensor& wq, const Tensor& scales, const Tensor& biases, int64_t group_size, int64_t bits,
                         at::ScalarType out_dtype) {
  check_packed(wq, scales, biases);
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(wq.device());
  const int64_t rows = wq.size(0), K = wq.size(1) * 32 / bits;
  Tensor out = at::empty({rows, K}, scales.options().dtype(out_dtype));
  if (rows == 0) return out;
  check_status("mfq_dequantize_affine",
               mfq_dequantize_affine(static_cast<const uint32_t*>(wq.data_ptr()), scales.data_ptr(), biases.data_ptr(),
                                     dtype_code(scales.scalar_type(), "scales"), rows, K, (int)group_size, (int)bits,
                                     out.data_ptr(), dtype_code(out_dtype, "the output"), stream_of(wq)));
  return out;
}

Tensor dequantize_rows(const Tensor& wq, const Tensor& scales, const Tensor& biases, const Tensor& indices,
                       int64_t group_size, int64_t bits, at::ScalarType out_dtype) {
  check_packed(wq, scales, biases);
  TORCH_CHECK(indices.scalar_type() == at::kLong && indices.dim() == 1 && indices.is_contiguous() &&
                  indices.device() == wq.device(),
              "mfq::dequantize_rows: indices must be a contiguous int64 vector on the table's device");
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(wq.device());
  const int64_t K = wq.size(1) * 32 / bits;
  Tensor out = at::empty({indices.size(0), K}, scales.options().dtype(out_dtype));
  if (indices.size(0) == 0) return out;
  check_status("mfq_dequantize_rows",
               mfq_dequantize_rows(static_cast<const uint32_t*>(wq.data_ptr()), scales.data_ptr(), biases.data_ptr(),
                                   dtype_code(scales.scalar_type(), "scales"), indices.data_ptr<int64_t>(),
                                   indices.size(0), wq.size(0), K, (int)group_size, (int)bits, out.data_ptr(),
                                   dtype_code(out_dtype, "the output"), stream_of(wq)));
  return out;
}

struct Matmul {
  int64_t M, K, N;
  int sb;
  const void* bias;
};

// common checks of the products; x is [M, K] in the scales' dtype
Matmul check_matmul(const char* fn, const Tensor& x, const Tensor& wq, const Tensor& scales, const Tensor& biases,
                    const c10::optional<Tensor>& bias, int64_t bits) {
  check_packed(wq, scales, biases);
  TORCH_CHECK(x.dim() == 2 && x.is_contiguous() && x.device() == wq.device(), fn, ": x must be a contiguous matrix on ",
              wq.device());
  TORCH_CHECK(x.scalar_type() == scales.scalar_type(), fn, ": x and scales must share a 16-bit dtype");
  Matmul m{x.size(0), wq.size(1) * 32 / bits, wq.size(0), dtype_code(scales.scalar_type(), "scales"), nullptr};
  TORCH_CHECK(x.size(1) == m.K, fn, ": x has ", x.size(1), " columns, the weight ", m.K);
  if (bias.has_value()) {
    TORCH_CHECK(bias->dim() == 1 && bias->size(0) == m.N && bias->scalar_type() == scales.scalar_type() &&
                    bias->is_contiguous() && bias->device() == wq.device(),
                fn, ": bias must be a contiguous [N] vector of the scales' dtype");
    m.bias = bias->data_ptr();
  }
  return m;
}

// y = x @ dequantize(wq)^T (+ t @ bs^T) (+ bias); the float32 planes of a K
// split come from torch's allocator on the current stream, so their reuse is
// ordered after this call.  `ok` is false (and y undefined) when the library
// has no kernel for the combination (MFQ_EUNSUPPORTED).
std::tuple<Tensor, bool> qmm_t(const Tensor& x, const Tensor& wq, const Tensor& scales, const Tensor& biases,
             const c10::optional<Tensor>& bias, int64_t group_size, int64_t bits, at::ScalarType out_dtype,
             const c10::optional<Tensor>& lr_t, const c10::optional<Tensor>& lr_bs) {
  const Matmul m = check_matmul("mfq::qmm_t", x, wq, scales, biases, bias, bits);
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor y = at::empty({m.M, m.N}, x.options().dtype(out_dtype));
  if (m.M == 0) return {y, true};
  const void *t = nullptr, *bs = nullptr;
  int64_t rank = 0;
  if (lr_t.has_value() || lr_bs.has_value()) {
    TORCH_CHECK(lr_t.has_value() && lr_bs.has_value(), "mfq::qmm_t: the low-rank update needs both t and bs");
    rank = lr_bs->size(1);
    TORCH_CHECK(lr_t->dim() == 2 && lr_bs->dim() == 2 && lr_t->size(0) == m.M && lr_t->size(1) == rank &&
                    lr_bs->size(0) == m.N && lr_t->scalar_type() == x.scalar_type() &&
                    lr_bs->scalar_type() == x.scalar_type() && lr_t->is_contiguous() && lr_bs->is_contiguous(),
                "mfq::qmm_t: the low-rank update is t [M, R], bs [N, R], contiguous, in x's dtype");
    t = lr_t->data_ptr();
    bs = lr_bs->data_ptr();
  }
  size_t ws_bytes = 0;
  if (rank && out_dtype == at::kFloat)  // (an update with a float32 result: the kernels that dequantise in the GEMM)
    ws_bytes = mfq_qmm_t_workspace_bytes(m.M, m.K, m.N, (int)group_size, (int)bits);
  else
    mfq_qmm_t_plan(m.M, m.K, m.N, (int)group_size, (int)bits, 0, nullptr, nullptr, nullptr, &ws_bytes);
  Tensor ws;
  if (ws_bytes) ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
  const int rc = mfq_qmm_t_low_rank(x.data_ptr(), m.sb, m.M, m.K, static_cast<const uint32_t*>(wq.data_ptr()),
                                    scales.data_ptr(), biases.data_ptr(), m.sb, m.bias, m.N, (int)group_size, (int)bits,
                                    t, bs, rank, y.data_ptr(), dtype_code(out_dtype, "the output"),
                                    ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, stream_of(x));
  if (rc == MFQ_EUNSUPPORTED) return {y, false};
  check_status("mfq_qmm_t_low_rank", rc);
  return {y, true};
}

// qmm_t with an epilogue of include/mfq.h's mfq_qmm_t_epilogue (1: gelu_approx from column act_from on,
// 2: residual + gate * y, 3: SwiGLU of gate / up rows stacked in blocks of 32, y is [M, N/2]); `ok` is false
// (and y undefined) when no kernel fuses it for the shape
std::tuple<Tensor, bool> qmm_t_epilogue(const Tensor& x, const Tensor& wq, const Tensor& scales, const Tensor& biases,
                                        const c10::optional<Tensor>& bias, int64_t group_size, int64_t bits,
                                        int64_t epilogue, const c10::optional<Tensor>& gate,
                                        const c10::optional<Tensor>& residual, int64_t act_from) {
  const Matmul m = check_matmul("mfq::qmm_t_epilogue", x, wq, scales, biases, bias, bits);
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const void *gate_p = nullptr, *res_p = nullptr;
  if (epilogue == MFQ_EPILOGUE_GATE_RESIDUAL) {
    TORCH_CHECK(gate.has_value() && residual.has_value(), "mfq::qmm_t_epilogue: gate and residual are required");
    TORCH_CHECK(gate->dim() == 1 && gate->size(0) == m.N && gate->scalar_type() == x.scalar_type() &&
                    gate->is_contiguous() && gate->device() == x.device(),
                "mfq::qmm_t_epilogue: gate must be a contiguous [N] vector of x's dtype");
    TORCH_CHECK(residual->dim() == 2 && residual->size(0) == m.M && residual->size(1) == m.N &&
                    residual->scalar_type() == x.scalar_type() && residual->is_contiguous() &&
                    residual->device() == x.device(),
                "mfq::qmm_t_epilogue: residual must be a contiguous [M, N] matrix of x's dtype");
    gate_p = gate->data_ptr();
    res_p = residual->data_ptr();
  }
  const int64_t n_out = epilogue == MFQ_EPILOGUE_SWIGLU ? m.N / 2 : m.N;
  Tensor y = at::empty({m.M, n_out}, x.options());
  if (m.M == 0) return {y, true};
  size_t ws_bytes = 0;
  mfq_qmm_t_plan(m.M, m.K, m.N, (int)group_size, (int)bits, (int)epilogue, nullptr, nullptr, nullptr, &ws_bytes);
  Tensor ws;
  if (ws_bytes) ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
  const int rc = mfq_qmm_t_epilogue(x.data_ptr(), m.sb, m.M, m.K, static_cast<const uint32_t*>(wq.data_ptr()),
                                    scales.data_ptr(), biases.data_ptr(), m.sb, m.bias, m.N, (int)group_size,
                                    (int)bits, (int)epilogue, gate_p, res_p, act_from, y.data_ptr(), m.sb,
                                    ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, stream_of(x));
  if (rc == MFQ_EUNSUPPORTED) return {y, false};
  check_status("mfq_qmm_t_epilogue", rc);
  return {y, true};
}

// y[M, K] = x[M, N] @ dequantize(wq[N, K]) (+ t @ bs^T); `ok` is false when N is not a multiple of 8
std::tuple<Tensor, bool> qmm_n(const Tensor& x, const Tensor& wq, const Tensor& scales, const Tensor& biases,
                               int64_t group_size, int64_t bits, at::ScalarType out_dtype,
                               const c10::optional<Tensor>& lr_t, const c10::optional<Tensor>& lr_bs) {
  check_packed(wq, scales, biases);
  TORCH_CHECK(x.dim() == 2 && x.is_contiguous() && x.device() == wq.device() && x.size(1) == wq.size(0) &&
                  x.scalar_type() == scales.scalar_type(),
              "mfq::qmm_n: x must be a contiguous [M, N] matrix of the scales' dtype on the weight's device");
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const int64_t M = x.size(0), N = wq.size(0), K = wq.size(1) * 32 / bits;
  Tensor y = at::empty({M, K}, x.options().dtype(out_dtype));
  if (M == 0) return {y, true};
  const int sb = dtype_code(scales.scalar_type(), "scales");
  const void *t = nullptr, *bs = nullptr;
  int64_t rank = 0;
  if (lr_t.has_value() || lr_bs.has_value()) {
    TORCH_CHECK(lr_t.has_value() && lr_bs.has_value(), "mfq::qmm_n: the low-rank update needs both t and bs");
    TORCH_CHECK(lr_t->dim() == 2 && lr_bs->dim() == 2 && lr_t->size(0) == M && lr_bs->size(0) == K &&
                    lr_t->size(1) == lr_bs->size(1) && lr_t->scalar_type() == x.scalar_type() &&
                    lr_bs->scalar_type() == x.scalar_type() && lr_t->is_contiguous() && lr_bs->is_contiguous() &&
                    lr_t->device() == x.device() && lr_bs->device() == x.device(),
                "mfq::qmm_n: the low-rank update is t [M, R], bs [K, R], contiguous, in x's dtype");
    rank = lr_bs->size(1);
    t = lr_t->data_ptr();
    bs = lr_bs->data_ptr();
  }
  // the transposed 16-bit copy of the two-kernel path (and the planes of its K cut), where that is used
  const size_t ws_bytes = mfq_qmm_n_workspace_bytes(M, N, K, (int)group_size, (int)bits);
  Tensor ws;
  if (ws_bytes) ws = at::empty({(int64_t)ws_bytes}, x.options().dtype(at::kByte));
  const int rc = mfq_qmm_n_low_rank(x.data_ptr(), sb, M, N, static_cast<const uint32_t*>(wq.data_ptr()),
                                    scales.data_ptr(), biases.data_ptr(), sb, K, (int)group_size, (int)bits, t, bs, rank,
                                    y.data_ptr(), dtype_code(out_dtype, "the output"),
                                    ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, stream_of(x));
  if (rc == MFQ_EUNSUPPORTED) return {y, false};
  check_status("mfq_qmm_n", rc);
  return {y, true};
}

// one to four rows of silu(x) against the weights in one kernel; `ok` is false
// (and y undefined) when no fused kernel takes the shape
std::tuple<Tensor, bool> qmv_silu(const Tensor& x, const Tensor& wq, const Tensor& scales, const Tensor& biases,
                                  const c10::optional<Tensor>& bias, int64_t group_size, int64_t bits) {
  const Matmul m = check_matmul("mfq::qmv_silu", x, wq, scales, biases, bias, bits);
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor y = at::empty({m.M, m.N}, x.options());
  const int rc = mfq_qmv_silu(x.data_ptr(), m.sb, m.M, m.K, static_cast<const uint32_t*>(wq.data_ptr()),
                              scales.data_ptr(), biases.data_ptr(), m.sb, m.bias, m.N, (int)group_size, (int)bits,
                              y.data_ptr(), m.sb, stream_of(x));
  if (rc == MFQ_EUNSUPPORTED) return {y, false};
  check_status("mfq_qmv_silu", rc);
  return {y, true};
}

// LayerNorm(x, eps) * (1 + scale) + shift over the rows of x [M, K]; scale and shift [B, K] with M % B == 0 (or
// neither); `ok` is false when the rows are too long for the kernel
std::tuple<Tensor, bool> layer_norm_modulate(const Tensor& x, const c10::optional<Tensor>& scale,
                                             const c10::optional<Tensor>& shift, double eps) {
  TORCH_CHECK(x.dim() == 2 && x.is_contiguous(), "mfq::layer_norm_modulate: x must be a contiguous matrix");
  TORCH_CHECK(scale.has_value() == shift.has_value(), "mfq::layer_norm_modulate: scale and shift come together");
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const int64_t M = x.size(0), K = x.size(1);
  int64_t rows_per_vector = M;
  const void *sc = nullptr, *sh = nullptr;
  if (scale.has_value()) {
    TORCH_CHECK(scale->dim() == 2 && scale->size(1) == K && scale->sizes() == shift->sizes() && scale->size(0) > 0 &&
                    M % scale->size(0) == 0 && scale->scalar_type() == x.scalar_type() &&
                    shift->scalar_type() == x.scalar_type() && scale->is_contiguous() && shift->is_contiguous() &&
                    scale->device() == x.device() && shift->device() == x.device(),
                "mfq::layer_norm_modulate: scale and shift must be contiguous [B, K] matrices of x's dtype, M % B == 0");
    rows_per_vector = M / scale->size(0);
    sc = scale->data_ptr();
    sh = shift->data_ptr();
  }
  Tensor y = at::empty_like(x);
  if (M == 0) return {y, true};
  const int rc = mfq_layer_norm_modulate(x.data_ptr(), dtype_code(x.scalar_type(), "x"), M, K, sc, sh, rows_per_vector,
                                         (float)eps, y.data_ptr(), stream_of(x));
  if (rc == MFQ_EUNSUPPORTED) return {y, false};
  check_status("mfq_layer_norm_modulate", rc);
  return {y, true};
}

// t = x @ A, A in the fragment order of mfq_low_rank_down ([R/16, K/32, 4, 16, 8])
Tensor low_rank_down(const Tensor& x, const Tensor& af) {
  TORCH_CHECK(x.dim() == 2 && af.dim() == 5 && x.is_contiguous() && af.is_contiguous() && af.size(2) == 4 &&
                  af.size(3) == 16 && af.size(4) == 8 && x.size(1) == 32 * af.size(1) &&
                  x.scalar_type() == af.scalar_type(),
              "mfq::low_rank_down: x [M, K], af [R/16, K/32, 4, 16, 8], contiguous, of one 16-bit type");
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const int64_t R = 16 * af.size(0);
  Tensor t = at::empty({x.size(0), R}, x.options());
  check_status("mfq_low_rank_down", mfq_low_rank_down(x.data_ptr(), af.data_ptr(), dtype_code(x.scalar_type(), "x"),
                                                      x.size(0), x.size(1), R, t.data_ptr(), stream_of(x)));
  return t;
}

// ---- a trainable adapter's products (include/mfq.h, mfq_low_rank_pack and what follows it)
int64_t training_rank(int64_t rank) { return rank <= 16 ? 16 : 32; }

void check_factor(const char* fn, const Tensor& t, int64_t rows, int64_t columns, const Tensor& like) {
  TORCH_CHECK(t.dim() == 2 && t.size(0) == rows && t.size(1) == columns && t.is_contiguous() &&
                  t.scalar_type() == like.scalar_type() && t.device() == like.device(),
              fn, ": expected a contiguous [", rows, ", ", columns, "] matrix of ", like.scalar_type(), " on ", like.device());
}

void check_fragments(const char* fn, const Tensor& t, int64_t steps, const Tensor& like) {
  TORCH_CHECK(t.dim() == 5 && t.size(1) == steps && t.size(2) == 4 && t.size(3) == 16 && t.size(4) == 8 && t.is_contiguous() &&
                  t.scalar_type() == like.scalar_type() && t.device() == like.device(),
              fn, ": expected fragments [R/16, ", steps, ", 4, 16, 8] of ", like.scalar_type(), " on ", like.device());
}

// lora_A [K, rank], lora_B [rank, N] -> their fragments, scale lora_B^T [N, R] and lora_A [K, R]: new tensors all, also at the
// ranks where lora_A needs no padding, so that backward sees the factors that forward saw, whatever is written to them between
std::tuple<Tensor, Tensor, Tensor, Tensor> low_rank_pack(const Tensor& a, const Tensor& b, double scale) {
  TORCH_CHECK(a.dim() == 2 && b.dim() == 2, "mfq::low_rank_pack: lora_A [K, rank], lora_B [rank, N]");
  const int64_t K = a.size(0), rank = a.size(1), N = b.size(1), R = training_rank(rank);
  check_factor("mfq::low_rank_pack", a, K, rank, a);
  check_factor("mfq::low_rank_pack", b, rank, N, a);
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(a.device());
  Tensor af = at::empty({R / 16, K / 32, 4, 16, 8}, a.options()), bf = at::empty({R / 16, N / 32, 4, 16, 8}, a.options());
  Tensor bs = at::empty({N, R}, a.options()), ap = at::empty({K, R}, a.options());
  check_status("mfq_low_rank_pack",
               mfq_low_rank_pack(a.data_ptr(), b.data_ptr(), dtype_code(a.scalar_type(), "lora_A"), K, N, rank, R, (float)scale,
                                 af.data_ptr(), bf.data_ptr(), bs.data_ptr(), ap.data_ptr(), stream_of(a)));
  return {af, bf, bs, ap};
}

// t [M, R] = x @ lora_A and its fragments
std::tuple<Tensor, Tensor> low_rank_forward(const Tensor& x, const Tensor& af, int64_t rank) {
  TORCH_CHECK(x.dim() == 2, "mfq::low_rank_forward: x [M, K]");
  const int64_t M = x.size(0), K = x.size(1);
  check_factor("mfq::low_rank_forward", x, M, K, x);
  check_fragments("mfq::low_rank_forward", af, K / 32, x);
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const int64_t R = 16 * af.size(0);
  Tensor t = at::empty({M, R}, x.options()), tf = at::empty({R / 16, (M + 31) / 32, 4, 16, 8}, x.options());
  check_status("mfq_low_rank_forward", mfq_low_rank_forward(x.data_ptr(), af.data_ptr(), dtype_code(x.scalar_type(), "x"), M, K,
                                                            rank, R, t.data_ptr(), tf.data_ptr(), stream_of(x)));
  return {t, tf};
}

// (gt [M, R], its fragments, the gradient of lora_B [rank, N]); what is not wanted comes back empty
std::tuple<Tensor, Tensor, Tensor> low_rank_gradient(const Tensor& g, const Tensor& bf, const Tensor& tf, int64_t rank, double scale,
                                                     bool want_gt, bool want_db) {
  TORCH_CHECK(g.dim() == 2, "mfq::low_rank_gradient: g [M, N]");
  const int64_t M = g.size(0), N = g.size(1);
  check_factor("mfq::low_rank_gradient", g, M, N, g);
  check_fragments("mfq::low_rank_gradient", bf, N / 32, g);
  check_fragments("mfq::low_rank_gradient", tf, (M + 31) / 32, g);
  TORCH_CHECK(tf.size(0) == bf.size(0), "mfq::low_rank_gradient: fragments of different ranks");
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(g.device());
  const int64_t R = 16 * bf.size(0);
  Tensor gt, gtf, db;
  if (want_gt) {
    gt = at::empty({M, R}, g.options());
    gtf = at::empty({R / 16, (M + 31) / 32, 4, 16, 8}, g.options());
  } else {
    gt = gtf = at::empty({0}, g.options());
  }
  db = at::empty({want_db ? rank : 0, N}, g.options());
  if (!want_gt && !want_db) return {gt, gtf, db};
  check_status("mfq_low_rank_gradient",
               mfq_low_rank_gradient(g.data_ptr(), bf.data_ptr(), tf.data_ptr(), dtype_code(g.scalar_type(), "g"), M, N, rank, R,
                                     (float)scale, want_gt ? gt.data_ptr() : nullptr, want_gt ? gtf.data_ptr() : nullptr,
                                     want_db ? db.data_ptr() : nullptr, stream_of(g)));
  return {gt, gtf, db};
}

// x^T @ t [K, rank], t in fragments
Tensor low_rank_up(const Tensor& x, const Tensor& tf, int64_t rank) {
  TORCH_CHECK(x.dim() == 2, "mfq::low_rank_up: x [M, K]");
  const int64_t M = x.size(0), K = x.size(1);
  check_factor("mfq::low_rank_up", x, M, K, x);
  check_fragments("mfq::low_rank_up", tf, (M + 31) / 32, x);
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor out = at::empty({K, rank}, x.options());
  check_status("mfq_low_rank_up", mfq_low_rank_up(x.data_ptr(), tf.data_ptr(), dtype_code(x.scalar_type(), "x"), M, K, rank,
                                                  16 * tf.size(0), out.data_ptr(), stream_of(x)));
  return out;
}

// y += t @ bs^T in place
void low_rank_add_(Tensor& y, const Tensor& t, const Tensor& bs) {
  TORCH_CHECK(y.dim() == 2 && t.dim() == 2 && bs.dim() == 2 && y.is_contiguous() && t.is_contiguous() &&
                  bs.is_contiguous() && t.size(0) == y.size(0) && bs.size(0) == y.size(1) && t.size(1) == bs.size(1) &&
                  t.scalar_type() == bs.scalar_type(),
              "mfq::low_rank_add_: y [M, N], t [M, R], bs [N, R], contiguous");
  const c10::hip::HIPGuardMasqueradingAsCUDA guard(y.device());
  check_status("mfq_low_rank_add",
               mfq_low_rank_add(t.data_ptr(), bs.data_ptr(), dtype_code(t.scalar_type(), "t"), y.size(0), y.size(1),
                                t.size(1), y.data_ptr(), dtype_code(y.scalar_type(), "y"), stream_of(y)));
}

}  // namespace

TORCH_LIBRARY(mfq, m) {
  m.def("quantize_affine(Tensor w, int group_size, int bits) -> (Tensor, Tensor, Tensor)");
  m.def("dequantize_affine(Tensor wq, Tensor scales, Tensor biases, int group_size, int bits, ScalarType out_dtype) -> Tensor");
  m.def("dequantize_rows(Tensor wq, Tensor scales, Tensor biases, Tensor indices, int group_size, int bits, ScalarType out_dtype) -> Tensor");
  m.def("qmm_t(Tensor x, Tensor wq, Tensor scales, Tensor biases, Tensor? bias, int group_size, int bits, ScalarType out_dtype, Tensor? lr_t, Tensor? lr_bs) -> (Tensor, bool)");
  m.def("qmm_t_epilogue(Tensor x, Tensor wq, Tensor scales, Tensor biases, Tensor? bias, int group_size, int bits, int epilogue, Tensor? gate, Tensor? residual, int act_from) -> (Tensor, bool)");
  m.def("qmm_n(Tensor x, Tensor wq, Tensor scales, Tensor biases, int group_size, int bits, ScalarType out_dtype, Tensor? lr_t=None, Tensor? lr_bs=None) -> (Tensor, bool)");
  m.def("qmv_silu(Tensor x, Tensor wq, Tensor scales, Tensor biases, Tensor? bias, int group_size, int bits) -> (Tensor, bool)");
  m.def("layer_norm_modulate(Tensor x, Tensor? scale, Tensor? shift, float eps) -> (Tensor, bool)");
  m.def("low_rank_add_(Tensor(a!) y, Tensor t, Tensor bs) -> ()");
  m.def("low_rank_down(Tensor x, Tensor af) -> Tensor");
  m.def("low_rank_pack(Tensor lora_a, Tensor lora_b, float scale) -> (Tensor, Tensor, Tensor, Tensor)");
  m.def("low_rank_forward(Tensor x, Tensor af, int rank) -> (Tensor, Tensor)");
  m.def("low_rank_gradient(Tensor g, Tensor bf, Tensor tf, int rank, float scale, bool want_gt, bool want_db) -> (Tensor, Tensor, Tensor)");
  m.def("low_rank_up(Tensor x, Tensor tf, int rank) -> Tensor");
}

TORCH_LIBRARY_IMPL(mfq, CUDA, m) {  // the HIP backend answers to torch's CUDA dispatch key
  m.impl("quantize_affine", quantize_affine);
  m.impl("dequantize_affine", dequantize_affine);
  m.impl("dequantize_rows", dequantize_rows);
  m.impl("qmm_t", qmm_t);
  m.impl("qmm_t_epilogue", qmm_t_epilogue);
  m.impl("qmm_n", qmm_n);
  m.impl("qmv_silu", qmv_silu);
  m.impl("layer_norm_modulate", layer_norm_modulate);
  m.impl("low_rank_add_", low_rank_add_);
  m.impl("low_rank_down", low_rank_down);
  m.impl("low_rank_pack", low_rank_pack);
  m.impl("low_rank_forward", low_rank_forward);
  m.impl("low_rank_gradient", low_rank_gradient);
  m.impl("low_rank_up", low_rank_up);
}
