// Operators of the `cornserve_amd` namespace that an encoder issues once or more per block, implemented natively.
//
// A forward pass of few rows is a chain of about 130 launches of 6 to 10 us each, so what the host spends between two of
// them is what the pass takes: a Python implementation (argument checks, a ctypes structure, a foreign call) costs 20 us a
// launch and left the GPU idle for most of it.  These check the same arguments in the same order with the same messages,
// fill CsGemmArgs from the tensors and call the C ABI on the current stream.  The schemas (and fake implementations) are
// those of cornserve_amd/ops.py, which loads this library after it has defined them; the operators that a pass issues once
// are implemented there.
//
// Everything reaches a kernel as a raw pointer: shapes, dtypes and devices are checked before anything is enqueued, because
// an undersized or mistyped buffer would be an out-of-bounds device access.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/Exception.h>
#include <pybind11/pybind11.h>
#include <torch/library.h>

#include <set>
#include <sstream>
#include <string>

#include "cornserve_amd.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

constexpr int64_t WATTN_TILE_ROWS = 256, WATTN_HEAD_DIM = 80, WATTN_WINDOW = 64;

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

const Tensor* get(const OptTensor& t) { return t.has_value() && t->defined() ? &*t : nullptr; }
void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

// Status codes as the exception categories of the model API (the same mapping as lib.check)
void check_status(int status, const char* what) {
  if (status == CS_OK) return;
  TORCH_CHECK_VALUE(status != CS_ERR_INVALID_ARG, what, ": invalid argument");
  TORCH_CHECK(status != CS_ERR_UNSUPPORTED, what, ": unsupported configuration");
  TORCH_CHECK(status != CS_ERR_TOO_LARGE, what, ": problem exceeds a fixed capacity");
  std::ostringstream msg;
  msg << what << ": HIP launch failed (status " << status << ")";
  pybind11::gil_scoped_acquire gil;
  const pybind11::object error = pybind11::module_::import("cornserve_amd.lib").attr("KernelLibraryError");
  PyErr_SetString(error.ptr(), msg.str().c_str());
  throw pybind11::error_already_set();
}

// What Python prints for a dtype, a shape and a set of devices
std::string py(at::ScalarType dt) { return "torch." + c10::getDtypeNames(dt).first; }

std::string py(at::IntArrayRef sizes) {
  std::ostringstream s;
  s << "(";
  for (size_t i = 0; i < sizes.size(); ++i) s << (i ? ", " : "") << sizes[i];
  s << (sizes.size() == 1 ? ",)" : ")");
  return s.str();
}

std::string py(const std::set<std::string>& devices) {
  std::string s;
  for (const std::string& d : devices) s += (s.empty() ? "['" : ", '") + d + "'";
  return s + "]";
}

void require(const Tensor& t, at::ScalarType dt, const char* name) {
  TORCH_CHECK_VALUE(t.is_cuda(), name, " must be a device tensor");
  TORCH_CHECK_VALUE(t.scalar_type() == dt, name, " must be ", py(dt), ", got ", py(t.scalar_type()));
  TORCH_CHECK_VALUE(t.dim() < 1 || t.stride(-1) == 1, name, " must be contiguous in its last dimension");
}

void require_rows(const Tensor& t, at::ScalarType dt, const char* name) {
  require(t, dt, name);
  TORCH_CHECK_VALUE(t.dim() == 2, name, " must be 2-D");
}

void require_sums(const Tensor* t, int64_t rows, const char* name) {
  if (!t) return;
  require(*t, at::kFloat, name);
  TORCH_CHECK_VALUE(t->dim() == 2 && t->size(1) == CS_SUMSQ_PARTS && t->is_contiguous() && t->size(0) >= rows, name,
                    " must be a contiguous fp32 [>=M, ", CS_SUMSQ_PARTS, "] tensor");
}

// A contiguous vector of exactly n elements
bool is_vector(const Tensor& t, int64_t n) { return t.dim() == 1 && t.size(0) == n && t.is_contiguous(); }

void one_device(std::initializer_list<const Tensor*> operands, const char* op) {
  const Tensor& first = **operands.begin();
  for (const Tensor* t : operands) {
    if (!t || t->device() == first.device()) continue;
    std::set<std::string> on;
    for (const Tensor* o : operands)
      if (o) on.insert(o->device().str());
    TORCH_CHECK_VALUE(false, op, " operands live on different devices: ", py(on));
  }
}

void set_prefetch(CsGemmArgs& args, const Tensor* prefetch, at::Device device) {
  if (!prefetch) return;
  TORCH_CHECK_VALUE(prefetch->is_cuda() && prefetch->device() == device && prefetch->is_contiguous() &&
                        (uintptr_t)prefetch->data_ptr() % 16 == 0,
                    "prefetch must be a contiguous, 16-byte aligned tensor on the operands' device");
  args.prefetch = prefetch->data_ptr();
  args.prefetch_bytes = prefetch->numel() * prefetch->element_size();
}

// Output rows of a product: A's rows, the gathered rows, or the patches of NCHW pixels
int64_t gemm_rows(const Tensor& a, const Tensor* a_rows, int64_t conv_patch) {
  if (conv_patch) {
    TORCH_CHECK_VALUE(a.dim() == 4 && conv_patch >= 1, "with conv_patch, `a` must be NCHW pixels [B,C,H,W]");
    return a.size(0) * (a.size(2) / conv_patch) * (a.size(3) / conv_patch);
  }
  TORCH_CHECK_VALUE(a.dim() == 2, "gemm operands must be 2-D");
  return a_rows ? a_rows->size(0) : a.size(0);
}

void gemm_(const Tensor& out, const Tensor& a, const Tensor& w, const OptTensor& bias_, int64_t epilogue, const OptTensor& residual_,
           const OptTensor& w_scale_, const OptTensor& pos_, const OptTensor& a_rows_, const OptTensor& c_rows_,
           std::optional<int64_t> k, const OptTensor& a_row_sumsq_, const OptTensor& c_row_sumsq_, double norm_eps,
           const OptTensor& a_row_sum_, const OptTensor& c_row_sum_, const OptTensor& w_col_sum_, const OptTensor& residual_lo_,
           const OptTensor& out_lo_, int64_t conv_patch, const OptTensor& prefetch_, bool norm_inline) {
  const Tensor *bias = get(bias_), *residual = get(residual_), *w_scale = get(w_scale_), *pos = get(pos_), *a_rows = get(a_rows_),
               *c_rows = get(c_rows_), *a_row_sumsq = get(a_row_sumsq_), *c_row_sumsq = get(c_row_sumsq_), *a_row_sum = get(a_row_sum_),
               *c_row_sum = get(c_row_sum_), *w_col_sum = get(w_col_sum_), *residual_lo = get(residual_lo_), *out_lo = get(out_lo_);
  CsGemmArgs args = {};
  require(a, at::kBFloat16, "a");
  TORCH_CHECK_VALUE(w.dim() == 2, "gemm operands must be 2-D");
  int64_t a_count, a_cols;
  if (conv_patch) {
    TORCH_CHECK_VALUE(a.dim() == 4 && a.is_contiguous() && conv_patch >= 2 && conv_patch % 2 == 0 && a.size(3) % 2 == 0,
                      "with conv_patch, `a` must be contiguous NCHW pixels with an even width and patch size");
    TORCH_CHECK_VALUE(!a_rows && !k.has_value() && epilogue == CS_EPI_BIAS,
                      "the strided-gather product takes no a_rows / k and only the bias epilogue");
    const int64_t kreal = a.size(1) * conv_patch * conv_patch, kpad = (kreal + 7) / 8 * 8;
    TORCH_CHECK_VALUE(w.size(1) == kpad, "w must have ", kpad, " columns (C*patch*patch = ", kreal, " rounded up to a multiple of 8)");
    a_count = gemm_rows(a, nullptr, conv_patch);
    a_cols = w.size(1);
    args.conv_c = (int32_t)a.size(1);
    args.conv_h = (int32_t)a.size(2);
    args.conv_w = (int32_t)a.size(3);
    args.conv_patch = (int32_t)conv_patch;
  } else {
    TORCH_CHECK_VALUE(a.dim() == 2, "gemm operands must be 2-D");
    a_count = a.size(0);
    a_cols = a.size(1);
    args.lda = a.stride(0);
  }
  const bool fp8 = w.scalar_type() == at::kFloat8_e4m3fn || w.scalar_type() == at::kByte;
  if (!fp8) require(w, at::kBFloat16, "w");
  TORCH_CHECK_VALUE(!fp8 || w_scale, "fp8 weights need w_scale");
  if (a_rows) {
    require(*a_rows, at::kInt, "a_rows");
    TORCH_CHECK_VALUE(a_rows->dim() == 1 && a_rows->is_contiguous(), "a_rows must be a contiguous int32 vector");
  }
  if (c_rows) {
    require(*c_rows, at::kInt, "c_rows");
    TORCH_CHECK_VALUE(c_rows->dim() == 1 && c_rows->is_contiguous(), "c_rows must be a contiguous int32 vector");
  }
  const int64_t M = a_rows ? a_rows->size(0) : a_count, K = k.value_or(a_cols), N = w.size(0);
  TORCH_CHECK_VALUE(K <= a_cols && K >= 1, "k=", K, " exceeds the ", a_cols, " columns of a");
  TORCH_CHECK_VALUE(w.size(1) >= K, "w has ", w.size(1), " columns, need at least K=", K);
  TORCH_CHECK_VALUE(!c_rows || c_rows->size(0) >= M, "c_rows has ", c_rows->size(0), " entries for ", M, " output rows");
  const int64_t n_out = epilogue == CS_EPI_SWIGLU ? N / 2 : N;
  require(out, at::kBFloat16, "out");
  TORCH_CHECK_VALUE(out.dim() == 2 && out.size(1) >= n_out && (c_rows || out.size(0) >= M), "out must be bf16 [>=", M, ", >=", n_out,
                    "], got ", py(out.sizes()));
  if (bias) {
    require(*bias, at::kBFloat16, "bias");
    TORCH_CHECK_VALUE(bias->dim() == 1 && bias->size(0) >= N, "bias must be bf16 [", N, "], got ", py(bias->sizes()));
  }
  TORCH_CHECK_VALUE(epilogue != CS_EPI_RESIDUAL || residual, "EPI_RESIDUAL needs `residual`");
  if (residual) {
    require(*residual, at::kBFloat16, "residual");
    TORCH_CHECK_VALUE(residual->dim() == 2 && residual->size(0) >= M && residual->size(1) >= N, "residual must be bf16 [>=", M, ", >=", N,
                      "], got ", py(residual->sizes()));
  }
  if (pos) {
    require(*pos, at::kBFloat16, "pos");
    TORCH_CHECK_VALUE(pos->dim() == 2 && pos->size(0) >= 1 && pos->size(1) >= N, "pos must be bf16 [period, >=", N, "], got ", py(pos->sizes()));
  }
  if (w_scale) {
    require(*w_scale, at::kFloat, "w_scale");
    TORCH_CHECK_VALUE(w_scale->dim() == 1 && w_scale->size(0) >= N && w_scale->is_contiguous(), "w_scale must be a contiguous fp32 [", N,
                      "] tensor");
  }
  if (residual_lo || out_lo) {
    TORCH_CHECK_VALUE(epilogue == CS_EPI_RESIDUAL && out_lo, "residual_lo / out_lo belong to EPI_RESIDUAL, and residual_lo needs out_lo");
    require(*out_lo, at::kByte, "out_lo");
    TORCH_CHECK_VALUE(out_lo->sizes() == out.sizes() && out_lo->strides() == out.strides(), "out_lo must have the shape and strides of out");
    if (residual_lo) {
      require(*residual_lo, at::kByte, "residual_lo");
      TORCH_CHECK_VALUE(residual_lo->sizes() == residual->sizes() && residual_lo->strides() == residual->strides(),
                        "residual_lo must have the shape and strides of residual");
    }
  }
  one_device({&a, &w, &out, bias, residual, pos, w_scale, a_rows, c_rows, residual_lo, out_lo}, "gemm");
  require_sums(a_row_sumsq, M, "a_row_sumsq");
  require_sums(c_row_sumsq, M, "c_row_sumsq");
  require_sums(a_row_sum, M, "a_row_sum");
  require_sums(c_row_sum, M, "c_row_sum");
  if (w_col_sum) {
    require(*w_col_sum, at::kFloat, "w_col_sum");
    TORCH_CHECK_VALUE(is_vector(*w_col_sum, N), "w_col_sum must be a contiguous fp32 [", N, "] tensor");
  }
  args.A = a.data_ptr();
  args.W = w.data_ptr();
  args.ldw = w.stride(0);
  args.w_scale = (const float*)ptr(w_scale);
  args.bias = ptr(bias);
  args.residual = ptr(residual);
  args.ldr = residual ? residual->stride(0) : 0;
  args.pos = ptr(pos);
  args.ldpos = pos ? pos->stride(0) : 0;
  args.pos_period = pos ? (int32_t)pos->size(0) : 0;
  args.C = out.data_ptr();
  args.ldc = out.stride(0);
  args.a_rows = (const int32_t*)ptr(a_rows);
  args.c_rows = (const int32_t*)ptr(c_rows);
  args.M = (int32_t)M;
  args.N = (int32_t)N;
  args.K = (int32_t)K;
  args.epilogue = (int32_t)epilogue;
  args.w_fp8 = fp8;
  args.a_row_sumsq = (const float*)ptr(a_row_sumsq);
  args.c_row_sumsq = (float*)ptr(c_row_sumsq);
  args.norm_eps = (float)norm_eps;
  args.a_row_sum = (const float*)ptr(a_row_sum);
  args.c_row_sum = (float*)ptr(c_row_sum);
  args.w_col_sum = (const float*)ptr(w_col_sum);
  args.residual_lo = (const uint8_t*)ptr(residual_lo);
  args.c_lo = (uint8_t*)ptr(out_lo);
  args.a_norm_inline = norm_inline;
  set_prefetch(args, get(prefetch_), a.device());
  check_status(cs_gemm(&args, current_stream()), "cs_gemm");
}

Tensor gemm(const Tensor& a, const Tensor& w, const OptTensor& bias, int64_t epilogue, const OptTensor& residual, const OptTensor& w_scale,
            const OptTensor& pos, const OptTensor& a_rows, const OptTensor& c_rows, std::optional<int64_t> k,
            const OptTensor& a_row_sumsq, double norm_eps, const OptTensor& a_row_sum, const OptTensor& w_col_sum, int64_t conv_patch) {
  TORCH_CHECK_VALUE(w.dim() == 2, "gemm operands must be 2-D");
  const int64_t M = gemm_rows(a, get(a_rows), conv_patch);
  Tensor out = at::empty({M, epilogue == CS_EPI_SWIGLU ? w.size(0) / 2 : w.size(0)}, a.options().dtype(at::kBFloat16));
  gemm_(out, a, w, bias, epilogue, residual, w_scale, pos, a_rows, c_rows, k, a_row_sumsq, {}, norm_eps, a_row_sum, {}, w_col_sum, {}, {},
        conv_patch, {}, false);
  return out;
}

void qkv_window_attn_(const Tensor& out, const Tensor& x, const Tensor& w_packed, const Tensor& b_packed, const Tensor& cos_sin,
                      int64_t heads, double scale, const OptTensor& a_row_sumsq_, double norm_eps, const OptTensor& win_start_,
                      const OptTensor& w_scale_, const OptTensor& prefetch, bool norm_inline) {
  const Tensor *a_row_sumsq = get(a_row_sumsq_), *win_start = get(win_start_), *w_scale = get(w_scale_);
  require_rows(x, at::kBFloat16, "x");
  require_rows(w_packed, w_scale ? at::kByte : at::kBFloat16, "w_packed");
  const int64_t M = x.size(0), K = x.size(1), d = WATTN_HEAD_DIM, w_rows = heads * WATTN_TILE_ROWS;
  if (w_scale) {
    require(*w_scale, at::kFloat, "w_scale");
    TORCH_CHECK_VALUE(is_vector(*w_scale, w_rows), "w_scale must be a contiguous fp32 [", w_rows, "] tensor");
    TORCH_CHECK_VALUE(!a_row_sumsq, "the folded norm (a_row_sumsq) does not exist for fp8 weights");
  }
  require_rows(out, at::kBFloat16, "out");
  require(b_packed, at::kBFloat16, "b_packed");
  require(cos_sin, at::kFloat, "cos_sin");
  TORCH_CHECK_VALUE(heads >= 1 && w_packed.size(0) == w_rows && w_packed.size(1) == K, "w_packed must be [", heads, "*", WATTN_TILE_ROWS,
                    ", ", K, "], got ", py(w_packed.sizes()));
  TORCH_CHECK_VALUE(is_vector(b_packed, w_rows), "b_packed must be a contiguous [", w_rows, "] tensor");
  CsGemmArgs args = {};
  if (!win_start) {
    TORCH_CHECK_VALUE(M % WATTN_WINDOW == 0, "the rows of x (", M, ") must be a whole number of ", WATTN_WINDOW, "-row windows");
  } else {
    require(*win_start, at::kInt, "win_start");
    const int64_t n_win = win_start->numel() - 1;
    TORCH_CHECK_VALUE(win_start->dim() == 1 && win_start->is_contiguous() && n_win >= 1 && 4 * n_win <= M &&
                          M <= WATTN_WINDOW * n_win && M % 4 == 0,
                      "win_start must be a contiguous int32 [windows + 1] tensor whose windows of 4 .. ", WATTN_WINDOW,
                      " rows add up to the ", M, " rows of x");
    args.attn_win_start = (const int32_t*)win_start->data_ptr();
    args.attn_n_win = (int32_t)n_win;
  }
  TORCH_CHECK_VALUE(cos_sin.dim() == 2 && cos_sin.size(0) == M && cos_sin.size(1) == d && cos_sin.is_contiguous(),
                    "cos_sin must be a contiguous fp32 [", M, ", ", d, "] table");
  TORCH_CHECK_VALUE(out.size(0) >= M && out.size(1) >= heads * d, "out must be bf16 [>=", M, ", >=", heads * d, "], got ", py(out.sizes()));
  require_sums(a_row_sumsq, M, "a_row_sumsq");
  one_device({&x, &out, &w_packed, &b_packed, &cos_sin, a_row_sumsq, win_start, w_scale}, "qkv_window_attn");
  args.A = x.data_ptr();
  args.lda = x.stride(0);
  args.W = w_packed.data_ptr();
  args.ldw = w_packed.stride(0);
  args.bias = b_packed.data_ptr();
  args.C = out.data_ptr();
  args.ldc = out.stride(0);
  args.M = (int32_t)M;
  args.N = (int32_t)w_rows;
  args.K = (int32_t)K;
  args.a_row_sumsq = (const float*)ptr(a_row_sumsq);
  args.norm_eps = (float)norm_eps;
  args.a_norm_inline = norm_inline;
  if (w_scale) {
    args.w_fp8 = 1;
    args.w_scale = (const float*)w_scale->data_ptr();
  }
  set_prefetch(args, get(prefetch), x.device());
  // (a workspace of the allocator's: its memory is handed on in the order of the current stream)
  const int64_t windows = win_start ? win_start->numel() - 1 : M / WATTN_WINDOW;
  const int32_t need = cs_qkv_window_attn_workspace((int32_t)M, (int32_t)windows, (int32_t)heads, (int32_t)K, w_scale ? 1 : 0);
  const Tensor workspace = need ? at::empty({need}, x.options().dtype(at::kByte)) : Tensor();
  check_status(cs_qkv_window_attn_ws(&args, (const float*)cos_sin.data_ptr(), (float)scale, (int32_t)heads, (int32_t)d,
                                     need ? workspace.data_ptr() : nullptr, need, current_stream()),
               "cs_qkv_window_attn");
}

void attn_varlen_(const Tensor& out, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& work, int64_t n_work,
                  int64_t max_seqlen, int64_t heads, int64_t head_dim, double scale, const OptTensor& cos_sin_, bool keys_rotated) {
  const Tensor* cos_sin = get(cos_sin_);
  const std::pair<const char*, const Tensor*> operands[] = {{"q", &q}, {"k", &k}, {"v", &v}, {"out", &out}};
  for (const auto& [name, t] : operands) {
    require_rows(*t, at::kBFloat16, name);
    TORCH_CHECK_VALUE(t->size(1) >= heads * head_dim && t->device() == q.device(), name, " must hold ", heads, " heads of ", head_dim,
                      " values per row on q's device");
  }
  TORCH_CHECK_VALUE(q.stride(0) == k.stride(0) && k.stride(0) == v.stride(0), "q, k, v must share a row stride");
  const int64_t L = q.size(0);
  TORCH_CHECK_VALUE(k.size(0) == L && v.size(0) == L && out.size(0) >= L, "q, k, v and out must have one row per token");
  require(work, at::kInt, "work");
  TORCH_CHECK_VALUE(work.dim() == 2 && work.size(1) == 4 && work.is_contiguous() && work.size(0) >= n_work && work.device() == q.device(),
                    "work must be a contiguous int32 [>=n_work, 4] tensor on q's device");
  if (cos_sin) {
    require(*cos_sin, at::kFloat, "cos_sin");
    TORCH_CHECK_VALUE(cos_sin->dim() == 2 && cos_sin->size(0) == L && cos_sin->size(1) == head_dim && cos_sin->is_contiguous() &&
                          cos_sin->device() == q.device(),
                      "cos_sin must be contiguous [L, head_dim] on q's device");
  }
  auto* const entry = keys_rotated ? cs_attn_varlen_keys_rotated : cs_attn_varlen;
  check_status(entry(q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(0), out.data_ptr(), out.stride(0), (const int32_t*)work.data_ptr(),
                     (int32_t)n_work, (int32_t)heads, (int32_t)head_dim, (float)scale, (const float*)ptr(cos_sin), (int32_t)max_seqlen,
                     current_stream()),
               keys_rotated ? "cs_attn_varlen_keys_rotated" : "cs_attn_varlen");
}

void rope_qk_(const Tensor& qkv, const Tensor& cos_sin, int64_t heads, int64_t head_dim) {
  require_rows(qkv, at::kBFloat16, "qkv");
  require(cos_sin, at::kFloat, "cos_sin");
  TORCH_CHECK_VALUE(cos_sin.dim() == 2 && cos_sin.size(0) == qkv.size(0) && cos_sin.size(1) == head_dim && cos_sin.is_contiguous() &&
                        cos_sin.device() == qkv.device(),
                    "cos_sin must be contiguous [L, head_dim] on qkv's device");
  TORCH_CHECK_VALUE(heads >= 1 && qkv.size(1) >= 2 * heads * head_dim, "qkv rows hold ", qkv.size(1),
                    " values, fewer than the q and k blocks of ", heads, " heads");
  check_status(cs_rope_qk(qkv.data_ptr(), qkv.stride(0), (const float*)cos_sin.data_ptr(), (int32_t)qkv.size(0), (int32_t)heads,
                          (int32_t)head_dim, current_stream()),
               "cs_rope_qk");
}

void norm_args(const Tensor& out, const Tensor& x, const Tensor& w, const Tensor* b) {
  require_rows(x, at::kBFloat16, "x");
  require_rows(out, at::kBFloat16, "out");
  const int64_t H = x.size(1);
  TORCH_CHECK_VALUE(out.size(0) >= x.size(0) && out.size(1) >= H && out.device() == x.device(), "out must be bf16 [>=", x.size(0), ", >=", H,
                    "] on x's device");
  const std::pair<const char*, const Tensor*> vectors[] = {{"w", &w}, {"b", b}};
  for (const auto& [name, t] : vectors) {
    if (!t) continue;
    require(*t, at::kBFloat16, name);
    TORCH_CHECK_VALUE(t->dim() == 1 && t->size(0) >= H && t->device() == x.device(), name, " must be bf16 [", H, "] on x's device");
  }
}

void rmsnorm_(const Tensor& out, const Tensor& x, const Tensor& w, double eps, bool gemma) {
  norm_args(out, x, w, nullptr);
  check_status(cs_rmsnorm(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), out.stride(0), (int32_t)x.size(0), (int32_t)x.size(1),
                          (float)eps, gemma, current_stream()),
               "cs_rmsnorm");
}

void layernorm_(const Tensor& out, const Tensor& x, const Tensor& w, const Tensor& b, double eps) {
  norm_args(out, x, w, &b);
  check_status(cs_layernorm(x.data_ptr(), x.stride(0), w.data_ptr(), b.data_ptr(), out.data_ptr(), out.stride(0), (int32_t)x.size(0),
                            (int32_t)x.size(1), (float)eps, current_stream()),
               "cs_layernorm");
}

}  // namespace

// The layout of CsGemmArgs is compiled in here as well as in the kernel library: lib.py compares the versions before it has
// the operators registered.
extern "C" int cs_torch_ops_abi_version(void) { return CS_ABI_VERSION; }

// Registers the implementations, once.  (For every backend key, as the operators that cornserve_amd/ops.py implements: the
// checks above turn host tensors away.)  While nothing was built yet, ops.py has put implementations in their place that
// come here at their first call; the dispatcher's remark that these are now overridden is no news.
extern "C" void cs_torch_ops_register(void) {
  struct : c10::WarningHandler {
    void process(const c10::Warning&) override {}
  } quiet;
  c10::WarningUtils::WarningHandlerGuard guard(&quiet);
  static torch::Library* const library = [] {
    auto* m = new torch::Library(torch::Library::IMPL, "cornserve_amd", c10::DispatchKey::CompositeExplicitAutograd, __FILE__, __LINE__);
    m->impl("gemm", gemm);
    m->impl("gemm_", gemm_);
    m->impl("qkv_window_attn_", qkv_window_attn_);
    m->impl("attn_varlen_", attn_varlen_);
    m->impl("rope_qk_", rope_qk_);
    m->impl("rmsnorm_", rmsnorm_);
    m->impl("layernorm_", layernorm_);
    return m;
  }();
  (void)library;   // (for the life of the process)
}
