// QKV projection with rotary and window attention as its epilogue: the 256x256 tile with one window of up to 64 rows per
// wavefront (waves 4 x 1) and one head per column tile.  The kernel is gemm_fast_kernel (gemm_fast_impl.h).  The
// accumulators live in accumulation registers that only inline assembly touches (CS_ALL_ACC_REGS: the build checks this
// file's compiler output for stray uses of them).
#include "gemm_fast_impl.h"

int cs_qkv_window_attn_small(const CsGemmArgs& a, int rows, hipStream_t stream);
// Whether a launch of `windows` windows takes that form (gemm_small.hip).
bool cs_qkv_window_attn_few(int64_t windows, int heads, int K);
// The two-launch form, and whether it is the faster one.
int cs_qkv_window_attn_two(const CsGemmArgs& a, int rows, int windows, float* x, hipStream_t stream);
bool cs_qkv_window_attn_two_pays(int64_t rows, int64_t windows, int heads, int K, bool w_fp8);

namespace {

int big_tiles(CsGemmArgs a, bool ragged, hipStream_t stream) {
  if (ragged) {
    a.M = a.attn_n_win * 64;   // virtual rows: one 64-row slot per window
    if (a.w_fp8) return launch<256, 256, 4, 1, CS_EPI_QKV_WATTN_RAGGED, true, 0>(a, stream);
    if (a.a_row_sumsq) return launch<256, 256, 4, 1, CS_EPI_QKV_WATTN_RAGGED, false, FUSE_NORM_A>(a, stream);
    return launch<256, 256, 4, 1, CS_EPI_QKV_WATTN_RAGGED, false, 0>(a, stream);
  }
  if (a.w_fp8) return launch<256, 256, 4, 1, CS_EPI_QKV_WATTN, true, 0>(a, stream);
  if (a.a_row_sumsq) return launch<256, 256, 4, 1, CS_EPI_QKV_WATTN, false, FUSE_NORM_A>(a, stream);
  return launch<256, 256, 4, 1, CS_EPI_QKV_WATTN, false, 0>(a, stream);
}

// Windows behind the last whole round of big tiles (256 workgroups of four windows and a head) cost a round of their own; few enough
// for a workgroup per window and head go to a second launch, which finds the weights in the caches.  Weights from HBM, K = 1280, whole
// rounds | with the windows that are split | with one more, in one launch again.  bf16 and folded norm: 16 heads 64 windows 42 us | 65 to 80
// 56 to 59 | 81 67, 128 76 | 144 94 | 145 104; 32 heads 32 43 | 33 to 40 57 to 60 | 41 69; 10 100 42 | 125 57 | 126 68; 8 128 40 | 160 59 |
// 161 66; 4 256 40 | 320 58 | 321 66; 2 512 40 | 640 57 | 641 66; 3 340 41 | 425 57 | 426 64.  fp8: 16 heads 64 46 | 80 59 | 81 74; 8 128 41 | 160
// 60 | 161 75; 3 340 42 | 425 59 | 426 73; 24 heads, K = 1920, 40 61 | 50 77 | 51 101.  K = 640, 8 heads: 128 25 | 160 39 | 161 43.
// Returns the windows of the first launch, 0 for one launch.
int64_t lead_windows(int64_t windows, int heads, int K) {
  if (cs_qkv_window_attn_few(windows, heads, K)) return 0;
  const int64_t round = 256 / heads * 4, rest = round ? windows % round : 0;
  return rest && rest < windows && cs_qkv_window_attn_few(rest, heads, K) ? windows - rest : 0;
}

}  // namespace

extern "C" int cs_qkv_window_attn_lead_windows(int32_t windows, int32_t heads, int32_t K) {
  return windows < 1 || heads < 1 || K < 1 ? 0 : (int)lead_windows(windows, heads, K);
}

extern "C" int cs_qkv_window_attn_workspace(int32_t rows, int32_t windows, int32_t heads, int32_t K, int32_t w_fp8) {
  if (rows < 1 || windows < 1 || heads < 1 || K < 1 || !cs_qkv_window_attn_two_pays(rows, windows, heads, K, w_fp8 != 0)) return 0;
  return rows * heads * 256 * (int32_t)sizeof(float);   // (at most 8 MB)
}

extern "C" int cs_qkv_window_attn(const CsGemmArgs* gemm, const float* cos_sin, float scale, int32_t heads,
                                  int32_t head_dim, void* stream) {
  return cs_qkv_window_attn_ws(gemm, cos_sin, scale, heads, head_dim, nullptr, 0, stream);
}

extern "C" int cs_qkv_window_attn_ws(const CsGemmArgs* gemm, const float* cos_sin, float scale, int32_t heads, int32_t head_dim,
                                     void* workspace, int64_t workspace_bytes, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!gemm || !cos_sin || heads <= 0) return CS_ERR_INVALID_ARG;
  CsGemmArgs a = *gemm;
  if (!a.A || !a.W || !a.C || !a.bias || a.M < 0 || a.K <= 0) return CS_ERR_INVALID_ARG;
  const bool ragged = a.attn_win_start != nullptr;
  if (ragged ? (a.attn_n_win < 1 || a.M < 4 * a.attn_n_win || a.M > 64 * (int64_t)a.attn_n_win || a.M % 4) : a.attn_n_win != 0)
    return CS_ERR_INVALID_ARG;
  if (head_dim != 80 || a.N != heads * 256 || (!ragged && a.M % 64) || a.K % csgemm::BK || a.K < 3 * csgemm::BK) return CS_ERR_UNSUPPORTED;
  if (a.residual || a.pos || a.a_rows || a.c_rows || a.c_row_sumsq || a.a_row_sum || a.c_row_sum || a.c_lo || a.residual_lo ||
      a.conv_patch)
    return CS_ERR_INVALID_ARG;
  // fp8 weights: e4m3 bytes packed like the bf16 rows, with their per-output-channel scales packed like the bias; no
  // folded norm with them (as for cs_gemm)
  if (a.w_fp8 ? (!a.w_scale || ((uintptr_t)a.w_scale & 15)) : (a.w_scale != nullptr)) return CS_ERR_INVALID_ARG;
  if (a.w_fp8 && a.a_row_sumsq) return CS_ERR_UNSUPPORTED;
  if (a.lda % 8 || a.ldw % (a.w_fp8 ? 16 : 8) || a.ldc % 4 || a.ldc < heads * 80) return CS_ERR_INVALID_ARG;
  if (((uintptr_t)a.A | (uintptr_t)a.W | (uintptr_t)cos_sin | (uintptr_t)a.a_row_sumsq) & 15) return CS_ERR_INVALID_ARG;
  if (((uintptr_t)a.C | (uintptr_t)a.bias) & 7) return CS_ERR_INVALID_ARG;
  if (a.prefetch ? (((uintptr_t)a.prefetch & 15) || a.prefetch_bytes < 0) : a.prefetch_bytes != 0) return CS_ERR_INVALID_ARG;
  // per-lane source offsets of the direct loads are 32-bit byte offsets from the matrix bases
  if ((int64_t)a.M * a.lda * 2 >= (int64_t)UINT32_MAX || (int64_t)a.N * a.ldw * (a.w_fp8 ? 1 : 2) >= (int64_t)UINT32_MAX)
    return CS_ERR_UNSUPPORTED;
  if (workspace && (((uintptr_t)workspace & 15) ||
                    workspace_bytes < cs_qkv_window_attn_workspace(a.M, ragged ? a.attn_n_win : a.M / 64, heads, a.K, a.w_fp8)))
    return CS_ERR_INVALID_ARG;
  if (a.M == 0) return CS_OK;
  a.attn_cos_sin = cos_sin;
  a.attn_scale_log2e = scale * 1.4426950408889634f;
  a.epilogue = CS_EPI_BIAS;
  if (ragged && ((uintptr_t)a.attn_win_start & 3 || (int64_t)a.attn_n_win * 64 > INT32_MAX)) return CS_ERR_INVALID_ARG;
  if (a.a_norm_inline && (a.a_norm_inline != 1 || a.a_row_sumsq || a.w_fp8 || a.w_col_sum)) return CS_ERR_INVALID_ARG;
  if (a.a_norm_inline && !csgemm::inline_norm_width(a.K)) return CS_ERR_UNSUPPORTED;
  // few windows: a workgroup per window and head
  if (cs_qkv_window_attn_few(ragged ? a.attn_n_win : a.M / 64, heads, a.K)) {
    const int rows = a.M, windows = ragged ? a.attn_n_win : a.M / 64;
    const int32_t need = workspace ? cs_qkv_window_attn_workspace(rows, windows, heads, a.K, a.w_fp8) : 0;
    if (ragged) a.M = a.attn_n_win * 64;   // (tiles_m counts windows; the operand ends with its last real row)
    if (need) return cs_qkv_window_attn_two(a, rows, windows, (float*)workspace, stream);
    return cs_qkv_window_attn_small(a, rows, stream);
  }
  if (a.a_norm_inline) return CS_ERR_UNSUPPORTED;
  const int64_t windows = ragged ? a.attn_n_win : a.M / 64, lead = lead_windows(windows, heads, a.K), rest = windows - lead;
  if (lead) {
    CsGemmArgs first = a, second = a;
    first.prefetch = nullptr;
    first.prefetch_bytes = 0;
    if (ragged) {
      first.attn_n_win = (int32_t)lead;
      second.attn_win_start = a.attn_win_start + lead;   // (whose starts are rows of the whole matrix)
      second.attn_n_win = (int32_t)rest;
      second.M = (int32_t)rest * 64;
    } else {
      first.M = (int32_t)lead * 64;
      second.M = (int32_t)rest * 64;
      second.A = (const bf16_t*)a.A + lead * 64 * a.lda;
      second.C = (bf16_t*)a.C + lead * 64 * a.ldc;
      second.attn_cos_sin = a.attn_cos_sin + lead * 64 * head_dim;
      if (a.a_row_sumsq) second.a_row_sumsq = a.a_row_sumsq + lead * 64 * CS_SUMSQ_PARTS;
    }
    const int status = big_tiles(first, ragged, stream);
    return status == CS_OK ? cs_qkv_window_attn_small(second, ragged ? a.M : second.M, stream) : status;
  }
  return big_tiles(a, ragged, stream);
}
