// QKV projection + rotary + window attention for few windows: one workgroup per window and head (64 rows x 240 columns, a
// ring of four K tiles) where the big tile of gemm_fast_qkv_wattn.hip gives four windows to a workgroup.  See
// gemm_small_impl.h.
#include "gemm_small_impl.h"

// a.M = 64 x windows, `rows` the rows that A really has (fewer where windows are short).
int cs_qkv_window_attn_small(const CsGemmArgs& a, int rows, hipStream_t stream) {
  CsGemmArgs p = a;
  p.tiles_m = a.M / 64;
  p.M = rows;
  csgemm::fit_hint(p, p.tiles_m * (a.N / 256), 20.0);
  if (a.w_fp8) return launch_small<64, 240, 1, 4, 1, 4, SM_EPI_QKV_WATTN, true, NORM_NONE, false>(p, stream);
  if (a.a_norm_inline) return launch_small<64, 240, 1, 4, 1, 4, SM_EPI_QKV_WATTN, false, NORM_RMS, false>(p, stream);
  return launch_small<64, 240, 1, 4, 1, 4, SM_EPI_QKV_WATTN, false, NORM_NONE, false>(p, stream);
}
