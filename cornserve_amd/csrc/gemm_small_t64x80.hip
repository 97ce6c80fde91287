// The 64x80 tile form (4x1 waves) of the few-row GEMM: 1024 rows of 1280 columns are exactly 256 workgroups.  Plain and
// residual epilogues (what an encoder has at that width), bf16 weights; see gemm_small_impl.h.
#include "gemm_small_impl.h"

int cs_gemm_small_tile_64x80(const CsGemmArgs& a, hipStream_t stream) {
  if (a.w_fp8 || a.a_norm_inline || a.pos) return CS_ERR_UNSUPPORTED;
  if (a.epilogue == CS_EPI_BIAS) return launch_small<64, 80, 4, 1, 2, 4, CS_EPI_BIAS, false, NORM_NONE, false>(a, stream);
  if (a.epilogue == CS_EPI_RESIDUAL && a.c_lo) return launch_small<64, 80, 4, 1, 2, 4, CS_EPI_RESIDUAL, false, NORM_NONE, true>(a, stream);
  return CS_ERR_UNSUPPORTED;
}
