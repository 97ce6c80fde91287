// The 32x160 tile form (2x2 waves) of the few-row GEMM: the residual GEMM that also emits its output's row sums in parts
// of 160 columns (split residual stream, bf16 weights); see gemm_small_impl.h.
#include "gemm_small_impl.h"

int cs_gemm_small_tile_32x160(const CsGemmArgs& a, hipStream_t stream) {
  if (a.w_fp8 || a.epilogue != CS_EPI_RESIDUAL || !a.c_lo || !a.c_row_sumsq) return CS_ERR_UNSUPPORTED;
  return a.c_row_sum ? launch_small<32, 160, 2, 2, 2, 3, CS_EPI_RESIDUAL, false, NORM_NONE, true, SUMS_BOTH>(a, stream)
                     : launch_small<32, 160, 2, 2, 2, 3, CS_EPI_RESIDUAL, false, NORM_NONE, true, SUMS_SQ>(a, stream);
}
