// The 64x160 tile form (4x2 waves) of the few-row GEMM: like the 32x160 form (gemm_small_t32x160.hip) for more rows.
#include "gemm_small_impl.h"

int cs_gemm_small_tile_64x160(const CsGemmArgs& a, hipStream_t stream) {
  if (a.w_fp8 || a.epilogue != CS_EPI_RESIDUAL || !a.c_lo || !a.c_row_sumsq) return CS_ERR_UNSUPPORTED;
  return a.c_row_sum ? launch_small<64, 160, 4, 2, 1, 4, CS_EPI_RESIDUAL, false, NORM_NONE, true, SUMS_BOTH>(a, stream)
                     : launch_small<64, 160, 4, 2, 1, 4, CS_EPI_RESIDUAL, false, NORM_NONE, true, SUMS_SQ>(a, stream);
}
