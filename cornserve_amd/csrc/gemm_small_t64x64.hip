// The 64x64 tile form (4x2 waves) of the few-row GEMM, with a ring of 4 K stages (see gemm_small_impl.h).
#include "gemm_small_impl.h"

int cs_gemm_small_tile_64x64(const CsGemmArgs& a, hipStream_t stream) { return dispatch_small<64, 64, 4, 2, 2, 4>(a, stream); }
