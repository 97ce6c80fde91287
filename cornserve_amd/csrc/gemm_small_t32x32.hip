// The 32x32 tile form (2x2 waves) of the few-row GEMM, with a ring of 8 K stages (see gemm_small_impl.h).
#include "gemm_small_impl.h"

int cs_gemm_small_tile_32x32(const CsGemmArgs& a, hipStream_t stream) { return dispatch_small<32, 32, 2, 2, 2, 8>(a, stream); }
