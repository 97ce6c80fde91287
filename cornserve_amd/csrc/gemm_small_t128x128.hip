// The 128x128 tile form (4x2 waves) of the few-row GEMM, with a ring of four stages of one K tile (see gemm_small_impl.h).
#include "gemm_small_impl.h"

int cs_gemm_small_tile_128x128(const CsGemmArgs& a, hipStream_t stream) { return dispatch_small<128, 128, 4, 2, 1, 4>(a, stream); }
