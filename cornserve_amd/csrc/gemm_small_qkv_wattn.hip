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

namespace {

// Rotary and attention of one window and one head from the projection's fp32 values, the lanes' fragments laid out as in
// small_wattn_epilogue.  Bound by latency: 61 KB in one round of loads, a barrier, short chains of MFMAs (5.6 us).
__global__ __launch_bounds__(256) void window_attn_f32_kernel(const CsGemmArgs p, const float* __restrict__ x, int64_t ldx, int windows) {
  constexpr int HD = 80, HALF = 40, VT_ROW = 144;
  __shared__ __attribute__((aligned(16))) char vt[HD * VT_ROW];
  __shared__ __attribute__((aligned(16))) char ks[4 * 2560];
  const int ntiles = windows * (p.N / 256);
  if ((int)blockIdx.x >= ntiles) {
    read_hint<256>(p, ntiles);
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, kq = lane >> 4;
  const int win = blockIdx.x % windows, n0 = blockIdx.x / windows * 256;
  int m0 = win * 64, cnt = 64;
  if (p.attn_win_start) {
    m0 = p.attn_win_start[win];
    cnt = min(max(p.attn_win_start[win + 1] - m0, 1), 64);
  }
  const int row = m0 + min(16 * wave + lr, cnt - 1);   // (a short window's last row stands for the missing ones)
  const float* const src = x + (int64_t)row * ldx + n0 + 8 * kq;
  f32x4_t f[15];
#pragma unroll
  for (int J = 0; J < 15; ++J) f[J] = *(const f32x4_t*)(src + (J / 2) * 32 + (J % 2) * 4);
  const float* const cs = p.attn_cos_sin + (int64_t)row * HD + 10 * kq;
  float co[10], si[10];
#pragma unroll
  for (int t = 0; t < 10; t += 2) {
    const f32x2_t c2 = *(const f32x2_t*)(cs + t), s2 = *(const f32x2_t*)(cs + HALF + t);
    co[t] = c2[0];
    co[t + 1] = c2[1];
    si[t] = s2[0];
    si[t + 1] = s2[1];
  }
#pragma unroll
  for (int d = 0; d < 5; ++d) {
#pragma unroll
    for (int r = 0; r < 4; ++r) *(bf16_t*)(vt + (16 * d + 4 * kq + r) * VT_ROW + (16 * wave + lr) * 2) = f2bf(f[10 + d][r]);
  }
  window_attention(p, vt, ks, [&](int J) { return f[J]; }, co, si, m0, n0, cnt, wave, lane);
}

template <int NORM>
int launch_projection(const CsGemmArgs& p, int bm, int bn, hipStream_t stream) {
  if (bm == 32) return launch_small<32, 64, 2, 2, 2, 6, SM_EPI_QKV_F32, false, NORM, false>(p, stream);
  if (bn == 64) return launch_small<64, 64, 4, 2, 2, 4, SM_EPI_QKV_F32, false, NORM, false>(p, stream);
  return launch_small<64, 128, 4, 2, 2, 3, SM_EPI_QKV_F32, false, NORM, false>(p, stream);
}
// ... and of the hint that it has, the bytes that this launch leaves
int64_t projection_leaves(int64_t hint, int tiles, int bm, int bn) {
  if (bm == 32) return hint_left_of<SmallShape<32, 64, 2, 6, false, NORM_NONE, SUMS_NONE>, 4>(hint, tiles);
  if (bn == 64) return hint_left_of<SmallShape<64, 64, 2, 4, false, NORM_NONE, SUMS_NONE>, 8>(hint, tiles);
  return hint_left_of<SmallShape<64, 128, 2, 3, false, NORM_NONE, SUMS_NONE>, 8>(hint, tiles);
}

}  // namespace

// The same in two launches over a workspace of rows x a.N floats.  With one workgroup per window and head a launch lasts 23 to 25
// us however few they are: each of them has 800 KB of operands to take in, and most of the chip is idle.  Here the projection
// runs in few-row tiles, whose columns fill the chip, and the kernel above does the rest; the values between are fp32 (the
// rotary takes unrounded ones) and every one is computed by the same operations, so the bits are the same.  128 rows 24.8 -> 16.0
// us, 256 24.0 -> 18.0; an image of 96 patches through the encoder 1.77 -> 1.49 ms.
int cs_qkv_window_attn_two(const CsGemmArgs& a, int rows, int windows, float* x, hipStream_t stream) {
  CsGemmArgs p = a;
  p.M = rows;
  p.C = x;
  p.ldc = a.N;
  // (the smallest tile that is one round)
  auto tiles_of = [&](int bm, int bn) { return (rows + bm - 1) / bm * (a.N / bn); };
  const int bn = tiles_of(64, 64) <= 256 ? 64 : 128, bm = bn == 64 && tiles_of(32, 64) <= 256 ? 32 : 64;
  csgemm::fit_hint(p, tiles_of(bm, bn), bm == 32 ? 9.0 : 10.0);
  const int status = a.a_norm_inline ? launch_projection<NORM_RMS>(p, bm, bn, stream) : launch_projection<NORM_NONE>(p, bm, bn, stream);
  if (status != CS_OK) return status;
  // (the hint's rest)
  CsGemmArgs q = a;
  if (a.prefetch && p.prefetch) {
    const int64_t done = (p.prefetch_bytes - projection_leaves(p.prefetch_bytes, tiles_of(bm, bn), bm, bn)) & ~(int64_t)15;
    q.prefetch = (const char*)a.prefetch + done;
    q.prefetch_bytes = a.prefetch_bytes - done;
  }
  const int tiles = windows * (a.N / 256);
  csgemm::fit_hint(q, tiles, 8.0);
  hipLaunchKernelGGL(window_attn_f32_kernel, dim3(tiles + (q.prefetch ? csgemm::hint_workgroups(tiles) : 0)), dim3(256), 0, stream, q, x,
                     (int64_t)a.N, windows);
  return cs_launch_status();
}
