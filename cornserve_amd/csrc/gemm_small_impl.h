// bf16 MFMA GEMM for launches of few rows:  C[M,N] = epilogue(A[M,K] . W[N,K]^T),  K % 128 == 0.
//
// With few rows the big tiles of gemm_fast_impl.h leave most of the 256 compute units without work (1280 columns in tiles
// of 160 are 8 workgroups per 128 rows), and the ones that have some walk the whole of K one big K tile after the other.
// This kernel trades operand reuse for parallelism: tiles of 32 to 128 rows by 32 to 160 columns, one workgroup of four
// or eight waves per tile, and as deep a ring of K stages in LDS as fits, so that most of a tile's operands are in
// flight at once.  What bounds it is the LDS: per stage of 128 k it takes in (BM + BN) x 256 bytes and hands out
// waves x (MT + NT) x 4 KB of fragments, and time per stage follows that sum at about 270 KB a microsecond and compute
// unit (128 bytes a clock) in the GEMM's tile forms; the rest of a launch is 4 to 5 us of launch, first loads and epilogue.
// (The window attention form, one wave a SIMD, takes 17 us with weights in the caches, 8 of them launch, first loads and the
// attention; 21 with the inline norm, 23 with its 10 MB of weights from HBM.)
// Measured on an MI355X with weights that no cache holds: 1280 columns, K = 3456: 96 rows 34.3 -> 8.7 us (32x32 tiles),
// 1024 rows 38 -> 20 us (64x80); K = 1280: 96 rows 19 -> 6 us, 1024 rows 19 -> 11 us.  The big tiles are the faster ones from
// about 2000 rows on at K = 1280, from 3100 (128x128 tiles until then) at K = 3456 to 5120: the choice is in gemm_small.hip.
//
// The arithmetic of an output element is the same sequence of operations as in gemm_fast_impl.h (v_mfma_f32_16x16x32_bf16
// over ascending K from a zero accumulator, W as the first operand, the same epilogue functions in the same order), so an
// element's bits do not depend on which of the two kernels a launch selects.
//
// Folded norms.  With CsGemmArgs.a_norm_inline the per-row sums over A that the big tiles read from the producing GEMM's
// arrays are taken from the operand fragments on their way to the matrix cores: every workgroup streams whole rows of A
// anyway.  The fragment of k-step s holds, in lane (row, q), columns 32 s + 8 q .. + 7: the columns that lane q of the
// producing epilogue sums in its s-th pair of pieces.  So the same chain of v_dot2 over five k-steps, and the same sum
// over the four lanes of a row, give the bits of the producer's 160-column parts.  The 160-column form also produces them
// (CsGemmArgs.c_row_sumsq): two waves share a row, the second continues the first one's chain through LDS.
#pragma once

#include <type_traits>
#include <utility>

#include "gemm_common.h"
#include "hint_ring.h"

namespace {

using namespace csgemm;

constexpr int SM_EPI_BIAS_POS = 100;  // internal: CS_EPI_BIAS plus the (row % pos_period) position addend
constexpr int SM_EPI_QKV_WATTN = 101; // internal: QKV projection + rotary + window attention of one head and one window
constexpr int SM_EPI_QKV_F32 = 103;   // internal: the QKV projection of such a launch alone, fp32 output (see gemm_small_qkv_wattn.hip)
enum { NORM_NONE = 0, NORM_RMS = 1, NORM_LN = 2 };   // inline norm of A's rows
enum { SUMS_NONE = 0, SUMS_SQ = 1, SUMS_BOTH = 2 };  // row sums of the output

typedef __attribute__((address_space(3))) void sm_lds_void_t;

// (Plain functions around device-only builtins: inside a generic lambda the host pass would reject them.)
CS_DEVICE float sm_dot2(uint32_t a, uint32_t b, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), acc, false);
}
CS_DEVICE f32x4_t sm_mfma(bf16x8_t w, bf16x8_t x, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, c, 0, 0, 0); }
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short sm_short4_t;
CS_DEVICE f32x4_t sm_mfma16(bf16x4_t w, bf16x4_t x, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(sm_short4_t, w), __builtin_bit_cast(sm_short4_t, x), c, 0, 0, 0);
}
constexpr uint32_t SM_ONE_PAIR = 0x3F803F80u;   // {1.0, 1.0}

// Wait until at most N of this wave's vector memory operations are outstanding and its LDS reads have returned, then
// meet the other waves.  (s_waitcnt encoding of gfx9: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8.)
template <int N>
CS_DEVICE void sm_wait_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(((N & 0xF) | ((N >> 4) << 14)) | 0x0070);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// The same for a wave-uniform number of stages of NLD loads each, 0 .. sizeof...(I) - 1
template <int NLD, int... I>
CS_DEVICE void small_wait(int stages, std::integer_sequence<int, I...>) {
  ((stages == I ? sm_wait_barrier<I * NLD>() : void()), ...);
}
// f(<0>), f(<1>), ...
template <class F, int... I>
CS_DEVICE void small_for(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// Schedule of a steady (half) iteration: LDS reads and direct loads go between the MFMAs, which do not depend on them.  The
// loads must not come in a burst: the waves of a workgroup leave the barrier together, a load occupies the memory pipeline
// for 16 clocks, and MFMAs behind ten loads of every wave in program order would start only when those have been issued
// (the reads of a half come first: the next half waits for them).
template <int MASK, int N>
CS_DEVICE void sched_group() {
#ifdef __HIP_DEVICE_COMPILE__
  if constexpr (N > 0) __builtin_amdgcn_sched_group_barrier(MASK, N, 0);
#endif
}
// N instructions of kind MASK spread over the slots 0 .. sizeof...(I) - 1, an MFMA before each slot
template <int MASK, int N, int... I>
CS_DEVICE void sched_spread(std::integer_sequence<int, I...>) {
  constexpr int SLOTS = sizeof...(I);
  ((sched_group<0x008, 1>(), sched_group<MASK, (I + 1) * N / SLOTS - I * N / SLOTS>()), ...);
}
template <int READS, int LOADS, int MFMAS>
CS_DEVICE void small_schedule() {
  // the LDS reads over the first MFMAs (one each, if there are enough of them), then the loads over the others
  constexpr int FIRST = MFMAS / 2 < READS ? (MFMAS + 1) / 2 : READS;
  sched_spread<0x100, READS>(std::make_integer_sequence<int, FIRST>{});
  if constexpr (MFMAS > FIRST) sched_spread<0x010, LOADS>(std::make_integer_sequence<int, MFMAS - FIRST>{});
#ifdef __HIP_DEVICE_COMPILE__
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// Row sums of A in LDS, [part][row][lane q]; the parts of a row are added in the order of gemm_fast_impl.h.
CS_DEVICE float sm_total_of_parts(const float* base, int rows, int row, int parts) {
  float v[CS_SUMSQ_PARTS];
#pragma unroll
  for (int q = 0; q < CS_SUMSQ_PARTS; ++q) {
    const f32x4_t s = *(const f32x4_t*)(base + (min(q, parts - 1) * rows + row) * 4);
    v[q] = q < parts ? (s[0] + s[1]) + (s[2] + s[3]) : 0.f;
  }
  return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
}

// A workgroup past the `ntiles` computing ones: reads its share of the hinted bytes, 16 per lane and four loads in flight, and
// is done.  (The big tiles' kernel spells the same loop out: called from there, it moves that kernel's register allocation.)
template <int THREADS>
CS_DEVICE void read_hint(const CsGemmArgs& p, int ntiles) {
  const int pw = (int)blockIdx.x - ntiles, npw = (int)gridDim.x - ntiles;
  const char* const base = (const char*)p.prefetch;
  const int64_t n16 = p.prefetch_bytes >> 4, stride = (int64_t)npw * THREADS;
  u32x4_t sink = {0u, 0u, 0u, 0u};
  for (int64_t i = (int64_t)pw * THREADS + threadIdx.x; i < n16; i += 4 * stride) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t j = i + u * stride;
      if (j < n16) {
        const u32x4_t v = *(const u32x4_t*)(base + 16 * j);
        sink[0] |= v[0] & v[1] & v[2] & v[3];
      }
    }
  }
  // (a store that never happens -- M is positive -- keeps the loads alive)
  if (sink[0] == 0xFFFFFFFFu && p.M < 0) *(volatile uint32_t*)p.C = sink[0];
}

// KS: K tiles of 64 per stage of the ring.
template <int BM, int BN, int KS, int STAGES, bool W_FP8, int NORM, int SUMS>
struct SmallShape {
  static constexpr int W_ROW = W_FP8 ? 64 : 128;                       // bytes per tile row and K tile of 64
  static constexpr int A_SUB = BM * 128, W_SUB = BN * W_ROW;           // one K tile of each operand
  static constexpr int STAGE = KS * (A_SUB + W_SUB);
  static constexpr int NORM_BYTES = NORM == NORM_NONE ? 0 : BM * CS_SUMSQ_PARTS * 16 * (NORM == NORM_LN ? 2 : 1);
  static constexpr int SUMS_BYTES = SUMS == SUMS_NONE ? 0 : BM * 16 * SUMS;
  static constexpr int LDS = STAGES * STAGE + NORM_BYTES + SUMS_BYTES;
  static_assert(LDS <= 160 * 1024, "the ring fits the LDS");
  static constexpr int NLD_OF(int waves) { return KS * (BM / 8) / waves + (KS * (BN * W_ROW / 1024) + waves - 1) / waves; }   // direct loads per wave and stage
  // A prefetch hint behind the last stage (see hint_rows_of): rows of one segment, as wide as a stage's step, per stage
  // (not in 128x128 tiles, with their launches of 20 us and more: the branch to it costs 0.8 % of them)
  static constexpr bool RING_HINT = !W_FP8 && BM * BN < 128 * 128;
  static constexpr int HINT_SEG = cshint::small_segment(KS), HINT_PITCH = cshint::small_segments(KS, STAGES) * HINT_SEG;
};

// What follows the projection in a window (see small_wattn_epilogue), 16 queries a wave: `qk(f)` is fragment f (0 .. 4 q, 5 .. 9
// k) of the window's row 16 wave + lane % 16, `vt` holds the transposed values, `ks` takes the keys (both the workgroup's).
template <class Fragment>
CS_DEVICE void window_attention(const CsGemmArgs& p, const char* vt, char* ks, Fragment qk, const float (&co)[10], const float (&si)[10],
                                int m0, int n0, int cnt, int wave, int lane) {
  constexpr int HD = 80, VT_ROW = 144;
  const int lr = lane & 15, kq = lane >> 4;
  // ---- rotary of this wave's q and k rows; the keys go back to LDS as operand fragments
  bf16x8_t q8[2];
  bf16x4_t q4;
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    float x[20], o[20];
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      const f32x4_t v = qk(which * 5 + f);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[4 * f + r] = v[r];
    }
#pragma unroll
    for (int t = 0; t < 10; ++t) {
      o[t] = __builtin_fmaf(x[t], co[t], -(x[t + 10] * si[t]));
      o[t + 10] = __builtin_fmaf(x[t + 10], co[t], x[t] * si[t]);
    }
    bf16x8_t f0, f1;
    bf16x4_t f2;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      f0[e] = f2bf(o[e]);
      f1[e] = f2bf(o[8 + e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) f2[e] = f2bf(o[16 + e]);
    if (which == 0) {
      q8[0] = f0;
      q8[1] = f1;
      q4 = f2;
    } else {
      char* const dst = ks + wave * 2560;
      *(bf16x8_t*)(dst + lane * 16) = f0;
      *(bf16x8_t*)(dst + 1024 + lane * 16) = f1;
      *(bf16x4_t*)(dst + 2048 + lane * 8) = f2;
    }
  }
  __syncthreads();
  // ---- S^T[key][query] = K.Q^T for this wave's 16 queries, softmax over the 64 keys (16 per lane, 4 lanes per query)
  const float sl2 = p.attn_scale_log2e;
  f32x4_t st[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const char* const src = ks + kb * 2560;
    st[kb] = sm_mfma(*(const bf16x8_t*)(src + lane * 16), q8[0], f32x4_t{0.f, 0.f, 0.f, 0.f});
    st[kb] = sm_mfma(*(const bf16x8_t*)(src + 1024 + lane * 16), q8[1], st[kb]);
    st[kb] = sm_mfma16(*(const bf16x4_t*)(src + 2048 + lane * 8), q4, st[kb]);
  }
  float sv[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) sv[e] = 16 * (e / 4) + 4 * kq < cnt ? st[e / 4][e % 4] : -__builtin_inff();
  float mx = sv[0];
#pragma unroll
  for (int e = 1; e < 16; ++e) mx = fmaxf(mx, sv[e]);
  mx = fmaxf(mx, __shfl_xor(mx, 16));
  mx = fmaxf(mx, __shfl_xor(mx, 32));
  const float mb = mx * sl2;
  bf16x8_t pf[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) pf[e >> 3][e & 7] = f2bf(__builtin_amdgcn_exp2f(sv[e] * sl2 - mb));
  // ---- O^T[dim][query] = V^T.P^T, the softmax denominators from the matrix cores as well (a row block of ones)
  f32x4_t ot[5], den = {0.f, 0.f, 0.f, 0.f};
  bf16x8_t ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = f2bf(1.0f);
#pragma unroll
  for (int d = 0; d < 5; ++d) ot[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int d = 0; d < 5; ++d) {
      const char* const src = vt + (16 * d + lr) * VT_ROW + (32 * t + 4 * kq) * 2;
      const u32x2_t lo = *(const u32x2_t*)src, hi = *(const u32x2_t*)(src + 32);
      ot[d] = sm_mfma(__builtin_bit_cast(bf16x8_t, u32x4_t{lo[0], lo[1], hi[0], hi[1]}), pf[t], ot[d]);
    }
    den = sm_mfma(ones, pf[t], den);
  }
  const float inv = 1.0f / den[0];
  const int row = 16 * wave + lr;
  if (row < cnt) {
    bf16_t* const out = (bf16_t*)p.C + (int64_t)(m0 + row) * p.ldc + (n0 / 256) * HD + 4 * kq;
#pragma unroll
    for (int d = 0; d < 5; ++d) {
      bf16x4_t o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = f2bf(ot[d][r] * inv);
      *(bf16x4_t*)(out + 16 * d) = o;
    }
  }
}

// QKV projection + rotary + window attention: the epilogue of a tile of one window (64 rows, `cnt` of them real) and one
// head (15 fragments: q 0..4, k 5..9, v 10..14; see cs_qkv_window_attn for the packed row order).  In the main loop wave w
// has computed fragments 4w .. 4w+3 of all rows; from here on wave w owns the window's rows 16w .. 16w+15 as queries.
// What changes hands goes through LDS (the ring is free by now): q and k in fp32 with norm and bias applied (a rotary
// pair's halves sit in different fragments), v rounded and transposed, then the rotated keys.  Every operation on a value
// is the one of the big tile's epilogue (gemm_fast_impl.h), in its order.
template <int MT, int NT, bool W_FP8>
CS_DEVICE void small_wattn_epilogue(const CsGemmArgs& p, char* smem, const f32x4_t (&acc)[MT][NT], const float (&rstd)[MT], const u32x2_t (&bias_w)[NT],
                                    const float (&co)[10], const float (&si)[10], int m0, int n0, int cnt, int wave, int lane) {
  static_assert(MT == 4 && NT == 4, "all four row blocks, four fragments per wave");
  constexpr int HD = 80, X_BYTES = 4 * 10 * 1024, VT_ROW = 144, VT_BYTES = HD * VT_ROW;
  const int lr = lane & 15, kq = lane >> 4;
  char* const xs = smem;                              // [row block][fragment 0..9][lane]: 4 fp32
  char* const vt = smem + X_BYTES;                    // [head dim][key]: bf16, 144-byte rows
  char* const ks = smem + X_BYTES + VT_BYTES;         // [row block][part 0, 1: 16 bytes, part 2: 8 bytes][lane]
  __syncthreads();   // (nobody reads operands from the ring any more)
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int J = 4 * wave + j;
    if (J >= 15) break;
    const int ch = n0 + (J / 2) * 32 + 8 * kq + (J % 2) * 4;
    const bf16x4_t bias_b = __builtin_bit_cast(bf16x4_t, bias_w[j]);
    f32x4_t wsc = {1.f, 1.f, 1.f, 1.f};
    if constexpr (W_FP8) wsc = *(const f32x4_t*)(p.w_scale + ch);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      f32x4_t x;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[r] = __builtin_fmaf(acc[i][j][r], W_FP8 ? wsc[r] : rstd[i], bf2f(bias_b[r]));   // (no folded norm with fp8 weights)
      }
      if (J < 10) {
        *(f32x4_t*)(xs + ((i * 10 + J) * 64 + lane) * 16) = x;
      } else {   // head dims 16 (J - 10) + 4 kq + r of key 16 i + lr
#pragma unroll
        for (int r = 0; r < 4; ++r) *(bf16_t*)(vt + (16 * (J - 10) + 4 * kq + r) * VT_ROW + (16 * i + lr) * 2) = f2bf(x[r]);
      }
    }
  }
  __syncthreads();
  window_attention(p, vt, ks, [&](int f) { return *(const f32x4_t*)(xs + ((wave * 10 + f) * 64 + lane) * 16); }, co, si, m0, n0, cnt, wave, lane);
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int KS, int STAGES, int EPI, bool W_FP8, int NORM, bool SPLIT, int SUMS>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, EPI == SM_EPI_QKV_WATTN ? 1 : 2) void gemm_small_kernel(const CsGemmArgs p, const int hint_rows) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  using Shape = SmallShape<BM, BN, KS, STAGES, W_FP8, NORM, SUMS>;
  constexpr bool WATTN = EPI == SM_EPI_QKV_WATTN;
  constexpr int NWAVES = WAVES_M * WAVES_N;
  constexpr int W_ROW = Shape::W_ROW, A_SUB = Shape::A_SUB, W_SUB = Shape::W_SUB, STAGE = Shape::STAGE;
  constexpr int FRAGS_N = BN / 16;   // W fragments of the tile; the last wave repeats the last one where they do not divide
  constexpr int WTM = BM / WAVES_M, MT = WTM / 16, NT = (FRAGS_N + WAVES_N - 1) / WAVES_N, WTN = 16 * NT;
  constexpr bool WHOLE = FRAGS_N % WAVES_N == 0;
  static_assert(WHOLE || (WATTN && FRAGS_N == NT * WAVES_N - 1), "at most the last fragment is missing");
  constexpr int A_BLK = BM / 8, W_BLK = BN * W_ROW / 1024;               // direct loads (1 KB) per K tile
  constexpr int A_LD = KS * A_BLK / NWAVES, W_LD = (KS * W_BLK + NWAVES - 1) / NWAVES;  // ... per wave and stage
  constexpr int NLD = A_LD + W_LD;
  // (every wave issues the same number of loads, because the waits count them: a wave without a block of W left repeats the
  // last one, the same bytes to the same place)
  static_assert(KS * A_BLK % NWAVES == 0, "every wave issues the same number of direct loads");
  static_assert((STAGES - 1) * NLD < 64, "the waits count outstanding loads in six bits");
  static_assert(SUMS == SUMS_NONE || (BN == 160 && WAVES_N == 2 && EPI == CS_EPI_RESIDUAL && SPLIT), "a part of the row sums is 160 columns");
  // Columns of fragment J of the tile: with an even number of fragments they come in pairs of 32 columns, of which lane q
  // holds 8 consecutive ones (4 in each fragment): the order in which the big tiles' epilogue holds and sums them.
  constexpr bool PAIRED = BN % 32 == 0 || WATTN;
  auto frag_col = [](int J, int q) { return PAIRED ? (J / 2) * 32 + 8 * q + (J % 2) * 4 : 16 * J + 4 * q; };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WAVES_M, wn = wave / WAVES_M;
  const int fa = lane & 15, kq = lane >> 4;

  // Workgroups past the computing ones read a prefetch hint (see fit_hint): no tile, no barriers.  Their code lies behind the
  // kernel's, and the arguments that the others start with are asked for ahead of the branch: a launch of 6 to 10 us feels one
  // more line of instructions or a second round of argument loads (with both, passes of 16 to 144 patches took 3 to 8 % longer).
  const int ntiles = p.tiles_m * p.tiles_n;
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" ::"s"(p.A), "s"(p.lda), "s"(p.W), "s"(p.ldw), "s"(p.bias), "s"(p.residual), "s"(p.c_rows), "s"(p.M), "s"(p.N), "s"(p.K));
#endif
  if (__builtin_expect((int)blockIdx.x >= ntiles, 0)) {
    read_hint<64 * NWAVES>(p, ntiles);
    return;
  }

  // Tile of this workgroup: every XCD gets a contiguous run of tiles, bands of 8 tile rows walked column by column.
  int m0, n0;
  int cnt = BM;   // WATTN: rows m0 .. m0 + cnt - 1 are the window
  if constexpr (WATTN) {   // one window and one head; windows of a head follow each other
    const int vb = (int)xcd_contiguous(blockIdx.x, ntiles);
    const int win = vb % p.tiles_m;
    n0 = (vb / p.tiles_m) * 256;
    m0 = win * 64;
    if (p.attn_win_start) {
      m0 = p.attn_win_start[win];
      cnt = min(max(p.attn_win_start[win + 1] - m0, 1), 64);
    }
  } else {
    const int vb = (int)xcd_contiguous(blockIdx.x, ntiles);
    constexpr int GM = 8;
    const int band_sz = GM * p.tiles_n, band = vb / band_sz, within = vb - band * band_sz;
    const int rows_in_band = min(GM, p.tiles_m - band * GM);
    m0 = (band * GM + within % rows_in_band) * BM;
    n0 = (within / rows_in_band) * BN;
  }

  // ---- what the epilogue adds, requested before the operands: the lane's outputs are rows m0 + wm*WTM + 16 i + fa and,
  //      per fragment j, four columns.  (No branches around the loads: the compiler would wait at the end of each; a
  //      missing operand is loaded from another one that is at least as large and masked.)
  constexpr bool ADDEND = EPI == CS_EPI_RESIDUAL || EPI == SM_EPI_BIAS_POS;
  int mrow[MT], crow[MT];
  bool mok[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int local = wm * WTM + 16 * i + fa, m = m0 + local;
    mok[i] = m < p.M;
    mrow[i] = WATTN ? m0 + min(local, cnt - 1) : min(m, p.M - 1);   // (a short window's last row stands for the missing ones)
  }
  {
    const int32_t* const rows_src = p.c_rows ? p.c_rows : (const int32_t*)p.A;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int mapped = rows_src[p.c_rows ? mrow[i] : 0];
      crow[i] = p.c_rows ? mapped : mrow[i];
    }
  }
  int col[NT], ncol[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    col[j] = n0 + frag_col(wn * NT + j, kq);
    ncol[j] = min(col[j], p.N - 4);
  }
  u32x2_t bias_w[NT];
  const bf16_t* const bias_src = (const bf16_t*)(p.bias ? p.bias : p.W);
  const uint32_t bias_mask = p.bias ? 0xFFFFFFFFu : 0u, lo_mask = p.residual_lo ? 0xFFFFFFFFu : 0u;
  u32x2_t add_hi[ADDEND ? MT : 1][ADDEND ? NT : 1];
  uint32_t add_lo[SPLIT ? MT : 1][SPLIT ? NT : 1];
#pragma unroll
  for (int j = 0; j < NT; ++j) bias_w[j] = *(const u32x2_t*)(bias_src + ncol[j]);
  // WATTN: the rotary table's rows of this wave's queries, and the row sums of the folded RMSNorm (from arrays) of the window's rows
  float co[WATTN ? 10 : 1], si[WATTN ? 10 : 1];
  f32x4_t row_parts[WATTN && NORM == NORM_NONE ? MT : 1][2] = {};
  if constexpr (WATTN) {
    const float* cs = p.attn_cos_sin + (int64_t)(m0 + min(16 * wave + fa, cnt - 1)) * 80 + 10 * kq;
#pragma unroll
    for (int t = 0; t < 10; t += 2) {
      const f32x2_t c2 = *(const f32x2_t*)(cs + t), s2 = *(const f32x2_t*)(cs + 40 + t);
      co[WATTN ? t : 0] = c2[0];
      co[WATTN ? t + 1 : 0] = c2[1];
      si[WATTN ? t : 0] = s2[0];
      si[WATTN ? t + 1 : 0] = s2[1];
    }
    if constexpr (NORM == NORM_NONE) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {   // (without a norm the table's rows stand in for them)
        const float* parts = p.a_row_sumsq ? p.a_row_sumsq + (int64_t)mrow[i] * CS_SUMSQ_PARTS : p.attn_cos_sin + (int64_t)mrow[i] * 80;
        row_parts[WATTN && NORM == NORM_NONE ? i : 0][0] = *(const f32x4_t*)parts;
        row_parts[WATTN && NORM == NORM_NONE ? i : 0][1] = *(const f32x4_t*)(parts + 4);
      }
    }
  }
  if constexpr (ADDEND) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const bf16_t* row = EPI == CS_EPI_RESIDUAL ? (const bf16_t*)p.residual + (int64_t)mrow[i] * p.ldr
                                                 : (const bf16_t*)p.pos + (int64_t)(mrow[i] % p.pos_period) * p.ldpos;
#pragma unroll
      for (int j = 0; j < NT; ++j) add_hi[ADDEND ? i : 0][ADDEND ? j : 0] = *(const u32x2_t*)(row + ncol[j]);
      if constexpr (SPLIT) {
        const uint8_t* row_lo = (p.residual_lo ? p.residual_lo : (const uint8_t*)p.residual) + (int64_t)mrow[i] * p.ldr;
#pragma unroll
        for (int j = 0; j < NT; ++j) add_lo[SPLIT ? i : 0][SPLIT ? j : 0] = *(const uint32_t*)(row_lo + ncol[j]);
      }
    }
  }
  asm volatile("" ::: "memory");   // (the loads above stay above)

  // ---- direct global -> LDS loads.  Tile rows of 128 bytes (64 for fp8 weights), 16-byte chunk c of row r in slot
  //      c ^ key(r) (conflict-free: 16 lanes read 16 consecutive rows of one chunk); the hardware places a wave's 64
  //      chunks one after the other, so the swizzle sits on the global side.  W rows are stored in fragment order.
  uint32_t a_src[A_LD], w_src[W_LD];
  uint32_t a_dst[A_LD], w_dst[W_LD];
#pragma unroll
  for (int j = 0; j < A_LD; ++j) {
    const int b = j * NWAVES + wave, sub = b / A_BLK, blk = b % A_BLK;
    const int row = blk * 8 + (lane >> 3), r = WATTN ? m0 + min(row, cnt - 1) : min(m0 + row, p.M - 1);
    a_src[j] = (uint32_t)(((int64_t)r * p.lda + (((lane & 7) ^ ((row >> 1) & 7)) << 3)) * 2) + sub * 128;
    a_dst[j] = sub * A_SUB + blk * 1024;
  }
  auto w_row = [&](int row) {   // matrix row of tile row `row`
    const int J = row >> 4, q = (row >> 2) & 3, r = row & 3;
    return min(n0 + (PAIRED ? (J / 2) * 32 + 8 * q + (J % 2) * 4 + r : row), p.N - 1);
  };
#pragma unroll
  for (int j = 0; j < W_LD; ++j) {
    const int b = min(j * NWAVES + wave, KS * W_BLK - 1), sub = b / W_BLK, blk = b % W_BLK;
    if constexpr (W_FP8) {
      const int row = blk * 16 + (lane >> 2);
      w_src[j] = (uint32_t)((int64_t)w_row(row) * p.ldw + (((lane & 3) ^ ((row >> 2) & 3)) << 4)) + sub * 64;
    } else {
      const int row = blk * 8 + (lane >> 3);
      w_src[j] = (uint32_t)(((int64_t)w_row(row) * p.ldw + (((lane & 7) ^ ((row >> 1) & 7)) << 3)) * 2) + sub * 128;
    }
    w_dst[j] = KS * A_SUB + sub * W_SUB + blk * 1024;
  }
  __amdgpu_buffer_rsrc_t rsrc_a =
      __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, (int)(uint32_t)(((int64_t)(p.M - 1) * p.lda + p.K) * 2), 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.W, 0, (int)(uint32_t)(((int64_t)(p.N - 1) * p.ldw + p.K) * (W_FP8 ? 1 : 2)), 0x00020000);
  // (the device-only builtin with nothing template-dependent around it: else the host pass drops the kernel)
  auto load_a = [&](char* lds_dst, uint32_t off, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (sm_lds_void_t*)lds_dst, 16, off, soff, 0, 0);
  };
  auto load_w = [&](char* lds_dst, uint32_t off, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (sm_lds_void_t*)lds_dst, 16, off, soff, 0, 0);
  };
  // direct loads FROM .. TO - 1 of a stage (the activation rows first)
  auto issue = [&](int stage, int slot_off, auto from_c, auto to_c) {
    constexpr int FROM = decltype(from_c)::value, TO = decltype(to_c)::value;
    char* const base = smem + slot_off;
#pragma unroll
    for (int n = FROM; n < TO; ++n) {
      if (n < A_LD) load_a(base + a_dst[n < A_LD ? n : 0], a_src[n < A_LD ? n : 0], stage * (KS * 128));
      else load_w(base + w_dst[n < A_LD ? 0 : n - A_LD], w_src[n < A_LD ? 0 : n - A_LD], stage * (KS * W_ROW));
    }
  };

  // ---- fragments: lane (fa, kq) of k-step ks reads chunk 4 ks + kq of row fa of each 16-row block
  int x_off[2], w_off[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    x_off[ks] = (wm * WTM + fa) * 128 + (((ks * 4 + kq) ^ ((fa >> 1) & 7)) << 4);
    w_off[ks] = W_FP8 ? (wn * WTN + fa) * 64 + (((ks * 2 + (kq >> 1)) ^ ((fa >> 2) & 3)) << 4) + (kq & 1) * 8
                      : (wn * WTN + fa) * 128 + (((ks * 4 + kq) ^ ((fa >> 1) & 7)) << 4);
  }
  const int w_last = (min(wn * NT + NT - 1, FRAGS_N - 1) - wn * NT) * (16 * W_ROW);   // offset of the wave's last fragment
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // ---- inline norms: sums of squares (and sums) of the lane's columns, five k-steps to a part
  //      (WATTN: every wave holds all four row blocks; each takes the sums of one, from a fragment read for that)
  constexpr int NORM_MT = WATTN ? 1 : MT;
  float ss[NORM != NORM_NONE ? NORM_MT : 1], sm[NORM == NORM_LN ? NORM_MT : 1];
  const int norm_row = WATTN ? wave * 16 + fa : wm * WTM + fa;
  bf16x8_t xn[2][2];
  int phase = 0, part = 0;
  float* const parts_ss = (float*)(smem + STAGES * STAGE);
  float* const parts_sm = parts_ss + BM * CS_SUMSQ_PARTS * 4;
  // A K tile is two k-steps, a part five: of five K tiles the third closes a part after its first k-step, the fifth after its second.
  // The tile only sets the chains aside (`ss0`); they are stored behind it, where no branch cuts an iteration's schedule (WATTN, 16
  // windows, weights from HBM: 24.9 -> 23.3 us).
  constexpr int NS = NORM != NORM_NONE ? NORM_MT : 1, NM = NORM == NORM_LN ? NORM_MT : 1;
  float ss0[NS], sm0[NM];
  auto store_part = [&](bool aside) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      // (the waves that share a tile row write the same values)
      const int at = (part * BM + norm_row + 16 * i) * 4 + kq;
      parts_ss[at] = aside ? ss0[i] : ss[i];
      ss[i] = aside ? ss[i] : 0.f;
      if constexpr (NORM == NORM_LN) {
        parts_sm[at] = aside ? sm0[i < NM ? i : 0] : sm[i < NM ? i : 0];
        sm[i < NM ? i : 0] = aside ? sm[i < NM ? i : 0] : 0.f;
      }
    }
    ++part;
  };
  auto end_of_step = [&](int step) {
    if (step == 0) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        ss0[i] = ss[i];
        ss[i] = phase == 2 ? 0.f : ss[i];
      }
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        sm0[i] = sm[i];
        sm[i] = phase == 2 ? 0.f : sm[i];
      }
    }
  };
  auto end_of_tile = [&]() {
    if constexpr (NORM != NORM_NONE) {
      if (phase == 2 || phase == 4) store_part(phase == 2);
      phase = phase == 4 ? 0 : phase + 1;
    }
  };
#pragma unroll
  for (int i = 0; i < NS; ++i) ss[i] = 0.f;
#pragma unroll
  for (int i = 0; i < NM; ++i) sm[i] = 0.f;

  // ---- operand fragments of one K tile, two sets: one is read while the matrix cores work on the other
  bf16x8_t xf[2][2][MT], wf[2][W_FP8 ? 1 : 2][W_FP8 ? 1 : NT];
  i32x2_t wraw[2][W_FP8 ? 2 : 1][W_FP8 ? NT : 1];
  auto read_tile = [&](int slot_off, auto sub_c, auto set_c) {   // K tile `sub` of the slot's stage into fragment set `set`
    constexpr int SUB = decltype(sub_c)::value, SET = decltype(set_c)::value;
    const char* const base = smem + slot_off;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const char* const a_tile = base + SUB * A_SUB + x_off[s];
      const char* const w_tile = base + KS * A_SUB + SUB * W_SUB + w_off[s];
#pragma unroll
      for (int i = 0; i < MT; ++i) xf[SET][s][i] = *(const bf16x8_t*)(a_tile + i * (16 * 128));
      if constexpr (WATTN && NORM != NORM_NONE) xn[SET][s] = *(const bf16x8_t*)(a_tile + wave * (16 * 128));
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const char* const src = WHOLE || j < NT - 1 ? w_tile + j * (16 * W_ROW) : w_tile + w_last;
        if constexpr (W_FP8) wraw[SET][W_FP8 ? s : 0][W_FP8 ? j : 0] = *(const i32x2_t*)src;
        else wf[SET][W_FP8 ? 0 : s][W_FP8 ? 0 : j] = *(const bf16x8_t*)src;
      }
    }
  };
  auto multiply = [&](auto set_c) {
    constexpr int SET = decltype(set_c)::value;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        bf16x8_t w;
        if constexpr (W_FP8) w = fp8x8_to_bf16(wraw[SET][W_FP8 ? s : 0][W_FP8 ? j : 0]);
        else w = wf[SET][W_FP8 ? 0 : s][W_FP8 ? 0 : j];
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i][j] = sm_mfma(w, xf[SET][s][i], acc[i][j]);
      }
    }
    if constexpr (NORM != NORM_NONE) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int i = 0; i < NORM_MT; ++i) {
            const u32x4_t x = __builtin_bit_cast(u32x4_t, WATTN ? xn[SET][s] : xf[SET][s][i]);
            ss[i] = sm_dot2(x[q], x[q], ss[i]);
            if constexpr (NORM == NORM_LN) sm[i] = sm_dot2(x[q], SM_ONE_PAIR, sm[i]);
          }
        }
        end_of_step(s);
      }
    }
  };
  const int nst = p.K / (BK * KS);
  constexpr std::integral_constant<int, 0> C0{};
  constexpr std::integral_constant<int, 1> C1{};
  constexpr std::integral_constant<int, NLD / 2> CMID{};
  constexpr std::integral_constant<int, NLD> CEND{};
  auto wait_landed = [&](int later) {   // at most the loads of the `later` stages requested after the needed one remain
    small_wait<NLD>(later, std::make_integer_sequence<int, STAGES>{});
  };
  // Slots by their byte offset in the ring: of stage kt - 1, kt and kt + 1
  int prev = (STAGES - 1) * STAGE, slot = 0, next = STAGE;
  auto turn = [&]() {
    prev = slot;
    slot = next;
    next = next == (STAGES - 1) * STAGE ? 0 : next + STAGE;
  };
  // With a share of the prefetch hint the ring runs on into it behind the last stage (see hint_rows_of): the loads' sources move.
  // The slots of the ring are free by then, and nobody reads what arrives.
  const bool reads_hint = Shape::RING_HINT && hint_rows > 0 && nst >= STAGES;
  auto switch_to_hint = [&]() {
    if constexpr (Shape::RING_HINT) {
      const cshint::Share share = cshint::share_of((uint32_t)p.prefetch_bytes, Shape::HINT_PITCH, hint_rows, (int)blockIdx.x);
      const char* const base = (const char*)p.prefetch + (int64_t)share.first * Shape::HINT_PITCH - nst * Shape::HINT_SEG;
      rsrc_a = rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, share.rows * Shape::HINT_PITCH, 0x00020000);
#pragma unroll
      for (int n = 0; n < NLD; ++n) {
        const uint32_t off = cshint::small_offset(KS, STAGES, NLD, wave, n, lane);
        if (n < A_LD) a_src[n < A_LD ? n : 0] = off;
        else w_src[n < A_LD ? 0 : n - A_LD] = off;
      }
    }
  };
  int kt = 0;
  // STEADY iterations have a stage to request and no branch that would interrupt their schedule.  Their loop is rolled: a launch of
  // few rows runs through some ten iterations, and unrolled over the ring each of them fetches its instructions for the first
  // time (256 rows x 1280 x 1280 7.1 -> 6.6 us).  Only the smallest tiles, whose iterations are a handful of MFMAs, save more
  // with the slots' addresses as constants where the loop is long (96 rows x 1280 x 3456 8.1 us rolled, 7.7).
  constexpr bool UNROLLED = BM == 32 && BN <= 64;
  constexpr std::true_type T{};
  constexpr std::false_type F{};
  if constexpr (KS == 2) {
    // Main loop, one barrier per stage of two K tiles.  First half of iteration kt: tile 0 of stage kt is multiplied while
    // tile 1 is read.  The barrier in the middle says that stage kt + 1 has landed for every wave and that nobody reads
    // stage kt's slot any more.  Second half: tile 1 is multiplied while tile 0 of stage kt + 1 is read.  Stage kt + STAGES
    // goes into the freed slot, half of its loads in this half and half in the next.
    small_for([&](auto s_c) {
      constexpr int S = decltype(s_c)::value;
      if (S < nst) issue(S, S * STAGE, C0, std::integral_constant<int, S < STAGES - 1 ? NLD : NLD / 2>{});
    }, std::make_integer_sequence<int, STAGES>{});
    if (nst >= STAGES) sm_wait_barrier<(STAGES - 2) * NLD + NLD / 2>();
    else wait_landed(nst - 1);
    read_tile(0, C0, C0);
    auto iteration = [&](auto steady_c) {
      constexpr bool STEADY = decltype(steady_c)::value;
      read_tile(slot, C1, C1);
      if (STEADY || cshint::small_second_half(kt, STAGES, nst, reads_hint)) issue(kt + STAGES - 1, prev, CMID, CEND);
      multiply(C0);
      if constexpr (STEADY) {
        small_schedule<2 * (MT + NT), NLD - NLD / 2, 2 * MT * NT>();
        end_of_tile();
        if (Shape::RING_HINT && kt + STAGES == nst) switch_to_hint();
        sm_wait_barrier<(STAGES - 2) * NLD>();
        read_tile(next, C0, C0);
        issue(kt + STAGES, slot, C0, CMID);
      } else {
        end_of_tile();
        if (kt + 1 < nst) {
          wait_landed(min(STAGES - 2, nst - kt - 2));
          read_tile(next, C0, C0);
        }
      }
      multiply(C1);
      if constexpr (STEADY) small_schedule<2 * (MT + NT), NLD / 2, 2 * MT * NT>();
      end_of_tile();
      ++kt;
      turn();
    };
    const int steady = cshint::small_steady(KS, STAGES, nst, reads_hint);
    if (UNROLLED && steady >= 2 * STAGES)
      while (kt + STAGES <= steady) small_for([&](auto) { iteration(T); }, std::make_integer_sequence<int, STAGES>{});
    while (kt < steady) iteration(T);
    while (kt < nst) iteration(F);
  } else {
    // One K tile per stage (tiles so large that a stage of two would leave a ring of two): the fragments of tile kt are in
    // registers at the top of iteration kt, the barrier frees its slot for tile kt + STAGES.  K is a multiple of 128, so
    // the tiles go in pairs, one for each fragment set.
    small_for([&](auto s_c) {
      constexpr int S = decltype(s_c)::value;
      if (S < nst) issue(S, S * STAGE, C0, CEND);
    }, std::make_integer_sequence<int, STAGES>{});
    wait_landed(min(STAGES, nst) - 1);
    read_tile(0, C0, C0);
    auto iteration = [&](auto steady_c, auto set_c) {
      constexpr bool STEADY = decltype(steady_c)::value;
      constexpr std::integral_constant<int, 1 - decltype(set_c)::value> OTHER{};
      if constexpr (STEADY) {
        if (Shape::RING_HINT && kt + STAGES == nst) switch_to_hint();
        sm_wait_barrier<(STAGES - 2) * NLD>();
        read_tile(next, C0, OTHER);
        issue(kt + STAGES, slot, C0, CEND);
      } else if (kt + 1 < nst) {
        // (behind a hint, whose loads are not waited for, the needed stage was requested before them)
        if (reads_hint) sm_wait_barrier<(STAGES - 2) * NLD>();
        else wait_landed(min(STAGES - 2, nst - kt - 2));
        if (!reads_hint && kt + STAGES < nst) issue(kt + STAGES, slot, C0, CEND);
        read_tile(next, C0, OTHER);
      }
      multiply(set_c);
      if constexpr (STEADY) small_schedule<2 * (MT + NT + (WATTN && NORM != NORM_NONE ? 1 : 0)), NLD, 2 * MT * NT>();
      end_of_tile();
      ++kt;
      turn();
    };
    const int steady = cshint::small_steady(KS, STAGES, nst, reads_hint);   // (the last of an odd count goes with the others)
    while (kt < steady) {
      iteration(T, C0);
      iteration(T, C1);
    }
    while (kt < nst) {
      iteration(F, C0);
      if (kt < nst) iteration(F, C1);
    }
  }

  // (the LDS that loads in flight write must stay this workgroup's; without a hint nobody waits here for the stores)
  auto end_of_hint = [&]() {
    if (reads_hint) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  // ---- epilogue
  float rstd[NORM != NORM_NONE ? MT : 1], nmean_rstd[NORM == NORM_LN ? MT : 1];
  if constexpr (NORM != NORM_NONE) {
    if ((2 * nst * KS) % 5) store_part(false);   // (the last part is narrower)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (this wave's own values: no barrier)
    if constexpr (WATTN) __syncthreads();                // (each row block's are another wave's)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int r = wm * WTM + 16 * i + fa;
      if constexpr (NORM == NORM_RMS) {
        rstd[i] = rsqrtf(sm_total_of_parts(parts_ss, BM, r, part) / (float)p.K + p.norm_eps);
      } else {
        const float mean = sm_total_of_parts(parts_sm, BM, r, part) / (float)p.K;
        const float var = fmaxf(__builtin_fmaf(-mean, mean, sm_total_of_parts(parts_ss, BM, r, part) / (float)p.K), 0.f);
        rstd[i] = rsqrtf(var + p.norm_eps);
        nmean_rstd[NORM == NORM_LN ? i : 0] = -mean * rstd[i];
      }
    }
  }
  if constexpr (WATTN) {
    float row_scale[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      row_scale[i] = 1.0f;
      if constexpr (NORM != NORM_NONE) {
        row_scale[i] = rstd[NORM != NORM_NONE ? i : 0];
      } else if (p.a_row_sumsq) {
        const f32x4_t s0 = row_parts[NORM == NORM_NONE ? i : 0][0], s1 = row_parts[NORM == NORM_NONE ? i : 0][1];
        const float total = ((s0[0] + s0[1]) + (s0[2] + s0[3])) + ((s1[0] + s1[1]) + (s1[2] + s1[3]));
        row_scale[i] = rsqrtf(total / (float)p.K + p.norm_eps);
      }
    }
    // (in the two slots that the hint's last loads, which may be in flight, do not go to: the last two stages', neighbours because
    // their number is even)
    small_wattn_epilogue<MT, NT, W_FP8>(p, smem + (W_FP8 ? 0 : (nst - 2) % STAGES * STAGE), acc, row_scale, bias_w, co, si, m0, n0, cnt, wave, lane);
    end_of_hint();
    return;
  }
  f32x4_t scale_v[W_FP8 ? NT : 1], csum_v[NORM == NORM_LN ? NT : 1];   // (all loads ahead of the first store)
  if constexpr (W_FP8) {
#pragma unroll
    for (int j = 0; j < NT; ++j) scale_v[W_FP8 ? j : 0] = *(const f32x4_t*)(p.w_scale + ncol[j]);
  }
  if constexpr (NORM == NORM_LN) {
#pragma unroll
    for (int j = 0; j < NT; ++j) csum_v[NORM == NORM_LN ? j : 0] = *(const f32x4_t*)(p.w_col_sum + ncol[j]);
  }
  if constexpr (EPI == SM_EPI_QKV_F32) {   // (the arithmetic of small_wattn_epilogue; C is fp32, W is not fp8)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      float row_scale = 1.0f;
      if constexpr (NORM != NORM_NONE) {
        row_scale = rstd[NORM != NORM_NONE ? i : 0];
      } else if (p.a_row_sumsq) {
        const float* parts = p.a_row_sumsq + (int64_t)mrow[i] * CS_SUMSQ_PARTS;
        const f32x4_t s0 = *(const f32x4_t*)parts, s1 = *(const f32x4_t*)(parts + 4);
        const float ss = ((s0[0] + s0[1]) + (s0[2] + s0[3])) + ((s1[0] + s1[1]) + (s1[2] + s1[3]));
        row_scale = rsqrtf(ss / (float)p.K + p.norm_eps);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const bf16x4_t bias_b = __builtin_bit_cast(bf16x4_t, bias_w[j]);
        f32x4_t x;
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = __builtin_fmaf(acc[i][j][r], row_scale, bf2f(bias_b[r]));
        if (mok[i]) *(f32x4_t*)((float*)p.C + (int64_t)mrow[i] * p.ldc + col[j]) = x;
      }
    }
    end_of_hint();
    return;
  }
  bf16_t* const pC = (bf16_t*)p.C;
  float oss[SUMS != SUMS_NONE ? MT : 1], osm[SUMS == SUMS_BOTH ? MT : 1];
  float* const chain_ss = (float*)(smem + STAGES * STAGE + Shape::NORM_BYTES);   // [row][lane q]
  float* const chain_sm = chain_ss + BM * 4;
  // One fragment's four values per row block; with SUMS the two halves of a row follow each other (see below).
  auto finish = [&]() {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const bool nok = col[j] < p.N;
      const bf16x4_t bias_b = __builtin_bit_cast(bf16x4_t, u32x2_t{bias_w[j][0] & bias_mask, bias_w[j][1] & bias_mask});
      float bias_f[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) bias_f[r] = bf2f(bias_b[r]);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float t = acc[i][j][r];
          if constexpr (W_FP8) t *= scale_v[W_FP8 ? j : 0][r];
          if constexpr (NORM == NORM_LN) {
            v[r] = layernorm_scaled(t, rstd[NORM != NORM_NONE ? i : 0], nmean_rstd[NORM == NORM_LN ? i : 0],
                                    csum_v[NORM == NORM_LN ? j : 0][r], bias_f[r]);
          } else {
            if constexpr (NORM == NORM_RMS) t *= rstd[NORM != NORM_NONE ? i : 0];
            v[r] = t + bias_f[r];
          }
        }
        const int64_t at = (int64_t)crow[i] * p.ldc + col[j];
        const bool ok = mok[i] && nok;
        if constexpr (EPI == CS_EPI_SWIGLU) {
          bf16x2_t o;
          o[0] = f2bf(silu(v[0]) * v[1]);
          o[1] = f2bf(silu(v[2]) * v[3]);
          if (ok) *(bf16x2_t*)(pC + (int64_t)crow[i] * p.ldc + (col[j] >> 1)) = o;
        } else if constexpr (SPLIT) {
          u32x2_t hi;
          uint32_t lo;
          add_split24(v, add_hi[ADDEND ? i : 0][ADDEND ? j : 0], add_lo[SPLIT ? i : 0][SPLIT ? j : 0] & lo_mask, hi, lo);
          if (ok) {
            *(u32x2_t*)(pC + at) = hi;
            *(uint32_t*)(p.c_lo + at) = lo;
          }
          if constexpr (SUMS != SUMS_NONE) {   // (a piece outside the matrix adds exact zeros)
            const uint32_t w0 = nok ? hi[0] : 0u, w1 = nok ? hi[1] : 0u;
            oss[i] = sm_dot2(w1, w1, sm_dot2(w0, w0, oss[i]));
            if constexpr (SUMS == SUMS_BOTH) osm[SUMS == SUMS_BOTH ? i : 0] = sm_dot2(w1, SM_ONE_PAIR, sm_dot2(w0, SM_ONE_PAIR, osm[SUMS == SUMS_BOTH ? i : 0]));
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (EPI == CS_EPI_GELU_ERF) v[r] = gelu_erf(v[r]);
            if constexpr (EPI == CS_EPI_GELU_TANH) v[r] = gelu_tanh(v[r]);
            if constexpr (EPI == CS_EPI_QUICK_GELU) v[r] = quick_gelu(v[r]);
          }
          if constexpr (ADDEND) {
            const bf16x4_t a = __builtin_bit_cast(bf16x4_t, add_hi[ADDEND ? i : 0][ADDEND ? j : 0]);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = rbf(v[r]) + bf2f(a[r]);
          }
          bf16x4_t o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = f2bf(v[r]);
          if (ok) *(bf16x4_t*)(pC + at) = o;
        }
      }
    }
  };
  if constexpr (SUMS == SUMS_NONE) {
    finish();
  } else {
    // The 160 columns of a row belong to two waves.  The sums are chains over ascending columns within each lane q: the
    // wave with the first 80 columns hands its chains over through LDS, the other one continues them and adds the lanes.
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      oss[i] = 0.f;
      if constexpr (SUMS == SUMS_BOTH) osm[SUMS == SUMS_BOTH ? i : 0] = 0.f;
    }
    if (wn == 0) {
      finish();
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int at = (wm * WTM + 16 * i + fa) * 4 + kq;
        chain_ss[at] = oss[i];
        if constexpr (SUMS == SUMS_BOTH) chain_sm[at] = osm[SUMS == SUMS_BOTH ? i : 0];
      }
    }
    __syncthreads();
    if (wn == 1) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int at = (wm * WTM + 16 * i + fa) * 4 + kq;
        oss[i] = chain_ss[at];
        if constexpr (SUMS == SUMS_BOTH) osm[SUMS == SUMS_BOTH ? i : 0] = chain_sm[at];
      }
      finish();
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        float s = oss[i];
        s += __shfl_xor(s, 16);
        s += __shfl_xor(s, 32);
        if (mok[i] && kq == 0) p.c_row_sumsq[(int64_t)crow[i] * CS_SUMSQ_PARTS + n0 / BN] = s;
        if constexpr (SUMS == SUMS_BOTH) {
          float u = osm[SUMS == SUMS_BOTH ? i : 0];
          u += __shfl_xor(u, 16);
          u += __shfl_xor(u, 32);
          if (mok[i] && kq == 0) p.c_row_sum[(int64_t)crow[i] * CS_SUMSQ_PARTS + n0 / BN] = u;
        }
      }
    }
  }
  end_of_hint();
}

// A launch with a tile for every compute unit has nobody idle to read its hint, but nothing to request in its last STAGES - 1
// iterations and its epilogue either: its workgroups read a share each with the ring's own loads, into slots that are free by then
// (hint_ring.h).  Returns the rows of a workgroup, at most what its loads cover; what is left of the hint is not read.
template <class Shape, int WAVES>
int hint_rows_of(int64_t bytes, int tiles) {
  if (!Shape::RING_HINT) return 0;
  return cshint::rows_of(bytes, Shape::HINT_PITCH, tiles, cshint::small_rows(Shape::HINT_SEG / 128, WAVES, Shape::NLD_OF(WAVES)));
}

// Bytes of a hint of `bytes` that a launch of so many tiles leaves at its end: none with idle workgroups, else what the shares do not
// reach (less than a row is not worth another launch's while).
template <class Shape, int WAVES>
int64_t hint_left_of(int64_t bytes, int tiles) {
  if (hint_workgroups(tiles)) return 0;
  if (!Shape::RING_HINT) return bytes;
  const int64_t left = bytes - cshint::bytes_of(bytes, Shape::HINT_PITCH, tiles, cshint::small_rows(Shape::HINT_SEG / 128, WAVES, Shape::NLD_OF(WAVES)));
  return left < Shape::HINT_PITCH ? 0 : left;
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int KS, int STAGES, int EPI, bool W_FP8, int NORM, bool SPLIT, int SUMS = SUMS_NONE>
int launch_small(const CsGemmArgs& a, hipStream_t stream) {
  CsGemmArgs p = a;
  if (EPI == SM_EPI_QKV_WATTN) {   // (tiles_m = windows: the caller's)
    p.tiles_n = p.N / 256;
  } else {
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
  }
  constexpr int lds = SmallShape<BM, BN, KS, STAGES, W_FP8, NORM, SUMS>::LDS;
  auto kern = gemm_small_kernel<BM, BN, WAVES_M, WAVES_N, KS, STAGES, EPI, W_FP8, NORM, SPLIT, SUMS>;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return CS_ERR_LAUNCH;
    attr_set = true;
  }
  const int tiles = p.tiles_m * p.tiles_n, extra = p.prefetch ? hint_workgroups(tiles) : 0;   // (a hint that is still there is one to be read)
  const int hint_rows = p.prefetch && !extra ? hint_rows_of<SmallShape<BM, BN, KS, STAGES, W_FP8, NORM, SUMS>, WAVES_M * WAVES_N>(p.prefetch_bytes, tiles) : 0;
  hipLaunchKernelGGL(kern, dim3(tiles + extra), dim3(64 * WAVES_M * WAVES_N), lds, stream, p, hint_rows);
  return cs_launch_status();
}

// Epilogue / norm dispatch of one tile form.
template <int BM, int BN, int WAVES_M, int WAVES_N, int KS, int STAGES>
int dispatch_small(const CsGemmArgs& a, hipStream_t s) {
#define CS_SMALL(EPI, FP8, NORM, SPLIT) launch_small<BM, BN, WAVES_M, WAVES_N, KS, STAGES, EPI, FP8, NORM, SPLIT>(a, s)
  if (a.w_fp8) {
    switch (a.epilogue) {
      case CS_EPI_BIAS: return CS_SMALL(CS_EPI_BIAS, true, NORM_NONE, false);
      case CS_EPI_RESIDUAL: return a.c_lo ? CS_SMALL(CS_EPI_RESIDUAL, true, NORM_NONE, true) : CS_SMALL(CS_EPI_RESIDUAL, true, NORM_NONE, false);
      case CS_EPI_SWIGLU: return CS_SMALL(CS_EPI_SWIGLU, true, NORM_NONE, false);
      case CS_EPI_GELU_ERF: return CS_SMALL(CS_EPI_GELU_ERF, true, NORM_NONE, false);
      case CS_EPI_GELU_TANH: return CS_SMALL(CS_EPI_GELU_TANH, true, NORM_NONE, false);
      case CS_EPI_QUICK_GELU: return CS_SMALL(CS_EPI_QUICK_GELU, true, NORM_NONE, false);
      default: return CS_ERR_INVALID_ARG;
    }
  }
  if (a.a_norm_inline && a.w_col_sum) {
    switch (a.epilogue) {
      case CS_EPI_BIAS: return CS_SMALL(CS_EPI_BIAS, false, NORM_LN, false);
      case CS_EPI_GELU_TANH: return CS_SMALL(CS_EPI_GELU_TANH, false, NORM_LN, false);
      case CS_EPI_QUICK_GELU: return CS_SMALL(CS_EPI_QUICK_GELU, false, NORM_LN, false);
      default: return CS_ERR_UNSUPPORTED;
    }
  }
  if (a.a_norm_inline) {
    switch (a.epilogue) {
      case CS_EPI_BIAS: return CS_SMALL(CS_EPI_BIAS, false, NORM_RMS, false);
      case CS_EPI_SWIGLU: return CS_SMALL(CS_EPI_SWIGLU, false, NORM_RMS, false);
      default: return CS_ERR_UNSUPPORTED;
    }
  }
  switch (a.epilogue) {
    case CS_EPI_BIAS: return a.pos ? CS_SMALL(SM_EPI_BIAS_POS, false, NORM_NONE, false) : CS_SMALL(CS_EPI_BIAS, false, NORM_NONE, false);
    case CS_EPI_RESIDUAL: return a.c_lo ? CS_SMALL(CS_EPI_RESIDUAL, false, NORM_NONE, true) : CS_SMALL(CS_EPI_RESIDUAL, false, NORM_NONE, false);
    case CS_EPI_SWIGLU: return CS_SMALL(CS_EPI_SWIGLU, false, NORM_NONE, false);
    case CS_EPI_GELU_ERF: return CS_SMALL(CS_EPI_GELU_ERF, false, NORM_NONE, false);
    case CS_EPI_GELU_TANH: return CS_SMALL(CS_EPI_GELU_TANH, false, NORM_NONE, false);
    case CS_EPI_QUICK_GELU: return CS_SMALL(CS_EPI_QUICK_GELU, false, NORM_NONE, false);
    default: return CS_ERR_INVALID_ARG;
  }
#undef CS_SMALL
}

}  // namespace
