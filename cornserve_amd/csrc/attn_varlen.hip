// Variable-length, non-causal flash attention on MFMA for gfx950.
//
// Replaces flash_attn_varlen_func (eric/models/qwen2_5_vl.py:110-120: block-diagonal attention over
// cu_seqlens segments, softmax scale head_dim^-0.5, no dropout, no mask inside a segment) and
// xformers memory_efficient_attention_forward (eric/models/layers/attention.py:51, one segment per
// image).  Optionally applies the Qwen2.5-VL rotary embedding (qwen2_5_vl.py:26-33) to q and k while
// they are staged into LDS, so the rotated tensors never exist in HBM.
//
// Decomposition.  A workgroup owns one query block (<= 32*NWAVES rows of one segment) of one head and
// streams that segment's keys/values through LDS in tiles of 64.  Each wave owns 32 query rows.
// Both products are computed TRANSPOSED so that a lane owns one query column of every accumulator:
//     S^T[key][q] = K[key][:] . Q[q][:]      (MFMA A operand = K rows, B operand = Q rows, k = head dim)
//     O^T[d][q]  += V^T[d][key] . P^T[key][q] (A operand = V^T rows, B operand = P, k = keys)
// With the 32x32 accumulator layout (lane -> column q = lane%32, 16 rows per lane) the online-softmax
// max / sum over keys is 32 in-register operations plus one exchange with lane^32, the rescale of O is
// a per-lane scalar, and P goes from the S accumulators straight into the B operand of the second
// product without touching LDS: accumulator rows 8kk..8kk+7 of a lane are keys
// {16kk+4h+0..3, 16kk+8+4h+0..3} (h = lane/32); the V^T fragment is read from LDS with the same key
// order, which is legal because a dot product does not care about the order of its terms.
// V goes to LDS row-major like K; the transposition happens in the LDS read: ds_read_b64_tr_b16 hands each
// lane of a 16-lane group four 16-bit values gathered from four other lanes' addresses, which turns a
// [4 keys x 16 dims] block into "lane l holds 4 consecutive keys of dim l".
// Head dims that are not multiples of 16 (SigLIP's 72) are zero-padded in LDS only.
#include <type_traits>

#include "common.h"

namespace {

constexpr int BKV = 64;        // keys per LDS tile
constexpr int V_RS = 192;      // bytes per key row of a V tile in LDS (96 head-dim slots).  192 = 64 mod 256: the four
                               // key rows x 64 bytes that 32 lanes of a transposing read touch fall into distinct banks.

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

// A-operand fragment of V^T for the 32x32x16 MFMA: lane (fr = lane%32, hf = lane/32) gets dim 32t + fr and the
// keys {16g + 4hf + 0..3, 16g + 8 + 4hf + 0..3} of key group g -- the key order in which the S^T accumulators
// hold P.  ds_read_b64_tr_b16 works on groups of 16 lanes: destination lane l receives element l%4 of the
// 8 bytes addressed by source lanes l/4 + 4e, e = 0..3.  So source lane s = 4e + j of a group addresses key
// k0 + e, dims d0 + 4j .. 4j+3, and destination lane l ends up with dim d0 + l, keys k0 .. k0+3.
CS_DEVICE bf16x8_t read_vt_frag(const char* v_tile, int t, int g, int lane) {
  const int hf = lane >> 5, s = lane & 15;
  const int key = 16 * g + 4 * hf + (s >> 2);
  const int dim = 32 * t + 16 * ((lane >> 4) & 1) + 4 * (s & 3);
  const char* p = v_tile + key * V_RS + dim * 2;
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)p);
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 8 * V_RS));
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

struct AttnArgs {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  int64_t ld;
  bf16_t* out;
  int64_t ldo;
  const int32_t* work;
  const float* cos_sin;
  float scale_log2e;
  // full-attention kernel only: 1-D launch, see its workgroup mapping
  int n_work, heads, chunk, n_chunks_x;
};

// ---- pieces shared by the attention kernels.  A wave owns 32 query rows (lane % 32 = query, lane / 32 = which
//      half of the 8-row groups of a 32x32 MFMA result it holds) and works on tiles of BKV = 64 keys.

// S^T = K.Q^T for one key tile in LDS (row stride RS bytes), keys past `nvalid` masked to -inf.
template <int KS, int RS>
CS_DEVICE void score_tile(f32x16_t (&sacc)[2], const char* k_tile, const bf16x8_t (&qf)[KS], int nvalid, int fr, int hf) {
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[kt][r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8_t kf = *(const bf16x8_t*)(k_tile + (kt * 32 + fr) * RS + (2 * ks + hf) * 16);
      sacc[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], sacc[kt], 0, 0, 0);
    }
  }
  if (nvalid < BKV) {  // uniform: only the last tile of a segment can be partial
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kt * 32 + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (key >= nvalid) sacc[kt][r] = -INFINITY;
      }
  }
}

// Online softmax of one tile's scores -> P (bf16 fragments for the P.V product).
// Lazy reference maximum: P = exp2((s - m_run) * scale) with an m_run that is only raised when some query of the
// wave sees a score more than LAZY_LOG2 (in log2 units) above it.  P then ranges up to 2^LAZY_LOG2 instead of 1,
// which fp32 accumulation and bf16's exponent range do not care about, the final division by the denominator
// (built from the same P) cancels the reference, and the rescale of O -- DT*16 multiplies and an exponential per
// tile -- runs only in the first tiles of a segment.  The whole wave is raised, each query to its own maximum so far: the
// nearer the reference is to a query's largest scores, the less their P is rounded (scores of standard deviation 9, largest
// weights near 1: error against 64 bits 1.63e-3 at d = 80 and 1.71e-3 at d = 64, where raising only the queries that ask for
// it gives 1.66e-3 and 1.86e-3).  m_run starts at -inf, so the first tile always sets it to its own maximum.  With
// L_FROM_MFMA the denominator is not summed here (see attn_full_kernel).
// FIRST_TILE: the caller knows that nothing has been accumulated yet (O = 0, m_run = -inf): no rescale to consider.
constexpr float LAZY_LOG2 = 6.0f;
template <int DT, bool L_FROM_MFMA, bool FIRST_TILE = false>
CS_DEVICE void softmax_tile(const f32x16_t (&sacc)[2], bf16x8_t (&pf)[2][2], f32x16_t (&oacc)[DT], float& m_run,
                            float& l_run, float sl2) {
  float mx = -INFINITY;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt)
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sacc[kt][r]);
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  float alpha = 1.0f;
  if constexpr (FIRST_TILE) {
    m_run = mx;
  } else if (__any((mx - m_run) * sl2 > LAZY_LOG2)) {
    const float m_new = fmaxf(m_run, mx);
    alpha = __builtin_amdgcn_exp2f((m_run - m_new) * sl2);
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[t][r] *= alpha;
    m_run = m_new;
  }
  const float mb = m_run * sl2;
  float psum = 0.f;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float pv = __builtin_amdgcn_exp2f(sacc[kt][r] * sl2 - mb);
      if constexpr (!L_FROM_MFMA) psum += pv;
      pf[kt][r >> 3][r & 7] = f2bf(pv);
    }
  if constexpr (!L_FROM_MFMA) {
    psum += __shfl_xor(psum, 32, 64);
    l_run = l_run * alpha + psum;
  }
}

// O^T[d][q] / l -> out[q][d0 ...]: a lane owns query `qi` and 4 consecutive d per 8-row group.  With L_FROM_MFMA the
// denominator is row D of O^T (block D/32, row D%32 = 8g + 4*half + e), held by the lanes of one half.
template <int D, int DT, bool L_FROM_MFMA>
CS_DEVICE void write_output(const f32x16_t (&oacc)[DT], float l_run, bf16_t* orow, bool valid, int hf) {
  if constexpr (L_FROM_MFMA) {
    constexpr int RR = D % 32, G_L = RR / 8, HF_L = (RR % 8) / 4, E_L = RR % 4;
    const float mine = oacc[D / 32][4 * G_L + E_L];
    const float other = __shfl_xor(mine, 32, 64);
    l_run = hf == HF_L ? mine : other;
  }
  if (!valid) return;
  const float inv = 1.0f / l_run;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = t * 32 + 8 * g + 4 * hf;
      if (d0 < D) {
        bf16x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f2bf(oacc[t][4 * g + e] * inv);
        *(bf16x4_t*)(orow + d0) = o;
      }
    }
}

// ---- softmax_tile in the pieces that the pipeline of attn_full_direct_kernel works on, half a key tile (32 keys) at a time: the
//      same operations on a query's values in the same order, so that a query has the same bits in every kernel.
CS_DEVICE float row_max(const f32x16_t& s) {
  float mx = s[0];
#pragma unroll
  for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
  return mx;
}
// over the two lanes that hold a query's scores (lane, lane ^ 32)
CS_DEVICE float pair_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  const uint32_t lower = r[0], upper = r[1];   // (named: a bit cast of a vector element takes the vector's first)
  return fmaxf(__builtin_bit_cast(float, lower), __builtin_bit_cast(float, upper));
}

template <int D, int NWAVES, bool ROPE, int HPW>
__global__ __launch_bounds__(NWAVES * 64, 2) void attn_kernel(const AttnArgs a) {
  constexpr int NT = NWAVES * 64;
  constexpr int BQ = NWAVES * 32;
  constexpr int KS = (D + 15) / 16;    // MFMA k-steps over the head dim
  constexpr int DT = (D + 31) / 32;    // 32-row tiles of O^T
  constexpr int DC = D / 8;            // real 16-byte chunks per row
  constexpr int DKC = KS * 2;          // chunks per row after zero padding
  constexpr int RS = (DKC | 1) * 16;   // LDS row stride in bytes, odd chunk count: conflict-free b128 reads
  static_assert(D % 8 == 0 && D <= 96, "head dim");
  static_assert(!ROPE || D % 16 == 0, "rotary needs an even number of chunks per half");
  // The softmax denominator comes out of the P.V product through a column of ones in the V tile when the head
  // dim leaves spare rows in the last 32-row block of O^T (see attn_full_kernel; the same arithmetic in every
  // attention kernel keeps an item's result independent of which of them a batch's longest segment selects).
  constexpr bool L_FROM_MFMA = (D % 32) != 0;

  __shared__ __attribute__((aligned(16))) char q_lds[BQ * RS];
  __shared__ __attribute__((aligned(16))) char k_lds[BKV * RS];
  __shared__ __attribute__((aligned(16))) char v_lds[BKV * V_RS];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 31, hf = lane >> 5;
  const int head0 = blockIdx.y * HPW;  // this workgroup's HPW consecutive heads
  const int seg_start = a.work[blockIdx.x * 4 + 0];
  const int seg_end = a.work[blockIdx.x * 4 + 1];
  const int q0 = a.work[blockIdx.x * 4 + 2];
  const int nq = a.work[blockIdx.x * 4 + 3];
  int64_t hoff = (int64_t)head0 * D;  // column offset of the head being processed
  if constexpr (L_FROM_MFMA) {  // chunk DC of every V row := (1, 0, ..., 0); the staging below never writes there
    bf16x8_t one = {0, 0, 0, 0, 0, 0, 0, 0};
    one[0] = f2bf(1.0f);
    for (int r = tid; r < BKV; r += NT) *(bf16x8_t*)(v_lds + r * V_RS + DC * 16) = one;
  }

  // Stage `nrows` rows starting at global row g0 (valid rows: < g0 + nvalid) of a [*, ld] tensor into an
  // LDS tile with row stride RS, zero-filling invalid rows and pad chunks, optionally rotating.
  auto stage_rows = [&](const bf16_t* src, char* dst, int g0, int nrows, int nvalid) {
    const bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
    if (ROPE) {
      constexpr int HC = DC / 2;  // chunks per half
      for (int i = tid; i < nrows * HC; i += NT) {
        const int r = i / HC, jc = i - r * HC;
        bf16x8_t o1 = zero, o2 = zero;
        if (r < nvalid) {
          const int64_t g = g0 + r;
          const bf16_t* p = src + g * a.ld + hoff + jc * 8;
          const bf16x8_t x1 = *(const bf16x8_t*)p;
          const bf16x8_t x2 = *(const bf16x8_t*)(p + D / 2);
          const float* cs = a.cos_sin + g * D + jc * 8;
          const f32x4_t c0 = *(const f32x4_t*)cs, c1 = *(const f32x4_t*)(cs + 4);
          const f32x4_t s0 = *(const f32x4_t*)(cs + D / 2), s1 = *(const f32x4_t*)(cs + D / 2 + 4);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float co = e < 4 ? c0[e] : c1[e - 4];
            const float si = e < 4 ? s0[e] : s1[e - 4];
            const float xa = bf2f(x1[e]), xb = bf2f(x2[e]);
            o1[e] = f2bf(rot_first(xa, xb, co, si));
            o2[e] = f2bf(rot_second(xa, xb, co, si));
          }
        }
        *(bf16x8_t*)(dst + r * RS + jc * 16) = o1;
        *(bf16x8_t*)(dst + r * RS + (jc + HC) * 16) = o2;
      }
    } else {
      for (int i = tid; i < nrows * DKC; i += NT) {
        const int r = i / DKC, c = i - r * DKC;
        bf16x8_t x = zero;
        if (r < nvalid && c < DC) x = *(const bf16x8_t*)(src + (int64_t)(g0 + r) * a.ld + hoff + c * 8);
        *(bf16x8_t*)(dst + r * RS + c * 16) = x;
      }
    }
    if (ROPE && DKC > DC) {
      for (int i = tid; i < nrows * (DKC - DC); i += NT) {
        const int r = i / (DKC - DC), c = DC + i % (DKC - DC);
        *(bf16x8_t*)(dst + r * RS + c * 16) = zero;
      }
    }
  };

  // V tile -> LDS, row-major; rows past the segment end are zero (they meet P = 0, which must not be 0 * NaN).
  auto stage_v = [&](int g0, int nvalid) {
    const bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = tid; i < BKV * DC; i += NT) {
      const int r = i / DC, c = i - r * DC;
      bf16x8_t x = zero;
      if (r < nvalid) x = *(const bf16x8_t*)(a.v + (int64_t)(g0 + r) * a.ld + hoff + c * 8);
      *(bf16x8_t*)(v_lds + r * V_RS + c * 16) = x;
    }
  };

  f32x16_t oacc[DT];
  float m_run, l_run;
  auto reset_state = [&]() {
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[t][r] = 0.f;
    m_run = -INFINITY;
    l_run = 0.f;
  };
  const bool wave_active = wave * 32 < nq;
  auto write_out = [&]() {
    const int qi = wave * 32 + fr;
    write_output<D, DT, L_FROM_MFMA>(oacc, l_run, a.out + (int64_t)(q0 + min(qi, nq - 1)) * a.ldo + hoff, qi < nq, hf);
  };
  bf16x8_t qf[KS];
  auto load_q_frags = [&]() {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const bf16x8_t*)(q_lds + (wave * 32 + fr) * RS + (2 * ks + hf) * 16);
  };

  // One K/V tile in LDS (nvalid keys): S^T = K Q^T, online softmax, O^T += V^T P^T.
  auto compute_tile = [&](int nvalid, auto first_c) {
    f32x16_t sacc[2];
    bf16x8_t pf[2][2];
    score_tile<KS, RS>(sacc, k_lds, qf, nvalid, fr, hf);
    softmax_tile<DT, L_FROM_MFMA, decltype(first_c)::value>(sacc, pf, oacc, m_run, l_run, a.scale_log2e);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const bf16x8_t vf = read_vt_frag(v_lds, t, kt * 2 + kk, lane);
          oacc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[kt][kk], oacc[t], 0, 0, 0);
        }
    }
  };

  const int seg_len = seg_end - seg_start;
  if (ROPE && BQ == BKV && seg_len <= BKV && q0 == seg_start) {
    // A whole segment in one tile (window attention): the query rows ARE the key rows.  Every global load
    // of a head -- q, k, v -- is issued in one batch into registers, the rotary table is fetched once
    // for all HPW heads, and the batch of head h+1 is requested before the matrix-core work on head h,
    // so after the first head the memory latency hides behind compute.
    constexpr int HC = DC / 2;
    constexpr int NI = (BKV * HC + NT - 1) / NT, NV = (BKV * DC + NT - 1) / NT;
    const bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
    bf16x8_t q1[NI], q2[NI], k1[NI], k2[NI], vx[NV];
    f32x4_t c0[NI], c1[NI], s0[NI], s1[NI];
    // Unconditional loads from clamped rows (no branch between them, so they are all in flight together).
    // Rows past the segment end therefore hold copies of the last row: as keys they are masked (P = 0, and
    // 0 times a finite V row is 0), as queries their outputs are never written.
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int i = min(tid + it * NT, BKV * HC - 1), r = i / HC, jc = i - r * HC;
      const float* cs = a.cos_sin + (int64_t)(seg_start + min(r, seg_len - 1)) * D + jc * 8;
      c0[it] = *(const f32x4_t*)cs;
      c1[it] = *(const f32x4_t*)(cs + 4);
      s0[it] = *(const f32x4_t*)(cs + D / 2);
      s1[it] = *(const f32x4_t*)(cs + D / 2 + 4);
    }
    auto issue_qkv = [&](int64_t ho) {
#pragma unroll
      for (int it = 0; it < NI; ++it) {
        const int i = min(tid + it * NT, BKV * HC - 1), r = i / HC, jc = i - r * HC;
        const int64_t off = (int64_t)(seg_start + min(r, seg_len - 1)) * a.ld + ho + jc * 8;
        q1[it] = *(const bf16x8_t*)(a.q + off);
        q2[it] = *(const bf16x8_t*)(a.q + off + D / 2);
        k1[it] = *(const bf16x8_t*)(a.k + off);
        k2[it] = *(const bf16x8_t*)(a.k + off + D / 2);
      }
#pragma unroll
      for (int it = 0; it < NV; ++it) {
        const int i = min(tid + it * NT, BKV * DC - 1), r = i / DC, c = i - r * DC;
        vx[it] = *(const bf16x8_t*)(a.v + (int64_t)(seg_start + min(r, seg_len - 1)) * a.ld + ho + c * 8);
      }
    };
    issue_qkv(hoff);
    if (DKC > DC) {  // pad chunks of the q and k tiles: written once, never overwritten
      for (int i = tid; i < BKV * (DKC - DC); i += NT) {
        const int r = i / (DKC - DC), c = DC + i % (DKC - DC);
        *(bf16x8_t*)(q_lds + r * RS + c * 16) = zero;
        *(bf16x8_t*)(k_lds + r * RS + c * 16) = zero;
      }
    }
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
      if (hh > 0) __syncthreads();  // every wave is done reading the previous head's tiles
#pragma unroll
      for (int it = 0; it < NI; ++it) {
        const int i = tid + it * NT, r = i / HC, jc = i - r * HC;
        if (i < BKV * HC) {
          bf16x8_t qa, qb, ka, kb;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float co = e < 4 ? c0[it][e] : c1[it][e - 4];
            const float si = e < 4 ? s0[it][e] : s1[it][e - 4];
            const float xa = bf2f(q1[it][e]), xb = bf2f(q2[it][e]);
            qa[e] = f2bf(rot_first(xa, xb, co, si));
            qb[e] = f2bf(rot_second(xa, xb, co, si));
            const float ya = bf2f(k1[it][e]), yb = bf2f(k2[it][e]);
            ka[e] = f2bf(rot_first(ya, yb, co, si));
            kb[e] = f2bf(rot_second(ya, yb, co, si));
          }
          *(bf16x8_t*)(q_lds + r * RS + jc * 16) = qa;
          *(bf16x8_t*)(q_lds + r * RS + (jc + HC) * 16) = qb;
          *(bf16x8_t*)(k_lds + r * RS + jc * 16) = ka;
          *(bf16x8_t*)(k_lds + r * RS + (jc + HC) * 16) = kb;
        }
      }
#pragma unroll
      for (int it = 0; it < NV; ++it) {
        const int i = tid + it * NT, r = i / DC, c = i - r * DC;
        if (i < BKV * DC) *(bf16x8_t*)(v_lds + r * V_RS + c * 16) = vx[it];
      }
      __syncthreads();
      if (hh + 1 < HPW) issue_qkv(hoff + D);  // the staging registers are free again
      reset_state();
      if (wave_active) {
        load_q_frags();
        compute_tile(seg_len, std::true_type{});
      }
      write_out();
      hoff += D;
    }
  } else {
    for (int hh = 0; hh < HPW; ++hh) {
      if (hh > 0) __syncthreads();
      reset_state();
      stage_rows(a.q, q_lds, q0, BQ, nq);
      __syncthreads();
      load_q_frags();
      for (int kv0 = 0; kv0 < seg_len; kv0 += BKV) {
        const int nvalid = min(BKV, seg_len - kv0);
        __syncthreads();  // previous tile fully consumed
        stage_rows(a.k, k_lds, seg_start + kv0, BKV, nvalid);
        stage_v(seg_start + kv0, nvalid);
        __syncthreads();
        if (!wave_active) continue;
        compute_tile(nvalid, std::false_type{});
      }
      write_out();
      hoff += D;
    }
  }
}

// Full-attention variant (segments longer than 64 rows): 4 waves x 32 query rows, K/V tiles double-buffered.
// The global loads of tile t+1 are issued before the matrix-core work on tile t and land in registers;
// rotary (K) and the transpose (V) are applied when those registers are written to the other LDS buffer
// after the compute, so one barrier per tile is enough and memory latency hides behind the MFMAs.  The Q
// tile shares its LDS region with the second K/V buffer: Q is only needed until its fragments are in
// registers.
template <int D, bool ROPE>
__global__ __launch_bounds__(256, 2) void attn_full_kernel(const AttnArgs a) {
  constexpr int NT = 256, BQ = 128;
  constexpr int KS = (D + 15) / 16, DT = (D + 31) / 32, DC = D / 8, DKC = KS * 2;
  constexpr int RS = (DKC | 1) * 16;
  constexpr int HC = DC / 2;
  static_assert(D % 8 == 0 && D <= 96, "head dim");
  static_assert(!ROPE || D % 16 == 0, "rotary needs an even number of chunks per half");
  // When the head dim does not fill its last 32-row block of O^T, one of the spare V columns is set to 1:
  // row D of O^T is then sum_k P[k], the softmax denominator, accumulated (and rescaled) by the matrix cores
  // together with O instead of 32 vector additions and a shuffle per tile.
  constexpr bool L_FROM_MFMA = (D % 32) != 0;
  constexpr int K_BYTES = BKV * RS, V_BYTES = BKV * V_RS, Q_BYTES = BQ * RS;
  constexpr int REGION_B = (K_BYTES + V_BYTES) > Q_BYTES ? (K_BYTES + V_BYTES) : Q_BYTES;
  __shared__ __attribute__((aligned(16))) char lds[K_BYTES + V_BYTES + REGION_B];
  auto k_buf = [&](int b) -> char* { return lds + b * (K_BYTES + V_BYTES); };
  auto v_buf = [&](int b) -> char* { return lds + b * (K_BYTES + V_BYTES) + K_BYTES; };
  char* const q_lds = lds + K_BYTES + V_BYTES;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 31, hf = lane >> 5;
  // Workgroup mapping.  Workgroup i runs on XCD i % 8, each with its own L2.  Query blocks of one segment
  // and head read the same K/V, so they should meet in one L2: the (work item, head) space is cut into
  // chunks of `chunk` consecutive work items of one head (a segment's query blocks are consecutive work
  // items), chunk c goes to XCD c % 8, and an XCD walks its chunks in order.
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  // The chunks of all heads come first item by item: with the longest segments in front of the work list (ops.attn_plan), the
  // long workgroups start first, and every XCD gets its share of them (with heads outermost and two chunks, one long and one
  // short, all long ones met on four of the eight XCDs: segments of 3300, 1196, 1024 and 720 rows, d = 72, 131 -> 105 us).
  const int cid = (j / a.chunk) * 8 + xcd;           // chunk id in [0, n_chunks_x * heads)
  const int item = (cid / a.heads) * a.chunk + j % a.chunk;
  const int head = cid % a.heads;
  if (item >= a.n_work) return;                      // padding of the last chunks (uniform per workgroup)
  const int seg_start = a.work[item * 4 + 0];
  const int seg_end = a.work[item * 4 + 1];
  const int q0 = a.work[item * 4 + 2];
  const int nq = a.work[item * 4 + 3];
  const int64_t hoff = (int64_t)head * D;
  const int seg_len = seg_end - seg_start;
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const f32x4_t zero4 = {0, 0, 0, 0};

  // ---- register staging of one K/V tile
  constexpr int K_ITEMS = ROPE ? BKV * HC : BKV * DC;
  constexpr int K_PER = (K_ITEMS + NT - 1) / NT;
  constexpr int V_ITEMS = BKV * DC;
  constexpr int V_PER = (V_ITEMS + NT - 1) / NT;
  bf16x8_t kx1[K_PER], kx2[ROPE ? K_PER : 1];
  f32x4_t kc0[ROPE ? K_PER : 1], kc1[ROPE ? K_PER : 1], ks0[ROPE ? K_PER : 1], ks1[ROPE ? K_PER : 1];
  bf16x8_t vx[V_PER];

  // Unconditional loads from clamped rows and items (no branch between them, so they are all in flight
  // together).  Rows past the segment end then hold copies of the last valid row: as keys they are masked
  // (P = 0, and 0 times a finite V row is 0).
  auto gload_tile = [&](int kv0, int nvalid) {
#pragma unroll
    for (int u = 0; u < K_PER; ++u) {
      const int i = min(tid + u * NT, K_ITEMS - 1);
      constexpr int PER_ROW = ROPE ? HC : DC;
      const int r = i / PER_ROW, jc = i - r * PER_ROW;
      const int64_t g = seg_start + kv0 + min(r, nvalid - 1);
      const bf16_t* p = a.k + g * a.ld + hoff + jc * 8;
      kx1[u] = *(const bf16x8_t*)p;
      if (ROPE) {
        kx2[u] = *(const bf16x8_t*)(p + D / 2);
        const float* cs = a.cos_sin + g * D + jc * 8;
        kc0[u] = *(const f32x4_t*)cs;
        kc1[u] = *(const f32x4_t*)(cs + 4);
        ks0[u] = *(const f32x4_t*)(cs + D / 2);
        ks1[u] = *(const f32x4_t*)(cs + D / 2 + 4);
      }
    }
#pragma unroll
    for (int u = 0; u < V_PER; ++u) {
      const int i = min(tid + u * NT, V_ITEMS - 1);
      const int r = i / DC, c = i - r * DC;   // consecutive lanes: consecutive chunks of one key row
      vx[u] = *(const bf16x8_t*)(a.v + (int64_t)(seg_start + kv0 + min(r, nvalid - 1)) * a.ld + hoff + c * 8);
    }
  };
  auto lstore_tile = [&](int b) {
    char* kd = k_buf(b);
    char* vd = v_buf(b);
#pragma unroll
    for (int u = 0; u < K_PER; ++u) {
      const int i = tid + u * NT;
      if (i < K_ITEMS) {
        constexpr int PER_ROW = ROPE ? HC : DC;
        const int r = i / PER_ROW, jc = i - r * PER_ROW;
        if (ROPE) {
          bf16x8_t o1, o2;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float co = e < 4 ? kc0[u][e] : kc1[u][e - 4];
            const float si = e < 4 ? ks0[u][e] : ks1[u][e - 4];
            const float xa = bf2f(kx1[u][e]), xb = bf2f(kx2[u][e]);
            o1[e] = f2bf(rot_first(xa, xb, co, si));
            o2[e] = f2bf(rot_second(xa, xb, co, si));
          }
          *(bf16x8_t*)(kd + r * RS + jc * 16) = o1;
          *(bf16x8_t*)(kd + r * RS + (jc + HC) * 16) = o2;
        } else {
          *(bf16x8_t*)(kd + r * RS + jc * 16) = kx1[u];
        }
      }
    }
    if (!ROPE && DKC > DC) {  // zero the pad chunks of the K rows (head dims that are not multiples of 16)
      for (int i = tid; i < BKV * (DKC - DC); i += NT) {
        const int r = i / (DKC - DC), c = DC + i % (DKC - DC);
        *(bf16x8_t*)(kd + r * RS + c * 16) = zero8;
      }
    }
#pragma unroll
    for (int u = 0; u < V_PER; ++u) {
      const int i = tid + u * NT;
      if (i < V_ITEMS) {
        const int r = i / DC, c = i - r * DC;
        *(bf16x8_t*)(vd + r * V_RS + c * 16) = vx[u];
      }
    }
  };

  // chunk DC (dims D .. D+7) of every key row of V buffer b := (1, 0, ..., 0); lstore_tile never writes there
  auto store_ones_column = [&](int b) {
    if constexpr (L_FROM_MFMA) {
      bf16x8_t one = zero8;
      one[0] = f2bf(1.0f);
      for (int r = tid; r < BKV; r += NT) *(bf16x8_t*)(v_buf(b) + r * V_RS + DC * 16) = one;
    }
  };

  // ---- prologue: Q -> LDS (rotated), tile 0 -> LDS buffer 0
  gload_tile(0, min(BKV, seg_len));
  {
    if (ROPE) {
      for (int i = tid; i < BQ * HC; i += NT) {
        const int r = i / HC, jc = i - r * HC;
        bf16x8_t o1 = zero8, o2 = zero8;
        if (r < nq) {
          const int64_t g = q0 + r;
          const bf16_t* p = a.q + g * a.ld + hoff + jc * 8;
          const bf16x8_t x1 = *(const bf16x8_t*)p;
          const bf16x8_t x2 = *(const bf16x8_t*)(p + D / 2);
          const float* cs = a.cos_sin + g * D + jc * 8;
          const f32x4_t c0 = *(const f32x4_t*)cs, c1 = *(const f32x4_t*)(cs + 4);
          const f32x4_t s0 = *(const f32x4_t*)(cs + D / 2), s1 = *(const f32x4_t*)(cs + D / 2 + 4);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float co = e < 4 ? c0[e] : c1[e - 4];
            const float si = e < 4 ? s0[e] : s1[e - 4];
            const float xa = bf2f(x1[e]), xb = bf2f(x2[e]);
            o1[e] = f2bf(rot_first(xa, xb, co, si));
            o2[e] = f2bf(rot_second(xa, xb, co, si));
          }
        }
        *(bf16x8_t*)(q_lds + r * RS + jc * 16) = o1;
        *(bf16x8_t*)(q_lds + r * RS + (jc + HC) * 16) = o2;
      }
    } else {
      for (int i = tid; i < BQ * DKC; i += NT) {
        const int r = i / DKC, c = i - r * DKC;
        bf16x8_t x = zero8;
        if (r < nq && c < DC) x = *(const bf16x8_t*)(a.q + (int64_t)(q0 + r) * a.ld + hoff + c * 8);
        *(bf16x8_t*)(q_lds + r * RS + c * 16) = x;
      }
    }
  }
  lstore_tile(0);
  store_ones_column(0);
  __syncthreads();
  bf16x8_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const bf16x8_t*)(q_lds + (wave * 32 + fr) * RS + (2 * ks + hf) * 16);
  __syncthreads();  // every wave holds its Q fragments: the Q region may now become K/V buffer 1
  store_ones_column(1);  // (ordered before the first read of buffer 1 by the barrier that ends iteration 0)

  f32x16_t oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[t][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const bool wave_active = wave * 32 < nq;
  const float sl2 = a.scale_log2e;

  int buf = 0;
  for (int kv0 = 0; kv0 < seg_len; kv0 += BKV, buf ^= 1) {
    const int nvalid = min(BKV, seg_len - kv0);
    const bool more = kv0 + BKV < seg_len;
    if (more) gload_tile(kv0 + BKV, min(BKV, seg_len - kv0 - BKV));
    if (wave_active) {
      const char* kd = k_buf(buf);
      const char* vd = v_buf(buf);
      f32x16_t sacc[2];
      bf16x8_t pf[2][2];
      score_tile<KS, RS>(sacc, kd, qf, nvalid, fr, hf);
      softmax_tile<DT, L_FROM_MFMA>(sacc, pf, oacc, m_run, l_run, sl2);
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) {
            const bf16x8_t vf = read_vt_frag(vd, t, kt * 2 + kk, lane);
            oacc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[kt][kk], oacc[t], 0, 0, 0);
          }
      }
    }
    if (more) lstore_tile(buf ^ 1);
    __syncthreads();
  }

  const int qi = wave * 32 + fr;
  write_output<D, DT, L_FROM_MFMA>(oacc, l_run, a.out + (int64_t)(q0 + min(qi, nq - 1)) * a.ldo + hoff, qi < nq, hf);
}

// Full attention without rotary on the keys (SigLIP; the Qwen families after cs_rope_qk): a software pipeline over half tiles of
// 32 keys.  One step issues the matrix instructions of two different half tiles -- P.V of the previous one and the scores of one
// of the next tile -- while the vector unit works on the softmax of the one between them.  Nothing in a step waits for a matrix
// result of the same step, so the matrix cores run under the softmax of the SAME wave: with the three phases one after the
// other, three waves per SIMD took 1,370 clocks of a SIMD per wave and 64-key tile, 704 of them matrix instructions.  The
// arithmetic is softmax_tile's, bit for bit: scores run a whole tile ahead, because a tile's reference maximum is that of all its 64
// keys, and a half tile's scores stay in their registers until the products of the same half of the next tile overwrite them
// (the exponents are taken out in phase 1, P.V; those products are phase 2).  How the instructions of a phase interleave is
// laid down with scheduling groups; two waves per SIMD (two workgroups per CU) use what a wave leaves free.  V fragments live
// in two register sets, the next step's being read during this one; K fragments are read at the start of their own step.
//   16 heads, back to back, one phase after the other -> this kernel, d = 72: 4 x 4096 rows 376 -> 356 us, 4096 rows 105 -> 94,
//   3300 + 1196 + 1024 + 720 rows 142 -> 85, 7 x 729 rows 33.5 -> 33.5, 2 x 729 rows 18.5 -> 14.4; d = 80: 8 x 1024 rows 59.5 -> 60.6, 1024
//   rows 22.4 -> 17.1, 1380 + 816 rows 38.9 -> 26.1, 4888 rows 206 -> 160, 9000 + 5000 + 3000 + 1000 + 432 rows 725 -> 643, 16 x 1008 rows 113 ->
//   117; d = 64: 2 x 1500 rows 37.5 -> 31.4; d = 96: 46.8 -> 40.9 us.  (A launch that fills the chip with equal segments gains
//   nothing; 6 to 12 instead of 4 exponentials in phase 1 take the same to 3 % longer.)
// A reference that is the first tile's maximum plus a margin, whose overrun shows in the packed words, needs no maximum of a tile:
// 2 to 4 % faster at d = 72 and 80, but P is rounded elsewhere and less exactly (wide scores, d = 80: error against 64 bits 1.67e-3
// instead of 1.63e-3, d = 64: 1.97e-3 instead of 1.71e-3).
// What bounds it is power: the shader clock falls from 1.9 to 1.4 .. 1.7 GHz under such a pipeline, and a build without the LDS reads
// ran as many clocks at a higher clock rate.  Also measured: 64 query rows per wave and one wave per SIMD (half the LDS reads,
// but a lone wave issues an instruction every five clocks: 2,630 clocks per 64 rows and tile against 1,930), eight waves around
// one K/V stream (the same time within 3 %; 7 x 729 rows 41 us), and dims 64 .. 79 of O^T in 16x16 blocks (a sixth less V read and
// multiplied, eight lane swaps more: no faster).
//
// K and V tiles go global -> LDS directly (buffer_load ... lds: no staging registers, no LDS store instructions, no
// address arithmetic per tile) into a ring of three tile buffers, requested two tiles ahead.  A direct load fixes the LDS
// side -- the 64 lanes of a wave fill 1 KB of consecutive LDS -- so the padded row layout is produced on the global side: a
// tile is the flat sequence of 16-byte chunk slots (row, slot), lane l of load j owns slot j*64 + l and fetches chunk
// `slot % slots_per_row` of row `slot / slots_per_row`; lanes that own padding slots are switched off for the load, which
// leaves the padding as initialised once per buffer (zeros behind the K rows that the last k-step reads, the ones
// column of V that yields the softmax denominator).  The loads are written in assembly, which writes LDS only: behind the
// builtin, the compiler takes every transposing LDS read for a possible reader of the bytes in flight and waits for
// ALL outstanding loads in front of it.  The kernel's own waits are explicit (one per tile, in front of its barrier).
typedef __attribute__((address_space(3))) void lds_void_t;
typedef int i32x4_sgpr_t __attribute__((ext_vector_type(4)));

template <int D>
struct AttnDirectShape {
  static constexpr int KS = (D + 15) / 16, DKC = KS * 2, DC = D / 8;
  static constexpr int K_SLOTS = DKC | 1, V_SLOTS = V_RS / 16;      // 16-byte slots per tile row
  static constexpr int RS = K_SLOTS * 16;
  static constexpr int K_BYTES = BKV * RS, V_BYTES = BKV * V_RS, TILE_BYTES = K_BYTES + V_BYTES;
  static constexpr int K_LOADS = BKV * K_SLOTS / 64, V_LOADS = BKV * V_SLOTS / 64;   // BKV == 64: one load per slot column
  static constexpr int LOADS = K_LOADS + V_LOADS, PER_WAVE = (LOADS + 3) / 4;
  static constexpr int Q_BYTES = 128 * RS;                          // the Q tile starts out in the third buffer
  static constexpr int LDS = 2 * TILE_BYTES + (Q_BYTES > TILE_BYTES ? Q_BYTES : TILE_BYTES);
  static_assert(2 * LDS <= 160 * 1024, "two workgroups per CU");
};

// ROPE_Q: the keys were rotated in place beforehand; the query rows are rotated here while they are staged (a
// query block is staged once, whereas every query block of a segment would rotate the segment's keys again).
template <int D, bool ROPE_Q = false>
__global__ __launch_bounds__(256, 2) void attn_full_direct_kernel(const AttnArgs a) {
  constexpr int NT = 256, BQ = 128;
  static_assert(!ROPE_Q || D % 16 == 0, "rotary needs an even number of 16-byte chunks per half");
  using Shape = AttnDirectShape<D>;
  constexpr int KS = Shape::KS, DT = (D + 31) / 32, DC = Shape::DC, DKC = Shape::DKC;
  constexpr int RS = Shape::RS, K_SLOTS = Shape::K_SLOTS, V_SLOTS = Shape::V_SLOTS;
  constexpr int K_BYTES = Shape::K_BYTES, TILE_BYTES = Shape::TILE_BYTES;
  constexpr int K_LOADS = Shape::K_LOADS, LOADS = Shape::LOADS, PER = Shape::PER_WAVE;
  static_assert(D % 8 == 0 && D <= 96 && BKV == 64, "head dim / tile");
  constexpr bool L_FROM_MFMA = (D % 32) != 0;   // see attn_full_kernel
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  auto k_buf = [&](int b) -> char* { return lds + b * TILE_BYTES; };
  auto v_buf = [&](int b) -> char* { return lds + b * TILE_BYTES + K_BYTES; };
  char* const q_lds = lds + 2 * TILE_BYTES;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, hf = lane >> 5;
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;   // workgroup mapping: see attn_full_kernel
  const int cid = (j / a.chunk) * 8 + xcd;
  const int item = (cid / a.heads) * a.chunk + j % a.chunk;
  const int head = cid % a.heads;
  if (item >= a.n_work) return;
  const int seg_start = a.work[item * 4 + 0];
  const int seg_end = a.work[item * 4 + 1];
  const int q0 = a.work[item * 4 + 2];
  const int nq = a.work[item * 4 + 3];
  const int64_t hoff = (int64_t)head * D;
  const int seg_len = seg_end - seg_start;
  const int n_tiles = (seg_len + BKV - 1) / BKV;
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};

  // ---- the wave's direct loads of a tile.  Load u of this wave is load number jl = min(4u + wave, LOADS-1) of the
  //      tile (the clamp makes a wave without a load of its own repeat the last one: every wave must issue the
  //      same number, because the waits count loads).  Byte offsets are relative to the segment's first row.
  const uint32_t row_bytes = (uint32_t)a.ld * 2u;
  const uint64_t k_base = (uint64_t)(a.k + (int64_t)seg_start * a.ld + hoff), v_base = (uint64_t)(a.v + (int64_t)seg_start * a.ld + hoff);
  uint32_t l_off[PER], l_dst[PER];   // offset in a whole tile, LDS address in buffer 0
  uint64_t l_mask[PER];              // the lanes that own data slots
  i32x4_sgpr_t l_rsrc[PER];
  // row and 16-byte column of this lane's slot of load u
  auto slot_of = [&](int u, int ln, int& row, int& chunk) {
    const int jl = min(4 * u + wave, LOADS - 1);
    const bool is_k = jl < K_LOADS;
    const int slot = (is_k ? jl : jl - K_LOADS) * 64 + ln;
    const int per_row = is_k ? K_SLOTS : V_SLOTS;
    row = slot / per_row;
    chunk = slot - row * per_row;
  };
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int jl = min(4 * u + wave, LOADS - 1);
    const bool is_k = jl < K_LOADS;
    int row, chunk;
    slot_of(u, lane, row, chunk);
    l_mask[u] = __ballot(chunk < DC);
    l_off[u] = (uint32_t)row * row_bytes + (uint32_t)chunk * 16u;
    const uint64_t base = is_k ? k_base : v_base;
    l_rsrc[u] = i32x4_sgpr_t{__builtin_amdgcn_readfirstlane((int)(uint32_t)base), __builtin_amdgcn_readfirstlane((int)((base >> 32) & 0xFFFFu)), -1, 0x00020000};
    l_dst[u] = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void_t*)lds + (uint32_t)(is_k ? jl * 1024 : K_BYTES + (jl - K_LOADS) * 1024));
  }
  auto issue_load = [&](uint32_t dst, uint64_t mask, uint32_t off, i32x4_sgpr_t rsrc, uint32_t soff) {
    uint64_t exec_was;   // (m0, the LDS address, is nobody else's in this kernel: no builtin that uses it is called)
    asm volatile("s_mov_b32 m0, %1\n\ts_and_saveexec_b64 %0, %2\n\tbuffer_load_dwordx4 %3, %4, %5 offen lds\n\ts_mov_b64 exec, %0"
                 : "=&s"(exec_was) : "s"(dst), "s"(mask), "v"(off), "s"(rsrc), "s"(soff) : "scc", "memory");
  };
  auto issue_tile = [&](int t, int b) {
    const int nvalid = min(BKV, seg_len - t * BKV);
    const uint32_t soff = (uint32_t)(t * BKV) * row_bytes, to = (uint32_t)(b * TILE_BYTES);
    if (nvalid == BKV) {
#pragma unroll
      for (int u = 0; u < PER; ++u) issue_load(l_dst[u] + to, l_mask[u], l_off[u], l_rsrc[u], soff);
    } else {   // rows past the segment end repeat the last valid row: as keys they are masked, and P = 0 times a finite V row is 0
      int lane_p = lane;
      asm volatile("" : "+v"(lane_p));   // (once a segment: its offsets are not kept in registers across the loop)
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        int row, chunk;
        slot_of(u, lane_p, row, chunk);
        issue_load(l_dst[u] + to, l_mask[u], (uint32_t)min(row, nvalid - 1) * row_bytes + (uint32_t)chunk * 16u, l_rsrc[u], soff);
      }
    }
  };
  auto init_padding = [&](int b) {
    if constexpr (DKC > DC) {
      for (int i = tid; i < BKV * (DKC - DC); i += NT) {
        const int r = i / (DKC - DC), c = DC + i % (DKC - DC);
        *(bf16x8_t*)(k_buf(b) + r * RS + c * 16) = zero8;
      }
    }
    // (V columns past the head dim: the column of ones, then zeros -- rows of O^T that nobody reads, but random bytes there would
    // cost the multipliers power)
    constexpr int VPAD = L_FROM_MFMA ? V_SLOTS - DC : 0;
    for (int i = tid; i < BKV * VPAD; i += NT) {
      const int r = i / (VPAD ? VPAD : 1), c = i - r * VPAD;
      bf16x8_t x = zero8;
      if (c == 0) x[0] = f2bf(1.0f);
      *(bf16x8_t*)(v_buf(b) + r * V_RS + (DC + c) * 16) = x;
    }
  };
  // every load of this wave has landed and every LDS access is done, in every wave
  auto sync_all = [&]() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ---- prologue: tiles 0 and 1 requested; Q, all of its loads in flight together, -> LDS (third buffer) -> fragments
  issue_tile(0, 0);
  if (n_tiles > 1) issue_tile(1, 1);
  if constexpr (ROPE_Q) {
    constexpr int HC = DC / 2, ITEMS = BQ * HC, N = (ITEMS + NT - 1) / NT;   // D % 16 == 0: no padding chunks (DKC == DC)
    bf16x8_t x1[N], x2[N];
    f32x4_t c0[N], c1[N], s0[N], s1[N];
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int i = min(tid + it * NT, ITEMS - 1), r = i / HC, jc = i - r * HC;
      const int64_t g = q0 + min(r, nq - 1);
      const bf16_t* p = a.q + g * a.ld + hoff + jc * 8;
      x1[it] = *(const bf16x8_t*)p;
      x2[it] = *(const bf16x8_t*)(p + D / 2);
      const float* cs = a.cos_sin + g * D + jc * 8;
      c0[it] = *(const f32x4_t*)cs;
      c1[it] = *(const f32x4_t*)(cs + 4);
      s0[it] = *(const f32x4_t*)(cs + D / 2);
      s1[it] = *(const f32x4_t*)(cs + D / 2 + 4);
    }
    init_padding(0);
    init_padding(1);
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int i = min(tid + it * NT, ITEMS - 1), r = i / HC, jc = i - r * HC;
      bf16x8_t o1, o2;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float co = e < 4 ? c0[it][e] : c1[it][e - 4];
        const float si = e < 4 ? s0[it][e] : s1[it][e - 4];
        const float xa = bf2f(x1[it][e]), xb = bf2f(x2[it][e]);
        o1[e] = f2bf(rot_first(xa, xb, co, si));
        o2[e] = f2bf(rot_second(xa, xb, co, si));
      }
      *(bf16x8_t*)(q_lds + r * RS + jc * 16) = o1;
      *(bf16x8_t*)(q_lds + r * RS + (jc + HC) * 16) = o2;
    }
  } else {
    constexpr int N = BQ * DKC / NT;
    static_assert(BQ * DKC % NT == 0, "whole batches");
    bf16x8_t x[N];
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int i = tid + it * NT, r = i / DKC, c = i - r * DKC;
      x[it] = *(const bf16x8_t*)(a.q + (int64_t)(q0 + min(r, nq - 1)) * a.ld + hoff + min(c, DC - 1) * 8);
    }
    init_padding(0);
    init_padding(1);
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int i = tid + it * NT, r = i / DKC, c = i - r * DKC;
      *(bf16x8_t*)(q_lds + r * RS + c * 16) = c < DC ? x[it] : zero8;
    }
  }
  sync_all();   // (tiles 0 and 1 have landed with the Q rows)
  bf16x8_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const bf16x8_t*)(q_lds + (wave * 32 + fr) * RS + (2 * ks + hf) * 16);

  f32x16_t oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[t][r] = 0.f;
  float mb = 0.f, l_run = 0.f;
  const float sl2 = a.scale_log2e;
  const int sg = lane & 15;
  const int k_lane = fr * RS + hf * 16;
  const int v_lane = (4 * hf + (sg >> 2)) * V_RS + (16 * ((lane >> 4) & 1) + 4 * (sg & 3)) * 2;   // see read_vt_frag

  auto read_k = [&](bf16x8_t (&kf)[KS], int b, int half) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = *(const bf16x8_t*)(k_buf(b) + k_lane + half * 32 * RS + ks * 32);
  };
  auto read_v = [&](bf16x8_t (&vf)[DT][2], int b, int half) {
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const char* p = v_buf(b) + v_lane + (32 * half + 16 * kk) * V_RS + t * 64;
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)p);
        const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 8 * V_RS));
        vf[t][kk] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
  };
  auto scores = [&](f32x16_t& s, const bf16x8_t (&kf)[KS]) {
    const f32x16_t z = {};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], qf[ks], ks == 0 ? z : s, 0, 0, 0);
  };
  auto pv = [&](const i32x4_t (&p)[2], const bf16x8_t (&vf)[DT][2]) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int t = 0; t < DT; ++t) oacc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t][kk], __builtin_bit_cast(bf16x8_t, p[kk]), oacc[t], 0, 0, 0);
  };
  // keys past `nvalid` of the tile (the last tile of a segment only)
  auto mask = [&](f32x16_t& s, int nvalid, int half) {
    int left = nvalid - half * 32 - 4 * hf;
    asm volatile("" : "+v"(left));   // one register compared with constants, not 32 loop-invariant comparisons kept in registers
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (8 * (r >> 2) + (r & 3) >= left) s[r] = -INFINITY;
  };
  // One step: O += V^T.P of p_in and vf (phase 1), then s_io, a half tile's scores, becomes those of half `half` of the tile in buffer k_b
  // (phase 2); p_out = exponentials of what s_io held, a part of them in either phase.  Meanwhile the V fragments of the next
  // step are read (half `half` of the tile in buffer v_b), and the maximum of s_max is taken, which `vote` gets between the phases.
  constexpr int EXP_1 = 4;   // exponentials of phase 1
  auto exponents = [&](float (&e)[16], const f32x16_t& s) {
#pragma unroll
    for (int r = 0; r < 16; ++r) e[r] = __builtin_fmaf(s[r], sl2, -mb);
#pragma unroll
    for (int r = 0; r < EXP_1; ++r) e[r] = __builtin_amdgcn_exp2f(e[r]);
  };
  auto step = [&](f32x16_t& s_io, i32x4_t (&p_out)[2], const i32x4_t (&p_in)[2], const bf16x8_t (&vf)[DT][2], bf16x8_t (&vf_next)[DT][2],
                  int k_b, int v_b, int half, const f32x16_t& s_max, float& psum, auto vote) {
    bf16x8_t kf[KS];
    float e[16];
    read_k(kf, k_b, half);
    read_v(vf_next, v_b, half);
    pv(p_in, vf);
    float mx = row_max(s_max);
    asm volatile("" : "+v"(mx));   // (here and below: what is used behind a branch is not moved there, out of the overlap)
    exponents(e, s_io);
#pragma unroll
    for (int i = 0; i < 2 * DT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, (KS + 4 * DT + 2 * DT - 1) / (2 * DT), 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 28 / (2 * DT), 0);
      __builtin_amdgcn_sched_group_barrier(0x400, (EXP_1 + 2 * DT - 1) / (2 * DT), 0);
    }
    vote(e, mx);
    __builtin_amdgcn_sched_barrier(0);
    scores(s_io, kf);
#pragma unroll
    for (int r = EXP_1; r < 16; ++r) e[r] = __builtin_amdgcn_exp2f(e[r]);
    if constexpr (!L_FROM_MFMA) {
#pragma unroll
      for (int r = 0; r < 16; ++r) psum += e[r];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      bf16x2_t w;
      w[0] = f2bf(e[2 * i]);
      w[1] = f2bf(e[2 * i + 1]);
      p_out[i >> 2][i & 3] = __builtin_bit_cast(int, w);
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x400, (16 - EXP_1 + KS - 1) / KS, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, L_FROM_MFMA ? 2 : 5, 0);
    }
    asm volatile("" : "+v"(p_out[0]), "+v"(p_out[1]));
  };

  // The next tile of the ring: tile t+1 has landed; every wave has read what it needs of tile t-1 (t == 0: of the Q tile), whose buffer
  // takes tile t+2.
  auto next_tile = [&](int t, int b) {
    sync_all();
    if (t == 0) init_padding(2);   // (first read in iteration 1, behind its barrier)
    if (t + 2 < n_tiles) issue_tile(t + 2, b);
  };
  if (wave * 32 >= nq) {   // a wave without queries: its share of the loads and the barriers
    for (int t = 0, b = 2; t < n_tiles; ++t, b = b == 2 ? 0 : b + 1) next_tile(t, b);
    return;
  }

  f32x16_t s0, s1;   // scores of both halves of a tile
  bf16x8_t vfa[DT][2], vfb[DT][2];
  i32x4_t p0[2], p1[2];
#pragma unroll
  for (int t = 0; t < DT; ++t) vfa[t][0] = vfa[t][1] = zero8;
  p1[0] = p1[1] = i32x4_t{0, 0, 0, 0};   // the first step multiplies zeros
  {
    bf16x8_t kfa[KS], kfb[KS];
    read_k(kfa, 0, 0);
    read_k(kfb, 0, 1);
    scores(s0, kfa);
    scores(s1, kfb);
    if (seg_len < BKV) {
      mask(s0, seg_len, 0);
      mask(s1, seg_len, 1);
    }
  }
  float mx_first = row_max(s0);   // maximum of the tile's first half (this lane's keys)
  // (a query without a score that is a number keeps -inf, as softmax_tile leaves it)
  float m_run = fmaxf(pair_max(fmaxf(mx_first, row_max(s1))), -INFINITY);
  mb = m_run * sl2;
  int b0 = 0, b1 = 1, b2 = 2;   // buffers of tiles t, t+1, t+2
  for (int t = 0; t < n_tiles; ++t) {
    next_tile(t, b2);
    const int left = seg_len - (t + 1) * BKV;   // keys of the tiles behind this one
    float psum = 0.f, alpha = 1.0f;
    // P.V: second half of t-1; softmax: first half of t; scores: first half of t+1
    // (behind the last tile, the scores of whatever the next buffer holds are computed and not used)
    step(s0, p0, p1, vfa, vfb, b1, b0, 0, s1, psum, [&](float (&e)[16], float mx_second) {
#pragma unroll
      for (int r = 0; r < EXP_1; ++r) asm volatile("" : "+v"(e[r]));
      const float mx = fmaxf(mx_first, mx_second);   // (of this lane's keys: the other lane of the query votes as well)
      if (__any((mx - m_run) * sl2 > LAZY_LOG2)) {   // (the whole wave: softmax_tile)
        const float m_new = fmaxf(m_run, pair_max(mx));
        alpha = __builtin_amdgcn_exp2f((m_run - m_new) * sl2);
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) oacc[d][r] *= alpha;
        m_run = m_new;
        mb = m_run * sl2;
        exponents(e, s0);
      }
    });
    if (left > 0 && left < BKV) mask(s0, left, 0);
    // P.V: first half of t; softmax: second half of t; scores: second half of t+1
    step(s1, p1, p0, vfb, vfa, b1, b0, 1, s0, psum, [&](float (&)[16], float mx) { mx_first = mx; });
    if (left > 0 && left < BKV) mask(s1, left, 1);
    if constexpr (!L_FROM_MFMA) {
      psum += __shfl_xor(psum, 32, 64);
      l_run = __builtin_fmaf(l_run, alpha, psum);
    }
    const int bt = b0;
    b0 = b1;
    b1 = b2;
    b2 = bt;
  }
  pv(p1, vfa);

  const int qi = wave * 32 + fr;
  write_output<D, DT, L_FROM_MFMA>(oacc, l_run, a.out + (int64_t)(q0 + min(qi, nq - 1)) * a.ldo + hoff, qi < nq, hf);
}

template <int D, bool ROPE_Q = false>
int launch_attn_full_direct(const AttnArgs& a, dim3 grid, hipStream_t stream) {
  constexpr int lds = AttnDirectShape<D>::LDS;
  static bool attr_set = false;
  auto kern = attn_full_direct_kernel<D, ROPE_Q>;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return CS_ERR_LAUNCH;
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, grid, dim3(256), lds, stream, a);
  return cs_launch_status();
}

template <int D>
int launch_attn(AttnArgs a, int n_work, int heads, int block_q, int max_seqlen, bool rope, bool keys_rotated,
                hipStream_t stream) {
  const dim3 grid(n_work, heads);
  a.n_work = n_work;
  a.heads = heads;
  a.chunk = min(32, max(1, (max_seqlen + 127) / 128));  // query blocks of the longest segment
  a.n_chunks_x = (n_work + a.chunk - 1) / a.chunk;
  const int n_chunks = a.n_chunks_x * heads;
  const dim3 grid_full(((n_chunks + 7) / 8) * 8 * a.chunk);
  if (keys_rotated) {
    // only the long-segment kernel has this form (short segments rotate q and k while staging, one workgroup each)
    if constexpr (D % 16 == 0) {
      if (block_q != 64 && rope && (int64_t)max_seqlen * a.ld * 2 < (int64_t)1 << 31)
        return launch_attn_full_direct<D, true>(a, grid_full, stream);
    }
    return CS_ERR_UNSUPPORTED;
  }
  if (block_q == 64) {
    if (rope) {
      // two heads per workgroup when that still leaves several workgroups per CU
      const bool pair = heads % 2 == 0 && (int64_t)n_work * heads >= 2048;
      if constexpr (D % 16 == 0) {
        if (pair) hipLaunchKernelGGL((attn_kernel<D, 2, true, 2>), dim3(n_work, heads / 2), dim3(128), 0, stream, a);
        else hipLaunchKernelGGL((attn_kernel<D, 2, true, 1>), grid, dim3(128), 0, stream, a);
      } else {
        return CS_ERR_UNSUPPORTED;
      }
    } else {
      hipLaunchKernelGGL((attn_kernel<D, 2, false, 1>), grid, dim3(128), 0, stream, a);
    }
  } else {
    if (rope) {
      if constexpr (D % 16 == 0) hipLaunchKernelGGL((attn_full_kernel<D, true>), grid_full, dim3(256), 0, stream, a);
      else return CS_ERR_UNSUPPORTED;
    } else {
      // the direct-to-LDS kernel addresses a segment's K/V rows with 32-bit byte offsets
      if ((int64_t)max_seqlen * a.ld * 2 < (int64_t)1 << 31)
        return launch_attn_full_direct<D, false>(a, grid_full, stream);
      hipLaunchKernelGGL((attn_full_kernel<D, false>), grid_full, dim3(256), 0, stream, a);
    }
  }
  return cs_launch_status();
}

}  // namespace

// Query rows per workgroup: 64 (2 waves) when no segment is longer than 64 rows (window attention),
// else 128 (4 waves).
extern "C" int cs_attn_block_q(int32_t max_seqlen) { return max_seqlen <= 64 ? 64 : 128; }

extern "C" int cs_attn_work_host(const int32_t* cu_seqlens_host, int32_t n_seg, int32_t block_q,
                                 int32_t* work_host, int32_t cap_items, int32_t* n_work) {
  if (!cu_seqlens_host || n_seg < 0 || block_q <= 0 || !work_host || !n_work) return CS_ERR_INVALID_ARG;
  int n = 0;
  for (int s = 0; s < n_seg; ++s) {
    const int b = cu_seqlens_host[s], e = cu_seqlens_host[s + 1];
    if (e < b) return CS_ERR_INVALID_ARG;
    for (int q = b; q < e; q += block_q) {
      if (n >= cap_items) return CS_ERR_TOO_LARGE;
      work_host[4 * n + 0] = b;
      work_host[4 * n + 1] = e;
      work_host[4 * n + 2] = q;
      work_host[4 * n + 3] = e - q < block_q ? e - q : block_q;
      ++n;
    }
  }
  *n_work = n;
  return CS_OK;
}

static int attn_varlen_entry(const void* q, const void* k, const void* v, int64_t ld, void* out, int64_t ldo,
                             const int32_t* work, int32_t n_work, int32_t heads, int32_t head_dim, float scale,
                             const float* cos_sin, int32_t max_seqlen, bool keys_rotated, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (keys_rotated && !cos_sin) return CS_ERR_INVALID_ARG;
  if (!q || !k || !v || !out || !work || n_work < 0 || heads <= 0 || heads > 65535 || head_dim <= 0 ||
      max_seqlen <= 0)
    return CS_ERR_INVALID_ARG;
  if (ld % 8 || ldo % 4 || head_dim % 8) return CS_ERR_INVALID_ARG;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)cos_sin) & 15) return CS_ERR_INVALID_ARG;
  if ((uintptr_t)out & 7) return CS_ERR_INVALID_ARG;
  if (n_work == 0) return CS_OK;
  AttnArgs a;
  a.q = (const bf16_t*)q;
  a.k = (const bf16_t*)k;
  a.v = (const bf16_t*)v;
  a.ld = ld;
  a.out = (bf16_t*)out;
  a.ldo = ldo;
  a.work = work;
  a.cos_sin = cos_sin;
  a.scale_log2e = scale * 1.4426950408889634f;
  const int bq = cs_attn_block_q(max_seqlen);
  const bool rope = cos_sin != nullptr;
  switch (head_dim) {
    case 64: return launch_attn<64>(a, n_work, heads, bq, max_seqlen, rope, keys_rotated, stream);
    case 72: return launch_attn<72>(a, n_work, heads, bq, max_seqlen, rope, keys_rotated, stream);
    case 80: return launch_attn<80>(a, n_work, heads, bq, max_seqlen, rope, keys_rotated, stream);
    case 96: return launch_attn<96>(a, n_work, heads, bq, max_seqlen, rope, keys_rotated, stream);
    default: return CS_ERR_UNSUPPORTED;
  }
}

extern "C" int cs_attn_varlen(const void* q, const void* k, const void* v, int64_t ld, void* out, int64_t ldo,
                              const int32_t* work, int32_t n_work, int32_t heads, int32_t head_dim, float scale,
                              const float* cos_sin, int32_t max_seqlen, void* stream) {
  return attn_varlen_entry(q, k, v, ld, out, ldo, work, n_work, heads, head_dim, scale, cos_sin, max_seqlen, false, stream);
}

extern "C" int cs_attn_varlen_keys_rotated(const void* q, const void* k, const void* v, int64_t ld, void* out,
                                           int64_t ldo, const int32_t* work, int32_t n_work, int32_t heads,
                                           int32_t head_dim, float scale, const float* cos_sin, int32_t max_seqlen,
                                           void* stream) {
  return attn_varlen_entry(q, k, v, ld, out, ldo, work, n_work, heads, head_dim, scale, cos_sin, max_seqlen, true, stream);
}
