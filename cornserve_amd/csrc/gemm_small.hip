// Few-row GEMM for gfx950: choice of the tile form, and whether the launch is a few-row one at all.  The kernel is in
// gemm_small_impl.h; each tile form is built in its own translation unit (gemm_small_t*.hip).
#include "gemm_common.h"

double cs_gemm_fast_saves(const CsGemmArgs& a, int64_t* tiles);   // gemm_fast.hip
int cs_gemm_small_tile_32x32(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_small_tile_32x64(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_small_tile_64x64(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_small_tile_64x80(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_small_tile_64x128(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_small_tile_128x128(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_small_tile_32x160(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_small_tile_64x160(const CsGemmArgs& a, hipStream_t stream);

namespace {

// Time of a launch in microseconds: per round of 256 tiles, `fixed_us` (first loads, epilogue, and once 2 us of launch)
// plus `stage_us` per 128 k.  From launches of 1280 columns at K = 1280 and 3456 that are one round: 96 rows (32x32: 6.0
// and 8.6 us), 250 (32x64: 7.0, 10.6), 512 (64x64: 8.1, 14.6), 1024 (64x80: 10.2, 18.2; 32x160: 11.8, 22.6), 1500 (64x128:
// 13.1, 22.5), 2048 (64x160: 16.2, 30.5), 2744 (128x128: 20.3, 33.4).  With weights from HBM and longer K both kernels take up
// to a third longer than this says, and fp8 weights cost the big forms more than the small ones; the comparison holds all the
// same: of 29 products of the encoders at 44 row counts each, 581 launches come here, and the one that loses most against the big
// tiles takes 38.7 us instead of 38.2 (2048 rows x 1280 x 3456).
struct Form {
  int bm, bn;
  float fixed_us, stage_us;
  int (*run)(const CsGemmArgs&, hipStream_t);
};
const Form FORMS[] = {
    {32, 32, 4.5f, 0.153f, cs_gemm_small_tile_32x32},   {32, 64, 4.9f, 0.212f, cs_gemm_small_tile_32x64},
    {64, 64, 4.3f, 0.382f, cs_gemm_small_tile_64x64},   {64, 80, 5.5f, 0.470f, cs_gemm_small_tile_64x80},
    {64, 128, 7.6f, 0.553f, cs_gemm_small_tile_64x128}, {128, 128, 12.6f, 0.770f, cs_gemm_small_tile_128x128},
};
const Form SUMS_FORMS[] = {   // with row sums of the output
    {32, 160, 5.5f, 0.635f, cs_gemm_small_tile_32x160}, {64, 160, 7.8f, 0.841f, cs_gemm_small_tile_64x160},
};
// The big tiles of gemm_fast.hip, which run on from tile to tile without a gap: the fixed part counts once (same shapes at
// 1500, 2744, 4096 and 5104 rows, 3840 and 6912 columns at 1024 and 4096).  These four, timed where few rows have to choose; the
// table of gemm_fast.hip, fitted up to 20000 rows, is 15 % off at either end of these (2048 rows x 1280 x 1280, 640 x 3584 x 3584) and
// says here only what its other forms save over them.
struct FastForm {
  int bm, bn;
  float fixed_us, stage_us;
};
const FastForm F128x160 = {128, 160, 8.0f, 1.03f}, F256x160 = {256, 160, 7.0f, 1.50f}, F256x256 = {256, 256, 10.0f, 2.65f},
               F256x128 = {256, 128, 8.0f, 1.50f};

double rounds(int64_t M, int64_t N, int bm, int bn) {
  const int64_t tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  return (double)((tiles + 255) / 256);
}

double small_us(const Form& f, int M, int N, int K, bool norm) {
  const double r = rounds(M, N, f.bm, f.bn), stages = K / 128.0;
  // (an inline norm: 8.8 and 9.2 us at 96 and 250 rows x 3840 columns, K = 1280, where the plain product takes 8.0 and 8.2)
  return r * (f.fixed_us - 2.0 + stages * f.stage_us * (norm ? 1.15 : 1.0)) + 2.0;
}

double fast_us(const CsGemmArgs& a, int64_t* tiles) {
  const int M = a.M, N = a.N;
  const bool sums = a.c_row_sumsq != nullptr;
  const double stages = a.K / 128.0;
  auto us = [&](const FastForm& f) { return f.fixed_us + rounds(M, N, f.bm, f.bn) * stages * f.stage_us; };
  const bool few = (int64_t)((M + 255) / 256) * ((N + 159) / 160) <= 128;   // (the same rule as in cs_gemm_fast_saves)
  double t = us(few ? F128x160 : F256x160);
  if (!sums) t = us(F256x256) < t ? us(F256x256) : t;
  if (!sums && a.epilogue == CS_EPI_SWIGLU) t = us(F256x128) < t ? us(F256x128) : t;
  return t * cs_gemm_fast_saves(a, tiles);
}

// A launch of more than two rounds is no few-row launch: the times above are of one round, and five rounds of 64x64 take 33 us
// (28 without the byte planes) where they promise 30.7 and 256x160 takes 30 (22): 4160 and 4374 rows x 1152 x 1152.  Two rounds
// of 32x64 hold: 200 rows x 4352 x 1152 12.6 us against 16.0, 288 fp8 rows x 3584 x 5120 31.7 against 93.  (Inline norms have
// no other kernel.)
constexpr double MAX_ROUNDS = 2.0;

template <int COUNT>
const Form* best_form(const Form (&forms)[COUNT], const CsGemmArgs& a, double* us) {
  const Form* best = nullptr;
  *us = 0;
  for (const Form& f : forms) {
    if (f.bn == 80 && (a.w_fp8 || a.a_norm_inline || a.pos || !(a.epilogue == CS_EPI_BIAS || (a.epilogue == CS_EPI_RESIDUAL && a.c_lo)))) continue;
    if (!a.a_norm_inline && rounds(a.M, a.N, f.bm, f.bn) > MAX_ROUNDS) continue;
    const double t = small_us(f, a.M, a.N, a.K, a.a_norm_inline);
    if (!best || t < *us) {
      best = &f;
      *us = t;
    }
  }
  return best;
}

int tiles_of(const Form& f, const CsGemmArgs& a) { return ((a.M + f.bm - 1) / f.bm) * ((a.N + f.bn - 1) / f.bn); }

// Whether a launch has too many tiles for idle compute units to read its hint, where the big form has some.  Of 128x128 tiles nobody
// reads it then, and the launch that the hint is for
// finds its weights cold (2700 rows of Qwen2-VL: projection 24 us instead of 17), so such a launch goes to the few-row kernel only
// if it is 15 % faster there.  Passes with few-row tiles and the hint unread -> with the big form: Qwen2-VL 2700 patches (fc2: 220
// tiles of 128x128 or 176 of 128x160; 43 and 49 us by the table) 7.51 -> 7.31 ms, 3024 8.17 -> 7.93.  One image of 1024 rows has
// 256 small tiles that are 30 to 50 % faster, and keeps them.  Not so with row sums, where it goes either way (Qwen2.5-VL 1600
// patches 4.17 -> 4.14, 1764 4.22 -> 4.34, 1936 4.27 -> 4.13) and the few-row forms stay; nor with fp8 weights, where the big form
// is slower by more than that (2700 patches 5.78 -> 6.06).  A hint that the big form has no time for either, as that for the
// merger's 52 MB, would only make its launch longer.  Smaller tiles read it with the ring, and the line is the same for them: a product
// and the one that its hint of 4 MB is for, K = 2048, both with weights from HBM, 128x160 | 64x80 for the first: 2048 rows x 1152 36.7 | 39.1 us,
// 1280 x 1920 35.6 | 38.9, 832 x 2560 31.0 | 34.4, 1664 x 1280 35.7 | 35.7 (of the encoders' products only those of 128x128 tiles come this near).
constexpr double HINT_WORTH = 0.15;
bool loses_hint(const Form& f, const CsGemmArgs& a, double big_us, int64_t big_tiles) {
  if (!a.prefetch || a.prefetch_bytes < 16 || a.w_fp8 || a.c_row_sumsq || tiles_of(f, a) <= csgemm::HINT_MAX_TILES) return false;
  return big_tiles <= csgemm::HINT_MAX_TILES && a.prefetch_bytes <= csgemm::hint_workgroups((int)big_tiles) * 8192.0 * big_us;
}

// The form of a launch and its time, nullptr if it is not a few-row one.
const Form* few_row_form(const CsGemmArgs& a, double* us) {
  if (a.K % 128 || a.a_row_sumsq || a.a_row_sum || a.conv_patch) return nullptr;
  const Form* f;
  if (a.c_row_sumsq) {   // (other producers of row sums: the big tiles' 160-column forms)
    if (a.w_fp8 || a.epilogue != CS_EPI_RESIDUAL || !a.c_lo || a.N > 160 * CS_SUMSQ_PARTS) return nullptr;
    f = best_form(SUMS_FORMS, a, us);
  } else {
    if (a.a_norm_inline && (!csgemm::inline_norm_width(a.K) || a.w_fp8 || a.pos)) return nullptr;
    f = best_form(FORMS, a, us);
    if (a.a_norm_inline) return f;
  }
  if (!f) return nullptr;
  int64_t big_tiles;
  const double big_us = fast_us(a, &big_tiles);
  return *us < big_us * (loses_hint(*f, a, big_us, big_tiles) ? 1.0 - HINT_WORTH : 1.0) ? f : nullptr;
}

}  // namespace

// Called by cs_gemm for a shape that the direct-to-LDS kernels take (see cs_gemm_fast).  Sets *handled when the launch goes
// to the few-row kernel.
int cs_gemm_small(const CsGemmArgs& a, hipStream_t stream, bool* handled) {
  double us;
  const Form* f = few_row_form(a, &us);
  *handled = f != nullptr;
  if (!f) return CS_OK;
  CsGemmArgs p = a;
  csgemm::fit_hint(p, tiles_of(*f, a), us);
  return f->run(p, stream);
}

double cs_gemm_small_us(const CsGemmArgs& a) {
  double us;
  return few_row_form(a, &us) ? us : 0;
}

// Workgroups of such a launch, 0 if the big tiles take it.
int cs_gemm_small_workgroups(const CsGemmArgs& a) {
  double us;
  const Form* f = few_row_form(a, &us);
  if (!f) return 0;
  const int tiles = tiles_of(*f, a);
  CsGemmArgs p = a;
  csgemm::fit_hint(p, tiles, us);
  return tiles + (p.prefetch ? csgemm::hint_workgroups(tiles) : 0);
}

// One workgroup per window and head while the chip holds them all at once: 23 to 25 us up to 16 windows of 16 heads (inline norm,
// weights from HBM; 21 to 24 without norm), where a big tile (four windows) takes 32 to 35 us whatever the count; with a second
// round (24 windows: 39 us) it is the slower.  (The first 512 rows of bf16 weights go to two launches where there is a workspace, see
// below.)
bool cs_qkv_window_attn_few(int64_t windows, int heads, int K) { return K % 128 == 0 && windows * heads <= 256; }

// Of these the ones that two launches over a workspace serve better (gemm_small_qkv_wattn.hip): while the projection's tiles are
// one round.  One launch | two, 16 heads, K = 1280, weights from HBM, inline norm: 128 rows 24.8 | 16.0 us, 256 24.0 | 18.0, 320
// 23.7 | 21.3, 512 23.5 | 23.0 (64x128 tiles from 257 rows on); when one launch took 25.1 to 25.4, whole passes of Qwen2.5-VL, 256 patches 2.10 | 1.86 ms, 576 2.71 |
// 2.66.  Not with fp8 weights, half the bytes: 96 rows 14.8 | 12.9 us, 192 14.8 | 14.8, and at up to 128 rows, where it would be
// faster, a pass lasts as long as the host takes to launch it (1.87 | 1.90 ms).
bool cs_qkv_window_attn_two_pays(int64_t rows, int64_t windows, int heads, int K, bool w_fp8) {
  return !w_fp8 && cs_qkv_window_attn_few(windows, heads, K) && (rows + 63) / 64 * (heads * 2) <= 256;
}

// (Compared with the big forms as a SwiGLU launch would take them, a folded LayerNorm's among others 256x256, which it does not
// have, so it says no too early rather than too late: passes with the rule | both | neither inline, Qwen3-VL 256 patches 1.95 | 1.94 | 2.68 ms, 576 2.62 |
// 2.54 | 2.87, 896 3.17 | 2.94 | 3.17, 1280 4.03 | 4.59 | 4.03; Qwen2.5-VL 256 2.12 | 2.12 | 2.59, 432 2.57 | 2.42 | 2.61, 576 2.78 |
// 2.74 | 2.76, 896 2.95 | 3.24 | 2.93, 1280 3.89 | 4.60 | 3.88.)
extern "C" int cs_gemm_norm_inline_pays(int32_t M, int32_t N, int32_t K, int32_t window_attn) {
  if (M < 1 || N < 8 || N % 8 || K < 192 || !csgemm::inline_norm_width(K)) return 0;
  if (window_attn) return cs_qkv_window_attn_few(M / 64, N / 256, K) ? 1 : 0;
  CsGemmArgs a = {};
  a.M = M;
  a.N = N;
  a.K = K;
  a.a_norm_inline = 1;
  double us;
  best_form(FORMS, a, &us);
  a.a_norm_inline = 0;
  a.epilogue = CS_EPI_SWIGLU;
  int64_t big_tiles;
  return us < fast_us(a, &big_tiles) ? 1 : 0;
}
