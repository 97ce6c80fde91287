// Fast-path bf16 MFMA GEMM for gfx950: choice of the tile form.  The kernel itself is in gemm_fast_impl.h; each tile
// form is built in its own translation unit (gemm_fast_t*.hip).
#include <math.h>
#include <stdlib.h>

#include "gemm_common.h"

// Epilogue / folded-norm dispatch of one tile form each (gemm_fast_t<rows>x<cols>.hip).
int cs_gemm_fast_tile_256x256(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_fast_tile_256x160(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_fast_tile_256x128(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_fast_tile_224x192(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_fast_tile_192x192(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_fast_tile_192x160(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_fast_tile_128x192(const CsGemmArgs& a, hipStream_t stream);
int cs_gemm_fast_tile_128x160(const CsGemmArgs& a, hipStream_t stream);
// The few-row kernel (gemm_small.hip).
int cs_gemm_small(const CsGemmArgs& a, hipStream_t stream, bool* handled);
int cs_gemm_small_workgroups(const CsGemmArgs& a);

namespace {

using csgemm::BK;

// Time of a launch in microseconds: LAUNCH_US; per round of 256 tiles, and per K tile of 64, `stage` plus `flow` times the share of the
// compute units that have a tile (full launches draw more power and more bandwidth); and what the epilogues add -- per round: bias
// alone, SwiGLU, another activation, a folded LayerNorm; residual products: the workgroup's last tile, whose residual piece came
// through the ring, and the tiles before it.  Fitted to 27 products of the encoders at up to 34 row counts from 1100 to 20000, every
// form that takes them, weights from HBM (about 3,700 launches; root mean square error 2 to 3 % with fp8 weights, 8 to 10 % with
// bf16 ones, most of it common to all forms of a product), before edge tiles of residual products took the fast epilogue (3 to 7 us
// less than their entries say, in every form).  A launch is as long as its rounds, and a round as long as a tile of its form however
// few of the 256 compute units have one, so what counts is a form whose tiles fill whole rounds: 6240 rows x 3456 (folded
// LayerNorm) are 550 tiles of 256x160 in three rounds, 62.8 us, and 504 of 224x192 in two, 49.2 us.  Chosen by this table, launches
// take 1.009 of the time of the best form on average (33 products at 24 to 34 row counts on the present kernels; residual
// products from 2500 rows on, the others from 1000; the worst 1.10); with five forms (256x256, 256x160 and its 128-row half, 256x128
// and 128x192 behind whole rounds of 256x256) and tile area as the cost they took 1.062.
struct FormUs {
  float bias, swiglu, act, ln, res, res_more, stage, flow;
};
struct BigForm {
  int bm, bn;
  FormUs bf16, fp8;
  int (*run)(const CsGemmArgs&, hipStream_t);
};
constexpr float LAUNCH_US = 3.0f;
constexpr float NONE = INFINITY;   // not built: no launch may be costed with it (takes() below)
const BigForm FORMS[] = {
    {256, 256, {5.7f, 6.1f, 11.8f, NONE, 18.9f, 21.3f, 0.99f, 0.38f}, {6.5f, 6.0f, 8.6f, NONE, 20.2f, 18.9f, 1.08f, 0.29f}, cs_gemm_fast_tile_256x256},
    {256, 160, {4.2f, 4.4f, 8.4f, 6.5f, 12.1f, 12.9f, 0.61f, 0.30f}, {5.0f, 4.6f, 6.4f, NONE, 11.9f, 12.3f, 0.85f, 0.19f}, cs_gemm_fast_tile_256x160},
    {256, 128, {2.9f, 3.6f, 6.3f, 5.4f, 9.1f, 8.6f, 0.55f, 0.25f}, {3.7f, 3.3f, 4.7f, NONE, 10.5f, 8.9f, 0.59f, 0.20f}, cs_gemm_fast_tile_256x128},
    {224, 192, {4.4f, 4.7f, 8.6f, 7.0f, 14.5f, 13.9f, 0.67f, 0.28f}, {4.7f, 4.4f, 6.2f, NONE, 17.4f, 13.5f, 0.75f, 0.22f}, cs_gemm_fast_tile_224x192},
    {192, 192, {3.7f, 4.2f, 7.5f, 6.1f, 11.1f, 10.1f, 0.62f, 0.23f}, {4.1f, 3.8f, 5.0f, NONE, 14.1f, 10.0f, 0.68f, 0.19f}, cs_gemm_fast_tile_192x192},
    {192, 160, {3.1f, 3.5f, 6.5f, 4.9f, 9.1f, 9.7f, 0.52f, 0.22f}, {3.6f, 3.0f, 4.5f, NONE, 9.3f, 9.4f, 0.73f, 0.14f}, cs_gemm_fast_tile_192x160},
    {128, 192, {1.5f, 2.3f, 4.3f, 3.1f, 6.7f, 5.7f, 0.48f, 0.19f}, {3.1f, 2.8f, 3.7f, NONE, 9.9f, 6.5f, 0.56f, 0.12f}, cs_gemm_fast_tile_128x192},
    {128, 160, {1.3f, 2.0f, 3.9f, 2.7f, 6.1f, 5.9f, 0.41f, 0.20f}, {NONE, NONE, NONE, NONE, 7.3f, 7.2f, 0.57f, 0.09f}, cs_gemm_fast_tile_128x160},
};

int64_t tiles_of(const BigForm& f, int M, int N) { return (int64_t)(((uint32_t)M + f.bm - 1) / (uint32_t)f.bm) * (((uint32_t)N + f.bn - 1) / (uint32_t)f.bn); }

double form_us(const BigForm& f, const CsGemmArgs& a, int N) {
  const FormUs& u = a.w_fp8 ? f.fp8 : f.bf16;
  const int64_t tiles = tiles_of(f, a.M, N);
  const double rounds = (double)((tiles + 255) / 256);
  const double k = (a.K / BK) * (rounds * u.stage + tiles / 256.0 * u.flow);
  if (a.epilogue == CS_EPI_RESIDUAL) return LAUNCH_US + k + u.res + (rounds - 1) * u.res_more;
  return LAUNCH_US + k + rounds * (a.a_row_sum ? u.ln : a.epilogue == CS_EPI_BIAS ? u.bias : a.epilogue == CS_EPI_SWIGLU ? u.swiglu : u.act);
}

// Row sums come in CS_SUMSQ_PARTS parts, one per column tile of the 160-column forms.  A folded LayerNorm's per-column sums do not fit
// the registers of 256x256, and of 128x160 with fp8 weights only the residual products are built (see dispatch_epi_w, dispatch_epi).
// The accumulation order of an output element, and of a row-sum part, is the same in every form: the choice changes no bit.
bool takes(const BigForm& f, const CsGemmArgs& a) {
  if (a.c_row_sumsq && f.bn != 160) return false;
  if (a.a_row_sum && f.bm == 256 && f.bn == 256) return false;
  return !(a.w_fp8 && f.bm == 128 && f.bn == 160 && a.epilogue != CS_EPI_RESIDUAL);
}

// The form for the first N columns, and its time.
const BigForm* best_form(const CsGemmArgs& a, int N, double* us) {
  const BigForm* best = nullptr;
  for (const BigForm& f : FORMS) {
    if (!takes(f, a)) continue;
    const double t = form_us(f, a, N);
    if (!best || t < 0.98 * *us) {   // (largest tiles first; what is closer than this is a tie, and theirs)
      best = &f;
      *us = t;
    }
  }
  return best;
}

// How a launch is made: `form` alone (lead_cols == 0), or 256x256 tiles over the first lead_cols columns, which fill whole rounds or
// nearly, and `form` over the rest in a launch of its own.
struct Plan {
  const BigForm* form;
  int lead_cols;
  double us;
};
Plan plan_of(const CsGemmArgs& a) {
  Plan p = {nullptr, 0, 0};
  p.form = best_form(a, a.N, &p.us);
  if (tiles_of(*p.form, a.M, a.N) <= 256 || !takes(FORMS[0], a) || a.c_row_sumsq) return p;   // (one round: nothing to split)
  Plan split = p;
  const int tn = (a.N + 255) / 256;
  for (int c = tn - 1; c >= 1 && c >= tn - 12; --c) {
    double tail_us = 0;
    const BigForm* tail = best_form(a, a.N - c * 256, &tail_us);
    const double t = form_us(FORMS[0], a, c * 256) + tail_us;
    if (tail != &FORMS[0] && t < split.us) split = {tail, c * 256, t};
  }
  // (for a clear gain only: 4096 rows x 6912 x 1280 take 65 us as 256x256 in two rounds, and 72 in two launches of the same estimate)
  return split.us < 0.96 * p.us ? split : p;
}

// Whether the direct-to-LDS kernels (the big tiles and the few-row kernel) take a problem.
bool direct_shape(const CsGemmArgs& a) {
  if (a.M < 1 || a.N < 8) return false;
  if (a.w_fp8 ? (!a.w_scale || a.pos) : (a.w_scale != nullptr)) return false;
  if (a.K % BK || a.K < 3 * BK) return false;  // the ring pipeline is written for at least three K tiles
  if (a.N % 8 || a.ldc % 8 || ((uintptr_t)a.C & 15)) return false;  // 16-byte output stores
  if (a.pos && a.epilogue != CS_EPI_BIAS) return false;  // the position addend only pairs with the plain epilogue here
  if (a.a_rows) return false;  // gathered A rows can lie anywhere: the general kernel keeps 64-bit pointers
  // per-lane source offsets are 32-bit byte offsets from the matrix bases
  return (int64_t)a.M * a.lda * 2 < (int64_t)UINT32_MAX && (int64_t)a.N * a.ldw * (a.w_fp8 ? 1 : 2) < (int64_t)UINT32_MAX;
}

}  // namespace

extern "C" int cs_gemm_few_row_workgroups(const CsGemmArgs* args) {
  return args && !args->conv_patch && direct_shape(*args) ? cs_gemm_small_workgroups(*args) : 0;
}

extern "C" int cs_gemm_big_form(const CsGemmArgs* args, int32_t plan[3]) {
  if (!args || !plan) return CS_ERR_INVALID_ARG;
  plan[0] = plan[1] = plan[2] = 0;
  if (args->conv_patch || args->a_norm_inline || !direct_shape(*args) || cs_gemm_small_workgroups(*args)) return CS_OK;
  const Plan p = plan_of(*args);
  plan[0] = p.form->bm;
  plan[1] = p.form->bn;
  plan[2] = p.lead_cols;
  return CS_OK;
}

// Called by cs_gemm after argument validation.  Sets *handled when this path took the problem.
int cs_gemm_fast(const CsGemmArgs& a, hipStream_t stream, bool* handled) {
  *handled = false;
  if (!direct_shape(a)) return CS_OK;
  // Few rows: tiles small enough to give most compute units one.
  {
    const int st = cs_gemm_small(a, stream, handled);
    if (*handled) return st;
  }
  *handled = true;
  if (a.a_norm_inline) return CS_ERR_UNSUPPORTED;   // the inline norms exist in the few-row kernel only
  if (a.c_row_sumsq && (a.N > CS_SUMSQ_PARTS * 160 || a.w_fp8)) return CS_ERR_UNSUPPORTED;
  const Plan plan = plan_of(a);
  if (plan.lead_cols == 0) return plan.form->run(a, stream);
  // two launches that write disjoint column ranges of C
  const int n1 = plan.lead_cols;
  CsGemmArgs lo = a, hi = a;
  lo.N = n1;
  lo.prefetch = nullptr;  // the tail launch is the one with idle compute units
  hi.N = a.N - n1;
  hi.W = (const char*)a.W + (int64_t)n1 * a.ldw * (a.w_fp8 ? 1 : 2);
  if (a.w_scale) hi.w_scale = a.w_scale + n1;
  if (a.bias) hi.bias = (const char*)a.bias + (int64_t)n1 * 2;
  if (a.residual) hi.residual = (const char*)a.residual + (int64_t)n1 * 2;
  if (a.residual_lo) hi.residual_lo = a.residual_lo + n1;
  if (a.c_lo) hi.c_lo = a.c_lo + n1;
  if (a.pos) hi.pos = (const char*)a.pos + (int64_t)n1 * 2;
  hi.C = (char*)a.C + (int64_t)(a.epilogue == CS_EPI_SWIGLU ? n1 / 2 : n1) * 2;
  const int st = FORMS[0].run(lo, stream);
  return st != CS_OK ? st : plan.form->run(hi, stream);
}

// For the few-row kernel's choice: the time of a launch as a share of what the best of 256x256, 256x128 (SwiGLU), and 256x160 or, for at
// most 128 tiles of it, 128x160 would take, of those that take the launch; and the tiles of its (last) launch.  1 where 128x160 is the
// one to compare with and is not built: with fp8 weights, but for residual products, whose big tiles take longer than the times
// that the share is of, in gemm_small.hip, so that the few-row kernel was never the slower one where it was chosen.
double cs_gemm_fast_saves(const CsGemmArgs& a, int64_t* tiles) {
  const Plan p = plan_of(a);
  *tiles = tiles_of(*p.form, a.M, a.N - p.lead_cols);
  const int narrow_rows = (int64_t)((a.M + 255) / 256) * ((a.N + 159) / 160) <= 128 ? 128 : 256;
  double of = 0;
  for (const BigForm& f : FORMS) {
    const bool narrow = f.bn == 160 && f.bm == narrow_rows;
    if (!takes(f, a)) {
      if (narrow) return 1.0;
      continue;
    }
    if (!narrow && !(f.bm == 256 && (f.bn == 256 || (f.bn == 128 && a.epilogue == CS_EPI_SWIGLU)))) continue;
    const double t = form_us(f, a, a.N);
    if (of == 0 || t < of) of = t;
  }
  return p.us < of ? p.us / of : 1.0;
}
