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
double cs_gemm_small_us(const CsGemmArgs& a);   // its time if it is the one to take a launch, else 0

namespace {

using csgemm::BK;

// Time of a launch in microseconds: LAUNCH_US; per round of 256 tiles, and per K tile of 64, `stage` plus `flow` times the share of the
// compute units that have a tile (full launches draw more power and more bandwidth); and what the epilogues add -- per round: bias
// alone, SwiGLU, another activation, a folded LayerNorm; residual products: the first round and each further one.  Fitted to 27 products of the encoders at up to 34 row counts from 1100 to 20000, every
// form that takes them, weights from HBM (about 3,700 launches; root mean square error 2 to 3 % with fp8 weights, 8 to 10 % with
// bf16 ones, most of it common to all forms of a product); the residual entries anew since those products have a workgroup per ring-fed
// tile and a fast epilogue at edges (1,100 launches, 1500 to 24576 rows; 2 to 4 % with fp8 weights, 3 to 9 % with bf16 ones).  A launch is as long as its rounds, and a round as long as a tile of its form however
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
    {256, 256, {5.7f, 6.1f, 11.8f, NONE, 17.2f, 20.9f, 0.99f, 0.38f}, {6.5f, 6.0f, 8.6f, NONE, 17.4f, 21.3f, 1.08f, 0.29f}, cs_gemm_fast_tile_256x256},
    {256, 160, {4.2f, 4.4f, 8.4f, 6.5f, 7.8f, 10.3f, 0.61f, 0.30f}, {5.0f, 4.6f, 6.4f, NONE, 9.5f, 8.7f, 0.85f, 0.19f}, cs_gemm_fast_tile_256x160},
    {256, 128, {2.9f, 3.6f, 6.3f, 5.4f, 7.4f, 9.7f, 0.55f, 0.25f}, {3.7f, 3.3f, 4.7f, NONE, 8.6f, 9.2f, 0.59f, 0.20f}, cs_gemm_fast_tile_256x128},
    {224, 192, {4.4f, 4.7f, 8.6f, 7.0f, 12.6f, 14.2f, 0.67f, 0.28f}, {4.7f, 4.4f, 6.2f, NONE, 14.2f, 14.3f, 0.75f, 0.22f}, cs_gemm_fast_tile_224x192},
    {192, 192, {3.7f, 4.2f, 7.5f, 6.1f, 8.4f, 10.5f, 0.62f, 0.23f}, {4.1f, 3.8f, 5.0f, NONE, 10.4f, 10.6f, 0.68f, 0.19f}, cs_gemm_fast_tile_192x192},
    {192, 160, {3.1f, 3.5f, 6.5f, 4.9f, 4.9f, 7.5f, 0.52f, 0.22f}, {3.6f, 3.0f, 4.5f, NONE, 5.9f, 5.9f, 0.73f, 0.14f}, cs_gemm_fast_tile_192x160},
    {128, 192, {1.5f, 2.3f, 4.3f, 3.1f, 2.7f, 4.9f, 0.48f, 0.19f}, {3.1f, 2.8f, 3.7f, NONE, 5.1f, 5.4f, 0.56f, 0.12f}, cs_gemm_fast_tile_128x192},
    {128, 160, {1.3f, 2.0f, 3.9f, 2.7f, 2.4f, 4.2f, 0.41f, 0.20f}, {NONE, NONE, NONE, NONE, 5.9f, 5.6f, 0.57f, 0.09f}, cs_gemm_fast_tile_128x160},
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

// The arguments of the launch over rows m0 .. m0 + rows - 1 and columns n0 .. n0 + cols - 1 of C.
CsGemmArgs part_of(const CsGemmArgs& a, int m0, int rows, int n0, int cols) {
  CsGemmArgs p = a;
  p.M = rows;
  p.N = cols;
  auto at = [](const auto* base, int64_t bytes) { return base ? (const char*)base + bytes : nullptr; };
  // (scattered rows: the map moves, and C and what is stored beside it stay)
  const int64_t crow = a.c_rows ? 0 : m0, ncol = a.epilogue == CS_EPI_SWIGLU ? n0 / 2 : n0;
  p.A = at(a.A, (int64_t)m0 * a.lda * 2);
  p.W = at(a.W, (int64_t)n0 * a.ldw * (a.w_fp8 ? 1 : 2));
  p.w_scale = (const float*)at(a.w_scale, (int64_t)n0 * 4);
  p.w_col_sum = (const float*)at(a.w_col_sum, (int64_t)n0 * 4);
  p.bias = at(a.bias, (int64_t)n0 * 2);
  p.residual = at(a.residual, ((int64_t)m0 * a.ldr + n0) * 2);
  p.residual_lo = (const uint8_t*)at(a.residual_lo, (int64_t)m0 * a.ldr + n0);
  p.pos = at(a.pos, (int64_t)n0 * 2);
  p.C = (char*)a.C + (crow * a.ldc + ncol) * 2;
  p.c_lo = (uint8_t*)at(a.c_lo, crow * a.ldc + ncol);
  p.c_rows = (const int32_t*)at(a.c_rows, (int64_t)m0 * 4);
  const int64_t parts = CS_SUMSQ_PARTS * 4;
  p.a_row_sumsq = (const float*)at(a.a_row_sumsq, m0 * parts);
  p.a_row_sum = (const float*)at(a.a_row_sum, m0 * parts);
  p.c_row_sumsq = (float*)at(a.c_row_sumsq, crow * parts);
  p.c_row_sum = (float*)at(a.c_row_sum, crow * parts);
  return p;
}

// How a launch is made: `form` alone (lead_cols == lead_rows == 0); 256x256 tiles over the first lead_cols columns, which fill
// whole rounds or nearly, and `form` over the rest in a launch of its own; or `lead` over the first lead_rows rows likewise and,
// over the others, the few-row kernel (form == nullptr) or `form`.
constexpr float ROW_SPLIT_US = 3.0f;
struct Plan {
  const BigForm* form;
  int lead_cols;
  double us;
  int lead_rows;
  const BigForm* lead;
};
Plan plan_of(const CsGemmArgs& a) {
  Plan p = {nullptr, 0, 0, 0, nullptr};
  p.form = best_form(a, a.N, &p.us);
  if (tiles_of(*p.form, a.M, a.N) <= 256) return p;   // (one round: nothing to split)
  Plan split = p;
  if (takes(FORMS[0], a) && !a.c_row_sumsq) {
    const int tn = (a.N + 255) / 256;
    for (int c = tn - 1; c >= 1 && c >= tn - 12; --c) {
      double tail_us = 0;
      const BigForm* tail = best_form(a, a.N - c * 256, &tail_us);
      const double t = form_us(FORMS[0], a, c * 256) + tail_us;
      if (tail != &FORMS[0] && t < split.us) split = {tail, c * 256, t, 0, nullptr};
    }
  }
  // Rows behind the last whole round of a form's tiles cost a round of their own, however few they are; in a second launch they take
  // the form that suits so many rows.  One launch -> two, row sums, K = 1280 / 3456: 8800 rows x 1280 48.1 / 85.0 -> 43.1 / 76.8 us,
  // 20480 87.4 / 177.5 -> 74.7 / 165.8, 58648 266 / 508 -> 259 / 480; fp8 SwiGLU 17000 rows x 6912 x 1280 258 -> 236; GELU 12393 rows
  // x 4352 x 1152 121.2 -> 115.6.  ROW_SPLIT_US on top of both launches' estimates, but for residual products led by 160-column
  // tiles, whose times are the surest: without it 5400 rows x 6912 x 1280 (87.9 -> 90.0), 6240 x 4352 x 1152 (62.8 -> 65.1) and the fp8
  // residual product 19200 x 1280 x 1280 (77.6 -> 80.2) are split too.  (A position addend counts rows from the matrix's first.)
  // Over 960 launches (15 products, 64 row counts each from 2700 to 28000, one launch in every form and two in every pair of forms timed)
  // the choice takes 1.006 of the best of them in the mean, 1.04 at 95 %, 1.11 at worst; without row splits 1.013, 1.07 and 1.26.  With 0 us
  // for ROW_SPLIT_US 1.005, with 3 us for all products 1.008.  A few-row tail counts what its own table says: at 1.33 of that, which one shape
  // asks for (9792 x 1152 x 4352, 91.9 us so, 93.6 now), 27 launches are planned otherwise and 23 of them are slower: 27184 rows x 1280 x 5120
  // 317 -> 365 us, fp8 SwiGLU 7252 x 6912 x 1280 109 -> 122, row sums 25504 x 1280 x 1280 100 -> 104.  (A row split has to promise 3 % more
  // than a column split: a choice, no measurement.  Without it 11 of these launches are planned otherwise, all 2 to 10 % faster.)
  const auto tight = [&](const BigForm& f) { return a.epilogue == CS_EPI_RESIDUAL && f.bn == 160; };
  if (!a.pos) {
    for (const BigForm& f : FORMS) {
      if (!takes(f, a)) continue;
      const int tn = (a.N + f.bn - 1) / f.bn, whole = (int)(tiles_of(f, a.M, a.N) / 256);
      const int lead = (int)((int64_t)whole * 256 / tn) * f.bm;
      if (lead <= 0 || lead >= a.M) continue;
      const double lead_us = form_us(f, part_of(a, 0, lead, 0, a.N), a.N);
      if (lead_us >= split.us) continue;
      const CsGemmArgs rest = part_of(a, lead, a.M - lead, 0, a.N);
      double t;
      const double few = cs_gemm_small_us(rest);
      const BigForm* form = best_form(rest, a.N, &t);
      if (few > 0 && few < t) {
        t = few;
        form = nullptr;
      }
      t += lead_us + (tight(f) ? 0.0 : ROW_SPLIT_US);
      if (t < (split.lead_cols ? 0.97 : 1.0) * split.us) split = {form, 0, t, lead, &f};
    }
  }
  // (for a clear gain only: 4096 rows x 6912 x 1280 take 65 us as 256x256 in two rounds, and 72 in two launches of the same estimate)
  return split.us < (split.lead_rows && tight(*split.lead) ? 0.98 : 0.96) * p.us ? split : p;
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
  const BigForm* form = p.lead_rows ? p.lead : p.form;
  plan[0] = form->bm;
  plan[1] = form->bn;
  plan[2] = p.lead_cols;
  return CS_OK;
}

extern "C" int cs_gemm_lead_rows(const CsGemmArgs* args) {
  if (!args || args->conv_patch || args->a_norm_inline || !direct_shape(*args) || cs_gemm_small_workgroups(*args)) return 0;
  return plan_of(*args).lead_rows;
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
  if (plan.lead_rows) {
    CsGemmArgs lead = part_of(a, 0, plan.lead_rows, 0, a.N);
    lead.prefetch = nullptr;  // (the hint stays with the tail, whose few tiles leave compute units idle; the lead could read it with its ring)
    const CsGemmArgs rest = part_of(a, plan.lead_rows, a.M - plan.lead_rows, 0, a.N);
    const int st = plan.lead->run(lead, stream);
    if (st != CS_OK) return st;
    if (plan.form) return plan.form->run(rest, stream);
    bool taken;
    const int st_rest = cs_gemm_small(rest, stream, &taken);
    return taken ? st_rest : CS_ERR_UNSUPPORTED;   // (it is the one to take them: plan_of asked)
  }
  if (plan.lead_cols == 0) return plan.form->run(a, stream);
  // two launches that write disjoint column ranges of C
  CsGemmArgs lead = part_of(a, 0, a.M, 0, plan.lead_cols);
  lead.prefetch = nullptr;
  const int st = FORMS[0].run(lead, stream);
  return st != CS_OK ? st : plan.form->run(part_of(a, 0, a.M, plan.lead_cols, a.N - plan.lead_cols), stream);
}

// For the few-row kernel's choice: the time of a launch as a share of what the best of 256x256, 256x128 (SwiGLU), and 256x160 or, for at
// most 128 tiles of it, 128x160 would take, of those that take the launch; and the tiles of its (last) launch.  1 where 128x160 is the
// one to compare with and is not built: with fp8 weights, but for residual products, whose big tiles take longer than the times
// that the share is of, in gemm_small.hip, so that the few-row kernel was never the slower one where it was chosen.
double cs_gemm_fast_saves(const CsGemmArgs& a, int64_t* tiles) {
  const Plan p = plan_of(a);
  *tiles = p.form ? tiles_of(*p.form, a.M - p.lead_rows, a.N - p.lead_cols)
                  : cs_gemm_small_workgroups(part_of(a, p.lead_rows, a.M - p.lead_rows, 0, a.N));
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
