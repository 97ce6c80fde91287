// What the computing workgroups of a full launch read of its prefetch hint (CsGemmArgs.prefetch) with the ring's own loads, behind
// their last K tile: which loads of which K tile are still requested there, and the byte each lane of them takes.  Plain C++ that the
// kernels and their launchers share with a host-side check, which goes through every load of a launch and counts the bytes.
#pragma once
#include <cstdint>

namespace cshint {

// A hint is cut into rows of `pitch` bytes: one segment for each K tile that is requested WHOLE behind the last one.  A lane keeps its row
// and its place in it, and the K tiles walk along the row.  A workgroup's rows follow each other, at most `most` of them.
struct Share {
  int first, rows;   // of a workgroup
};
constexpr int rows_of(int64_t bytes, int pitch, int workgroups, int most) {
  const int64_t share = (bytes / pitch + workgroups - 1) / workgroups;
  return (int)(share < most ? share : most);
}
constexpr int64_t bytes_of(int64_t bytes, int pitch, int workgroups, int most) {   // what all of them read, from the hint's start
  const int64_t whole = bytes / pitch, reach = (int64_t)workgroups * most;
  return (whole < reach ? whole : reach) * pitch;
}
constexpr Share share_of(uint32_t bytes, int pitch, int hint_rows, int workgroup) {
  const int first = workgroup * hint_rows, left = (int)(bytes / (uint32_t)pitch) - first;
  return {first, left < 0 ? 0 : left < hint_rows ? left : hint_rows};
}

// ---- The big tiles (gemm_fast_impl.h).  The direct loads of a wave and K tile, activation rows first, go in two portions, one in each
// half of an iteration.  Five-unit ring: A(kt+2) in the first half, W(kt+2) in the second.  Three-stage ring: the second portion
// of K tile kt+2 in the first half, the first portion of K tile kt+3 in the second half.
struct BigRing {
  int a_ld, w_ld;
  bool five_units;
  constexpr int nld() const { return a_ld + w_ld; }
  constexpr int pa() const { return five_units ? a_ld : nld() - nld() / 2; }   // loads issued in a first half
  constexpr int pb() const { return nld() - pa(); }                            // ... in a second half
  constexpr int pa_first() const { return five_units ? 0 : pb(); }
  constexpr int pb_first() const { return five_units ? a_ld : 0; }
  constexpr int ahead_a() const { return 2; }
  constexpr int ahead_b() const { return five_units ? 2 : 3; }
};
// K tiles 0 and 1 behind the last one are requested whole by either ring; of K tile 2 the three-stage ring would request the first
// portion, and leaves it.
constexpr int BIG_SEGMENT = 128, BIG_SEGMENTS = 2, BIG_PITCH = BIG_SEGMENTS * BIG_SEGMENT;
// Rows that a workgroup of four waves covers.  (With fp8 weights only the activations' loads take part: the others' rows are half as wide.)
constexpr int big_loads(const BigRing& r, bool w_fp8) { return w_fp8 ? r.a_ld : r.nld(); }
constexpr int big_rows(const BigRing& r, bool w_fp8) { return 4 * big_loads(r, w_fp8) * 8; }
constexpr uint32_t big_offset(const BigRing& r, bool w_fp8, int wave, int load, int lane) {   // eight lanes to a segment
  return (uint32_t)(((wave * big_loads(r, w_fp8) + load) * 8 + (lane >> 3)) * BIG_PITCH + (lane & 7) * 16);
}

// ---- The few-row kernel (gemm_small_impl.h): a ring of `stages` slots, `ks` K tiles of 64 to a stage, `nst` stages of the matrix.  ks 1:
// iteration kt requests stage kt + stages whole, but for the last two (K tiles go in pairs), which request nothing.  ks 2: its loads'
// first half behind the barrier of iteration kt, the second half at the top of iteration kt + 1; the last iteration, which has no
// barrier, completes a stage of the hint.
constexpr int small_segment(int ks) { return ks * 128; }
constexpr int small_segments(int ks, int stages) { return ks == 2 ? stages - 1 : stages - 2; }
constexpr int small_steady(int ks, int stages, int nst, bool hint) {   // iterations that begin a stage
  return ks == 2 ? (hint ? nst - 1 : nst - stages) : (hint ? nst - 2 : nst - stages - 1);
}
// (ks 2) whether iteration kt requests the second half of stage kt + stages - 1
constexpr bool small_second_half(int kt, int stages, int nst, bool hint) { return hint || kt + stages - 1 < nst; }
constexpr int small_rows(int ks, int waves, int nld) { return waves * nld * (1024 / small_segment(ks)); }
constexpr uint32_t small_offset(int ks, int stages, int nld, int wave, int load, int lane) {   // a segment is 8 ks lanes
  return (uint32_t)((lane / (8 * ks) + (wave * nld + load) * (8 / ks)) * (small_segments(ks, stages) * small_segment(ks)) + lane % (8 * ks) * 16);
}

}  // namespace cshint
