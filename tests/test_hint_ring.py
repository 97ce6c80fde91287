"""What a full launch reads of its prefetch hint with the ring's own loads (csrc/hint_ring.h): every load of a launch is gone through on
the host, in the order in which the kernel's last iterations request them, and the bytes are counted."""

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "cornserve_amd" / "csrc"

_PRELUDE = r"""
#include "hint_ring.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace cshint;
// Of `bytes` hinted ones, read by `workgroups` of `waves` waves: the leading whole rows that the workgroups' loads cover are read once
// each, and nothing else.  `requests(f)` calls f(segment, load) for everything requested behind the last K tile.
template <class Requests, class Offset>
void check(const char* what, int64_t bytes, int workgroups, int waves, int segment, int segments, int most, Requests requests, Offset offset) {
  const int pitch = segment * segments, rows = rows_of(bytes, pitch, workgroups, most);
  std::vector<unsigned char> times(bytes, 0);
  int64_t covered = 0;
  for (int g = 0; g < workgroups; ++g) {
    const Share s = share_of((uint32_t)bytes, pitch, rows, g);
    covered += (int64_t)s.rows * pitch;
    for (int wave = 0; wave < waves; ++wave)
      requests([&](int seg, int load) {
        for (int lane = 0; lane < 64; ++lane) {
          const uint32_t off = offset(wave, load, lane);
          if (off >= (uint32_t)(s.rows * pitch)) continue;   // (behind the descriptor's end; the K tile's offset is not compared with it)
          const int64_t at = (int64_t)s.first * pitch + off + seg * segment;
          for (int b = 0; b < 16; ++b) {
            if (at + b >= bytes) { printf("%s, %ld bytes: byte %ld is read\n", what, (long)bytes, (long)(at + b)); exit(1); }
            ++times[at + b];
          }
        }
      });
  }
  if (covered != bytes_of(bytes, pitch, workgroups, most)) { printf("%s, %ld bytes: %ld in shares\n", what, (long)bytes, (long)covered); exit(1); }
  for (int64_t i = 0; i < bytes; ++i)
    if (times[i] != (i < covered)) { printf("%s, %ld bytes: byte %ld is read %d times\n", what, (long)bytes, (long)i, times[i]); exit(1); }
}
"""

# the last ahead_b() iterations of a workgroup's last tile; the sources move before the first load of the hint
_BIG = r"""
int main() {
  const int forms[][2] = {{256, 256}, {256, 160}, {256, 128}, {224, 192}, {192, 192}, {192, 160}, {128, 192}, {128, 160}};
  for (auto& f : forms)
    for (int fp8 = 0; fp8 < 2; ++fp8) {
      const int bm = f[0], bn = f[1];
      const BigRing r = {bm / 32, (bn / (fp8 ? 16 : 8) + 3) / 4, bm == 256 && bn == 256 && !fp8};
      auto requests = [&](auto&& read) {
        for (int tail = r.ahead_b(); tail >= 1; --tail) {
          if (r.ahead_a() >= tail)
            for (int n = 0; n < r.pa(); ++n)
              if (r.pa_first() + n < big_loads(r, fp8)) read(r.ahead_a() - tail, r.pa_first() + n);
          if (r.ahead_b() >= tail && r.ahead_b() - tail < BIG_SEGMENTS)
            for (int n = 0; n < r.pb(); ++n)
              if (r.pb_first() + n < big_loads(r, fp8)) read(r.ahead_b() - tail, r.pb_first() + n);
        }
      };
      char what[64];
      snprintf(what, sizeof what, "%dx%d %s", bm, bn, fp8 ? "fp8" : "bf16");
      for (int64_t bytes : {16l, 1000l, 256l * 193, 1000016l, 9l << 20, 16l << 20})
        for (int workgroups : {193, 224, 256})
          check(what, bytes, workgroups, 4, BIG_SEGMENT, BIG_SEGMENTS, big_rows(r, fp8), requests,
                [&](int wave, int load, int lane) { return big_offset(r, fp8, wave, load, lane); });
    }
}
"""

# a few-row launch's iterations in order, with the sources moved behind the top of iteration nst - stages
_FEW_ROWS = r"""
int main() {
  const int forms[][5] = {{32, 32, 4, 2, 8}, {32, 64, 4, 2, 6}, {64, 64, 8, 2, 4}, {64, 80, 4, 2, 4}, {64, 128, 8, 2, 3}, {32, 160, 4, 2, 3},
                          {64, 160, 8, 1, 4}, {64, 240, 4, 1, 4}};
  for (auto& f : forms) {
    const int bm = f[0], bn = f[1], waves = f[2], ks = f[3], stages = f[4];
    const int nld = ks * (bm / 8) / waves + (ks * (bn / 8) + waves - 1) / waves;
    for (int nst : {stages, stages + 2}) {
      if (ks == 1 && nst % 2) continue;
      auto requests = [&](auto&& read) {
        for (int kt = 0; kt < nst; ++kt) {
          const bool steady = kt < small_steady(ks, stages, nst, true);
          auto loads = [&](int stage, int from, int to) {
            if (stage < nst) return;
            if (stage - nst >= small_segments(ks, stages)) { printf("stage %d of %d\n", stage, nst); exit(1); }
            for (int n = from; n < to; ++n) read(stage - nst, n);
          };
          if (ks == 2) {
            if (steady || small_second_half(kt, stages, nst, true)) loads(kt + stages - 1, nld / 2, nld);
            if (steady) loads(kt + stages, 0, nld / 2);
          } else if (steady) {
            loads(kt + stages, 0, nld);
          }
        }
      };
      char what[64];
      snprintf(what, sizeof what, "%dx%d, %d stages", bm, bn, nst);
      for (int64_t bytes : {16l, 1000l, 768l * 193, 1000016l, 20l << 20})
        for (int workgroups : {193, 256, 480})
          check(what, bytes, workgroups, waves, small_segment(ks), small_segments(ks, stages), small_rows(ks, waves, nld), requests,
                [&](int wave, int load, int lane) { return small_offset(ks, stages, nld, wave, load, lane); });
    }
  }
}
"""


@pytest.mark.parametrize("kernel,main", [pytest.param("big", _BIG, id="big tiles"), pytest.param("few", _FEW_ROWS, id="few rows")])
def test_the_ring_reads_every_byte_of_its_share_once(tmp_path, kernel, main):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / f"{kernel}.cpp", tmp_path / kernel
    src.write_text(_PRELUDE + main)
    subprocess.run([gxx, "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert run.returncode == 0, run.stdout
