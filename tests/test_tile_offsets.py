"""Offsets of the power-of-two strided passes, on the CPU: every length,
elements per thread and value size, at the largest position pitch whose field
the element indices reach (2^31 values).

A pass addresses a value as a 64-bit base, uniform over the workgroup, plus a
32-bit byte offset of the lane into a buffer resource of kBufMax bytes, beyond
which loads read zero and stores are dropped.  The program below evaluates the
engine's own functions (fsx_tile.h) in a host build: the slots of the first
and last stage hold every position once, base and lane offset add up to the
position's address (whole and pruned axes), and no lane offset reaches
kBufMax.
"""

import shutil
import subprocess

import pytest

from fluidsim_amd.build import CSRC, hipcc

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "fsx_tile.h"
using namespace fsx;
static int bad = 0;
static void fail(const char* what, int logn, int loge, int bytes) {
  if (++bad < 20) std::printf("%s: N = 2^%d, E = 2^%d, %d bytes\n", what, logn, loge, bytes);
}

template <int LOGN, int LOGE, int S>
void stage(unsigned bytes) {
  constexpr int N = 1 << LOGN, E = 1 << LOGE;
  const int nl = 16;
  // the small form is not taken where its lanes would reach too far
  unsigned ps = (unsigned)(((1ull << 31) - 1) / N);
  if (LOGE == kSmallLogE && LOGN > kSmallLogE) {
    ps /= 4;
    if (small_loge(LOGN, LOGE + 1, 1, ps, bytes) != LOGE) fail("small form", LOGN, LOGE, bytes);
  }
  // a pruned axis, in memory or compact
  const int lo = N > 2 ? N / 2 - 1 : 1, hi = N / 4;
  const AxisMap whole{N, N / 2 + 1, N / 2 - 1}, pruned{N, lo, hi};
  const Lines sides[3] = {lines_of(ps, whole, false, nl), lines_of(ps, pruned, false, nl),
                          lines_of(ps, pruned, true, nl)};
  const unsigned long long reach = lane_reach(N, LOGE, ps, nl, bytes);
  if (reach >= kBufMax) fail("reach", LOGN, LOGE, bytes);
  std::vector<int> seen(N, 0);
  for (int j0 = 0; j0 < N / E; ++j0)
    for (int e = 0; e < E; ++e)
      for (int line = 0; line < nl; line += nl - 1) {
        const Slot t = tile_slot<LOGN, LOGE, S>(e, line, j0);
        const int p = t.pos();
        if (p < 0 || p >= N) {
          fail("position", LOGN, LOGE, bytes);
          continue;
        }
        if (line == 0) ++seen[p];
        for (int k = 0; k < 3; ++k) {
          const Lines& g = sides[k];
          const bool kept = k == 0 || p < lo || p >= N - hi;
          if (ln_kept<LOGN>(g, t) != kept) fail("kept", LOGN, LOGE, bytes);
          if (!kept) continue;
          const unsigned off = ln_lane(g, t, bytes);
          if (off > reach || off >= kBufMax) fail("lane offset", LOGN, LOGE, bytes);
          const int q = k < 2 || p < lo ? p : p - (N - lo - hi);
          const unsigned long long want = ((unsigned long long)q * ps + line) * bytes;
          if ((unsigned long long)ln_base<LOGN>(g, t) * bytes + off != want)
            fail("address", LOGN, LOGE, bytes);
        }
      }
  for (int p = 0; p < N; ++p)
    if (seen[p] != 1) fail("coverage", LOGN, LOGE, bytes);
}

template <int LOGN, int LOGE>
void plan(unsigned bytes) {
  stage<LOGN, LOGE, 0>(bytes);
  stage<LOGN, LOGE, TilePlan<LOGN, LOGE>::NS - 1>(bytes);
}

// Elements per thread the launcher takes for next to no lines of the largest
// field, and for many.
template <int LOGN>
void chosen(int loge, unsigned bytes) {
  const unsigned long long ps = ((1ull << 31) - 1) / (1 << LOGN);
  for (long long lines : {1LL, 1LL << 40}) {
    const int e = small_loge(LOGN, loge, lines, ps, bytes);
    if (e > loge || lane_reach(1 << LOGN, e, ps, 16, bytes) >= kBufMax)
      fail("chosen", LOGN, e, bytes);
  }
}

template <int LOGN>
void length() {
  constexpr int E3 = LOGN < 3 ? LOGN : 3, E4 = LOGN < 4 ? LOGN : 4;
  plan<LOGN, E3>(8);                     // FP32, several transforms of a line
  plan<LOGN, E4>(8);                     // FP32
  chosen<LOGN>(E3, 8);
  chosen<LOGN>(E4, 8);
  if (LOGN <= 12) {
    plan<LOGN, E3>(16);  // FP64
    chosen<LOGN>(E3, 16);
  }
  if constexpr (LOGN >= kSmallLogLo && LOGN <= kSmallLogHi) {
    plan<LOGN, kSmallLogE>(8);
    plan<LOGN, kSmallLogE>(16);
  }
}

int main() {
  static_assert(kOOB >= kBufMax && kOOB <= 0xffffffffu - 16, "");
  length<1>();
  length<2>();
  length<3>();
  length<4>();
  length<5>();
  length<6>();
  length<7>();
  length<8>();
  length<9>();
  length<10>();
  length<11>();
  length<12>();
  length<13>();
  std::printf("%d wrong\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_lane_offsets_of_every_length(tmp_path):
    src, exe = tmp_path / "offsets.hip", tmp_path / "offsets"
    src.write_text(PROGRAM)
    subprocess.run([hipcc(), "-O1", "--offload-arch=gfx950", "-std=c++17", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC, str(src), "-o",
                    str(exe)], check=True, capture_output=True, text=True, timeout=300)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout
