"""The row walk's 32-bit offsets at the largest lists (CPU: the kernels' own expressions, compiled
for the host)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "particledynamics.jl_amd", "csrc")

PROGRAM = r"""
#include "pdx_rowwalk.hpp"
#include <cstdio>
#include <initializer_list>
using namespace pdx::pairk;
int main() {
  const long long two28 = 1ll << 28;
  int bad = 0, narrow = 0, wide = 0;
  for (int lanes = 1; lanes <= 64; lanes <<= 1)
    for (long long around : {1ll, 1000ll, 486400ll, 1ll << 20, two28 / 64, two28 / 16, 45000000ll, two28 / 4, 179000000ll,
                             1ll << 27, two28 / 4 * 3, two28, 1ll << 30, (1ll << 31) - 2})
      for (long long d = -3; d <= 3; ++d) {
        const long long n = around + d;
        if (n < 1 || n >= (1ll << 31) - 1) continue;
        const int g = walk_shape(lanes, (int)n);
        bool ok = g >= 0 && g <= lanes;
        const bool fits1 = 16 * n < (1ll << 32) && 16 * (n + 1) < (1ll << 32);
        ok = ok && (g == 0) == !fits1;
        if (g == 0) {
          ++wide;
        } else {
          ++narrow;
          ok = ok && walk_records((int)n) == 16 * (n + 1);
          ok = ok && walk_gather((int)n) == 16 * n && 16 * n + 16 <= (long long)walk_records((int)n);
          const long long last = (long long)(g - 1) * n + n - 1, step = (long long)(WALK_U - 1) * g * n;
          ok = ok && walk_lane(g - 1, (int)n, (int)(n - 1)) == 4 * last;
          ok = ok && walk_step(WALK_U - 1, g, (int)n) == 4 * step && 4 * (last + step) + 4 <= (1ll << 32);
          ok = ok && (g == lanes || 4ll * WALK_U * 2 * g * n >= (1ll << 32));  // no fewer lanes than needed
        }
        if (!ok) { ++bad; std::printf("lanes %d n %lld: %d\n", lanes, n, g); }
      }
  for (int split : {-2, -4, -8, -16}) bad += walk_shape(split, 1 << 29) != split;
  std::printf("narrow %d wide %d bad %d\n", narrow, wide, bad);
  return bad != 0 || narrow == 0 || wide == 0;
}
"""


def test_offsets_fit_at_the_largest_lists(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    src = tmp_path / "rowwalk.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "rowwalk"
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
