"""The stream form's work (matfree_amd/csrc/matvec_plan.h) on the host: every
block of the matrix in one segment of one workgroup, each row block's segments
in planes 0, 1, .. below the number that the plan gives, the workgroups' shares
equal to a block.  Built with the sanitizers; no GPU needed."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <vector>
#include "matvec_plan.h"

using namespace slq;

static int check(int64_t n, int64_t P) {
  const F32Plan pl(n, P, false, false);
  if (pl.form != (n >= 32 && n <= 96 ? F32Plan::kWave : F32Plan::kStream)) return 1;
  if (pl.form != F32Plan::kStream) return 0;
  const int64_t tiles = (n + kMvTile - 1) / kMvTile, rows = (n + 31) / 32, runs = stream_runs(n);
  const int64_t groups = pl.even ? pl.even : rows * pl.S;
  if (pl.even && pl.S > choose_splitk(n, P, int64_t(1) << 60, true)) return 2;
  std::vector<int64_t> next(rows, 0);  // the row block's next block
  std::vector<int> planes(rows, 0);
  int64_t least = int64_t(1) << 60, most = 0, at = 0;
  for (int64_t g = 0; g < groups; ++g) {
    const int64_t rb = g / pl.S, z = g % pl.S;
    const int64_t u0 = pl.even ? stream_split(n, groups, g) : rb * runs + runs * z / pl.S;
    const int64_t u1 = pl.even ? stream_split(n, groups, g + 1) : rb * runs + runs * (z + 1) / pl.S;
    if (u0 != at || u1 < u0) return 3;
    at = u1;
    least = std::min(least, u1 - u0);
    most = std::max(most, u1 - u0);
    for (int64_t u = u0; u < u1;) {
      const StreamSegment s = stream_segment(n, u / runs, u % runs, u1 - u);
      if (s.rb < 0 || s.rb >= rows || s.k0 != next[s.rb] || s.k1 <= s.k0 || s.k1 > runs) return 4;
      next[s.rb] = s.k1;
      const int plane = pl.even ? stream_plane(n, groups, g, s.rb) : int(z);
      if (plane != planes[s.rb]++ || plane >= pl.S) return 5;
      // its tiles: whole ones up to the next segment's, the partial one with the last
      const int64_t end = s.tile0 + s.nwhole + (s.part ? 1 : 0);
      if (s.tile0 != s.k0 * kStreamTiles) return 6;
      if (end != std::min(tiles, s.k1 * kStreamTiles)) return 7;
      if (s.part != (s.k1 == runs && n % kMvTile != 0)) return 8;
      if ((s.tile0 + s.nwhole) * kMvTile > n) return 9;
      if (s.nblocks != (s.nwhole + kStreamTiles - 1) / kStreamTiles || s.nblocks > s.k1 - s.k0)
        return 10;
      u += s.k1 - s.k0;
    }
  }
  if (at != rows * runs) return 11;
  for (int64_t r = 0; r < rows; ++r)
    if (next[r] != runs || planes[r] < 1) return 12;
  return most - least > 1 ? 13 : 0;
}

int main() {
  for (int64_t n = 1; n < 140000; n += n < 9000 ? 1 : n < 20000 ? 7 : 4001)
    for (int64_t P : {1, 32})
      if (const int why = check(n, P)) {
        std::printf("FAILED %d at n = %lld, P = %lld\n", why, (long long)n, (long long)P);
        return 1;
      }
  std::printf("OK\n");
  return 0;
}
"""


def test_every_block_once(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(DRIVER)
    subprocess.run([gxx, "-std=c++17", "-O2", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-I",
                    os.path.join(ROOT, "matfree_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300,
                         env=dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0"))
    assert run.returncode == 0 and run.stdout.startswith("OK"), run.stdout + run.stderr
