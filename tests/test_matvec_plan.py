"""The FP32 matvec's plan (matfree_amd/csrc/matvec_plan.h) on the host: its
slices tile the columns, its passes cover the slices and stay inside the
scratch, with the least scratch only the number of passes changes, and small
problems of more than 32 vectors read them as they are.  Built with the
sanitizers; no GPU needed."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "matvec_plan.h"

using namespace slq;

// the least scratch: partial sums, two planes and the point records
static int64_t least(int64_t n, int64_t P) {
  const int64_t unlimited = int64_t(1) << 60;
  const int S = std::max(choose_splitk(n, P, unlimited, true), choose_splitk(n, P, unlimited, false));
  const PlaneSizes z(n, P);
  return S * P * n + z.Ppad * z.npad + 16 * z.npad;
}

static int64_t cases = 0, several = 0;

static int check(int64_t n, int64_t P, bool rbf, bool planed) {
  const F32Plan pl(n, P, rbf, planed);
  const int64_t tiles = (n + kMvTile - 1) / kMvTile;
  if (pl.S < 1 || pl.slice_tile(0) != 0 || pl.slice_tile(pl.S) != tiles) return 1;
  for (int zi = 0; zi < pl.S; ++zi)
    if (pl.slice_tile(zi) >= pl.slice_tile(zi + 1)) return 2;  // no empty slice
  const int64_t lean = least(n, P);
  const int64_t full = std::max(lean, pl.input_floats() + lean - pl.z.Ppad * pl.z.npad - 16 * pl.z.npad);
  if (!pl.whole(full) || pl.pass_end(0, full) != pl.S) return 3;
  if (pl.input_floats() % 4 != 0) return 4;
  // a small problem of more than 32 probes: no launch for planes, 32 rows a workgroup
  const int64_t blocks = (P + 31) / 32;
  const bool small =
      P > 32 && n < 4096 && n * n * blocks <= (planed ? int64_t(3) << 23 : int64_t(1) << 25);
  if (small != (P > 32 && pl.form == F32Plan::kWave)) return 7;
  if (small && (pl.input != F32Plan::kRows || pl.S > 4)) return 8;
  int passes = 0;
  for (int z0 = 0, z1; z0 < pl.S; z0 = z1, ++passes) {
    z1 = pl.pass_end(z0, lean);
    if (z1 <= z0 || z1 > pl.S) return 5;
    const int64_t in = pl.form == F32Plan::kWorkgroup
                           ? pl.input_floats(pl.slice_tile(z0), pl.slice_tile(z1))
                           : pl.input_floats();
    if (in < 0 || in > (lean - pl.sum_floats()) / 4 * 4) return 6;
  }
  ++cases;
  several += passes > 1;
  return 0;
}

int main() {
  // (a call of fewer than 256 columns has less than the static scratch at any probe count)
  for (int64_t n = 256; n < 200000; n += n < 1000 ? 37 : n < 20000 ? 257 : 9973)
    for (int64_t P = 1; P <= 1100; P += P < 200 ? 1 : 13)
      for (int kind = 0; kind < 4; ++kind)
        if (const int why = check(n, P, kind & 1, kind & 2)) {
          std::printf("FAILED %d at n = %lld, P = %lld, kind %d\n", why, (long long)n,
                      (long long)P, kind);
          return 1;
        }
  std::printf("OK %lld %lld\n", (long long)cases, (long long)several);
  return several > 0 ? 0 : 1;
}
"""


def test_passes_over_the_slices(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(DRIVER)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-I",
                    os.path.join(ROOT, "matfree_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True,
                         env=dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0"))
    assert run.returncode == 0 and run.stdout.startswith("OK"), run.stdout + run.stderr
