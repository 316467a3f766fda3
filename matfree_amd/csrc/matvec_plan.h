// Which form the FP32 block matvec takes, its column slices and how they share
// the scratch.  Plain C++ (no HIP), so that the rules can be checked without a
// GPU (tests/test_matvec_plan.py).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace slq {

constexpr int kMvRows = 128;  // output elements per workgroup
constexpr int kMvTile = 32;   // contraction tile

// Largest split-K factor of the block matvec; its partial sums need up to
// kMaxSplitK * P * n floats of scratch (matvec_scratch_floats sizes it for
// the factor the launch will take).
constexpr int kMaxSplitK = 16;

inline int nacc_for(int64_t P) { return P <= 32 ? 1 : (P <= 64 ? 2 : 4); }

// Padded sizes of the planes of P probes.
struct PlaneSizes {
  int64_t npad, Ppad;
  PlaneSizes(int64_t n, int64_t P) {
    const int64_t bpw = 32 * nacc_for(P);
    npad = (n + kMvTile - 1) / kMvTile * kMvTile;
    Ppad = (P + bpw - 1) / bpw * bpw;
  }
};

// Split-K factor: enough workgroups for two per CU (256 CUs), as long as
// every slice keeps at least 8 tiles and the partial sums fit the scratch.
// The FP32 kernels for up to 32 probes use under 128 registers and hold four
// waves per SIMD, so they get twice the workgroups (more waves to hide the
// latency of their short per-tile chains).
inline int choose_splitk(int64_t n, int64_t P, int64_t avail_floats, bool fp32) {
  const int64_t nacc = nacc_for(P);
  const int64_t wgs = ((n + kMvRows - 1) / kMvRows) * ((P + 32 * nacc - 1) / (32 * nacc));
  const int64_t tiles = (n + kMvTile - 1) / kMvTile;
  const int64_t target = (fp32 && nacc == 1) ? 1024 : 512;
  int S = 1;
  while (S < kMaxSplitK && wgs * S < target && tiles / (2 * S) >= 8 &&
         int64_t(2 * S) * P * n <= avail_floats)
    S *= 2;
  return S;
}

// Column slices of the FP32 matvec, up to the factor above (which sizes the
// scratch).  Workgroup form: the last round of resident workgroups (two per
// CU) filled best.  Wave form: three per CU.  Stream form: one per CU runs
// faster than two that share the CU's part of the bandwidth (n = 4096, 32
// probes: 20 us in 256 workgroups, 27 in 512), so rounds of 256, by up to
// three slices (10413: 1, 2, 3 slices take 143, 121, 117 us).
inline int choose_splitk_f32(int64_t n, int64_t P, bool rbf) {
  const int most = choose_splitk(n, P, int64_t(1) << 60, true);
  const int64_t nacc = nacc_for(P);
  const bool stream = nacc == 1 && !rbf;
  const int64_t wgs = nacc == 1 ? (n + 31) / 32
                                : (n + kMvRows - 1) / kMvRows * ((P + 32 * nacc - 1) / (32 * nacc));
  const int64_t resident = stream ? 256 : (nacc == 1 ? 768 : 512);
  if (stream && wgs <= resident) return int(std::min<int64_t>(most, resident / wgs));
  int best = 1;
  double fill = 0.0;
  for (int S = 1; S <= (stream ? std::min(most, 3) : most); ++S) {
    const double rounds = double(wgs * S) / double(resident);
    const double f = rounds / std::ceil(rounds);
    if (f > fill + 0.02) {
      fill = f;
      best = S;
    }
  }
  return best;
}

// The FP32 matvec's planes hold V and -V in turns of this many tiles (see
// k_matvec_f32), times this power of two (see kSplitScale).
constexpr int kPlaneSignRun = 2;
constexpr float kPlaneScale = 65536.f;

// Floats of the FP32 matvec's three BF16 planes of `probes` (padded) probes.
inline int64_t f32_plane_floats(int64_t npad, int64_t probes) { return 3 * npad * probes / 2; }

// The FP32 matvec of P vectors.
struct F32Plan {
  enum Form { kWorkgroup, kWave, kStream };
  // what the kernel reads its vectors from: the rows as given, three BF16
  // planes (k_split3_probes), or the stream form's tiles (k_tile_probes)
  enum Input { kRows, kPlanes, kTiles };
  int64_t n, P;
  PlaneSizes z;
  Form form;
  Input input;
  int nacc;  // workgroup form: blocks of 32 probes a workgroup
  int S;     // column slices

  F32Plan(int64_t n_, int64_t P_, bool rbf) : n(n_), P(P_), z(n_, P_), nacc(nacc_for(P_)) {
    form = nacc > 1 ? kWorkgroup : rbf ? kWave : kStream;
    input = kRows;
    // The wave form reads rows at small n, where its waves split the vectors
    // themselves (the launch that writes the planes costs about 3.5 us,
    // splitting in the waves 0.2 us per 1000 columns).
    if (form == kWorkgroup || (form == kWave && n >= 4096)) input = kPlanes;
    // The stream form's tiles are written by the producer of the input where
    // there is one, in a launch of about 3.5 us otherwise.  With up to 16
    // probes most of a tile is padding, and its lines cost more than the rows'
    // (15001, 16 probes: 199 -> 208 us); up to n = 8400 the launch costs what
    // the tiles save.
    if (form == kStream && n > 8960 && P > 24) input = kTiles;
    S = choose_splitk_f32(n, P, rbf);
  }

  // First tile of slice z of the workgroup form: whole runs of one plane sign.
  int64_t slice_tile(int64_t zi) const {
    const int64_t tiles = (n + kMvTile - 1) / kMvTile, runs = (tiles + kPlaneSignRun - 1) / kPlaneSignRun;
    return std::min(runs * zi / S * kPlaneSignRun, tiles);
  }
  int64_t sum_floats() const { return S > 1 ? int64_t(S) * P * n : 0; }
  // Floats of the input of tiles [t0, t1).
  int64_t input_floats(int64_t t0, int64_t t1) const {
    if (input == kRows) return 0;
    if (input == kTiles) return (t1 - t0) * kMvTile * 32;
    return f32_plane_floats((t1 - t0) * kMvTile, z.Ppad);
  }
  int64_t input_floats() const { return input_floats(0, z.npad / kMvTile); }
  // Whether the whole input fits beside the partial sums.
  bool whole(int64_t scratch_floats) const {
    return input_floats() + sum_floats() <= scratch_floats;
  }
  // With less scratch (the least size) the workgroup form runs in passes over
  // its slices, the planes of a pass's columns in the scratch at a time: the
  // end of the pass that starts at slice z0, z0 if not even one fits.  The
  // form, the slices and every slice's sums are those of a single pass.
  int pass_end(int z0, int64_t scratch_floats) const {
    const int64_t room = scratch_floats - sum_floats();
    if (form != kWorkgroup) return input_floats() <= room ? S : z0;
    int z1 = z0;
    while (z1 < S && input_floats(slice_tile(z0), slice_tile(z1 + 1)) <= room) ++z1;
    return z1;
  }
};

}  // namespace slq
