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

// More than 32 probes of a small problem take the wave form (blocks of 32
// probes) as well.  The workgroup form there has a launch of its own for the
// planes and a few workgroups, each a chain of tiles as long as the row (stored
// n = 512, 64 probes: 23.0 us, wave form 7.0; RBF 23.8 and 7.7).  The wave
// form's work grows with n^2 and the blocks, every block forming and splitting
// the entries again: 2^25 is where the two meet (stored, wave and workgroup
// form: n = 2048, 256 probes 33.1 and 36.3 us, 3700, 40: 27.2 and 34.7; beyond,
// 4096, 40: 35.1 and 30.6, 3000, 128: 40.1 and 39.9, 2500, 256: 53.8 and 49.2).
// planed: calls of a loop whose inputs come with their planes, which saves the
// workgroup form 3.5 us; the two meet at three quarters of that (decomposition of
// 20 steps: n = 2048, 256 probes 1023 and 983 us, 3500, 64: 733 and 838).
inline bool wave_blocks(int64_t n, int64_t P, bool planed) {
  const int64_t blocks = (P + 31) / 32, limit = planed ? int64_t(3) << 23 : int64_t(1) << 25;
  return blocks > 1 && blocks <= 65535 && n < 4096 && n * n * blocks <= limit;
}

// Column slices of the FP32 matvec, up to the factor above (which sizes the
// scratch).  Workgroup form: the last round of resident workgroups (two per
// CU) filled best.  Wave form: three per CU.  Stream form: one per CU runs
// faster than two that share the CU's part of the bandwidth (n = 4096, 32
// probes: 20 us in 256 workgroups, 27 in 512), so as many slices as fit 256
// workgroups (larger matrices are split evenly: F32Plan).  Blocks of the wave
// form: rounds of 256 as well, by up to four (stored n = 2500, 128 probes: 1 to 4
// slices take 37.0, 33.8, 32.3, 31.1 us; 2048, 64: 17.7, 13.4, 15.6, 14.8), RBF,
// which computes more, of 512 (4095, 33 probes: 1 slice 33.1, 2 slices 31.0); more
// of them only for a sixth more of the round, which their sum costs (stored
// 2048, 224 probes: 1 slice 32.8, 4 slices 38.2).
inline int choose_splitk_f32(int64_t n, int64_t P, bool rbf, bool planed) {
  const int most = choose_splitk(n, P, int64_t(1) << 60, true);
  const int64_t nacc = nacc_for(P);
  const bool stream = nacc == 1 && !rbf, blocks = wave_blocks(n, P, planed);
  const int64_t wgs = nacc == 1 ? (n + 31) / 32
                      : blocks  ? (n + 31) / 32 * ((P + 31) / 32)
                                : (n + kMvRows - 1) / kMvRows * ((P + 32 * nacc - 1) / (32 * nacc));
  const int64_t resident = stream || (blocks && !rbf) ? 256 : (nacc == 1 ? 768 : 512);
  if (stream && wgs <= resident) return int(std::min<int64_t>(most, resident / wgs));
  int best = 1;
  double fill = 0.0;
  for (int S = 1; S <= (stream ? 1 : blocks ? std::min(most, 4) : most); ++S) {
    const double rounds = double(wgs * S) / double(resident);
    const double f = rounds / std::ceil(rounds);
    if (f > (blocks ? fill * 1.16 : fill + 0.02)) {
      fill = f;
      best = S;
    }
  }
  return best;
}

// The stream form's work: blocks of 32 rows x 128 columns, the row's last one
// whatever is left.  A workgroup takes blocks [u0, u1) in the order of the rows
// and goes through them in segments of one row block each.
constexpr int kStreamTiles = 4;    // tiles of a block
constexpr int kStreamGroups = 256;  // workgroups of the even split, one a CU
struct StreamSegment {
  int64_t rb, k0, k1;  // blocks [k0, k1) of row block rb
  int64_t tile0;       // first tile
  int64_t nwhole;      // whole tiles
  int64_t nblocks;     // blocks that hold whole tiles
  bool part;           // the matrix's partial last tile too
};
constexpr int64_t stream_runs(int64_t n) {
  return (n + kStreamTiles * kMvTile - 1) / (kStreamTiles * kMvTile);
}
// The segment from block k0 of row block rb on, of `left` blocks still to do.
constexpr StreamSegment stream_segment(int64_t n, int64_t rb, int64_t k0, int64_t left) {
  const int64_t tiles = (n + kMvTile - 1) / kMvTile, runs = stream_runs(n);
  StreamSegment s{};
  s.rb = rb;
  s.k0 = k0;
  s.k1 = left < runs - k0 ? k0 + left : runs;
  s.tile0 = s.k0 * kStreamTiles;
  const int64_t end = s.k1 == runs ? tiles : s.k1 * kStreamTiles;
  s.part = end == tiles && n % kMvTile != 0;
  s.nwhole = end - s.tile0 - (s.part ? 1 : 0);
  s.nblocks = (s.nwhole + kStreamTiles - 1) / kStreamTiles;
  return s;
}
// Even split of all blocks over G workgroups: workgroup g's first block, and
// the partial plane of its segment in row block rb (the row block's segments in
// order).
constexpr int64_t stream_split(int64_t n, int64_t G, int64_t g) {
  return (n + kMvTile - 1) / kMvTile * stream_runs(n) * g / G;
}
constexpr int stream_plane(int64_t n, int64_t G, int64_t g, int64_t rb) {
  const int64_t units = (n + kMvTile - 1) / kMvTile * stream_runs(n);
  // the workgroup that holds the row block's first block
  const int64_t first = ((rb * stream_runs(n) + 1) * G + units - 1) / units - 1;
  return int(g - first);
}
// Planes that the even split needs: the most segments of a row block.
inline int stream_planes(int64_t n, int64_t G) {
  const int64_t runs = stream_runs(n), units = (n + kMvTile - 1) / kMvTile * runs;
  if (units % G == 0 && units / G % runs == 0) return 1;
  const int64_t least = units / G;
  return least >= runs ? 2 : int((runs + least - 1) / least) + 1;
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
  int S;     // column slices (partial planes)
  int even;  // stream form: workgroups of the even split, 0: row blocks x slices

  // planed: one of a loop of calls whose inputs come with their planes
  F32Plan(int64_t n_, int64_t P_, bool rbf, bool planed)
      : n(n_), P(P_), z(n_, P_), nacc(nacc_for(P_)) {
    // a stored matrix of one to three tiles a row has no stream to speak of (n =
    // 32, 32 vectors: wave form 3.3 us, stream form 4.5; 96: 3.8 and 4.7; less
    // than a tile, n = 16: 4.3 and 3.7)
    const bool few = n >= kMvTile && n <= 3 * kMvTile;
    form = wave_blocks(n, P, planed) ? kWave
           : nacc > 1                ? kWorkgroup
           : rbf || few              ? kWave
                                     : kStream;
    input = kRows;
    // The wave form reads rows at small n, where its waves split the vectors
    // themselves (the launch that writes the planes costs about 3.5 us,
    // splitting in the waves 0.2 us per 1000 columns).
    if (form == kWorkgroup || (form == kWave && nacc == 1 && n >= 4096)) input = kPlanes;
    // The stream form's tiles are written by the producer of the input where
    // there is one, in a launch of about 3.5 us otherwise.  With few probes
    // most of a tile is padding, and its lines cost more than the rows' (a
    // product with that launch, rows and tiles: n = 10413, 16 probes 99.1 and
    // 105.9 us, 24: 105.3 and 105.8, 25: 108.2 and 105.3, 32: 114.0 and 109.9);
    // for less than n = 9000 the launch costs more than the tiles save (8600, 32
    // probes: 71.4 and 73.7; 8961: 88.5 and 81.6).
    if (form == kStream && n > 8960 && P > 24) input = kTiles;
    S = choose_splitk_f32(n, P, rbf, planed);
    even = 0;
    // Even split of a matrix beyond 4096, unless its row blocks nearly fill the
    // CUs once (n = 8000, 1 to 32 vectors: 49.5 to 53.8 us a row block each, 52.6
    // to 57.0 split; 7168: 44.2 to 45.6 and 43.4 to 46.0) or a partial plane more
    // is more than the scratch holds.
    if (form == kStream && n > 4096 && !(n <= 8192 && n > 7360)) {
      const int planes = stream_planes(n, kStreamGroups);
      if (planes <= choose_splitk(n, P, int64_t(1) << 60, true)) {
        even = kStreamGroups;
        S = planes;
      }
    }
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
