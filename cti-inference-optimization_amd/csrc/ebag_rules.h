// Dispatch rules that are arithmetic on sizes and alignments alone: plain C++, so that a test can hold
// them against what the kernels behind them assume, without a GPU.
#pragma once

#include <stdint.h>

#include <initializer_list>

namespace cti {

// Whether the ragged kernel may read a table of `rows` rows of `dim` elements of `elem_bytes`, `row_bytes`
// apart from `base` on, with buffer loads: rows of at least one 16-byte chunk, every chunk 4-byte aligned
// (the last one ends with the row, so the row's own length counts beside the base and the stride; it also
// keeps the table's end, where loads past a bag go, a whole number of words away), and no offset from the
// end on, by up to a row, wrapping around 32 bits.
inline bool ragged_buffer_loads(uint64_t base, int64_t rows, int64_t row_bytes, int64_t dim, int elem_bytes) {
  const int64_t len = dim * elem_bytes;
  const int64_t span = (rows - 1) * row_bytes + len;
  return len >= 16 && base % 4 == 0 && row_bytes % 4 == 0 && len % 4 == 0 && span + len < (int64_t{1} << 32);
}

// ---------------------------------------------------------------------------------------------
// LayerNorm-Linear: y [M, N] = a [M, K] w^T, K in steps of kLinearStep.
// ---------------------------------------------------------------------------------------------
constexpr int kLinearStep = 64;
constexpr int kLinearCus = 256;                 // one workgroup per CU
constexpr int kLinearBandParams = 28 * 1024;    // LDS of the band form for gamma and beta

enum LinearForm {
  kLinearGeneral,  // any K: 64 x 256 tiles
  kLinearTile128,  // K a multiple of 128, byte offsets below 2^31: 128 x 128 tiles, K split if they are few
  kLinearTile256,  // 128 x 256 tiles, from two per CU on
  kLinearBand,     // bands of 128 rows by 256, 384 or 512 columns, K split if they are few
};
struct LinearPlan {
  LinearForm form;
  int splits;  // of K: 1, or as many fp32 partial products as the workspace then has to hold
  int steps;   // per split (even)
};

inline int64_t linear_ceil(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Column fragments per wavefront of the band form: 8 wavefronts cover N = 256, 384 or 512 columns.
inline int linear_band_fragments(int32_t N) { return N <= 256 ? 2 : (N <= 384 ? 3 : 4); }
inline int64_t linear_band_tiles(int64_t M, int32_t N) {
  return linear_ceil(M, 128) * linear_ceil(N, 128 * linear_band_fragments(N));
}

// Splits K into at most `want` parts of even step counts, as many as `ws_bytes` of fp32 partials hold;
// 1 = no split. `steps` receives the steps per split.
inline int linear_split(int64_t want, int64_t M, int32_t N, int32_t K, int64_t ws_bytes, int* steps) {
  const int nk = K / kLinearStep;
  *steps = nk;
  if (want <= 1 || nk < 4) return 1;
  const int64_t fit = ws_bytes / (M * N * 4);
  if (want > fit) want = fit;
  if (want > nk / 2) want = nk / 2;
  if (want <= 1) return 1;
  const int per = static_cast<int>((linear_ceil(nk, want) + 1) / 2 * 2);
  *steps = per;
  return static_cast<int>(linear_ceil(nk, per));
}

// The form and the splits of K for a shape; param_bytes: an element of gamma and beta (0: the plain Linear).
//
// 128 x 256 tiles when there are at least two per CU, else 128 x 128, whole or split for one workgroup per CU
// (two measured slower: M = 1024, K = 3584, N = 512 took 28.0 against 18.7 us, the partials' HBM traffic
// outweighing the extra parallelism); or the band form, whole or split for at most one workgroup per CU:
// whichever has the lowest estimated time. The estimates: rounds of one workgroup per CU, each of a
// fixed and a per-step time (us; the band form's steps slow down by kFull as the chip fills, with x, the
// weight and the products each at a limit), the second launch of a split with its partial products, and the
// band form's stores of rows that are no multiple of 4 columns. Fitted to 2,000 shapes (K = 256 to 7168,
// M = 512 to 65,536, N = 64 to 1024); the choice is on average 1% off the better form's time. What decides,
// in measured us of the tiles | the band form whole | split:
//   enough rows           M = 30000, K = 3584, N = 256 / 384 / 512: 106 / 156 / 212 | 68 / 93 / 109
//                         M = 30000, K = 896, N = 256 / 384 / 512: 37 / 55 / 72 | 24 / 32 / 39
//   columns               M = 16384, K = 3584, N = 128: 50 (36 split) | 55 | 41: the band multiplies 256
//   partials of short K   M = 16384, K = 896, N = 512: 36 | 30 | 47
//   few bands, no split   M = 8192, K = 7168, N = 512, plain: 75 | 146; M = 8192, K = 3584, N = 384: 53 | 67 | 43
inline LinearPlan linear_choose(int64_t M, int32_t N, int32_t K, int param_bytes, int64_t ws_bytes) {
  const int nk = K / kLinearStep;
  constexpr int64_t kBytes = int64_t{1} << 31;
  if (K % (2 * kLinearStep) != 0 || M >= kBytes || (M + 128) * K * 2 >= kBytes || static_cast<int64_t>(N) * K * 2 >= kBytes)
    return {kLinearGeneral, 1, nk};
  struct Cost {
    double fixed, step;
  };
  const bool ln = param_bytes != 0;
  const Cost tile128 = ln ? Cost{4.4, 0.75} : Cost{3.2, 0.51};
  const Cost tile256 = ln ? Cost{9.4, 1.2} : Cost{9.1, 1.0};
  const Cost bands[3] = {ln ? Cost{4.3, 0.78} : Cost{3.6, 0.62}, ln ? Cost{6.6, 0.98} : Cost{6.0, 0.83},
                         ln ? Cost{9.2, 1.18} : Cost{9.2, 1.14}};
  constexpr double kLaunch = 3.0, kFull = 0.55, kReduce = 2.3, kPartial = 1.1e-6;
  const double odd_store = N % 2 ? (ln ? 0.6e-6 : 0.9e-6) : (N % 4 ? 0.15e-6 : 0.0);  // per element stored
  const double mn = static_cast<double>(M) * N;
  const auto split_time = [&](int splits) { return splits > 1 ? kReduce + kPartial * mn * splits : 0.0; };

  LinearPlan tiles{kLinearTile256, 1, nk};
  double tile_time;
  const int64_t t256 = linear_ceil(M, 128) * linear_ceil(N, 256);
  if (t256 >= 2 * kLinearCus) {
    tile_time = kLaunch + linear_ceil(t256, kLinearCus) * (tile256.fixed + tile256.step * nk);
  } else {
    const int64_t t128 = linear_ceil(M, 128) * linear_ceil(N, 128);
    const auto time128 = [&](int splits, int steps) {
      // plain tiles fit a CU twice: a half-filled round takes little more than half the time
      const double rounds = ln ? linear_ceil(t128 * splits, kLinearCus)
                               : t128 * splits <= kLinearCus ? 1.0 : 0.1 + 0.5 * linear_ceil(2 * t128 * splits, kLinearCus);
      return kLaunch + split_time(splits) + rounds * (tile128.fixed + tile128.step * steps);
    };
    tiles.form = kLinearTile128;
    tile_time = time128(1, nk);
    int steps = 0;
    const int splits = linear_split(linear_ceil(kLinearCus, t128), M, N, K, ws_bytes, &steps);
    if (splits > 1 && time128(splits, steps) < tile_time) {
      tiles = {kLinearTile128, splits, steps};
      tile_time = time128(splits, steps);
    }
  }
  if (static_cast<int64_t>(K) * 2 * param_bytes > kLinearBandParams) return tiles;

  const Cost band = bands[linear_band_fragments(N) - 2];
  const int64_t t_band = linear_band_tiles(M, N);
  const auto band_time = [&](int splits, int steps) {
    const int64_t full = t_band * splits / kLinearCus, last = t_band * splits % kLinearCus;
    const double filled = last > kLinearCus / 2 ? 2.0 * last / kLinearCus - 1.0 : 0.0;
    return kLaunch + split_time(splits) + odd_store * mn * splits +
           full * (band.fixed + band.step * steps * (1.0 + kFull)) +
           (last ? band.fixed + band.step * steps * (1.0 + kFull * filled) : 0.0);
  };
  if (band_time(1, nk) < (ln ? 0.97 : 0.93) * tile_time) {
    tiles = {kLinearBand, 1, nk};
    tile_time = band_time(1, nk);
  }
  int steps = 0;
  const int splits = linear_split(kLinearCus / t_band, M, N, K, ws_bytes, &steps);
  if (splits > 1 && band_time(splits, steps) < (ln ? 0.97 : 0.88) * tile_time) return {kLinearBand, splits, steps};
  return tiles;
}

// Bytes of workspace that a shape is given at most, whatever gamma and beta are: what the splits of the
// fastest choice need (0: it is whole).
inline int64_t linear_workspace_bytes(int64_t M, int32_t N, int32_t K) {
  int splits = 1;
  for (int param_bytes : {0, 2, 4}) {
    const LinearPlan plan = linear_choose(M, N, K, param_bytes, INT64_MAX);
    if (plan.splits > splits) splits = plan.splits;
  }
  return splits > 1 ? static_cast<int64_t>(splits) * M * N * 4 : 0;
}

inline LinearPlan linear_plan(int64_t M, int32_t N, int32_t K, int param_bytes, int64_t ws_bytes) {
  const int64_t most = ws_bytes > 0 ? linear_workspace_bytes(M, N, K) : 0;
  return linear_choose(M, N, K, param_bytes, ws_bytes < most ? ws_bytes : most);
}

}  // namespace cti
