// Split launches of the bit-plane GEMV (plz_gemv.hip): their LDS, their shape, and the sizes at
// which they are the faster ones. Host arithmetic only.
#pragma once
#include "plz_common.h"

namespace plz {
namespace gv {

// x prep, one chunk per linear and stage: A rows m = 2 t + piece, 256 B each (the fragments of both
// MFMA halves: 16-byte piece c = 8 h + 2 j + half, holding stage k = 128 h + 64 half + 16 j +
// (0..15), stored at c ^ (m & 15)); then the tokens' E8M0 scale bytes (16 B), their stage sums X
// as fp32 (64 B) and 48 B of padding.
__host__ __device__ constexpr int pl_chunk(int M) { return 512 * M + 128; }

constexpr int SP_WAVES = 16;           // most waves per workgroup
constexpr int SP_LDS = 160 * 1024;     // a CU's
constexpr int sp_ni(int M) { return M == 1 ? 2 : 4; }  // C rows per lane that hold a token's piece
__host__ __device__ constexpr int sp_sum_bytes(int ni, int rbw) {  // a wave's plane sums, lookup words
  return rbw * (3 * ni * 64 * 4 + 16 * 8);
}
__host__ __device__ constexpr int sp_wave_bytes(int ni, int rbw, int M) {
  return sp_sum_bytes(ni, rbw) + 2 * pl_chunk(M);
}

// rbw row blocks (16 rows) per workgroup, 0 to stream, and its waves.
struct SplitPlan {
  int rbw, waves;
};
// A launch of `items` (128 rows of one linear) for M tokens; stages (256 k): of the longest linear, a
// wave takes one per pass. Workgroups of 16 waves fill a CU at these register counts, so rbw is the
// least that leaves one round of them, and a launch of more workgroups than CUs gets at most 8
// waves each. Measured on 2560 -> 9728 (76 items) at M = 1 / 4: 7.3 / 11.4 us in one round of
// 152 / 304 workgroups of 10 waves, 8.1 / 9.2 us with 304 of 5.
//
// Every workgroup makes all of x's pieces, so the time grows with M, the passes and the rounds of
// workgroups: 2.5 us, then 0.9 us a pass and 0.01 + 0.05 rbw + 0.027 M for each wave on its CU
// (within 20% over 4 to 256 items, K 256 to 9728, M 1 to 8). The streaming launch walks a linear's
// stages as one chain: 6 + 0.25 M + 0.57 stages (its x prep included). Split and streaming as
// measured, weights from HBM, in us: K 9728, 140 items, M = 4 / 8 45.6 / 58.2 and 31.0 / 32.4;
// 76 items, M = 4 / 5 / 8 29.9 / 35.1 / 39.4 and 30.0 / 29.6 / 31.8; K 4096, 140 items, M = 3 / 5
// 16.8 / 25.3 and 20.2 / 20.7; K 2560, 160 items, M = 4 / 8 14.5 / 18.2 and 15.1 / 15.9; K 1024, 160
// items, M = 8 10.0 and 13.3. At M = 1 up to one item per CU (304 items of 2560 tie), from M = 2 up
// to 5/8.
inline SplitPlan split_plan_on(int64_t items, int64_t stages, int M, int64_t cus) {
  if (M > 8 || items > (M == 1 ? cus : cus * 5 / 8)) return SplitPlan{0, 0};
  const int ni = sp_ni(M), max_rbw = M == 1 ? 4 : 2;  // M > 1: the sums of 4 leave too few waves
  int rbw = items * 8 <= cus ? 1 : items * 4 <= cus ? 2 : 4;
  rbw = rbw < max_rbw ? rbw : max_rbw;
  const int64_t wgs = items * (8 / rbw);
  const int64_t cap = wgs <= cus ? SP_WAVES : SP_WAVES / 2;
  int64_t waves = (stages + (stages + cap - 1) / cap - 1) / ((stages + cap - 1) / cap);
  const int wave_bytes = sp_wave_bytes(ni, rbw, M);
  waves = waves < SP_LDS / wave_bytes ? waves : SP_LDS / wave_bytes;
  waves = waves < rbw * ni / 2 ? rbw * ni / 2 : waves;  // the folds take rbw * ni / 2 waves

  const int64_t passes = (stages + waves - 1) / waves;
  int64_t on_cu = SP_WAVES / waves, fit = SP_LDS / (waves * wave_bytes);
  on_cu = on_cu < fit ? on_cu : fit;
  const double per_wave = 0.01 + 0.05 * rbw + 0.027 * M;
  const int64_t rounds = wgs / (cus * on_cu), last = (wgs % (cus * on_cu) + cus - 1) / cus;
  double us = 2.5 + (double)(rounds * passes) * (0.9 + per_wave * (double)(on_cu * waves));
  if (last > 0) us += (double)passes * (0.9 + per_wave * (double)(last * waves));
  if (us > 6.0 + 0.25 * M + 0.57 * (double)stages) return SplitPlan{0, 0};
  return SplitPlan{rbw, (int)waves};
}

}  // namespace gv
}  // namespace plz
