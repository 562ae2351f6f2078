// Parameters of the few-row projections (linear_rows.hip).
#pragma once

#include "fa2_common.h"

namespace mi_fa2 {

enum LinearEpilogue { kOut = 0, kSilu = 1, kRope = 2 };

// Tokens per call, and hidden sizes a normalising or activating launch takes (one work-group's
// waves hold a whole row of x).
constexpr int kLrMaxRows = 64, kLrMaxNormRows = 16, kLrMaxK = 2048;

struct LinearParams {
  const uint16_t* x;       // [M][x_st], K used
  int64_t x_st;
  const uint16_t* norm_w;  // [K], or NULL: x is used as it is
  float eps;
  const uint16_t* w;       // [N][K] (kSilu: [2N][K], gate rows first)
  const uint16_t* bias;    // [N] or NULL
  const uint16_t* res;     // [M][res_st] added to the rounded product, or NULL; may be out
  int64_t res_st;
  uint16_t* out;           // [M][out_st] (kRope: the rotated q)
  int64_t out_st;
  int32_t M, N, K;
  int32_t tiles;           // 16-row tiles of W
  int32_t x_frag;          // x is in operand order, [MT][K / 32][64][8]
  // kOut with splits > 1: work-groups per unit, their fp32 partials, the units' arrival counts
  // (zero at launch)
  int32_t splits;
  uint64_t* part;
  uint32_t* count;
  // counters this launch zeroes for the next one
  uint32_t* zero;
  int32_t n_zero;
  // kRope
  const uint16_t* cos;     // [M][cs_st], 128 used
  const uint16_t* sin;
  int64_t cs_st;
  const int32_t* slots;    // [M]
  uint16_t* k_pool;
  uint16_t* v_pool;
  int64_t pool_st, pool_sh;
  int32_t num_slots, Hq, Hkv;
};

// Rotary tables of rows that append `T` tokens each from position starts[row] on.
struct RopeTableParams {
  const int32_t* starts;     // [rows]
  const uint16_t* inv_freq;  // [64]
  uint16_t* cos;             // [rows * T][128]
  uint16_t* sin;
  int32_t rows, T;
};
hipError_t launch_rope_table(const RopeTableParams& p, int dtype, hipStream_t stream);

// Work-groups that share a tile's K (1 for K <= 2048).
int linear_splits(int K);
hipError_t launch_linear_rows(LinearParams p, int dtype, int epi, int n_cus, hipStream_t stream);

}  // namespace mi_fa2
