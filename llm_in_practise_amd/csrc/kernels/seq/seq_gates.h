// Shared by the two forms of the recurrences with a scalar decay (seq_chunk.hip, seq_walk.hip).
#pragma once
#include "seq_common.h"

namespace lipa {

constexpr double LOG2E = 1.4426950408889634074;

__device__ __forceinline__ double shfl_up_d(double v, int o) {
  const long long b = __double_as_longlong(v);
  const int lo = __shfl_up((int)b, o, 64), hi = __shfl_up((int)(b >> 32), o, 64);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double last_lane_d(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// v of a lane further down (CTRL: by 1, 2, 4, 8 within a row of 16, or a row's last lane to the rows behind it), `none` where there is none
template <int CTRL, int ROWS>
__device__ __forceinline__ double from_below(double v, double none) {
  const long long b = __double_as_longlong(v), z = __double_as_longlong(none);
  const int lo = __builtin_amdgcn_update_dpp((int)z, (int)b, CTRL, ROWS, 0xF, false),
            hi = __builtin_amdgcn_update_dpp((int)(z >> 32), (int)(b >> 32), CTRL, ROWS, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// op over a lane and those in front of it: a scan without a trip through LDS per step (6.5 -> 3.5 thousand cycles for a chunk's gates)
template <typename Op>
__device__ __forceinline__ double scan_lanes(double v, double none, Op op) {
  v = op(v, from_below<0x111, 0xF>(v, none));      // row_shr 1, 2, 4, 8
  v = op(v, from_below<0x112, 0xF>(v, none));
  v = op(v, from_below<0x114, 0xF>(v, none));
  v = op(v, from_below<0x118, 0xF>(v, none));
  v = op(v, from_below<0x142, 0xA>(v, none));      // row_bcast 15 into rows 1 and 3, row_bcast 31 into rows 2 and 3
  v = op(v, from_below<0x143, 0xC>(v, none));
  return v;
}

struct GateArgs {
  // state space: dt (bf16, row stride lddt), per head bias and log rate
  const bf16* dt;
  int lddt;
  const float *dt_bias, *a_log, *dskip;
  // mLSTM: gate pre-activations [T, H], per head biases, cap
  const float *ipre, *fpre, *ib, *fb;
  float cap, qscale;
  int H;
};

// The 8-byte transposed read: of 16 lanes, lane l gets column l of the four rows that lanes 0, 4, 8, 12 point into.
__device__ __forceinline__ bf16x4 read_tr(const bf16* p) {
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}
}  // namespace lipa
