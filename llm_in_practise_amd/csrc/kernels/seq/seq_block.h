// Shared by the scans of prompts in blocks of tokens (seq_block.hip, seq_delta.hip).
#pragma once
#include "seq_common.h"

namespace lipa {

constexpr int BT = 16;      // tokens of a tile of the float matrix units

__device__ __forceinline__ float row16_sum(float v) {       // over the 16 lanes of a row, in all of them
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));    // quad_perm [1, 0, 3, 2]
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));    // quad_perm [2, 3, 0, 1]
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));   // row_half_mirror
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));   // row_mirror
  return v;
}

__device__ __forceinline__ f32x4 row4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 row4(const bf16* p) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

// How a walk takes the sequences: whole; in parts of `len` tokens without outputs and without a sequence's last one, which leaves what is
// behind each; in parts with the outputs.
enum { WHOLE, ENDS, PARTS };

// Part `id` of all that run, without a sequence's last one for `ends`; place: the sequence's first place.  (Counted, not bounded as the
// pieces are: blocks of threads that find nothing to do leave others side by side on one CU, 84 us for 45.)
// Parts and places are counted in the halves of an int: MOST_PARTS at most, T / len + B.
constexpr int MOST_PARTS = (1 << 15) - 1;
struct Part {
  int s, idx, place, t0, t1, end;
};
__device__ __forceinline__ bool find_part(const SeqDesc& d, int len, int id, bool ends, Part& p) {
  int before = 0;                                            // parts in the lower half, places in the upper one
  for (int b0 = 0; b0 < d.B; b0 += 64) {
    const int lane = threadIdx.x & 63, b = min(b0 + lane, d.B - 1);
    const int s0 = d.seq_off[b], s1 = d.seq_off[b + 1], on = d.live ? d.live[b] : 1;
    const int n = on && b0 + lane < d.B ? (s1 - s0 + len - 1) / len : 0, own = n + (max(n - 1, 0) << 16);
    int sum = own;
#pragma unroll
    for (int o = 1; o < 64; o *= 2) {
      const int x = __shfl_up(sum, o, 64);
      sum += lane >= o ? x : 0;
    }
    sum += before;
    const unsigned long long m = __ballot((ends ? sum >> 16 : sum & 0xffff) > id);
    if (m) {
      const int at = __builtin_ctzll(m), first = __builtin_amdgcn_readlane(sum - own, at);
      p.s = b0 + at;
      p.idx = id - (ends ? first >> 16 : first & 0xffff);
      p.place = first >> 16;
      p.end = __builtin_amdgcn_readlane(s1, at);
      p.t0 = __builtin_amdgcn_readlane(s0, at) + p.idx * len;
      p.t1 = min(p.t0 + len, p.end);
      return true;
    }
    before = __builtin_amdgcn_readlane(sum, 63);
  }
  return false;
}

}  // namespace lipa
