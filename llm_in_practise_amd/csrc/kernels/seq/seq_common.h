// Shared pieces of the sequence-state kernels (recurrent mixers, short convolutions, head-mixing and latent
// attention, routed experts, fp32-residual norms).  Activations are bf16 or float (template parameter T); the
// residual stream, every norm, softmax, gate and recurrent state is float.
//
// A step's tokens are packed back to back, [Ttot, features].  Sequence b owns tokens seq_off[b] .. seq_off[b+1]-1,
// lives in state slot slots[b] and starts this step at position pos0[b] (0 = a fresh sequence: its state is taken
// as zero, whatever the slot held before).  live (optional) marks rows whose state may be touched.
#pragma once
#include "../common.h"

namespace lipa {

struct SeqDesc {
  const int* seq_off;   // [B + 1]
  const int* slots;     // [B]
  const int* pos0;      // [B]
  const int* tok_seq;   // [Ttot] sequence of a token
  const int* tok_pos;   // [Ttot] absolute position of a token
  const int* live;      // [B] or null
  int B, Ttot;
};

// A step's sequences cut into pieces of LEN tokens (0: of `len`), each with a slot for what a kernel leaves of it.  count 0: every piece has
// one, sequence s owns the slots from seq_off[s] / LEN + s on (consecutive sequences never overlap).  Else the pieces [first, first +
// count) of every sequence, s owns the slots from s * count on: a step whose slots would take too much memory runs window after
// window, and the state goes from one to the next through the sequence's own place.
struct Pieces {
  int len, first, count;
};
struct Piece {
  int s, idx, t0, n;     // sequence, number within it, first token, tokens
  int pos0;              // the sequence's pos0
};
// False: the slot holds no piece (or one of an idle sequence).  A lane looks at one of up to 64 sequences at a time, so that everything
// comes in one round trip to memory: a search of eight sequences step by step takes four, 3 us where nothing else can start before.
template <int LEN>
__device__ __forceinline__ bool find_piece(const SeqDesc& d, const Pieces& p, int slot, Piece& c) {
  const int len = LEN > 0 ? LEN : p.len;
  int b0 = 0, lo = p.count > 0 ? slot / p.count : 0;
  if (p.count > 0) {
    b0 = lo;             // its lane is the first
  } else {
    for (int hi = d.B - 1; hi - b0 >= 64;) {          // until the sequence is one of 64 from b0 on
      const int mid = (b0 + hi + 1) >> 1;
      if (d.seq_off[mid] / len + mid <= slot)
        b0 = mid;
      else
        hi = mid - 1;
    }
  }
  const int b = min(b0 + ((int)threadIdx.x & 63), d.B - 1);
  const int s0 = d.seq_off[b], s1 = d.seq_off[b + 1], p0 = d.pos0[b], on = d.live ? d.live[b] : 1;
  if (p.count == 0) {
    const unsigned long long m = __ballot(s0 / len + b <= slot);       // (true in lane 0, and up to the sequence that owns the slot)
    lo = min(b0 + 63 - __builtin_clzll(m), d.B - 1);
  }
  const int at = __builtin_amdgcn_readfirstlane(lo) - b0;
  const int o0 = __builtin_amdgcn_readlane(s0, at), o1 = __builtin_amdgcn_readlane(s1, at);
  c.s = b0 + at;
  c.idx = slot - (p.count > 0 ? c.s * p.count - p.first : o0 / len + c.s);
  c.t0 = o0 + c.idx * len;
  c.n = min(len, o1 - c.t0);
  c.pos0 = __builtin_amdgcn_readlane(p0, at);
  return c.idx >= 0 && c.n > 0 && __builtin_amdgcn_readlane(on, at);
}
// a sequence's pieces here: how many, and the slot of the first
template <int LEN>
__device__ __forceinline__ int own_pieces(const SeqDesc& d, const Pieces& p, int s, int& slot) {
  const int len = LEN > 0 ? LEN : p.len, o0 = d.seq_off[s], all = (d.seq_off[s + 1] - o0 + len - 1) / len;
  slot = p.count > 0 ? s * p.count : o0 / len + s;
  return p.count > 0 ? min(all - p.first, p.count) : all;
}

// Slots and windows for at most `most` floats at `per` a slot; no slots: the token-by-token form is to run, at token_us a token of the
// mean length (a window costs 15 us at least, and one sequence may hold nearly all the tokens).
struct PiecePlan {
  size_t slots;
  int count, windows;
};
inline PiecePlan plan_pieces(int T_, int B, int len, size_t per, size_t most, float token_us) {
  const size_t all = (size_t)T_ / len + B;
  if (all * per <= most) return {all, 0, 1};
  const size_t count = most / (per * B);
  if (count == 0) return {0, 0, 0};
  const int windows = (int)((((size_t)T_ + len - 1) / len + count - 1) / count);
  if (15.f * windows > token_us * T_ / B) return {0, 0, 0};
  return {count * B, (int)count, windows};
}

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float softplusf_(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float gelu_tanhf_(float v) {
  return 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
}
__device__ __forceinline__ float logsigmoidf_(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

// ln(1 + e^-a) for a >= 0 as 2 atanh(e / (2 + e)), e = e^-a: the argument stays below 1/3, so eight terms of the odd series
// reach float accuracy without a table or a branch (the staging of a chunk evaluates one per element).
__device__ __forceinline__ float log1p_exp_neg(float a) {
  const float e = __builtin_amdgcn_exp2f(a * -1.4426950408889634f), s = e * __builtin_amdgcn_rcpf(2.f + e), q = s * s;
  float p = 1.f / 17.f;
  p = p * q + 1.f / 15.f;
  p = p * q + 1.f / 13.f;
  p = p * q + 1.f / 11.f;
  p = p * q + 1.f / 9.f;
  p = p * q + 1.f / 7.f;
  p = p * q + 1.f / 5.f;
  p = p * q + 1.f / 3.f;
  return 2.f * s * (p * q + 1.f);
}

// Two floats as sums of three bf16 numbers each, h + m + l, which hold their 24 bits exactly (an infinity stays one: what it leaves is
// no number, and is bounded).  By cutting, since packing the upper halves of two words is one instruction.
struct Split {
  unsigned h, m, l;
};
__device__ __forceinline__ Split split3(float x0, float x1) {
  const auto upper = [](float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); };
  const auto pack = [](float a, float b) { return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u); };
  const float r0 = __builtin_amdgcn_fmed3f(x0 - upper(x0), -0x1p120f, 0x1p120f),
              r1 = __builtin_amdgcn_fmed3f(x1 - upper(x1), -0x1p120f, 0x1p120f);
  return {pack(x0, x1), pack(r0, r1), pack(r0 - upper(r0), r1 - upper(r1))};
}

// sums of two values over exchanged lanes
__device__ __forceinline__ float swap32_add(float a, float b) {       // lanes 0-31: sum of a, lanes 32-63: sum of b
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap16_add(float a, float b) {       // even rows: sum of a over a pair of rows, odd: of b
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Entry c of a vector whose first `dims` entries are rotated by pos * inv_freq[pair]: neighbours (2i, 2i+1) form pair
// i, or with `half` entries (i, i + dims/2) do; the rest pass unchanged.  Sine and cosine are multiplied by mag.
// The pair (u, v) becomes (u cos - v sin, v cos + u sin); the angle is a float product.
template <typename T>
__device__ __forceinline__ float rotated_at(const T* __restrict__ v, int c, int dims, float pos,
                                            const float* __restrict__ inv_freq, int half, float mag) {
  const float a = (float)v[c];
  if (c >= dims) return a;
  const int hd = dims >> 1;
  const bool second = half ? c >= hd : (c & 1);
  const int pair = half ? (second ? c - hd : c) : (c >> 1);
  const float b = (float)v[half ? (second ? c - hd : c + hd) : (c ^ 1)];
  float sn, cs;
  sincosf(pos * inv_freq[pair], &sn, &cs);
  sn *= mag;
  cs *= mag;
  return second ? a * cs + b * sn : a * cs - b * sn;
}

// sum over a 256-thread block (4 waves); result in every thread
__device__ __forceinline__ float block_sum256(float v, float* scratch) { return block_sum<4>(v, scratch); }

}  // namespace lipa

#define SEQ_DISPATCH_T(code, ...)              \
  do {                                         \
    if ((code) == 0) {                         \
      using T = lipa::bf16;                    \
      __VA_ARGS__;                             \
    } else {                                   \
      using T = float;                         \
      __VA_ARGS__;                             \
    }                                          \
  } while (0)
