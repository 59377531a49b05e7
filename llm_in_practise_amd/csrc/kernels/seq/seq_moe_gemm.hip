// Routed experts of a prompt: every expert's products over its run of (token, expert) pairs in two launches, without a host
// round trip.  A first kernel orders the pairs by expert; the products then run over tiles of 128 pairs of one expert - the first
// gathers its rows of the input as it loads them and ends in the gated activation, so neither the gathered input nor the gate
// and up products ever stand in memory.
//
// 8000 tokens of width 2048, 8 experts of 384, top 2 (75 GFLOP): 638 -> 143 us with routing and the weighted sum: order 5, first
// products 60 (840 TFLOP/s), second 40 (630), sum 26, routing 13 (171 where the inputs come from memory).  100 tokens: 533 -> 40 us.  The sort, the host's read of the run lengths
// and a vendor product pair, an activation and their launch gaps per expert took 500 us at any number of tokens.
#include "seq_common.h"

#include <type_traits>

using namespace lipa;

namespace {

constexpr int BM = 128, BK = 64;                // pairs and depth of a tile

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __amdgpu_buffer_rsrc_t rsrc;

constexpr int PT = 1024;                        // threads of the ordering kernel

// Blocks (e, part): expert e's place in the order is the number of pairs of lower experts, that of a part of its pairs behind the
// ones in front of it; pairs keep their order.  perm: pair at a place; pos: place of a pair (0 for pairs of no expert); offs [E + 1].
// Every block counts over all pairs, four neighbouring ones a load and four loads on their way, then places its part: parts of 4096
// pairs, one turn of the block, as long as there are 256 blocks or fewer.  Bound by latency: one block an expert that read turn after
// turn, twice, took 14 us for 16000 pairs of 8 experts; this 5.5 (24000 pairs 7, 200 4).
typedef int int4u __attribute__((ext_vector_type(4), aligned(4)));
constexpr int TURN = 4 * PT;
__global__ __launch_bounds__(PT) void k_moe_order(const int* __restrict__ idx, int P, int E, int turns, int* __restrict__ offs,
                                                  int* __restrict__ perm, long* __restrict__ pos) {
  __shared__ int wsum[PT / 64], wlow[PT / 64], wall[PT / 64];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, first = blockIdx.y * turns, all = (P + TURN - 1) / TURN;
  auto load = [&](int turn) {
    const int p = turn * TURN + 4 * tid;
    int4u v = {-1, -1, -1, -1};
    if (p + 4 <= P) {
      v = *reinterpret_cast<const int4u*>(idx + p);
    } else {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (p + i < P) v[i] = idx[p + i];
    }
    return v;
  };
  const int4u mine = load(first);
  int low = 0, before = 0, eq = 0;                     // (eq: of the block that writes the last place)
  auto count = [&](const int4u& v, bool ahead) {
    int n = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      low += (unsigned)v[i] < (unsigned)e;
      n += v[i] == e;
    }
    eq += n;
    before += ahead ? n : 0;
  };
  for (int t = 0; t < all - 1; t += 4) {               // all turns but the block's own first one
    int4u v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = load(t + j + (t + j >= first));     // (turns past the last one load nothing)
#pragma unroll
    for (int j = 0; j < 4; ++j) count(v[j], t + j < first);
  }
  count(mine, false);
  auto total = [&](int v, int* part) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) part[w] = v;
  };
  const bool last = e == E - 1 && blockIdx.y == 0;
  total(low, wlow);
  if (first > 0) total(before, wsum);
  if (last) total(eq, wall);
  __syncthreads();
  int at = 0, ahead0 = 0, count0 = 0;
#pragma unroll
  for (int i = 0; i < PT / 64; ++i) {
    at += wlow[i];
    ahead0 += first > 0 ? wsum[i] : 0;
    count0 += last ? wall[i] : 0;
  }
  if (tid == 0 && blockIdx.y == 0) {
    offs[e] = at;
    if (last) offs[E] = at + count0;
  }
  at += ahead0;
  for (int t = first; t < min(first + turns, all); ++t) {
    const int4u v = t == first ? mine : load(t);
    const int p = t * TURN + 4 * tid;
    int ahead = 0, count = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned long long m = __ballot(v[i] == e);
      ahead += __popcll(m & ((1ull << lane) - 1));
      count += __popcll(m);
    }
    __syncthreads();                                  // the last counts are read
    if (lane == 0) wsum[w] = count;
    __syncthreads();
    int turn = 0;
#pragma unroll
    for (int i = 0; i < PT / 64; ++i) {
      ahead += i < w ? wsum[i] : 0;
      turn += wsum[i];
    }
    int place = at + ahead;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (v[i] == e) {
        perm[place] = p + i;
        pos[p + i] = place++;
      } else if (e == 0 && p + i < P && (v[i] < 0 || v[i] >= E)) {
        pos[p + i] = 0;
      }
    }
    at += turn;
  }
}

__device__ __forceinline__ rsrc window(const void* base, uint32_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p), hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0,
                                           __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}
// 64 lanes x 16 bytes from memory into LDS [dst, dst + 1 KB), lane after lane; M0 is put back
__device__ __forceinline__ void to_lds(const rsrc& rs, uint32_t dst, uint32_t voff, uint32_t soff) {
  uint32_t keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %2, %3, %4 offen lds\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(keep)
      : "s"(dst), "v"(voff), "s"(rs), "s"(soff)
      : "memory");
}

// 1 / (1 + e^-x) without a division's and expf's forty instructions (they took 5 of a tile's 30 us): e^-|x| with the exponent's rounding
// error put back, one Newton step behind the reciprocal.  Largest error from -86 to 88: 1.8e-7 of the value.
__device__ __forceinline__ float sigmoid_fast(float x) {
  const float a = fminf(fabsf(x), 126.f), t = -1.44269502f * a, lo = fmaf(-1.44269502f, a, -t) - 1.92596299e-8f * a;
  float e = __builtin_amdgcn_exp2f(t);
  e = fmaf(e, 0.69314718f * lo, e);
  const float d = 1.f + e, y = __builtin_amdgcn_rcpf(d), r = fmaf(y, fmaf(-d, y, 1.f), y);
  return x < 0.f ? e * r : r;
}
__device__ __forceinline__ float glu(float g, float u, float limit, int mode) {       // 1: clipped GLU, 2: SiLU GLU
  if (mode == 2) return g * sigmoid_fast(g) * u;
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoid_fast(1.702f * g) * (u + 1.f);
}

struct Rows {
  const int *offs, *perm;
  int E, P, top;
};

// UP: out[place, f] = glu(wg_f . x, wu_f . x) with x = the pair's row of the input, BN / 2 gate rows and their up rows a tile.
// Otherwise out[place, c] = w_c . x with x = the place's row.  K: depth; N: columns of out.
// 2 x WN waves; weights are the first operand, so a lane holds one pair's products for neighbouring columns, and the result goes
// through LDS to leave in whole rows.  RING stages of depth BK in LDS.
//
// A tile of the first products is 32 steps of 0.75 us against 0.6 of its products alone (the matrix cores' clock falls under load); what
// it waited for: rows on their way (two stages ahead 27 us a tile, one stage 34), the address unit taking eight loads in front of the
// products, a barrier and a round trip to LDS a step, half of LDS's cycles in bank conflicts (a wave's 16-byte reads of 32 rows of 128
// bytes are free of them when the chunk is turned by row / 2, not by row), expf and a division an element.  Tiles of 128 x 128 with two stages
// and none of this, two blocks a CU -> 128 x 256, three stages, us: 12000 tokens 104 -> 92, 8000 80 -> 61, 5000 59 -> 54.  256 x 256: 108,
// 59, 52.  The second products have a depth of 6 steps and are bound by their first loads and the
// results' way out: two blocks a CU of 128 x 128 and two stages 42 us at 8000 tokens, of 128 x 256 43, one block with three stages 53.
template <bool UP, int WN, int BN, int RING>
__global__ __launch_bounds__(128 * WN, 2) void k_moe_tiles(const bf16* __restrict__ x, const bf16* __restrict__ wt,
                                                      const float* __restrict__ rs, bf16* __restrict__ out, Rows r, int K, int N,
                                                      float limit, int mode) {
  constexpr int NW = 2 * WN;                    // waves
  constexpr int COLS = UP ? BN / 2 : BN;        // columns of out per tile
  constexpr int TN = BN / (32 * WN);            // tiles of 32 weight rows a wave
  constexpr int KS = BK / 16, ROW = 2 * BK;     // bytes of a staged row: eight lanes load it
  constexpr int WIMG = BN * ROW, STAGE = WIMG + BM * ROW, LDR = COLS + 8;
  constexpr int WP = WIMG / (1024 * NW), LOADS = STAGE / (1024 * NW);          // a wave's 1 KB pieces of a stage: weights, all
  static_assert(WP * 1024 * NW == WIMG && LOADS * 1024 * NW == STAGE);
  constexpr int LDS = RING * STAGE > BM * LDR * 2 ? RING * STAGE : BM * LDR * 2;
  __shared__ __attribute__((aligned(1024))) char lds[LDS];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int nt = (N + COLS - 1) / COLS, tile = xcd_remap(blockIdx.x, gridDim.x), mt = tile / nt, n0 = (tile % nt) * COLS;
  // expert e owns the row tiles offs[e] / BM + e, ..; a wave looks at 64 experts at a time
  int e = -1;
  for (int e0 = 0; e0 < r.E; e0 += 64) {
    const int j = min(e0 + lane, r.E - 1);
    e += __popcll(__ballot(e0 + lane < r.E && r.offs[j] / BM + j <= mt));
  }
  e = __builtin_amdgcn_readfirstlane(e);
  const int o0 = r.offs[e], m0 = o0 + (mt - (o0 / BM + e)) * BM, m = min(BM, r.offs[e + 1] - m0);
  if (m0 < o0 || m <= 0) return;
  // rows of the operands that this lane loads: neighbouring lanes load a row, chunk c of row i to slot c ^ swz(i) of the staged row
  auto swz = [](int i) { return i >> 1 & 7; };
  const size_t wbytes = (size_t)(UP ? 2 : 1) * N * K * 2;
  const rsrc wr = window(wt + (size_t)e * (UP ? 2 : 1) * N * K, (uint32_t)wbytes);
  const rsrc xr = window(x, 0xFFFFFFFFu);
  uint32_t off[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int i = 8 * (j < WP ? WP * w + j : (LOADS - WP) * w + j - WP) + (lane >> 3);
    int row;
    if (j < WP) {
      row = UP ? i / COLS * N + min(n0 + i % COLS, N - 1) : min(n0 + i, N - 1);
    } else {
      const int place = m0 + min(i, m - 1);
      row = UP ? r.perm[place] / r.top : place;
    }
    off[j] = (uint32_t)row * (uint32_t)K * 2 + ((lane & 7) ^ swz(i)) * 16;
  }
  const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)lds);
  auto load = [&](int j, int stage, int k0) {
    const uint32_t dst = base + stage * STAGE;
    if (j < WP)
      to_lds(wr, dst + (WP * w + j) * 1024, off[j], k0 * 2);
    else
      to_lds(xr, dst + WIMG + ((LOADS - WP) * w + j - WP) * 1024, off[j], k0 * 2);
  };
  const int l32 = lane & 31, half = lane >> 5, wm = w & 1, wn = w >> 1;
  f32x16 acc[TN][2];                            // [weight rows][pairs]
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
  // first of the 32 weight rows of tile t: gate rows, then their up rows
  auto first = [&](int t) {
    return UP ? t / (TN / 2) * COLS + COLS / WN * wn + 32 * (t % (TN / 2)) : COLS / WN * wn + 32 * t;
  };
  const int steps = K / BK;
#pragma unroll
  for (int s = 0; s < RING; ++s)
    if (s < steps)
#pragma unroll
      for (int j = 0; j < LOADS; ++j) load(j, s, s * BK);
  bf16x8 a[2][TN], b[2][2];                     // the operands of two neighbouring 16 of the depth
  auto read = [&](int stage, int ks) {
    const char *wp = lds + stage * STAGE + l32 * ROW, *xp = lds + stage * STAGE + WIMG + (64 * wm + l32) * ROW;
    const int c = ((2 * ks + half) ^ swz(l32)) * 16;
#pragma unroll
    for (int u = 0; u < 2; ++u) b[ks & 1][u] = *reinterpret_cast<const bf16x8*>(xp + u * 32 * ROW + c);
#pragma unroll
    for (int t = 0; t < TN; ++t) a[ks & 1][t] = *reinterpret_cast<const bf16x8*>(wp + first(t) * ROW + c);
  };
  // `later`: stages that may be on their way while this wave goes on
  auto arrive = [&](int later) {
    if (later == 2 && RING == 3)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * LOADS) : "memory");
    else if (later >= 1)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  arrive(min(RING, steps) - 1);
  read(0, 0);
  // A step multiplies stage i.  Its last operands are read in front of the last products; there the next stage is awaited and its first
  // operands are read, so that these products cover the barrier and the way out of LDS.  Then the stage is free: the loads that refill it
  // go out one by one between the next step's products (all at once they hold up the wave until the address unit has them).
  auto step = [&](int i, int st, auto refill, auto next) {
    const int prev = st == 0 ? RING - 1 : st - 1, succ = st == RING - 1 ? 0 : st + 1;
    constexpr int EACH = (LOADS + (KS - 1) * TN - 1) / ((KS - 1) * TN);      // loads behind a pair of products
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 1 < KS) {
        read(st, ks + 1);
      } else if constexpr (next) {
        arrive(refill ? RING - 2 : min(steps - i - 2, RING - 2));
        read(succ, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < TN; ++t) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks & 1][t], b[ks & 1][u], acc[t][u], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (refill)
#pragma unroll
          for (int j = (ks * TN + t) * EACH; j < min(LOADS, (ks * TN + t + 1) * EACH); ++j) load(j, prev, (i + RING - 1) * BK);
      }
    }
  };
  static_assert(KS % 2 == 0 && (RING == 2 || RING == 3));
  int i = 1, st = 1;
  if (steps > 1)
    step(0, 0, std::false_type{}, std::true_type{});
  for (; i + RING - 1 < steps; ++i, st = st == RING - 1 ? 0 : st + 1) step(i, st, std::true_type{}, std::true_type{});
  for (; i + 1 < steps; ++i, st = st == RING - 1 ? 0 : st + 1) step(i, st, std::false_type{}, std::true_type{});
  step(steps - 1, steps == 1 ? 0 : st, std::false_type{}, std::false_type{});
  __syncthreads();
  // results: staged as [pair][COLS] bf16 rows (16 bytes of padding), then stored 16 bytes a lane
  bf16* res = reinterpret_cast<bf16*>(lds);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = 64 * wm + 32 * u + l32;
    float s = 1.f;
    if (UP && rs != nullptr) s = rs[r.perm[m0 + min(i, m - 1)]];
    auto put = [&](auto value) {
#pragma unroll
      for (int t = 0; t < (UP ? TN / 2 : TN); ++t)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          bf16x4 v;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = (bf16)value(t, 4 * g4 + q);
          *reinterpret_cast<bf16x4*>(res + i * LDR + first(t) + 8 * g4 + 4 * half) = v;
        }
    };
    if (!UP)
      put([&](int t, int j) { return acc[t][u][j]; });
    else if (mode == 2)
      put([&](int t, int j) { return glu(s * acc[t][u][j], s * acc[TN - TN / 2 + t][u][j], limit, 2); });
    else
      put([&](int t, int j) { return glu(s * acc[t][u][j], s * acc[TN - TN / 2 + t][u][j], limit, 1); });
  }
  __syncthreads();
  constexpr int PER = COLS / 8;                 // lanes of a row
  for (int i = tid / PER; i < m; i += 64 * NW / PER) {
    const int c = (tid % PER) * 8;
    if (n0 + c < N)
      *reinterpret_cast<bf16x8*>(out + (size_t)(m0 + i) * N + n0 + c) = *reinterpret_cast<const bf16x8*>(res + i * LDR + c);
  }
}

template <bool UP, int WN, int BN, int RING>
void tiles(const void* x, const void* wt, const float* rs, void* out, const Rows& r, int K, int N, float limit, int mode, hipStream_t st) {
  constexpr int COLS = UP ? BN / 2 : BN;
  hipLaunchKernelGGL((k_moe_tiles<UP, WN, BN, RING>), dim3((r.P / BM + r.E) * ((N + COLS - 1) / COLS)), dim3(128 * WN), 0, st,
                     (const bf16*)x, (const bf16*)wt, rs, (bf16*)out, r, K, N, limit, mode);
}

}  // namespace

// bf16, depths that are multiples of 64, rows that 16-byte loads take, operands inside a 32-bit window
bool seq_moe_tiles_ok(int code, const void* h, const void* wgu, const void* wd, long T_, int top, int E, int F, int W) {
  const auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const long big = 1L << 32, P = T_ * top;
  return code == 0 && E >= 1 && F >= 64 && W >= 64 && F % 64 == 0 && W % 64 == 0 && aligned(h) && aligned(wgu) && aligned(wd) &&
         T_ * W * 2 < big && P * F * 2 < big && P * W * 2 < big && 2L * F * W * 2 < big;
}

// offs int [E + 1], perm int [T * top], pos [T * top], a [T * top, F], ys [T * top, W]; wts: a factor of every pair's input, or null
void seq_moe_tiles(const void* h, const void* wgu, const void* wd, const int* idx, const float* wts, int* offs, int* perm, long* pos,
                   void* a, void* ys, int T_, int top, int E, int F, int W, float limit, int mode, hipStream_t st) {
  const int P = T_ * top;
  if (P == 0) return;
  const Rows r = {offs, perm, E, P, top};
  const int mt = P / BM + E;
  const int all = (P + TURN - 1) / TURN, parts = min(all, max(1, 256 / E)), turns = (all + parts - 1) / parts;
  hipLaunchKernelGGL(k_moe_order, dim3(E, (all + turns - 1) / turns), dim3(PT), 0, st, idx, P, E, turns, offs, perm, pos);
  // Where every CU gets one tile of 128 x 128 at most, three stages; where there are more, tiles twice as wide unless they would pad
  // the columns by more than a twentieth, and two blocks a CU otherwise.  us, 2 x 128 two stages / 2 x 128 three / 4 x 256 three, with the
  // second products, routing and sum: 8 experts, width 2048, F 384, tokens 100 51 / 42 / 47, 1500 (186 blocks) 61 / 52 / 57, 3000 (324)
  // 80 / 83 / 74, 8000 154 / 163 / 147; width 1024, F 448, 1500 (217) 41 / 37 / 41, 3000 51 / 54 / 50, 8000 102 / 106 / 114, 12000 139 / 147 / 157;
  // top 4, F 512, width 2048, 700 (232) 65 / 57 / 63, 1500 (432) 82 / 85 / 78, 12000 465 / 485 / 449.  Second products at 200 tokens (176
  // blocks) 7.9 / 6.8, at 1500 (496) 11.7 / 12.9.
  const int wide = (F + 127) / 128 * 128;
  if (mt * ((F + 63) / 64) <= 256)
    tiles<true, 2, 128, 3>(h, wgu, wts, a, r, W, F, limit, mode, st);
  else if (20 * wide <= 21 * F)
    tiles<true, 4, 256, 3>(h, wgu, wts, a, r, W, F, limit, mode, st);
  else
    tiles<true, 2, 128, 2>(h, wgu, wts, a, r, W, F, limit, mode, st);
  if (mt * ((W + 127) / 128) <= 256)
    tiles<false, 2, 128, 3>(a, wd, nullptr, ys, r, F, W, limit, mode, st);
  else
    tiles<false, 2, 128, 2>(a, wd, nullptr, ys, r, F, W, limit, mode, st);
  LIPA_CHECK_LAUNCH();
}
