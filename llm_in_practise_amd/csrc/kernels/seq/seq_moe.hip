// Mixture-of-experts feed-forward for serving: group-limited top-k routing over softmax scores with a selection-only
// correction and identity experts; a few-token path in which every (token, chosen expert) pair streams its expert's
// rows (no sort, no host round trip: decode steps and hipGraphs); and the weighted combine of expert outputs.
// Routing variants (`kind` bits): scores as each output's own sigmoid instead of the softmax (1), a group ranked by the
// sum of its two largest choices instead of its largest (2), weights divided by their sum over the chosen (4), the
// correction added to the logits, so that it moves the scores and weights too (8).
// Experts are clipped GLUs or SiLU GLUs; a pair's weight multiplies the expert's output or its input; the shared expert may sit behind a per-token sigmoid gate.
// Router scores, weights and the combine are float; expert products read the activation type and accumulate in float.
#include "seq_common.h"

#include <type_traits>

using namespace lipa;

constexpr int RPL = 4;   // router outputs per lane: experts + identity experts <= 64 * RPL

// the value of lane ^ M inside rows of 16, by a move between lanes where one does it: a trip through LDS takes ten times as long,
// and routing is one chain of them
template <int M>
__device__ __forceinline__ int lane_xor(int v) {
  if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);          // quad_perm [1, 0, 3, 2]
  else if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);     // quad_perm [2, 3, 0, 1]
  else if constexpr (M == 4)                                                               // row_shl:4, row_shr:4 in lanes 4-7, 12-15
    return __builtin_amdgcn_update_dpp(__builtin_amdgcn_mov_dpp(v, 0x104, 0xF, 0xF, true), v, 0x114, 0xF, 0xA, false);
  else if constexpr (M == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);    // row_ror:8
  else return __shfl_xor(v, M, 64);
}
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
  return __int_as_float(lane_xor<M>(__float_as_int(v)));
}
// (value, index) maximum over GW lanes; ties go to the lower index
template <int GW>
__device__ __forceinline__ void group_argmax(float& v, int& i) {
  const float ov = lane_xor<GW / 2>(v);
  const int oi = lane_xor<GW / 2>(i);
  if (ov > v || (ov == v && oi < i)) {
    v = ov;
    i = oi;
  }
  if constexpr (GW > 2) group_argmax<GW / 2>(v, i);
}
template <int GW>
__device__ __forceinline__ float group_max(float v) {
  v = fmaxf(v, lane_xor<GW / 2>(v));
  if constexpr (GW > 2) v = group_max<GW / 2>(v);
  return v;
}
template <int GW>
__device__ __forceinline__ float group_add(float v) {
  v += lane_xor<GW / 2>(v);
  if constexpr (GW > 2) v = group_add<GW / 2>(v);
  return v;
}
// v[i] and v[i + HALF] of lanes `HALF` apart: a lane keeps the sum of the one that its bit names
template <int HALF>
__device__ __forceinline__ void fold(float (&v)[64], int lane) {
  const bool up = lane & HALF;
#pragma unroll
  for (int i = 0; i < HALF; ++i) {
    const float keep = up ? v[i + HALF] : v[i], send = up ? v[i] : v[i + HALF];
    v[i] = keep + lane_xor<HALF>(send);
  }
  if constexpr (HALF > 1) fold<HALF / 2>(v, lane);
}

// GW lanes route one token from its n router logits, RP a lane (z[i]: output lane + GW i).  s = softmax(z) over all n outputs;
// choice = s + corr; the n outputs form `groups` equal runs of neighbours, a group's score is its largest choice and
// only the `keep` best groups stay eligible; the `top` largest eligible choices are taken and weighted by s * scale
// (s without the correction, not renormalised).  `always` more ids n, n + 1, .. of weight 1 follow the chosen ones (experts
// that every token uses).
template <int GW, int RP>
__device__ __forceinline__ void route_lanes(const float (&z)[RP], const float* __restrict__ corr, int* __restrict__ idx,
                                           float* __restrict__ wout, int lane, int n, int top, int groups, int keep,
                                           float scale, int kind, int always) {
  float s[RP], ch[RP];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    const int e = lane + GW * i;
    // a row nobody reads (an idle decode row) may carry anything, NaN included: it still gets ids inside [0, n)
    s[i] = e < n ? (isfinite(z[i]) ? z[i] : 0.f) : -INFINITY;
    if ((kind & 8) && e < n && corr != nullptr) s[i] += corr[e];
    mx = fmaxf(mx, s[i]);
  }
  mx = group_max<GW>(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    if (kind & 1)
      s[i] = lane + GW * i < n ? sigmoidf_(s[i]) : 0.f;
    else
      s[i] = lane + GW * i < n ? expf(s[i] - mx) : 0.f;
    sum += s[i];
  }
  sum = (kind & 1) ? 1.f : group_add<GW>(sum);
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    const int e = lane + GW * i;
    s[i] /= sum;
    ch[i] = e < n ? s[i] + (corr != nullptr && !(kind & 8) ? corr[e] : 0.f) : -INFINITY;
  }
  if (groups > 1 && keep < groups && (kind & 2)) {
    // rank of group g = its largest choice + its second largest (a group of one: the one), held by lane g
    const int gs = n / groups;
    float rank = -INFINITY;
    for (int g = 0; g < groups; ++g) {
      float b1 = -INFINITY;
      int e1 = 1 << 30;
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        const int e = lane + GW * i;
        if (e < n && e / gs == g && (ch[i] > b1 || (ch[i] == b1 && e < e1))) {
          b1 = ch[i];
          e1 = e;
        }
      }
      group_argmax<GW>(b1, e1);
      float b2 = -INFINITY;
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        const int e = lane + GW * i;
        if (e < n && e / gs == g && e != e1) b2 = fmaxf(b2, ch[i]);
      }
      b2 = group_max<GW>(b2);
      if (lane == g) rank = b1 + (b2 == -INFINITY ? 0.f : b2);
    }
    unsigned long long kept = 0ull;               // groups <= GW
    for (int r = 0; r < keep; ++r) {
      float bv = rank;
      int bg = lane < groups ? lane : 1 << 30;
      group_argmax<GW>(bv, bg);
      if (bg < groups) kept |= 1ull << bg;
      if (lane == bg) rank = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      const int e = lane + GW * i;
      if (e < n && !((kept >> (e / gs)) & 1ull)) ch[i] = -INFINITY;
    }
  } else if (groups > 1 && keep < groups) {
    const int gs = n / groups;
    // a lane's outputs may lie in different groups: the kept-group mask is built by `keep` rounds of
    // "best remaining group", each an argmax over (choice, group) pairs
    unsigned long long kept = 0ull;               // groups <= GW
    for (int r = 0; r < keep; ++r) {
      float bv = -INFINITY;
      int bg = 1 << 30;
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        const int e = lane + GW * i, g = e / gs;
        if (e < n && !((kept >> g) & 1ull) && (ch[i] > bv || (ch[i] == bv && g < bg))) {
          bv = ch[i];
          bg = g;
        }
      }
      group_argmax<GW>(bv, bg);
      if (bg < groups) kept |= 1ull << bg;
    }
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      const int e = lane + GW * i;
      if (e < n && !((kept >> (e / gs)) & 1ull)) ch[i] = -INFINITY;
    }
  }
  unsigned taken = 0u;                            // bit i: this lane's output i is already chosen
  float tot = 0.f, myw = 0.f;                     // lane r keeps the r-th choice (top <= GW)
  int myid = 0;
  for (int r = 0; r < top; ++r) {
    float bv = -INFINITY;
    int be = 1 << 30;
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      const int e = lane + GW * i;
      if (e < n && !((taken >> i) & 1u) && (ch[i] > bv || (ch[i] == bv && e < be))) {
        bv = ch[i];
        be = e;
      }
    }
    group_argmax<GW>(bv, be);
    be = min(be, n - 1);                          // (only when fewer than `top` outputs are eligible)
    float cand = 0.f;
#pragma unroll
    for (int i = 0; i < RP; ++i)
      if (i == (be / GW)) cand = s[i];
    const float bs = __shfl(cand, be % GW, GW);
    if ((be % GW) == lane) taken |= 1u << (be / GW);
    tot += bs;
    if (lane == r) {
      myw = bs;
      myid = be;
    }
  }
  if (lane < top) {
    idx[lane] = myid;
    wout[lane] = ((kind & 4) ? myw / (tot + 1e-20f) : myw) * scale;
  } else if (lane < top + always) {
    idx[lane] = n + lane - top;
    wout[lane] = 1.f;
  }
}

// one wave per token, logits in memory or LDS
__device__ __forceinline__ void route_wave(const float* z, const float* __restrict__ corr, int* __restrict__ idx,
                                           float* __restrict__ wout, int lane, int n, int top, int groups, int keep,
                                           float scale, int kind, int always) {
  float v[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) v[i] = lane + 64 * i < n ? z[lane + 64 * i] : 0.f;
  route_lanes<64, RPL>(v, corr, idx, wout, lane, n, top, groups, keep, scale, kind, always);
}

// routing from given logits: one wave per token
__global__ __launch_bounds__(256) void k_route_grouped(const float* __restrict__ z, const float* __restrict__ corr,
                                                       int* __restrict__ idx, float* __restrict__ wout, int T_, int n,
                                                       int top, int groups, int keep, float scale, int kind) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T_) return;
  route_wave(z + (size_t)t * n, corr, idx + (size_t)t * top, wout + (size_t)t * top, lane, n, top, groups, keep, scale,
             kind, 0);
}

// four entries of an activation row as floats (16-byte rows when the width allows)
__device__ __forceinline__ f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 load4(const bf16* p) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

// router product and routing in one kernel: one block of NW waves per token (16 for the few tokens of a decode step,
// so that its few blocks have many loads in flight; 4 for prompts).  A work item is (four router rows, one interleaved
// quarter of the columns): four independent accumulators over 16-byte loads; float weights, activations as they are,
// float accumulation.  Partial sums meet in LDS, then wave 0 routes.
template <typename T, int NW>
__global__ __launch_bounds__(64 * NW) void k_route_fused(const T* __restrict__ h, int ldh, const float* __restrict__ router,
                                                      const float* __restrict__ corr, int* __restrict__ idx,
                                                      float* __restrict__ wout, int n, int W, int top, int groups,
                                                      int keep, float scale, int kind, int extra,
                                                      float* __restrict__ xout, int always) {
  // n counts all router rows; the last `extra` of them are not routed: their products go to xout [T, extra]
  __shared__ float part[64 * RPL][4];
  __shared__ float sz[64 * RPL];
  const int t = blockIdx.x, wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const T* x = h + (size_t)t * ldh;
  const bool vec = (W & 3) == 0 && (ldh & 3) == 0;
  const int items = ((n + 3) / 4) * 4;
  for (int it = wv; it < items; it += NW) {
    const int e0 = 4 * (it >> 2), qt = it & 3;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    const float* r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = router + (size_t)min(e0 + i, n - 1) * W;
    if (vec) {
#pragma unroll 2
      for (int c = 4 * lane + 256 * qt; c < W; c += 1024) {
        const f32x4 xv = load4(x + c);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 rv = load4(r[i] + c);
          acc[i] += rv[0] * xv[0] + rv[1] * xv[1] + rv[2] * xv[2] + rv[3] * xv[3];
        }
      }
    } else {
      for (int c = lane + 64 * qt; c < W; c += 256) {
        const float xv = (float)x[c];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += r[i][c] * xv;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = wave_sum(acc[i]);
      if (lane == 0 && e0 + i < n) part[e0 + i][qt] = v;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n; e += 64 * NW) sz[e] = (part[e][0] + part[e][1]) + (part[e][2] + part[e][3]);
  __syncthreads();
  for (int e = threadIdx.x; e < extra; e += 64 * NW) xout[(size_t)t * extra + e] = sz[n - extra + e];
  if (wv > 0) return;
  const size_t at = (size_t)t * (top + always);
  if (n - extra <= 16 && top + always <= 16) {             // (the same choices and weights; a chain of moves inside a row of 16 lanes)
    const float z[1] = {lane < n - extra ? sz[lane] : 0.f};
    if (lane < 16) route_lanes<16, 1>(z, corr, idx + at, wout + at, lane, n - extra, top, groups, keep, scale, kind, always);
  } else {
    route_wave(sz, corr, idx + at, wout + at, lane, n - extra, top, groups, keep, scale, kind, always);
  }
}

// The same for prompts and up to 16 outputs: a block takes four tokens, a wave a quarter of their columns, so that a router row
// read from the cache serves four tokens; the 4 x 16 sums over a wave's lanes leave (token, output) in lane 16 token + output, and
// after the four waves' sums meet in LDS each 16 lanes of the first route their token.  8000 float tokens or rows that the tiles below
// do not take, width 2048, 8 outputs: 41 -> 17 us (a block per token read the whole router from L2, 0.6 GB in all, and routed with 64
// lanes); moves between lanes through LDS instead of between registers 19.  Bound by issue, 8 waves a SIMD of 800 instructions; 6 blocks
// a CU spill and take 20 us, 8 32.
template <typename T, int NG>
__global__ __launch_bounds__(256) void k_route_rows(const T* __restrict__ h, int ldh, const float* __restrict__ router,
                                                    const float* __restrict__ corr, int* __restrict__ idx,
                                                    float* __restrict__ wout, int T_, int n, int W, int top, int groups, int keep,
                                                    float scale, int kind, int extra, float* __restrict__ xout, int always) {
  __shared__ float part[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t0 = blockIdx.x * 4;
  float v[64];
#pragma unroll
  for (int i = 0; i < 64; ++i) v[i] = 0.f;
#pragma unroll 2
  for (int c = 4 * lane + 256 * w; c < W; c += 1024) {
    f32x4 x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = load4(h + (size_t)min(t0 + i, T_ - 1) * ldh + c);
#pragma unroll
    for (int o = 0; o < 4 * NG; ++o) {
      const f32x4 r = load4(router + (size_t)min(o, n - 1) * W + c);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[16 * i + o] += r[0] * x[i][0] + r[1] * x[i][1] + r[2] * x[i][2] + r[3] * x[i][3];
    }
  }
#pragma unroll
  for (int i = 0; i < 32; ++i) v[i] = swap32_add(v[i], v[i + 32]);
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = swap16_add(v[i], v[i + 16]);
  fold<8>(v, lane);
  part[w][lane] = v[0];
  __syncthreads();
  const int t = t0 + (lane >> 4), o = lane & 15;
  if (w != 0 || t >= T_) return;
  const float z[1] = {(part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane])};
  if (o >= n - extra && o < n) xout[(size_t)t * extra + o - (n - extra)] = z[0];
  route_lanes<16, 1>(z, corr, idx + (size_t)t * (top + always), wout + (size_t)t * (top + always), o, n - extra, top, groups, keep,
                     scale, kind, always);
}

// The same of bf16 rows on the matrix units: a block takes 16 tokens, a wave every fourth 64 of their columns.  A router weight is the sum of
// three bf16 numbers (split3: its 24 bits), so a product of 32 columns is three of v_mfma_f32_16x16x32_bf16 with float sums.  Rows come
// in pieces of 128 bytes and turn into operands through 8 KB of LDS a wave (pieces of row r turned by r / 2: no bank conflicts);
// operands straight from memory, 64 lines a load, took 12.5 us.  The waves' sums meet in LDS and each 16 lanes route a token.
template <int U, int NG>                      // a wave's pieces of 64 columns on their way at once; router rows / 4
__global__ __launch_bounds__(256, 2) void k_route_tiles(const bf16* __restrict__ h, int ldh, const float* __restrict__ router,
                                                        const float* __restrict__ corr, int* __restrict__ idx,
                                                        float* __restrict__ wout, int T_, int n, int W, int top, int groups, int keep,
                                                        float scale, int kind, int extra, float* __restrict__ xout, int always) {
  __shared__ __attribute__((aligned(16))) bf16 buf[4][4][16 * 64];            // [wave][tokens, the weights' three parts][row][column]
  __shared__ float part[4][16][16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, q = lane >> 4, t0 = blockIdx.x * 16;
  const int r8 = lane >> 3, c8 = lane & 7, r4 = lane >> 4, c4 = lane & 15;    // in memory: rows of 8 or 16 lanes
  const bf16* x[2];
  const float* r[NG];
#pragma unroll
  for (int i = 0; i < 2; ++i) x[i] = h + (size_t)min(t0 + 8 * i + r8, T_ - 1) * ldh + 8 * c8;
#pragma unroll
  for (int g = 0; g < NG; ++g) r[g] = router + (size_t)min(4 * g + r4, n - 1) * W + 4 * c4;
  const auto piece = [](int row, int p) { return 64 * row + 8 * (p ^ ((row >> 1) & 7)); };
  f32x4 hi[4], lo[2];                         // (sums of few terms each: fewer roundings at the sum's size)
#pragma unroll
  for (int i = 0; i < 4; ++i) hi[i] = lo[i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c0 = 64 * w; c0 < W; c0 += 256 * U) {
    bf16x8 a[U][2];
    f32x4 b[2][NG];
    const auto weights = [&](int u) {
#pragma unroll
      for (int g = 0; g < NG; ++g) b[u & 1][g] = *reinterpret_cast<const f32x4*>(r[g] + min(c0 + 256 * u, W - 64));
    };
    weights(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) a[u][i] = *reinterpret_cast<const bf16x8*>(x[i] + min(c0 + 256 * u, W - 64));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u + 1 < U) weights(u + 1);
      const bool on = c0 + 256 * u < W;       // (past the row: its last columns again, which count as 0)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        u32x4 v = __builtin_bit_cast(u32x4, a[u][i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = on ? v[e] : 0u;
        *reinterpret_cast<u32x4*>(buf[w][0] + piece(8 * i + r8, c8)) = v;
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const f32x4 y = b[u & 1][g];
        const Split s0 = split3(y[0], y[1]), s1 = split3(y[2], y[3]);
        bf16* to = buf[w][1] + piece(4 * g + r4, c4 >> 1) + 4 * (c4 & 1);
        *reinterpret_cast<u32x2*>(to) = u32x2{s0.h, s1.h};
        *reinterpret_cast<u32x2*>(to + 1024) = u32x2{s0.m, s1.m};
        *reinterpret_cast<u32x2*>(to + 2048) = u32x2{s0.l, s1.l};
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto at = [&](int k) { return *reinterpret_cast<const bf16x8*>(buf[w][k] + piece(li, 4 * i + q)); };
        const bf16x8 t = at(0);
        f32x4& big = hi[2 * (u & 1) + i];
        big = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t, at(1), big, 0, 0, 0);
        lo[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t, at(3), lo[i], 0, 0, 0);
        lo[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t, at(2), lo[i], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) part[w][4 * q + i][li] = ((hi[0][i] + hi[1][i]) + (hi[2][i] + hi[3][i])) + (lo[0][i] + lo[1][i]);
  __syncthreads();
  const int tt = 4 * w + q, t = t0 + tt, o = li;
  if (t >= T_) return;
  float z[1] = {(part[0][tt][o] + part[1][tt][o]) + (part[2][tt][o] + part[3][tt][o])};
  if (o >= n - extra && o < n) {
    if (!isfinite(z[0])) {               // (an infinity meets weights' parts that are 0: what it is without parts)
      z[0] = 0.f;
      for (int c = 0; c < W; ++c) z[0] += router[(size_t)o * W + c] * (float)h[(size_t)t * ldh + c];
    }
    xout[(size_t)t * extra + o - (n - extra)] = z[0];
  }
  route_lanes<16, 1>(z, corr, idx + (size_t)t * (top + always), wout + (size_t)t * (top + always), o, n - extra, top, groups, keep,
                     scale, kind, always);
}

// g = min(g, limit), u = clamp(u, -limit, limit): g * sigmoid(1.702 g) * (u + 1)
__device__ __forceinline__ float clipped_glu(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoidf_(1.702f * g) * (u + 1.f);
}

// mode 1: the clipped GLU; mode 2: silu(g) * u; mode 3: gelu_tanh(g) * u
__device__ __forceinline__ float glu(float g, float u, float limit, int mode) {
  if (mode == 3) return gelu_tanhf_(g) * u;
  return mode == 2 ? g * sigmoidf_(g) * u : clipped_glu(g, u, limit);
}

template <typename T>
__device__ __forceinline__ float wave_dot(const T* __restrict__ a, const T* __restrict__ b, int n, int lane);

template <>
__device__ __forceinline__ float wave_dot<float>(const float* __restrict__ a, const float* __restrict__ b, int n,
                                                 int lane) {
  float acc = 0.f;
  if ((n & 3) == 0) {
    for (int c = 4 * lane; c < n; c += 256) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(a + c), y = *reinterpret_cast<const f32x4*>(b + c);
      acc += x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3];
    }
  } else {
    for (int c = lane; c < n; c += 64) acc += a[c] * b[c];
  }
  return wave_sum(acc);
}
template <>
__device__ __forceinline__ float wave_dot<bf16>(const bf16* __restrict__ a, const bf16* __restrict__ b, int n, int lane) {
  float acc = 0.f;
  if ((n & 7) == 0) {
    for (int c = 8 * lane; c < n; c += 512) {
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(a + c), y = *reinterpret_cast<const bf16x8*>(b + c);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc += (float)x[j] * (float)y[j];
    }
  } else {
    for (int c = lane; c < n; c += 64) acc += (float)a[c] * (float)b[c];
  }
  return wave_sum(acc);
}

// pairs path, stage 1.  One wave per (pair, hidden unit r): a[pair, r] = glu(Wg_e[r] . h_t, Wu_e[r] . h_t).
// wgu: [E, 2, F, W] (gate rows then up rows of every expert).  Identity pairs (e >= E) have nothing to compute.
// inw (or null): a weight per pair that multiplies the expert's input, applied to both float products.
template <typename T>
__global__ __launch_bounds__(256) void k_moe_pair_up(const T* __restrict__ h, int ldh, const T* __restrict__ wgu,
                                                     const int* __restrict__ idx, T* __restrict__ a, int npairs, int top,
                                                     int E, int F, int W, float limit, int mode,
                                                     const float* __restrict__ inw) {
  const int pair = blockIdx.x, r = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int e = idx[pair];
  if (r >= F || e < 0 || e >= E) return;
  const T* x = h + (size_t)(pair / top) * ldh;
  const T* wg = wgu + ((size_t)e * 2 * F + r) * W;
  const float iw = inw != nullptr ? inw[pair] : 1.f;
  const float g = iw * wave_dot<T>(wg, x, W, lane), u = iw * wave_dot<T>(wg + (size_t)F * W, x, W, lane);
  if (lane == 0) a[(size_t)pair * F + r] = (T)glu(g, u, limit, mode);
}

// pairs path, stage 2.  One wave per (token, output column c):
// out[t, c] = sum_j w[t, j] * (e_j < E ? Wd_e[c] . a[t, j] : h[t, c]) + shared[t, c]   (wts null: w = 1)
template <typename T>
__global__ __launch_bounds__(256) void k_moe_pair_down(const T* __restrict__ a, const T* __restrict__ wd,
                                                       const int* __restrict__ idx, const float* __restrict__ wts,
                                                       const T* __restrict__ h, int ldh, const T* __restrict__ shared,
                                                       const float* __restrict__ sgate, float* __restrict__ out, int top,
                                                       int E, int F, int W) {
  const int t = blockIdx.x, c = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (c >= W) return;
  float acc = shared != nullptr ? (float)shared[(size_t)t * W + c] * (sgate != nullptr ? sigmoidf_(sgate[t]) : 1.f) : 0.f;
  for (int j = 0; j < top; ++j) {
    const int e = idx[(size_t)t * top + j];
    const float w = wts != nullptr ? wts[(size_t)t * top + j] : 1.f;
    if (e >= E)
      acc += w * (float)h[(size_t)t * ldh + c];
    else if (e >= 0)
      acc += w * wave_dot<T>(wd + ((size_t)e * W + c) * F, a + ((size_t)t * top + j) * F, F, lane);
  }
  if (lane == 0) out[(size_t)t * W + c] = acc;
}

// ---- the same of a decode batch, bf16: an expert's rows are read once for all of its pairs, which share them on the matrix units, instead of once
// a pair.  Every block finds the pairs of its expert by itself, so there is no sort.  What stays: sums and the experts' outputs are float, a
// token's outputs are added in the order of its choices.  Bound by latency: ids, rows and weights are one round trip each, two launches.
constexpr int FEW = 512;                        // pairs

__device__ __forceinline__ void load_ids(const int* __restrict__ idx, int P, int lane, int (&v)[FEW / 64]) {
#pragma unroll
  for (int i = 0; i < FEW / 64; ++i) v[i] = idx[min(64 * i + lane, P - 1)];
  __builtin_amdgcn_sched_barrier(0);            // (in front of the weights: loads come back in order)
}
// The pairs of expert e in their order, in a wave's own place in LDS; their number.
__device__ __forceinline__ int list_pairs(const int (&v)[FEW / 64], int P, int e, int lane, unsigned short* list) {
  int n = 0;
#pragma unroll
  for (int i = 0; i < FEW / 64; ++i) {
    const unsigned long long m = __ballot(64 * i + lane < P && v[i] == e);
    if (m >> lane & 1) list[n + __popcll(m & ((1ull << lane) - 1))] = (unsigned short)(64 * i + lane);
    n += __popcll(m);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  return __builtin_amdgcn_readfirstlane(n);
}

// A row of lanes' operands over S steps of 32 of the depth, all on their way at once.  (Steps past the end are the last one again, and left out.)
template <int S>
__device__ __forceinline__ void load_steps(const bf16* p, int steps, bf16x8 (&v)[S]) {
#pragma unroll
  for (int s = 0; s < S; ++s) v[s] = *reinterpret_cast<const bf16x8*>(p + 32 * min(s, steps - 1));
}
template <int S>
__device__ __forceinline__ f32x4 multiply_steps(const bf16x8 (&a)[S], const bf16x8 (&x)[S], int steps, f32x4 acc) {
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < steps) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s], x[s], acc, 0, 0, 0);
  return acc;
}
// f(tiles) for the tiles of 16 that `left` pairs fill, four at most
template <typename F>
__device__ __forceinline__ void few_tiles(int left, F f) {
  if (left <= 16) f(std::integral_constant<int, 1>{});
  else if (left <= 32) f(std::integral_constant<int, 2>{});
  else if (left <= 48) f(std::integral_constant<int, 3>{});
  else f(std::integral_constant<int, 4>{});
}

// stage 1: a block 16 hidden units of an expert, gate and up rows, a wave a quarter of the depth.  Its weights are on their way before it
// knows its pairs, a tile's rows under the products of the tile before.
template <int S>
__global__ __launch_bounds__(256, 1) void k_moe_few_up(const bf16* __restrict__ h, int ldh, const bf16* __restrict__ wgu,
                                                       const int* __restrict__ idx, bf16* __restrict__ a, int P, int top, int F, int W,
                                                       float limit, int mode, const float* __restrict__ inw) {
  __shared__ unsigned short list[4][FEW];
  __shared__ f32x4 red[4][2][4][64];
  const int e = blockIdx.y, r0 = blockIdx.x * 16, w = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4;
  const int steps = W / 128, k0 = w * (W / 4) + 8 * q;
  const bf16* wg = wgu + ((size_t)e * 2 * F + r0 + li) * W + k0;
  bf16x8 gate[S], up[S], x[2][S];
  int ids[FEW / 64];
  load_ids(idx, P, lane, ids);
  load_steps<S>(wg, steps, gate);
  load_steps<S>(wg + (size_t)F * W, steps, up);
  __builtin_amdgcn_sched_barrier(0);
  const int n = list_pairs(ids, P, e, lane, list[w]);
  for (int g0 = 0; g0 < n; g0 += 64)
    few_tiles(n - g0, [&](auto tiles) {
      constexpr int NT = decltype(tiles)::value;
      const auto load = [&](int t) {
        load_steps<S>(h + (size_t)(list[w][min(g0 + 16 * t + li, n - 1)] / top) * ldh + k0, steps, x[t & 1]);
      };
      load(0);
      f32x4 acc[2][NT] = {};
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (t + 1 < NT) load(t + 1);
        acc[0][t] = multiply_steps<S>(gate, x[t & 1], steps, acc[0][t]);
        acc[1][t] = multiply_steps<S>(up, x[t & 1], steps, acc[1][t]);
      }
      if (g0 > 0) __syncthreads();              // (the last sums are read)
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) red[w][r][t][lane] = acc[r][t];
      __syncthreads();
      const int at = g0 + 16 * w + li;          // wave w finishes tile w: hidden units 4 q .. 4 q + 3 of pair li
      if (w >= NT || at >= n) return;
      f32x4 g = red[0][0][w][lane], u = red[0][1][w][lane];
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        g += red[i][0][w][lane];
        u += red[i][1][w][lane];
      }
      const int pair = list[w][at];
      const float iw = inw != nullptr ? inw[pair] : 1.f;
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (bf16)glu(iw * g[i], iw * u[i], limit, mode);
      *reinterpret_cast<bf16x4*>(a + (size_t)pair * F + r0 + 4 * q) = o;
    });
}

// stage 2: a block 16 output columns, a wave every eighth expert; the pairs' outputs stay float and meet in LDS
template <int S>
__global__ __launch_bounds__(512) void k_moe_few_down(const bf16* __restrict__ a, const bf16* __restrict__ wd, const int* __restrict__ idx,
                                                      const float* __restrict__ wts, const bf16* __restrict__ h, int ldh,
                                                      const bf16* __restrict__ shared, const float* __restrict__ sgate,
                                                      float* __restrict__ out, int T_, int top, int E, int F, int W) {
  constexpr int LDY = 20;
  __shared__ unsigned short list[8][FEW];
  __shared__ __attribute__((aligned(16))) float y[FEW * LDY];
  const int c0 = blockIdx.x * 16, w = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, q = lane >> 4, P = T_ * top, steps = F / 32;
  __shared__ int sid[FEW];
  __shared__ float swt[FEW];
  // a thread's first four outputs: what stands beside the experts' is on its way from here on
  const int i0 = min((int)threadIdx.x, 4 * T_ - 1);
  const int id0 = idx[min((int)threadIdx.x, P - 1)];
  const float wt0 = wts != nullptr ? wts[min((int)threadIdx.x, P - 1)] : 1.f;
  f32x4 beside = {0.f, 0.f, 0.f, 0.f};
  if (shared != nullptr) beside = load4(shared + (size_t)(i0 >> 2) * W + c0 + 4 * (i0 & 3));
  int ids[FEW / 64];
  load_ids(idx, P, lane, ids);
  if ((int)threadIdx.x < P) {
    sid[threadIdx.x] = id0;
    swt[threadIdx.x] = wt0;
  }
  for (int e = w; e < E; e += 8) {
    bf16x8 rows[S], x[2][S];
    load_steps<S>(wd + ((size_t)e * W + c0 + li) * F + 8 * q, steps, rows);
    __builtin_amdgcn_sched_barrier(0);
    const int n = list_pairs(ids, P, e, lane, list[w]);
    for (int g0 = 0; g0 < n; g0 += 64)
      few_tiles(n - g0, [&](auto tiles) {
        constexpr int NT = decltype(tiles)::value;
        int pair[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) pair[t] = list[w][min(g0 + 16 * t + li, n - 1)];
        load_steps<S>(a + (size_t)pair[0] * F + 8 * q, steps, x[0]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          if (t + 1 < NT) load_steps<S>(a + (size_t)pair[t + 1] * F + 8 * q, steps, x[(t + 1) & 1]);
          const f32x4 acc = multiply_steps<S>(rows, x[t & 1], steps, f32x4{0.f, 0.f, 0.f, 0.f});
          *reinterpret_cast<f32x4*>(y + pair[t] * LDY + 4 * q) = acc;           // (pairs past the end repeat the last)
        }
      });
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the list is read)
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 4 * T_; i += 512) {
    const int t = i >> 2, c = c0 + 4 * (i & 3);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (shared != nullptr) acc = (i < 512 ? beside : load4(shared + (size_t)t * W + c)) * (sgate != nullptr ? sigmoidf_(sgate[t]) : 1.f);
    for (int j = 0; j < top; ++j) {
      const int p = t * top + j, e = sid[p];
      const float wt = swt[p];
      if (e >= E)
        acc += load4(h + (size_t)t * ldh + c) * wt;
      else if (e >= 0)
        acc += *reinterpret_cast<const f32x4*>(y + p * LDY + 4 * (i & 3)) * wt;
    }
    *reinterpret_cast<f32x4*>(out + (size_t)t * W + c) = acc;
  }
}

// sorted path: out[t, c] = sum_j w[t, j] * (e_j < E ? ys[pos[t, j], c] : h[t, c]) + shared[t, c]
template <typename T>
__global__ __launch_bounds__(256) void k_moe_combine(const T* __restrict__ ys, const long* __restrict__ pos,
                                                     const int* __restrict__ idx, const float* __restrict__ wts,
                                                     const T* __restrict__ h, int ldh, const T* __restrict__ shared,
                                                     const float* __restrict__ sgate, float* __restrict__ out, int top,
                                                     int E, int W) {
  const size_t t = blockIdx.x;
  const float sg = sgate != nullptr ? sigmoidf_(sgate[t]) : 1.f;
  for (int c = threadIdx.x; c < W; c += 256) {
    float acc = shared != nullptr ? (float)shared[t * W + c] * sg : 0.f;
    for (int j = 0; j < top; ++j) {
      const int e = idx[t * top + j];
      const float w = wts[t * top + j];
      if (e >= 0) acc += w * (e >= E ? (float)h[t * ldh + c] : (float)ys[(size_t)pos[t * top + j] * W + c]);
    }
    out[t * W + c] = acc;
  }
}

// The same, four columns per thread (16-byte or 8-byte accesses); a token's ids, rows and weights are read once into LDS.  Its rows, N at a time (a
// choice of no expert reads h's and leaves it), are loaded together, and the sums leave nothing in the caches: one by one behind branches, and kept,
// 8000 tokens of 2048 with two choices took 28.0 µs, and take 22.9 (5.7 TB/s; 26 in a call, behind the experts'
// products); four and a shared expert 44.5 → 39.1, 3000 with two 10.3 → 9.4.
// (The rows as loads that leave nothing: 27.6, they have just been written.)
constexpr int MAXTOP = 64;
template <typename T, int N>
__global__ __launch_bounds__(256) void k_moe_combine4(const T* __restrict__ ys, const long* __restrict__ pos,
                                                      const int* __restrict__ idx, const float* __restrict__ wts,
                                                      const T* __restrict__ h, int ldh, const T* __restrict__ shared,
                                                      const float* __restrict__ sgate, float* __restrict__ out, int top,
                                                      int E, int W) {
  __shared__ const T* row[MAXTOP];
  __shared__ float sw[MAXTOP];
  __shared__ bool on[MAXTOP];
  const size_t t = blockIdx.x;
  const float sg = sgate != nullptr ? sigmoidf_(sgate[t]) : 1.f;
  if (threadIdx.x < top) {
    const size_t p = t * top + threadIdx.x;
    const int e = idx[p];
    row[threadIdx.x] = e >= 0 && e < E ? ys + (size_t)pos[p] * W : h + t * ldh;
    sw[threadIdx.x] = wts[p];
    on[threadIdx.x] = e >= 0;
  }
  __syncthreads();
  for (int c = 4 * threadIdx.x; c < W; c += 1024) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, v[N];
    if (shared != nullptr) acc = load4(shared + t * W + c) * sg;
    for (int j0 = 0; j0 < top; j0 += N) {
#pragma unroll
      for (int j = 0; j < N; ++j) v[j] = load4(row[min(j0 + j, top - 1)] + c);
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (j0 + j < top && on[j0 + j]) acc += v[j] * sw[j0 + j];
    }
    __builtin_nontemporal_store(acc, reinterpret_cast<f32x4*>(out + t * W + c));
  }
}

// feed-forward activations on a GEMM output: mode 0 tanh-form GELU of z [T, F]; mode 1 clipped GLU, mode 2 SiLU GLU,
// mode 3 tanh-form GELU GLU of the [gate | up] halves of z [T, 2F]
template <typename T>
__global__ __launch_bounds__(256) void k_ff_act(const T* __restrict__ z, T* __restrict__ out, size_t n, int F, int mode,
                                                float limit, const float* __restrict__ rs) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  if (mode == 0) {
    const float v = (float)z[i];
    out[i] = (T)gelu_tanhf_(v);
  } else {
    const size_t t = i / F, c = i % F;
    const float s = rs != nullptr ? rs[t] : 1.f;      // a weight per row on both halves
    out[i] = (T)glu(s * (float)z[t * 2 * F + c], s * (float)z[t * 2 * F + F + c], limit, mode);
  }
}

int seq_route_max_outputs() { return 64 * RPL; }

void seq_route_grouped(const float* z, const float* corr, int* idx, float* w, int T_, int n, int top, int groups,
                       int keep, float scale, int kind, hipStream_t st) {
  if (T_ == 0) return;
  hipLaunchKernelGGL(k_route_grouped, dim3((T_ + 3) / 4), dim3(256), 0, st, z, corr, idx, w, T_, n, top, groups, keep,
                     scale, kind);
  LIPA_CHECK_LAUNCH();
}

void seq_route_fused(int code, const void* h, int ldh, const float* router, const float* corr, int* idx, float* w,
                     int T_, int n, int W, int top, int groups, int keep, float scale, int kind, int extra, float* xout,
                     int always, hipStream_t st) {
  if (T_ == 0) return;
  const auto fits = [](const void* p, int b) { return ((uintptr_t)p & (b - 1)) == 0; };
  // us, a block's four tokens (rows above 8 KB and few tokens: a block per token) -> tiles of 16: 256 / 2000 / 8000 tokens of width 2048, 8
  // outputs 6.8 -> 6.4, 7.3 -> 6.7, 15.5 -> 9.7 (15.2 -> 9.1; 13 with rows that come from memory), 16 outputs 9.5 -> 8.3, 10.5 -> 8.7, 29.7 -> 12.2; 1000 of 8192 17.5 -> 14.8.
  // Short rows and few outputs give a wave too little to do to make up for the way through LDS: 1000 tokens of width 1024, 8 outputs 4.7 -> 5.2 (not
  // taken), 8000 8.6 -> 6.5; 4 outputs of 4096 7.7 -> 8.1 (not taken), 8000 17.5 -> 17.0.  Error of the weights against 64 bits as before (0.7e-7).
  if (T_ >= 256 && ((long)T_ * n >= 40000 || (W > 1024 && n > 4)) && code == 0 && n <= 16 && top + always <= 16 && W % 64 == 0 && ldh % 8 == 0 &&
      fits(h, 16) && fits(router, 16)) {
#define ROUTE_TILES(NG_)                                                                                                          \
  hipLaunchKernelGGL((W <= 1024 ? k_route_tiles<4, NG_> : k_route_tiles<8, NG_>), dim3((T_ + 15) / 16), dim3(256), 0, st, (const bf16*)h, \
                   ldh, router, corr, idx, w, T_, n, W, top, groups, keep, scale, kind, extra, xout, always)
    switch ((n + 3) / 4) {
      case 1: ROUTE_TILES(1); break;
      case 2: ROUTE_TILES(2); break;
      case 3: ROUTE_TILES(3); break;
      default: ROUTE_TILES(4); break;
    }
#undef ROUTE_TILES
    LIPA_CHECK_LAUNCH();
    return;
  }
  // (Below 256 tokens a block of 16 waves per token fills the chip better: 8 us at any number up to 200.  Rows above 8 KB are a long
  // way for four waves, which only pays with many tokens: 1000 of width 8192, 12 outputs, 32 against 24 us in bf16, 512 in float 28 against
  // 20; from 2000 on ahead.)
  if (T_ >= 256 && (W * (code == 0 ? 2 : 4) <= 8192 || T_ >= 2000) && n <= 16 && top + always <= 16 && W % 4 == 0 && ldh % 4 == 0 && fits(h, code == 0 ? 8 : 16) && fits(router, 16)) {
#define ROUTE_ROWS(NG_)                                                                                                      \
  hipLaunchKernelGGL((k_route_rows<T, NG_>), dim3((T_ + 3) / 4), dim3(256), 0, st, (const T*)h, ldh, router, corr, idx, w, T_, n,    \
                     W, top, groups, keep, scale, kind, extra, xout, always)
    SEQ_DISPATCH_T(code, {
      switch ((n + 3) / 4) {
        case 1: ROUTE_ROWS(1); break;
        case 2: ROUTE_ROWS(2); break;
        case 3: ROUTE_ROWS(3); break;
        default: ROUTE_ROWS(4); break;
      }
    });
#undef ROUTE_ROWS
    LIPA_CHECK_LAUNCH();
    return;
  }
  SEQ_DISPATCH_T(code, {
    if (T_ < 256)
      hipLaunchKernelGGL((k_route_fused<T, 16>), dim3(T_), dim3(1024), 0, st, (const T*)h, ldh, router, corr, idx, w, n,
                         W, top, groups, keep, scale, kind, extra, xout, always);
    else
      hipLaunchKernelGGL((k_route_fused<T, 4>), dim3(T_), dim3(256), 0, st, (const T*)h, ldh, router, corr, idx, w, n, W,
                         top, groups, keep, scale, kind, extra, xout, always);
  });
  LIPA_CHECK_LAUNCH();
}

// Where a decode batch's experts are read once: operands that 16-byte loads take, at most 2048 deep (512 the second products), pairs that LDS holds.
// us of a step in a captured graph, routing included (1.0 to 1.7 us shorter on both sides by now), a wave a (pair, row) -> here, 8 experts: width 2048, F
// 384, top 2, 12 / 16 / 32 / 48 / 128 pairs 22.9 -> 23.7 (not taken), 25.7 -> 24.1, 37 -> 24, 47 -> 25, 87 -> 29; width 1024, F 448, 16 / 32 / 128 pairs 18.1 ->
// 19.1 (not taken), 25 -> 20, 54 -> 23; F 512, top 4, width 2048, 12 / 16 / 64 / 256 26.0 -> 27.1 (not taken), 29.9 -> 28.0, 62 -> 29, 150 -> 37; width 1024, 16 / 24
// / 32 / 256 18.6 -> 20.8 (not taken), 23.3 -> 21.5, 25.4 -> 21.7, 91 -> 29.  With the ids' loads in front of the weights', and what stands beside the experts'
// outputs on its way from the start, half a us less.
// Where the line lies.  12.5 million: nothing between 10.5 (slower here) and 12.58 was timed.  1260 more steps, 1 to 16 experts, top 1 to 8, F 32 to 512,
// widths of 128 to 2048, weights from memory, experts alone, routed evenly: up to 10 experts all are ahead by then, whatever the depths (8 experts 1.05 to
// 9 times), but a single one of less than 640 columns (0.93).  With more, an expert's few pairs do not pay for blocks that fill the chip twice:
// 16 experts, F 512, width 1024, top 4, 32 pairs 20.7 -> 22.9, 36 26.5 -> 22.9; width 768 32 / 36 pairs 18.7 -> 21.6, 21.6 -> 21.9; F 448, width 640, 44 / 48
// 20.9 -> 22.0, 21.6 -> 22.3; F 384, width 1536, 32 / 40 / 48 26.7 -> 29.6, 29.0 -> 29.8, 34.7 -> 30.1; width 2048, 32 33.0 -> 31.7; up to F 256 always
// ahead.  Taken here: 1160 of the 1260, none slower by more than 1 %.  (Where all tokens choose the same experts the other form reads no others'
// rows: of 500 such steps 33 are slower here, by up to 13 %.)
bool seq_moe_few(int code, const void* h, int ldh, const void* wgu, const void* wd, const void* shared, int T_, int top, int E, int F, int W) {
  const auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const long P = (long)T_ * top, work = P * F * W;
  const bool many = E > 10 && F > 256 && W <= 1536;
  return code == 0 && P <= FEW && work >= 12500000 && P >= 2 * E && E <= 16 && (E > 1 || W >= 640) &&
         (!many || (W <= 1024 ? P > 32 && work >= 1000000l * E : P >= 3 * E)) && F % 32 == 0 && F <= 512 && W % 128 == 0 && W <= 2048 && ldh % 8 == 0 &&
         aligned(h) && aligned(wgu) && aligned(wd) && aligned(shared);
}

void seq_moe_pairs(int code, const void* h, int ldh, const void* wgu, const void* wd, const int* idx, const float* wts,
                   const void* shared, const float* sgate, void* a, float* out, int T_, int top, int E, int F, int W,
                   float limit, int mode, int weight_input, hipStream_t st) {
  if (T_ == 0) return;
  if (seq_moe_few(code, h, ldh, wgu, wd, shared, T_, top, E, F, W)) {
    hipLaunchKernelGGL(W <= 1024 ? k_moe_few_up<8> : k_moe_few_up<16>, dim3(F / 16, E), dim3(256), 0, st, (const bf16*)h, ldh, (const bf16*)wgu, idx,
                       (bf16*)a, T_ * top, top, F, W, limit, mode, weight_input ? wts : nullptr);
    hipLaunchKernelGGL(F <= 256 ? k_moe_few_down<8> : k_moe_few_down<16>, dim3(W / 16), dim3(512), 0, st, (const bf16*)a, (const bf16*)wd, idx,
                       weight_input ? nullptr : wts, (const bf16*)h, ldh, (const bf16*)shared, sgate, out, T_, top, E, F, W);
    LIPA_CHECK_LAUNCH();
    return;
  }
  SEQ_DISPATCH_T(code, {
    hipLaunchKernelGGL(k_moe_pair_up<T>, dim3(T_ * top, (F + 3) / 4), dim3(256), 0, st, (const T*)h, ldh, (const T*)wgu,
                       idx, (T*)a, T_ * top, top, E, F, W, limit, mode, weight_input ? wts : nullptr);
    hipLaunchKernelGGL(k_moe_pair_down<T>, dim3(T_, (W + 3) / 4), dim3(256), 0, st, (const T*)a, (const T*)wd, idx,
                       weight_input ? nullptr : wts,
                       (const T*)h, ldh, (const T*)shared, sgate, out, top, E, F, W);
  });
  LIPA_CHECK_LAUNCH();
}

void seq_moe_combine(int code, const void* ys, const long* pos, const int* idx, const float* wts, const void* h, int ldh,
                     const void* shared, const float* sgate, float* out, int T_, int top, int E, int W, hipStream_t st) {
  if (T_ == 0) return;
  const auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  if (W % 4 == 0 && ldh % 4 == 0 && top <= MAXTOP && aligned(ys) && aligned(h) && aligned(shared) && aligned(out)) {
#define C(N_)                                                                                                              \
  SEQ_DISPATCH_T(code, (k_moe_combine4<T, N_><<<dim3(T_), dim3(256), 0, st>>>((const T*)ys, pos, idx, wts, (const T*)h, ldh, \
                                                                              (const T*)shared, sgate, out, top, E, W)))
    if (top == 1) C(1);
    else if (top == 2) C(2);
    else if (top == 3) C(3);
    else C(4);
#undef C
    LIPA_CHECK_LAUNCH();
    return;
  }
  SEQ_DISPATCH_T(code, hipLaunchKernelGGL(k_moe_combine<T>, dim3(T_), dim3(256), 0, st, (const T*)ys, pos, idx, wts,
                                          (const T*)h, ldh, (const T*)shared, sgate, out, top, E, W));
  LIPA_CHECK_LAUNCH();
}

void seq_ff_act(int code, const void* z, void* out, int T_, int F, int mode, float limit, const float* row_scale,
                hipStream_t st) {
  const size_t n = (size_t)T_ * F;
  if (n == 0) return;
  SEQ_DISPATCH_T(code, hipLaunchKernelGGL(k_ff_act<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (const T*)z,
                                          (T*)out, n, F, mode, limit, row_scale));
  LIPA_CHECK_LAUNCH();
}
