// Routed experts of a prompt: every expert's products over its run of (token, expert) pairs in two launches, without a host
// round trip.  A first kernel orders the pairs by expert; the products then run over tiles of 128 pairs of one expert - the first
// gathers its rows of the input as it loads them and ends in the gated activation, so neither the gathered input nor the gate
// and up products ever stand in memory.
//
// 8000 tokens of width 2048, 8 experts of 384, top 2 (75 GFLOP): 638 -> 175 us with routing and the weighted sum: order 13, first
// products 71 (710 TFLOP/s), second 39 (650), sum 27, routing 18.  100 tokens: 533 -> 48 us.  The sort, the host's read of the run lengths
// and a vendor product pair, an activation and their launch gaps per expert took 500 us at any number of tokens.
#include "seq_common.h"

using namespace lipa;

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __amdgpu_buffer_rsrc_t rsrc;

constexpr int BM = 128, BN = 128, BK = 64;      // pairs x weight rows x depth of a tile
constexpr int IMG = 128 * BK * 2;               // bytes of a staged operand: 128 rows of 128 bytes
constexpr int PT = 1024;                        // threads of the ordering kernel

// One block per expert e: its place in the order is the number of pairs of lower experts; its pairs keep their order.
// perm: pair at a place; pos: place of a pair (0 for pairs of no expert); offs [E + 1].
__global__ __launch_bounds__(PT) void k_moe_order(const int* __restrict__ idx, int P, int E, int* __restrict__ offs,
                                                  int* __restrict__ perm, long* __restrict__ pos) {
  __shared__ int wsum[PT / 64], wlow[PT / 64];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int low = 0, eq = 0;
  for (int p = 4 * tid; p < P; p += 4 * PT)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int v = p + i < P ? idx[p + i] : -1;
      low += v >= 0 && v < e;
      eq += v == e;
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    low += __shfl_xor(low, o, 64);
    eq += __shfl_xor(eq, o, 64);
  }
  if (lane == 0) {
    wlow[w] = low;
    wsum[w] = eq;
  }
  __syncthreads();
  int at = 0, all = 0;
#pragma unroll
  for (int i = 0; i < PT / 64; ++i) {
    at += wlow[i];
    all += wsum[i];
  }
  if (tid == 0) {
    offs[e] = at;
    if (e == E - 1) offs[E] = at + all;
  }
  for (int p0 = 0; p0 < P; p0 += 4 * PT) {            // four neighbouring pairs a thread
    const int p = p0 + 4 * tid;
    int v[4], ahead = 0, count = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = p + i < P ? idx[p + i] : -1;
      const unsigned long long m = __ballot(v[i] == e);
      ahead += __popcll(m & ((1ull << lane) - 1));
      count += __popcll(m);
    }
    __syncthreads();                                  // the last turn's counts are read
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

__device__ __forceinline__ float glu(float g, float u, float limit, int mode) {       // 1: clipped GLU, 2: SiLU GLU
  if (mode == 2) return g * sigmoidf_(g) * u;
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoidf_(1.702f * g) * (u + 1.f);
}

struct Rows {
  const int *offs, *perm;
  int E, P, top;
};

// UP: out[place, f] = glu(wg_f . x, wu_f . x) with x = the pair's row of the input, 64 gate rows and their 64 up rows a tile.
// Otherwise out[place, c] = w_c . x with x = the place's row.  K: depth; N: columns of out.
// Four waves in a 2 x 2 grid; weights are the first operand, so a lane holds one pair's products for neighbouring columns, and the
// result goes through LDS to leave in whole rows.  Two stages in LDS, filled while the other is multiplied; two blocks a CU cover
// each other's waits.
template <bool UP>
__global__ __launch_bounds__(256, 2) void k_moe_tiles(const bf16* __restrict__ x, const bf16* __restrict__ wt,
                                                      const float* __restrict__ rs, bf16* __restrict__ out, Rows r, int K, int N,
                                                      float limit, int mode) {
  __shared__ __attribute__((aligned(1024))) char lds[4 * IMG];
  constexpr int COLS = UP ? BN / 2 : BN;        // columns of out per tile
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int nt = (N + COLS - 1) / COLS, tile = xcd_remap(blockIdx.x, gridDim.x), mt = tile / nt, n0 = (tile % nt) * COLS;
  int lo = 0, hi = r.E - 1;
  while (lo < hi) {                             // expert e owns the row tiles offs[e] / BM + e, ..
    const int mid = (lo + hi + 1) >> 1;
    if (r.offs[mid] / BM + mid <= mt)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int e = lo, o0 = r.offs[e], m0 = o0 + (mt - (o0 / BM + e)) * BM, m = min(BM, r.offs[e + 1] - m0);
  if (m0 < o0 || m <= 0) return;
  // rows of the operands that this lane loads: 8 lanes a row, chunk c of row i in slot c ^ (i & 7) of the staged row
  const size_t wbytes = (size_t)(UP ? 2 : 1) * N * K * 2;
  const rsrc wr = window(wt + (size_t)e * (UP ? 2 : 1) * N * K, (uint32_t)wbytes);
  const rsrc xr = window(x, 0xFFFFFFFFu);
  uint32_t wo[4], xo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = 32 * w + 8 * j + (lane >> 3), chunk = ((lane & 7) ^ (i & 7)) * 16;
    const int n = UP ? (i >> 6) * N + min(n0 + (i & 63), N - 1) : min(n0 + i, N - 1);
    wo[j] = (uint32_t)n * (uint32_t)K * 2 + chunk;
    const int place = m0 + min(i, m - 1), row = UP ? r.perm[place] / r.top : place;
    xo[j] = (uint32_t)row * (uint32_t)K * 2 + chunk;
  }
  const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)lds);
  auto fill = [&](int stage, int k0) {
    const uint32_t dst = base + stage * 2 * IMG + w * (IMG / 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      to_lds(wr, dst + j * 1024, wo[j], k0 * 2);
      to_lds(xr, dst + IMG + j * 1024, xo[j], k0 * 2);
    }
  };
  const int l32 = lane & 31, half = lane >> 5, wm = w & 1, wn = w >> 1;
  f32x16 acc[2][2];                             // [weight rows][pairs]
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
  const int wrow = UP ? 32 * wn + l32 : 64 * wn + l32, wstep = (UP ? 64 : 32) * 128, xrow = 64 * wm + l32;
  fill(0, 0);
  for (int k0 = 0, st = 0; k0 < K; k0 += BK, st ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                            // this stage stands; nobody reads the other one any more
    if (k0 + BK < K) fill(st ^ 1, k0 + BK);
    const char *wp = lds + st * 2 * IMG + wrow * 128, *xp = lds + st * 2 * IMG + IMG + xrow * 128;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int cw = ((2 * ks + half) ^ (wrow & 7)) * 16, cx = ((2 * ks + half) ^ (xrow & 7)) * 16;
      bf16x8 a[2], b[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        a[t] = *reinterpret_cast<const bf16x8*>(wp + t * wstep + cw);
        b[t] = *reinterpret_cast<const bf16x8*>(xp + t * 32 * 128 + cx);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[t], b[u], acc[t][u], 0, 0, 0);
    }
  }
  __syncthreads();
  // results: staged as [pair][COLS] bf16 rows (16 bytes of padding), then stored 16 bytes a lane
  constexpr int LDR = COLS + 8;
  bf16* res = reinterpret_cast<bf16*>(lds);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = 64 * wm + 32 * u + l32;
    float s = 1.f;
    if (UP && rs != nullptr) s = rs[r.perm[m0 + min(i, m - 1)]];
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int c = 8 * g4 + 4 * half;
      if (UP) {
        bf16x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = (bf16)glu(s * acc[0][u][4 * g4 + q], s * acc[1][u][4 * g4 + q], limit, mode);
        *reinterpret_cast<bf16x4*>(res + i * LDR + 32 * wn + c) = v;
      } else {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          bf16x4 v;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = (bf16)acc[t][u][4 * g4 + q];
          *reinterpret_cast<bf16x4*>(res + i * LDR + 64 * wn + 32 * t + c) = v;
        }
      }
    }
  }
  __syncthreads();
  constexpr int PER = COLS / 8;                 // lanes of a row
  for (int i = tid / PER; i < m; i += 256 / PER) {
    const int c = (tid % PER) * 8;
    if (n0 + c < N)
      *reinterpret_cast<bf16x8*>(out + (size_t)(m0 + i) * N + n0 + c) = *reinterpret_cast<const bf16x8*>(res + i * LDR + c);
  }
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
  hipLaunchKernelGGL(k_moe_order, dim3(E), dim3(PT), 0, st, idx, P, E, offs, perm, pos);
  hipLaunchKernelGGL(k_moe_tiles<true>, dim3(mt * ((F + 63) / 64)), dim3(256), 0, st, (const bf16*)h, (const bf16*)wgu, wts,
                     (bf16*)a, r, W, F, limit, mode);
  hipLaunchKernelGGL(k_moe_tiles<false>, dim3(mt * ((W + 127) / 128)), dim3(256), 0, st, (const bf16*)a, (const bf16*)wd,
                     (const float*)nullptr, (bf16*)ys, r, F, W, limit, mode);
  LIPA_CHECK_LAUNCH();
}
