// The gated product of 17 to 64 decode rows, h[M, F] = silu(x·Wgᵀ)·(x·Wuᵀ) of W [2 F, K] (gate above up), every sum one chain of MFMA over K in
// order, rounded as the product and the activation behind it would be.  What bounds it is W from memory and, beside it, x,
// which every workgroup reads whole: a workgroup takes as many columns as leave one workgroup for each CU, four tiles of 16 at most.
//
//  * a workgroup of 8 waves walks K in stages of 128: its rows of W and x come by LDS-DMA, 4 rows × 256 B an instruction (chunk c of row r
//    in slot c ^ r % 16: the fragments' reads are free of conflicts), into a ring of all LDS.  The waves share out a stage's loads and meet in one
//    barrier per stage, at which the stage read before it is free for the next loads.  (Stages of 64: 47.4 µs where these take 45.8.)
//  * W's lines leave nothing in the caches on their way (45.8 → 39.9 µs).
//  * wave w multiplies row tile w % 4 with the gate columns, or, from wave 4 on, with the up columns; they meet in LDS at the end.
//
// µs at 17 / 32 / 48 / 64 rows, W cold, the library's product and the activation → here: 2 × 12288 × 4096 48.0 / 47.7 / 48.2 / 49.0 → 39.6 / 38.9 /
// 39.1 / 39.9 (5.1 TB/s), 2 × 14336 × 4096 56 / 56 / 62 / 55 → 46 / 46 / 46 / 47, 2 × 9728 × 2560 27.4 / 29.0 / 29.5 / 30.0 → 20.7 / 21.9 / 21.7 / 23.1,
// 2 × 3072 × 1024 14 → 6.4 / 6.4 / 7.2 / 7.0.  Without the gated end it takes as long as the library's 6144 × 4096 (17.4 and 17.8 µs at 64 rows).
//
// The narrow product y[M, N] = x·Wᵀ (+ residual) of a deep weight has too few columns for that: 256 workgroups of 16 columns each read all of x,
// at 64 rows four times what they read of W.  There K is summed in four parts that take its units in turns, one workgroup a part and up to 64
// columns, and a second launch adds the parts in order.  µs at 17 / 32 / 48 / 64 rows, W cold, the library → here (both launches, residual
// included): 4096 × 12288 26.6 / 30.1 / 35.8 / 39.5 → 23.3 / 25.1 / 25.3 / 26.9, 2560 × 9728 22.4 / 23.6 / 23.7 / 30.9 → 15.8 / 16.9 / 19.0 / 19.5, 1024 × 12288
// 18.8 / 24.1 / 19.6 / 20.5 → 13.0 / 13.4 / 15.1 / 16.5; at 48 and 64 rows 4096 × 4096 16.2 / 17.8 → 12.2 / 12.8, 2560 × 4096 14.6 / 16.6 → 10.6 / 11.3.
// Units of 64 and of 128 take the same time within 5 %; a sum is a chain of K / 4 products with either, and off 64 bits by no more than the
// library's.  For many shapes these are the library's own sums, bit for bit (units of 128 of deep weights up to 32 rows, of 64 at 64 rows), for
// others not (1024 × 12288 at 64 rows, 4096 × 14336 at 64).
#include "lds_dma.h"

using namespace lipa;

namespace {

constexpr int ring_of(int stage) { return 163840 / stage < 8 ? 163840 / stage : 8; }

// MT: row tiles, CT: tiles of W's rows (GLU: half of them gate's, half up's), UNIT: 0 for the gated product, else how deep the units are that the
// four parts of K take in turns: workgroup 4 b + p sums part p of columns block b, and leaves it in part[p]
template <int MT, int CT, int UNIT>
__global__ __launch_bounds__(512) void rows_k(const bf16* __restrict__ X, int ldx, const bf16* __restrict__ W, bf16* __restrict__ out,
                                              float* __restrict__ part, int M, int N, int K) {
  constexpr bool GLU = UNIT == 0;
  constexpr int CO = GLU ? CT / 2 : CT, PIECES = 4 * (CT + MT), D = (PIECES + 7) / 8, SB = PIECES * 1024, RING = ring_of(SB);
  constexpr int HALF = (CT + 1) / 2;                       // tiles of the first four waves
  static_assert(RING >= 3 && (RING - 2) * D < 64 && (!GLU || MT * CO * 1024 <= RING * SB), "ring");
  __shared__ __attribute__((aligned(1024))) char smem[RING * SB];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
  const int n0 = (GLU ? blockIdx.x : blockIdx.x / 4) * 16 * CO, pt = GLU ? 0 : blockIdx.x % 4, r4 = lane >> 4;
  const rsrc wr = window(W + (size_t)n0 * K), ur = window(W + (size_t)(GLU ? N + n0 : n0) * K), xr = window(X);
  const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)smem);
  // pieces of a stage: 4 rows each, W's column tiles first (gate, up), then x; wave w brings pieces w, w + 8, ..
  const bool full = w + 8 * (D - 1) < PIECES;
  uint32_t vo[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const int p = min(w + 8 * j, PIECES - 1), c = li ^ (4 * (p & 3) + r4), ch = 16 * c + (UNIT == 64 && c >= 8 ? 384 : 0);
    vo[j] = p < 4 * CT ? (uint32_t)min(4 * (GLU && p >= 4 * CO ? p - 4 * CO : p) + r4, N - 1 - n0) * (uint32_t)K * 2 + ch
                       : (uint32_t)min(4 * (p - 4 * CT) + r4, M - 1) * (uint32_t)ldx * 2 + ch;
  }
  auto fill = [&](int slot, int stage) {
    const uint32_t dst = base + slot * SB + w * 1024;
    const uint32_t k = GLU ? stage * 256 : UNIT == 64 ? (8 * stage + pt) * 128 : (4 * stage + pt) * 256;
#pragma unroll
    for (int j = 0; j < D; ++j)
      if (j < D - 1 || full) {
        const int p = w + 8 * j;
        if (p >= 4 * CT) to_lds(xr, dst + j * 8192, vo[j], k);
        else if (GLU && p >= 4 * CO) to_lds_once(ur, dst + j * 8192, vo[j], k);
        else to_lds_once(wr, dst + j * 8192, vo[j], k);
      }
  };
  const int stages = (GLU ? K : K / 4) / 128, mt = w & 3, c0 = w < 4 ? 0 : HALF;
  const bool work = mt < MT;
  f32x4 acc[HALF];
#pragma unroll
  for (int t = 0; t < HALF; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < RING - 1; ++s)
    if (s < stages) fill(s, s);
  for (int s = 0, slot = 0; s < stages; ++s) {
    const int left = min(stages - 1 - s, RING - 2);
    if (full) wait_units<D, RING - 2>(left); else wait_units<D - 1, RING - 2>(left);
    __builtin_amdgcn_s_barrier();                          // the stage is here, and the one before it is read
    asm volatile("" ::: "memory");
    if (s + RING - 1 < stages) fill(slot == 0 ? RING - 1 : slot - 1, s + RING - 1);
    if (work) {
      const char* p = smem + slot * SB;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        bf16x8 a[2][HALF], b[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int c = li * 256 + ((8 * h2 + 4 * h + g) ^ li) * 16;
          b[h] = *reinterpret_cast<const bf16x8*>(p + (CT + mt) * 4096 + c);
#pragma unroll
          for (int t = 0; t < HALF; ++t)
            if (c0 + t < CT) a[h][t] = *reinterpret_cast<const bf16x8*>(p + (c0 + t) * 4096 + c);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < HALF; ++t)
            if (c0 + t < CT) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][t], b[h], acc[t], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    slot = slot + 1 == RING ? 0 : slot + 1;
  }
  const int m = 16 * mt + li;
  if constexpr (!GLU) {
    if (!work || m >= M) return;
    part += (size_t)pt * M * N + (size_t)m * N;
#pragma unroll
    for (int t = 0; t < HALF; ++t) {
      const int n = n0 + 16 * (c0 + t) + 4 * g;
      if (c0 + t < CT && n < N) *reinterpret_cast<f32x4*>(part + n) = acc[t];
    }
    return;
  }
  f32x4(*up)[CO][64] = reinterpret_cast<f32x4(*)[CO][64]>(smem);
  __syncthreads();
  if (work && w >= 4)
#pragma unroll
    for (int t = 0; t < CO; ++t) up[mt][t][lane] = acc[t];
  __syncthreads();
  if (!work || w >= 4 || m >= M) return;
#pragma unroll
  for (int t = 0; t < CO; ++t) {
    const int n = n0 + 16 * t + 4 * g;
    if (n >= N) continue;
    const f32x4 u = up[mt][t][lane];
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {                        // (rounded like the products they would have been)
      const float gt = (float)(bf16)acc[t][e], ut = (float)(bf16)u[e];
      o[e] = (bf16)(gt / (1.f + __expf(-gt)) * ut);
    }
    *reinterpret_cast<bf16x4*>(out + (size_t)m * N + n) = o;
  }
}

// y = part[0] + part[1] + part[2] + part[3] (+ res), four elements a thread
__global__ __launch_bounds__(256) void parts_sum_k(const float* __restrict__ part, const bf16* __restrict__ res, bf16* __restrict__ y, int n4) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const f32x4* p = reinterpret_cast<const f32x4*>(part) + i;
  f32x4 v = p[0];
#pragma unroll
  for (int s = 1; s < 4; ++s) v += p[(size_t)s * n4];
  if (res != nullptr) {
    const bf16x4 r = reinterpret_cast<const bf16x4*>(res)[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += (float)r[e];
  }
  reinterpret_cast<bf16x4*>(y)[i] = bf16x4{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
}

// The same sum and the RMSNorm of its rows in one launch: y as parts_sum_k and w4mm_reduce_k leave it, yn as the norm's own kernel forms it from
// that, bit for bit.  A workgroup owns a row, a thread eight columns; WAVES waves add up the squares, each in the order of the wave of that kernel
// that has its columns.  Bound by latency: 64
// rows of 4096 take 4.9 µs under a profiler, where the two launches took 4.95 and 5.1.  A captured step, the two launches → this one, µs: 8B bf16, 64 rows 6490 →
// 6381; 4B bf16, 24 / 48 rows 3220 → 3154, 3913 → 3774, W4A16 3292 → 3248, 4898 → 4762; a small model W4A16, 40 rows 299 → 285.
template <int WAVES>
__global__ __launch_bounds__(1024) void parts_norm_k(const float* __restrict__ part, int S, const bf16* __restrict__ res, const bf16* __restrict__ w,
                                                     bf16* __restrict__ y, bf16* __restrict__ yn, int M, int N, float eps) {
  __shared__ __attribute__((aligned(16))) bf16x8 row[1024];
  __shared__ float squares[WAVES];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const size_t at = (size_t)blockIdx.x * N + 8 * t, step = (size_t)M * N;
  const float* p = part + at;
  float v[8], f[4][8], r[8], g[8];
  load8(res + at, r);
  load8(w + 8 * t, g);
  load8(p, v);
  int s = 1;
  for (; s + 4 <= S; s += 4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) load8(p + (s + j) * step, f[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] += f[j][i];
  }
#pragma unroll
  for (int j = 0; j < 3; ++j)                              // (all at once; what there is not is read again and left)
    load8(p + min(s + j, S - 1) * step, f[j]);
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = s + j < S ? v[i] + f[j][i] : v[i];
  bf16x8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    o[i] = (bf16)(v[i] + r[i]);
    v[i] = (float)o[i];
  }
  row[t] = o;
  *reinterpret_cast<bf16x8*>(y + at) = o;
  __syncthreads();
  if (wave < WAVES) {
    float ss = 0.f;
    for (int c = t; c < N / 8; c += 64 * WAVES) {
      const bf16x8 x = row[c];
#pragma unroll
      for (int i = 0; i < 8; ++i) ss += (float)x[i] * (float)x[i];
    }
    ss = wave_sum(ss);
    if (lane == 0) squares[wave] = ss;
  }
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) tot += squares[i];
  const float rs = rsqrtf(tot / N + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = v[i] * rs * g[i];
  store8(yn + at, v);
}

}  // namespace

// Whether parts_norm_k takes rows of N: a thread eight columns, whole waves
bool parts_norm_ok(int N) { return N % 512 == 0 && N <= 8192; }

// Whether parts_norm_k is ahead of the sum's own launch and the norm's: a row's parts all come through one CU here, where the sum spreads them over the chip.
// Of W4A16 products of 5 to 64 rows (N 512 to 8192, K 1024 to 25600, 3 to 100 slices; the product included) the two launches -> this one, µs at 8 rows:
// 1024 × 4096 (16 slices) 9.8 → 8.6, 2560 × 9728 (38) 16.7 → 15.8, 1536 × 12288 (48) 16.6 → 15.8, at 17 rows 4096 × 12288 (24) 24.4 → 24.3; not taken: 4096 × 19456
// (38) 0.92 times as fast, 5120 × 9728 (19) 20.1 → 20.7, 8192 × 5120 (10) 0.93 times, 8192 × 12288 (24) 27.0 → 31.3, 1024 × 17408 (68, a long chain) 0.97 times.  Past
// 4096 columns a row has more than eight waves to bring its parts through.  Of 881 such products 583 are taken, none slower by more than 1.5 %; 221 of
// all were, by up to a third.  (bf16 products have four parts: 1.04 and more at every size.)
bool parts_norm_ahead(int N, int S) { return S <= 48 && (long)S * N <= (N <= 4096 ? 98304 : 65536); }

// y [M, N] = sum of S parts + res, yn = its RMSNorm with weight w
void launch_parts_norm(const float* part, int S, const void* res, const void* w, void* y, void* yn, int M, int N, float eps, hipStream_t st) {
  const int ch = N % 1024 ? 0 : N / 1024;                  // (the norm's kernel gives these widths two waves a row, others one)
  if (ch == 1 || ch == 2 || ch == 4 || ch == 8)
    parts_norm_k<2><<<M, N / 8, 0, st>>>(part, S, (const bf16*)res, (const bf16*)w, (bf16*)y, (bf16*)yn, M, N, eps);
  else
    parts_norm_k<1><<<M, N / 8, 0, st>>>(part, S, (const bf16*)res, (const bf16*)w, (bf16*)y, (bf16*)yn, M, N, eps);
  LIPA_CHECK_LAUNCH();
}

// F: columns of the result, a multiple of 16 (W has 2 F rows); K a multiple of 128; 17 <= M <= 64
void launch_rows_swiglu(const void* X, int ldx, const void* W, void* out, int M, int F, int K, hipStream_t st) {
  const int tiles = F / 16, t = tiles <= 256 ? 1 : tiles <= 512 ? 2 : tiles <= 768 ? 3 : 4;
#define L(MT_, CO_) rows_k<MT_, 2 * CO_, 0><<<(tiles + t - 1) / t, 512, 0, st>>>((const bf16*)X, ldx, (const bf16*)W, (bf16*)out, nullptr, M, F, K)
#define LT(MT_)               \
  do {                        \
    if (t == 1) L(MT_, 1);    \
    else if (t == 2) L(MT_, 2); \
    else if (t == 3) L(MT_, 3); \
    else L(MT_, 4);           \
  } while (0)
  if (M > 48) LT(4);
  else if (M > 32) LT(3);
  else LT(2);
#undef LT
#undef L
  LIPA_CHECK_LAUNCH();
}

// y [M, N] = x wᵀ (+ res): K in four parts of units in turns, a multiple of 512; N a multiple of 16; 17 <= M <= 64; part: 4 M N floats.  Without y the
// parts are left to launch_parts_norm.
void launch_rows_parts(const void* X, int ldx, const void* W, const void* res, void* y, float* part, int M, int N, int K, int unit, hipStream_t st) {
  const int tiles = N / 16, t = tiles <= 64 ? 1 : tiles <= 128 ? 2 : tiles <= 192 ? 3 : 4;
#define L(MT_, CT_, UNIT_) rows_k<MT_, CT_, UNIT_><<<(tiles + t - 1) / t * 4, 512, 0, st>>>((const bf16*)X, ldx, (const bf16*)W, nullptr, part, M, N, K)
#define LT(MT_, UNIT_)                 \
  do {                                 \
    if (t == 1) L(MT_, 1, UNIT_);      \
    else if (t == 2) L(MT_, 2, UNIT_); \
    else if (t == 3) L(MT_, 3, UNIT_); \
    else L(MT_, 4, UNIT_);             \
  } while (0)
#define LM(UNIT_)                     \
  do {                                \
    if (M > 32) LT(4, UNIT_);         \
    else LT(2, UNIT_);                \
  } while (0)
  if (unit == 64) LM(64);
  else LM(128);
#undef LM
#undef LT
#undef L
  LIPA_CHECK_LAUNCH();
  if (y == nullptr) return;
  const int n4 = M * N / 4;
  parts_sum_k<<<(n4 + 255) / 256, 256, 0, st>>>(part, (const bf16*)res, (bf16*)y, n4);
  LIPA_CHECK_LAUNCH();
}
