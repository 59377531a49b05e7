// Decode-shaped bf16 GEMM: y[M, N] = x[M, K] · W[N, K]ᵀ (+ residual) for few rows, and the same with the gated activation
// h[M, F] = silu(x·Wgᵀ)·(x·Wuᵀ) as its end — the weight-streaming regime, where the whole cost is reading W once from HBM and
// every launch beside it.
//
//  * a workgroup owns 16·CT rows of W and ALL of K, shared out to its NW waves; the partial sums meet in LDS and the one launch
//    ends in the residual (or the activation) and bf16.  (Split-K partials through memory took a second launch: 5.7 µs of the
//    18 of a 6144 × 4096 product.)
//  * up to 16 rows K is cut into the S pieces of skinny_splits, whose sums are added in order: the order, and so every bit of a
//    product, does not depend on how the pieces are shared out.  The gated form and more rows take units of 64 or 128 in turns.
//  * x and W come by LDS-DMA, 8 rows × 128 B an instruction, into a ring of RING 64-deep units that belongs to one wave: no barrier in
//    the loop, a wave waits for its own loads.  As MFMA fragments straight from memory, where neighbouring lanes stand in
//    different rows, a CU takes 37 KB/µs of them at most, wherever they are; in whole 64-byte pieces 110.
//  * chunk c (16 B) of row r of an 8-row image stands in slot c ^ r: the fragments' ds_read_b128 are free of conflicts.
//
// µs with fragments from memory → through LDS, W cold, bit for bit the same, at 1 / 12 / 16 rows: 4096 × 4096 9.0 / 10.4 / 11.0 → 9.1 / 9.4 /
// 9.6, 6144 × 4096 14.4 / 16.2 / 17.1 → 13.8 / 14.5 / 15.1, 1024 × 2048 4.6 / 5.7 / 6.0 → 3.9 / 4.1 / 4.2, 2 × 12288 × 4096 gated 40.7 / 45.6 /
// 48.7 → 37.6 / 37.0 / 37.3 (5.4 TB/s), 2 × 9728 × 2560 gated 26.0 / 28.7 / 30.1 → 22.9 / 22.7 / 23.1.
//
// W's lines, which one wave reads once, come by loads that leave nothing in the caches on their way.  1 / 16 rows, W cold: 4096 × 4096
// 9.3 / 10.1 → 8.3 / 9.3, 6144 × 4096 13.4 / 14.9 → 12.6 / 14.3, 8192 × 8192 26.5 / 27.6 → 23.9 / 26.1, 4096 × 12288 20.9 / 24.2 → 18.8 / 22.9, 1024 ×
// 1024 3.5 / 3.8 → 3.2 / 3.5, 2 × 12288 × 4096 gated 35.5 → 32.4 (6.2 TB/s), 2 × 9728 × 2560 gated 22.5 / 23.4 → 20.6 / 22.0.  Where a piece ends in the
// middle of a line the line is read twice and has to stay: 2560 × 9728 15.8 / 20.6 with, 16.1 / 21.6 without.  (Weights that a caller multiplies with
// again and again and that fit into L2 or the last cache lose: 6144 × 2560 alone 6.5 → 8.2, 4096 × 4096 7.8 → 7.4.  A model's layers do not fit; where they
// do, 4 of 25 MB, a decode step of 1 / 4 / 12 / 16 rows takes 140 / 152 / 172 / 175 µs, and took 147 / 157 / 173 / 175 before this and the other changes
// to a step's kernels: no loss that shows.)
#include "lds_dma.h"

using namespace lipa;

namespace {

// An RMSNorm in front of the product: the norm's weight (null: none).  A row is summed by wpr waves, 8 elements a lane and turn, as the norm's
// own kernel does (norm.hip), so that the normed rows, rounded to bf16 as it rounds them, are the same bit for bit.
struct Norm {
  const bf16* w;
  float eps;
  int wpr;
};

// How K is cut into parts, each a chain of products whose sums are added in order: S pieces, or a part per wave of units of 64 or 128 in turns
enum { PIECES, TURNS64, TURNS128 };

// NORM: the rows of x come first, are normed in LDS behind the static part (M rows of 2 K + 64 bytes, then the norm's weight) while W's first
// units are on their way, and stay there; the rings hold W alone.
template <int CT, int MT, int NW, int RING, bool GLU, int CUT, int PARTS, bool NORM>
__global__ __launch_bounds__(64 * NW) void gemm_skinny_k(const bf16* __restrict__ X, int ldx, const bf16* __restrict__ W,
                                                         const bf16* __restrict__ res, bf16* __restrict__ out, int M, int N,
                                                         int K, int S, Norm nrm) {
  constexpr int CO = GLU ? CT / 2 : CT, UB = (CT + (NORM ? 0 : MT)) * 2048, D = UB / 1024, RINGS = NW * RING * UB, SUMS = PARTS * CT * MT * 1024;
  constexpr bool BESIDE = CUT == PIECES;        // (sums are left while the rings run; else they take the rings' place)
  static_assert((NORM ? RING : RING - 1) * D < 64 && (!NORM || MT == 1), "the counter of outstanding loads");
  __shared__ __attribute__((aligned(1024))) char smem[BESIDE ? RINGS + SUMS : RINGS > SUMS ? RINGS : SUMS];
  extern __shared__ __attribute__((aligned(16))) char rows[];
  f32x4(*red)[CT * MT][64] = reinterpret_cast<f32x4(*)[CT * MT][64]>(smem + (BESIDE ? RINGS : 0));
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * CO;
  const rsrc wr = window(W + (size_t)n0 * K), ur = window(W + (size_t)(GLU ? N + n0 : n0) * K), xr = window(X);
  uint32_t wo[2 * CO], xo[2 * MT];
  const int r8 = lane >> 3, ch = ((lane & 7) ^ r8) * 16;
#pragma unroll
  for (int j = 0; j < 2 * CO; ++j) wo[j] = (uint32_t)min(8 * j + r8, N - 1 - n0) * (uint32_t)K * 2 + ch;
#pragma unroll
  for (int j = 0; j < 2 * MT; ++j) xo[j] = (uint32_t)min(8 * j + r8, M - 1) * (uint32_t)ldx * 2 + ch;
  const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)smem) + w * RING * UB;
  // 64-deep units of a part in a row (per), of this wave (cnt), and the next one to load: part or turn lp, place lb in it.  A piece may
  // end in half a unit: the one that ends there is loaded, and its second half multiplied.
  const int len = CUT == PIECES ? K / S : CUT == TURNS64 ? 64 : 128, per = (len + 63) / 64, turns = CUT == PIECES ? S : K / len;
  const int odd = CUT == PIECES ? len & 32 : 0;
  const int cnt = (turns - w + NW - 1) / NW * per;
  int lp = w, lb = 0;
  auto fill = [&](int slot) {
    const uint32_t dst = base + slot * UB, k = (lp * len + 64 * lb - (lb == per - 1 ? odd : 0)) * 2;
    if (CUT == PIECES && odd) {                          // (a line of W that two units share is found in L2 the second time)
#pragma unroll
      for (int j = 0; j < 2 * CT; ++j) to_lds(GLU && j >= 2 * CO ? ur : wr, dst + j * 1024, wo[j % (2 * CO)], k);
    } else {
#pragma unroll
      for (int j = 0; j < 2 * CT; ++j) to_lds_once(GLU && j >= 2 * CO ? ur : wr, dst + j * 1024, wo[j % (2 * CO)], k);
    }
    if (!NORM)
#pragma unroll
      for (int j = 0; j < 2 * MT; ++j) to_lds(xr, dst + (2 * CT + j) * 1024, xo[j], k);
    if (++lb == per) lb = 0, lp += NW;
  };
  f32x4 acc[CT][MT];
  auto clear = [&] {
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto leave = [&](int part) {
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[part][t * MT + m][lane] = acc[t][m];
  };
  clear();
  // a wave brings the 1 KB pieces that it will read itself: row m's and the weight's, pieces p, p + wpr, ..
  const int stride = 2 * K + 64, pieces = NORM ? K / (512 * nrm.wpr) : 0, p0 = NORM ? w % nrm.wpr : 0;
  const int step = NORM ? NW / nrm.wpr : 1;
  if (NORM) {
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)rows);
    const rsrc gr = window(nrm.w);
    for (int c = 0; c < pieces; ++c) {
      const uint32_t o = (c * nrm.wpr + p0) * 1024;
      to_lds(gr, at + M * stride + o, lane * 16, o);
      for (int m = w / nrm.wpr; m < M; m += step) to_lds(xr, at + m * stride + o, (uint32_t)m * (uint32_t)ldx * 2 + lane * 16, o);
    }
  }
  for (int i = 0; i < min(RING, cnt); ++i) fill(i);
  if (NORM) {
    __shared__ float part[4][2];
    wait_units<D, RING>(min(RING, cnt));
    for (int m = w / nrm.wpr; m < M; m += step) {
      float ss = 0.f;
#pragma unroll 4
      for (int c = 0; c < pieces; ++c) {
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(rows + m * stride + (c * nrm.wpr + p0) * 1024 + lane * 16);
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += (float)v[i] * (float)v[i];
      }
      ss = wave_sum(ss);
      if (lane == 0) part[m][p0] = ss;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                 // (not a fence: it would wait for W's units too)
    asm volatile("" ::: "memory");
    for (int m = w / nrm.wpr; m < M; m += step) {
      float tot = 0.f;
      for (int i = 0; i < nrm.wpr; ++i) tot += part[m][i];
      const float r = rsqrtf(tot / K + nrm.eps);
#pragma unroll 4
      for (int c = 0; c < pieces; ++c) {
        const int o = (c * nrm.wpr + p0) * 1024 + lane * 16;
        bf16x8* at = reinterpret_cast<bf16x8*>(rows + m * stride + o);
        const bf16x8 v = *at, wv = *reinterpret_cast<const bf16x8*>(rows + M * stride + o);
        bf16x8 y;
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = (bf16)((float)v[i] * r * (float)wv[i]);
        *at = y;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  int cp = w, cb = 0;                             // (NORM: the part and the place in it of the unit that is multiplied)
  int rp = w, rb = 0;
  for (int i = 0, slot = 0; i < cnt; ++i) {
    wait_units<D, RING - 1>(cnt - 1 - i);
    const char* p = smem + (w * RING + slot) * UB;
    bf16x8 a[2][CT], b[2][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = li * 128 + ((4 * h + g) ^ (li & 7)) * 16;
#pragma unroll
      for (int t = 0; t < CT; ++t) a[h][t] = *reinterpret_cast<const bf16x8*>(p + t * 2048 + c);
      if (NORM) {
        const int k = cp * len + 64 * cb - (cb == per - 1 ? odd : 0);
        b[h][0] = *reinterpret_cast<const bf16x8*>(rows + min(li, M - 1) * stride + 2 * k + 64 * h + 16 * g);
      } else {
#pragma unroll
        for (int m = 0; m < MT; ++m) b[h][m] = *reinterpret_cast<const bf16x8*>(p + (CT + m) * 2048 + c);
      }
    }
    if (NORM && ++cb == per) cb = 0, cp += NW;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // the unit is in registers: its place is free
    if (i + RING < cnt) fill(slot);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (CUT == PIECES && h == 0 && odd && rb == per - 1) continue;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < CT; ++t) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][t], b[h][m], acc[t][m], 0, 0, 0);
    }
    if (CUT == PIECES && ++rb == per) {
      leave(rp);
      clear();
      rb = 0, rp += NW;
    }
    slot = slot + 1 == RING ? 0 : slot + 1;
  }
  if (!BESIDE) {
    __syncthreads();
    leave(w);
  }
  const int parts = CUT == PIECES ? S : NW;
  __syncthreads();
  // lane holds C[n = n0 + 16 t + 4 g + i][m = 16 mt + li]
  for (int c = w; c < CO * MT; c += NW) {
    const int t = c / MT, m = 16 * (c % MT) + li, n = n0 + 16 * t + 4 * g;
    f32x4 v = red[0][c][lane], up = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 1; s < parts; ++s) v += red[s][c][lane];
    if (GLU) {
#pragma unroll 4
      for (int s = 0; s < parts; ++s) up += red[s][c + CO * MT][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {          // (rounded like the products they would have been)
        const float gt = (float)(bf16)v[e], ut = (float)(bf16)up[e];
        v[e] = gt / (1.f + __expf(-gt)) * ut;
      }
    }
    if (m >= M || n >= N) continue;
    if (res != nullptr) {
      const bf16x4 r = *reinterpret_cast<const bf16x4*>(res + (size_t)m * N + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += (float)r[e];
    }
    *reinterpret_cast<bf16x4*>(out + (size_t)m * N + n) = bf16x4{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
  }
}

}  // namespace

// Pieces of K: about 512 pairs of 128 rows and a piece, each piece 256 or more.
static int skinny_splits(int N, int K) {
  const int nblk = (N + 127) / 128;
  int s = 1;
  while (nblk * s < 512 && K % (64 * s) == 0 && K / (2 * s) >= 256) s *= 2;
  return s;
}

// Rows that gemm_skinny norms itself, the norm's weight and the rows beside the rings in LDS: as many as leave the workgroups a CU holds where
// they were, and where a workgroup norms them in the time that W takes to come.  µs, norm and product → here, 1 / 2 / 3 / 4 rows: 6144 × 4096
// 15.4 → 12.5 / 12.7 / 19.3 / 19.6, 2 × 12288 × 4096 gated 39.8 → 37.3 / 40.0 / 39.4 / 38.3, 2 × 9728 × 2560 gated 25.8 → 22.0 / 21.1 / 22.7 / 26.0,
// 6144 × 2560 12.9 → 9.6 to 4 rows; 4096 × 1024 5.8 → 4.6 / 4.8 / 5.5 / 5.5, at 5 rows 6.2, at 8 7.0.
static size_t norm_bytes(int M, int K) { return (size_t)M * (2 * K + 64) + 2 * K; }
bool skinny_norms(int M, int K, bool glu) { return M <= 4 && K <= 4096 && K % 512 == 0 && norm_bytes(M, K) <= (glu ? 21 : 30) * 1024; }

// One tile of W a workgroup (GLU: 16 gate and 16 up rows).  Eight waves where one workgroup a CU holds all of W's tiles, else four, so
// that two fit into a CU's LDS (6144 × 4096, 12 rows: 12.3 µs against 13.5 with two tiles of 8 waves); the gated form takes three of them.
template <bool NORM>
static void launch_rows(const void* X, int ldx, const void* W, const void* res, void* out, int M, int N, int K, bool glu, const Norm& nrm,
                        hipStream_t st) {
  const int pieces = skinny_splits(N, K);
  const size_t extra = NORM ? norm_bytes(M, K) : 0;
#define L(CT_, NW_, RING_, GLU_, CUT_, PARTS_)                                                                             \
  gemm_skinny_k<CT_, 1, NW_, RING_, GLU_, CUT_, PARTS_, NORM><<<(N + 15) / 16, 64 * NW_, extra, st>>>(                     \
      (const bf16*)X, ldx, (const bf16*)W, (const bf16*)res, (bf16*)out, M, N, K, pieces, nrm)
  if constexpr (!NORM) {                        // (rows that are normed here have 4096 elements at most: 16 pieces of 256)
    // Deep weights: four parts of 128-deep units in turns, a wave each with a long ring (one workgroup a CU, with
    // all of its LDS).  In pieces 4096 × 12288 took 18.0 / 21.2 µs at 1 / 16 rows, and takes 18.0 / 20.3; 2560 × 9728 16.0 / 20.2, and 12.1 / 15.0.
    if (!glu && K > 8192 && K % 128 == 0) {
      L(1, 4, 8, false, TURNS128, 4);
      return;
    }
    if (!glu && pieces > 16) {                  // (32, of K = 8192 alone: any K with more of them is deeper and a multiple of 128)
      L(1, 8, 3, false, PIECES, 32);
      return;
    }
  }
  if (glu) {
    if (N > 4096 && K % 2048 && K % 128 == 0) L(2, 2, 4, true, TURNS128, 2);
    else L(2, 4, 2, true, TURNS64, 4);
  } else if (pieces >= 8 && N <= 4096) {
    L(1, 8, 4, false, PIECES, 16);
  } else {
    L(1, 4, 4, false, PIECES, 16);
  }
#undef L
}

// norm: the weight of an RMSNorm in front of the product, or null (else skinny_norms(M, K, glu))
void launch_gemm_skinny(const void* X, int ldx, const void* W, const void* res, void* out, int M, int N, int K, bool glu,
                        const void* norm, float eps, hipStream_t st) {
  const Norm nrm = {(const bf16*)norm, eps, K == 1024 || K == 2048 || K == 4096 ? 2 : 1};
#define L(CT_, MT_, RING_, GLU_)                                                                                          \
  gemm_skinny_k<CT_, MT_, 4, RING_, GLU_, TURNS64, 4, false><<<(N + 15) / 16, 256, 0, st>>>(                              \
      (const bf16*)X, ldx, (const bf16*)W, (const bf16*)res, (bf16*)out, M, N, K, 1, nrm)
  if (M > 32) {
    if (glu) L(2, 4, 3, true);
    else L(1, 4, 3, false);
  } else if (M > 16) {
    if (glu) L(2, 2, 3, true);
    else L(1, 2, 4, false);
  } else if (norm != nullptr) {
    launch_rows<true>(X, ldx, W, res, out, M, N, K, glu, nrm, st);
  } else {
    launch_rows<false>(X, ldx, W, res, out, M, N, K, glu, nrm, st);
  }
#undef L
  LIPA_CHECK_LAUNCH();
}
