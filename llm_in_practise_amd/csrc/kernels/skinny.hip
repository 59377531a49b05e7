// Decode-shaped bf16 GEMM: y[M, N] = x[M, K] · W[N, K]ᵀ (+ residual) for few rows, and the same with the gated activation
// h[M, F] = silu(x·Wgᵀ)·(x·Wuᵀ) as its end — the weight-streaming regime, where the whole cost is reading W once from HBM and
// every launch beside it.
//
//  * a workgroup owns 16·CT rows of W and ALL of K, shared out to its NW waves; the partial sums meet in LDS and the one launch
//    ends in the residual (or the activation) and bf16.  (Split-K partials through memory took a second launch: 5.7 µs of the
//    18 of a 6144 × 4096 product.)
//  * up to 16 rows K is cut into the S pieces of skinny_splits, whose sums are added in order: the order, and so every bit of a
//    product, does not depend on how the pieces are shared out.  The gated form and more rows take units of 64 or 128 in turns.
//  * W fragments are the MFMA A operands, loaded straight from HBM (16 B per lane, whole 128-byte lines per row); one batch
//    of steps per wave is in flight while another is multiplied.  x (tiny, L2-resident) supplies the B operands.
//  * no load sits behind a branch: a partial batch loads its last step again and does not multiply it.
#include "common.h"

using namespace lipa;

namespace {

// CUT: S pieces of kc, each with its own sum (red: S tiles); else units of UNIT in turns, a sum per wave (red: NW tiles).
// B: 32-deep steps per batch; FULL: every piece is whole batches.
template <int CT, int MT, int NW, int B, bool GLU, bool CUT, bool FULL, int UNIT>
__global__ __launch_bounds__(64 * NW) void gemm_skinny_k(const bf16* __restrict__ X, int ldx, const bf16* __restrict__ W,
                                                         const bf16* __restrict__ res, bf16* __restrict__ out, int M, int N,
                                                         int K, int S) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f32x4(*red)[CT * MT][64] = reinterpret_cast<f32x4(*)[CT * MT][64]>(smem);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * (GLU ? CT / 2 : CT);
  const bf16 *wr[CT], *xr[MT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const int n = GLU ? (t < CT / 2 ? 0 : N) + min(n0 + 16 * (t % (CT / 2 > 0 ? CT / 2 : 1)) + li, N - 1) : min(n0 + 16 * t + li, N - 1);
    wr[t] = W + (size_t)n * K + 8 * g;
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) xr[m] = X + (size_t)min(16 * m + li, M - 1) * ldx + 8 * g;
  f32x4 acc[CT][MT];
  auto clear = [&] {
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto leave = [&](int slot) {
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[slot][t * MT + m][lane] = acc[t][m];
  };
  struct Batch {
    bf16x8 a[B][CT], b[B][MT];
  };
  // steps of one piece (of the whole wave, if not CUT), batches of one piece, batches of this wave
  const int kc = CUT ? K / S : K, steps = CUT ? kc / 32 : UNIT / 32 * ((K / UNIT - w + NW - 1) / NW), per = (steps + B - 1) / B;
  const int nb = CUT ? (S - w + NW - 1) / NW * per : per;
  int lp = w, lb = 0;                            // the next batch to load: its piece, its place in it
  auto load = [&](Batch& s) {
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int e = FULL ? lb * B + u : min(lb * B + u, steps - 1);
      const int k = CUT ? lp * kc + 32 * e : UNIT * (w + NW * (e / (UNIT / 32))) + 32 * (e % (UNIT / 32));
#pragma unroll
      for (int t = 0; t < CT; ++t) s.a[u][t] = *reinterpret_cast<const bf16x8*>(wr[t] + k);
#pragma unroll
      for (int m = 0; m < MT; ++m) s.b[u][m] = *reinterpret_cast<const bf16x8*>(xr[m] + k);
    }
    if (++lb == per) lb = 0, lp += NW;
  };
  int rp = w, rb = 0;                            // the next batch to multiply
  auto run = [&](const Batch& s) {
#pragma unroll
    for (int u = 0; u < B; ++u) {
      if (!FULL && rb * B + u >= steps) break;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < CT; ++t)
          acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.a[u][t], s.b[u][m], acc[t][m], 0, 0, 0);
    }
    if (++rb == per && CUT) {
      leave(rp);
      clear();
      rb = 0, rp += NW;
    }
  };
  clear();
  if (nb > 0) {
    Batch p, q;
    load(p);
    int i = 0;
    for (; i + 2 < nb; i += 2) {
      load(q);
      run(p);
      load(p);
      run(q);
    }
    if (i + 1 < nb) {
      load(q);
      run(p);
      run(q);
    } else {
      run(p);
    }
  }
  if (!CUT) leave(w);
  const int parts = CUT ? S : NW;
  __syncthreads();
  // lane holds C[n = n0 + 16 t + 4 g + i][m = 16 mt + li]
  for (int c = w; c < (GLU ? CT / 2 : CT) * MT; c += NW) {
    const int t = c / MT, m = 16 * (c % MT) + li, n = n0 + 16 * t + 4 * g;
    f32x4 v = red[0][c][lane], up = {0.f, 0.f, 0.f, 0.f};
    for (int s = 1; s < parts; ++s) v += red[s][c][lane];
    if (GLU) {
      for (int s = 0; s < parts; ++s) up += red[s][c + CT / 2 * MT][lane];
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

// Column tiles and waves per workgroup, us at 1 / 8 / 16 rows: two tiles of 8 waves take 13.2 / 13.9 / 15.1 for 6144 x 4096 (one tile
// of 4 waves 13.7 / 15.5 / 17.5) and 9.7 / 10.8 / 12.3 for 6144 x 2560 (10.7 / 12.3 / 14.4), but 4096 rows of W fill half the CUs with
// them: 11.9 / 13.2 / 14.9 for K = 4096 against 9.0 / 9.7 / 10.9.  Batches of 5 steps where the pieces divide by them (2560: whole
// batches 9.7, partial ones 11.8).
// The gated form pairs 16 gate with 16 up rows.  4 waves of 64-deep units against 2 of 128-deep ones: with few workgroups the
// waves count, 2 x 3072 x 1024 5.3 / 5.7 / 6.0 against 6.1 / 6.3 / 6.4, 2 x 2048 x 4096 12.4 / 13.7 / 14.9 against 15.7 / 16.5 / 17.2; with
// many, the longer units: 2 x 8192 x 3072 20.7 / 22.5 / 24.9 against 19.8 / 20.5 / 22.4, 2 x 6912 x 2304 16.2 / 18.7 / 20.7 against 14.6 / 15.3
// / 16.6.  Where K is a multiple of 2048 the four waves are ahead at one row all the same (2 x 12288 x 4096 39.1 / 40.8 / 45.7 against
// 40.2 / 39.4 / 42.1, 2 x 8192 x 2048 16.5 / 17.6 / 17.9 against 17.1 / 17.3 / 16.5) and stay, since one row is where latency counts.
void launch_gemm_skinny(const void* X, int ldx, const void* W, const void* res, void* out, int M, int N, int K, bool glu,
                        hipStream_t st) {
  const int pieces = skinny_splits(N, K), kc = K / pieces;        // (one tile of 1 KB of LDS each: up to 32)
#define L(CT_, MT_, NW_, B_, GLU_, CUT_, FULL_, UNIT_)                                                                          \
  gemm_skinny_k<CT_, MT_, NW_, B_, GLU_, CUT_, FULL_, UNIT_>                                                                       \
      <<<(N + 16 * (GLU_ ? CT_ / 2 : CT_) - 1) / (16 * (GLU_ ? CT_ / 2 : CT_)), 64 * NW_, (CUT_ ? pieces : NW_) * CT_ * MT_ * 1024, \
         st>>>((const bf16*)X, ldx, (const bf16*)W, (const bf16*)res, (bf16*)out, M, N, K, pieces)
#define PIECES(CT_, NW_, B_)                                                                         \
  do {                                                                                               \
    if (kc % (32 * B_) == 0) L(CT_, 1, NW_, B_, false, true, true, 64);                              \
    else if (kc % 160 == 0) L(CT_, 1, NW_, 5, false, true, true, 64);                                \
    else L(CT_, 1, NW_, 4, false, true, false, 64);                                                  \
  } while (0)
#define TURNS(CT_, NW_, B_, GLU_, UNIT_)                                                             \
  do {                                                                                               \
    if (M <= 16 && K % (UNIT_ * NW_) == 0 && K % (32 * B_ * NW_) == 0) L(CT_, 1, NW_, B_, GLU_, false, true, UNIT_); \
    else if (M <= 16) L(CT_, 1, NW_, 4, GLU_, false, false, UNIT_);                                  \
    else if (M <= 32) L(CT_, 2, NW_, 4, GLU_, false, false, UNIT_);                                  \
    else L(CT_, 4, NW_, 4, GLU_, false, false, UNIT_);                                               \
  } while (0)
  if (glu) {
    if (N > 4096 && K % 2048 && K % 128 == 0) TURNS(2, 2, 4, true, 128);
    else TURNS(2, 4, 4, true, 64);
  } else if (pieces <= 32 && M <= 16) {
    if (N >= 6144) PIECES(2, 8, 4);
    else PIECES(1, 4, 8);
  } else {
    if (N >= 6144) TURNS(2, 8, 4, false, 64);
    else TURNS(1, 4, 8, false, 64);
  }
#undef TURNS
#undef PIECES
#undef L
  LIPA_CHECK_LAUNCH();
}
