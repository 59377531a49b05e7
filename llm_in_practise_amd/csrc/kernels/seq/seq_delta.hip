// Prompts through the gated delta rule in blocks of 32 tokens, two tiles of 16.  With G_t the product of the decays from the block's first
// token up to t (per key channel) and S the state in front of the block,
//   u_t = beta_t (v_t - (k_t G_t)^T S - sum_{j<t} A_tj u_j),   A_tj = sum_d k_td k_jd G_td / G_jd
//   o_t = (q_t G_t)^T S + sum_{j<=t} B_tj u_j,                 B_tj = sum_d q_td k_jd G_td / G_jd
//   S  <- G_32 S + sum_j (k_j G_32 / G_j) u_j^T.
// A first kernel forms, for all blocks at once, everything that does not read the state: the scaled rows, B, and - with T = (I + beta A)^-1
// beta - the rows W = T (k G) and U = T v, so that u = U - W S and one product with the state stands between two states.  Every tile
// of 16 is solved by itself; the second one's rows then take what the first one's u adds, A_21 = (k G)_2 (k G_16 / G)_1^T.  The
// ratios G_t / G_j are running products of the decays themselves, never quotients, so a decay of 0 (or any other value) is what
// it is in the token-by-token scan.  The second kernel walks a sequence's blocks with the state in registers; all products are float on
// the float matrix units (v_mfma_f32_16x16x4_f32), whose result layout is also its operand layout.
//
// Measured, blocks of 16 -> of 32 tokens: three sequences of 1500, 700 and 97 tokens, 8 heads of 128 x 128: 112 -> 90 us (26 for the first
// kernel - 32 with two blocks a CU and rows that left four bytes a lane - and 64 for the walk, which is bound by the longest sequence's
// chain: 1.3 us a block of 32, 0.7 of them products of a wave on the float matrix unit; 0.94 us a block of 16; with the 1500 tokens in four parts and the 700 in two,
// 25 for the ends and 40 for the parts, 84 us in all).  Error against 64 bits of
// outputs, blocks of 16 -> 32: 3.2 -> 2.6e-7 where decays are next to 1, 1.6 -> 1.55 at 0.95, 1.25 -> 1.28 at 0.8, 1.08 -> 1.10 at 0.4:
// the state and a tile's sums are added up by themselves and rounded once at the size of what they are added to.
#include "seq_block.h"

#include <algorithm>
#include <type_traits>

using namespace lipa;

namespace {

constexpr int LEN = 2 * BT;

// what the first kernel leaves per (block, head): W | q G | k G_32 / G in operand order (two tiles each), G_32, B of the tiles 1-1, 2-1 and 2-2,
// U in result order (two tiles of every 16 columns); and behind these, per (block, head) and wave, whether it met a value that is
// infinite or NaN
__host__ __device__ constexpr int cell_floats(int dk, int dv) { return 3 * LEN * dk + dk + 3 * BT * BT + LEN * ((dv + 15) & ~15); }
constexpr int SEEN = 8;

__device__ __forceinline__ f32x4 mfma4(const f32x4& a, const f32x4& b, f32x4 c) {      // c + a b over 16 k, lane group g holding 4g .. 4g+3
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
  return c;
}

// element e of lane row r <-> element r of lane row e
__device__ __forceinline__ f32x4 turn_rows(const f32x4& v) {
  auto u = [](float f) { return __float_as_uint(f); };
  const auto a = __builtin_amdgcn_permlane32_swap(u(v[0]), u(v[2]), false, false), b = __builtin_amdgcn_permlane32_swap(u(v[1]), u(v[3]), false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return f32x4{__uint_as_float(c[0]), __uint_as_float(c[1]), __uint_as_float(d[0]), __uint_as_float(d[1])};
}

// 512 threads, half of them a tile: token j = tid / 16 of it, and the four channels 4 x .. of every 64 (x = tid % 16).  A thread carries
// its token's key times the decays of the tokens behind it; at token s the 16 threads of a row sum k_s and q_s against it, and lane
// s keeps the sums.
template <typename T, int NS>
__global__ __launch_bounds__(512, 6) void k_delta_prep(const T* __restrict__ q, int ldq, const T* __restrict__ k, int ldk,
                                                    const T* __restrict__ v, int ldv, int dv, const float* __restrict__ decay,
                                                    const float* __restrict__ beta, float* __restrict__ ws,
                                                    unsigned* __restrict__ seen, int H, int G, Pieces pc, SeqDesc d) {
  constexpr int DK = 64 * NS, ROWS = BT * DK;
  __shared__ __attribute__((aligned(16))) float sg[2 * ROWS];        // decays, then k G_16 / G of the first tile
  __shared__ __attribute__((aligned(16))) float sk[2 * ROWS];        // keys, then k G
  __shared__ __attribute__((aligned(16))) float sq[2 * ROWS];        // queries, then q G of the second tile and G_16 of both
  __shared__ __attribute__((aligned(16))) float sT[2][BT * BT];
  __shared__ __attribute__((aligned(16))) float sA[2][BT * BT];      // A; then A_21 in place of the first
  __shared__ float sb[LEN];
  __shared__ int sbad[LEN];
  // G_16 of the tiles, where the second tile's queries stood: with a place of its own a CU holds two of these blocks, not three
  float(*sG)[DK] = reinterpret_cast<float(*)[DK]>(sq + ROWS);
  const int slot = blockIdx.y, hd = blockIdx.x, tid = threadIdx.x;
  Piece blk;
  if (!find_piece<LEN>(d, pc, slot, blk)) return;
  const int t0 = blk.t0, n = blk.n;
  const int half = tid >> 8, j = (tid >> 4) & 15, x = tid & 15, tok = BT * half + j, kh = hd / (H / G);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, g4 = lane >> 4, vtiles = (dv + 15) / 16;
  const bool on = tok < n;
  const size_t t = t0 + (on ? tok : 0);
  // the wave's first tile of values is on its way from here on
  T vraw[2][4];
  auto load_values = [&](int vt) {
    const int c = hd * dv + min(16 * vt + li, dv - 1);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) vraw[h][e] = v[(size_t)(t0 + min(BT * h + 4 * g4 + e, n - 1)) * ldv + c];
  };
  if (w < vtiles) load_values(w);
  f32x4 kj[NS], qj[NS], W[NS], Gm[NS];
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    const int D = 64 * c + 4 * x;
    f32x4 g = row4(decay + (t * H + hd) * DK + D);
    kj[c] = row4(k + t * ldk + kh * DK + D);
    qj[c] = row4(q + t * ldq + kh * DK + D);
    if (!on) {                                               // past the end: tokens that change nothing
      kj[c] = qj[c] = f32x4{0.f, 0.f, 0.f, 0.f};
      g = f32x4{1.f, 1.f, 1.f, 1.f};
    }
    *reinterpret_cast<f32x4*>(sg + tok * DK + D) = g;
    *reinterpret_cast<f32x4*>(sk + tok * DK + D) = kj[c];
    *reinterpret_cast<f32x4*>(sq + tok * DK + D) = qj[c];
    W[c] = kj[c];
    Gm[c] = f32x4{1.f, 1.f, 1.f, 1.f};
  }
  if (tid < LEN) sb[tid] = tid < n ? sigmoidf_(beta[(size_t)(t0 + tid) * H + hd]) : 0.f;
  __syncthreads();
  float ra = 0.f, rb = 0.f;                                  // A and B of (token x, token j)
#pragma unroll 2
  for (int s = 0; s < BT; ++s) {
    float pa = 0.f, pb = 0.f;
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      const int D = half * ROWS + s * DK + 64 * c + 4 * x;
      const f32x4 g = row4(sg + D);
      if (s <= j)
        Gm[c] *= g;
      else
        W[c] *= g;
      const f32x4 qs = row4(sq + D), ks = row4(sk + D);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pb += qs[e] * W[c][e];
        pa += ks[e] * W[c][e];
      }
    }
    pb = row16_sum(pb);
    pa = row16_sum(pa);
    if (x == s) {
      rb = pb;
      ra = pa;
    }
  }
  // From the first token on whose key, decays or beta are no numbers everything is NaN.  In front of it T and B are 0 there, and
  // 0 x NaN is NaN: such rows of k G and T are 0, and NaN stands in B's rows, which reach the outputs of these tokens, and in the key
  // that is written to the state - and to the second tile, all of which is behind.
  float z = 0.f;
#pragma unroll
  for (int c = 0; c < NS; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) z += 0.f * (kj[c][e] * Gm[c][e]);
  const bool bad = !(row16_sum(z) == 0.f && isfinite(sb[tok]));
  if (x == 0) sbad[tok] = bad ? j : BT;
  sA[half][x * BT + j] = ra;
  __syncthreads();                                           // keys, queries and decays are read
  int first = sbad[BT * half + x];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o, 16));
  float* cell = ws + ((size_t)slot * H + hd) * cell_floats(DK, dv);
  float *ck = cell, *cq = ck + 2 * ROWS, *cp = cq + 2 * ROWS, *cg = cp + 2 * ROWS, *cB = cg + DK, *cU = cB + 3 * BT * BT;
  cB[2 * half * BT * BT + x * BT + j] = x >= first ? NAN : x >= j ? rb : 0.f;
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    const int D = 64 * c + 4 * x;
    *reinterpret_cast<f32x4*>(sk + tok * DK + D) = bad ? f32x4{0.f, 0.f, 0.f, 0.f} : kj[c] * Gm[c];
    if (half == 1) *reinterpret_cast<f32x4*>(sq + j * DK + D) = qj[c] * Gm[c];
    if (half == 0) *reinterpret_cast<f32x4*>(sg + j * DK + D) = bad ? f32x4{NAN, NAN, NAN, NAN} : W[c];
    if (j == BT - 1) *reinterpret_cast<f32x4*>(&sG[half][D]) = Gm[c];
  }
  if ((tid & 255) < BT) {                                    // column x of (I + beta A)^-1 beta, row after row
    float r[BT];
#pragma unroll
    for (int s = 0; s < BT; ++s) {
      float acc = s == x ? 1.f : 0.f;
#pragma unroll
      for (int i = 0; i < s; ++i) acc -= sA[half][s * BT + i] * r[i];
      r[s] = s >= first ? 0.f : sb[BT * half + s] * acc;
      sT[half][s * BT + x] = r[s];
    }
  }
  __syncthreads();
  // the scaled rows that leave as they are
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    // operand order of the 16x16x4 products: [tile of 16 channels][4 channels][token][channel of the 4] for the rows, and
    // [tile][4 tokens][channel][token of the 4] for the keys that are written to the state
    const int D = 64 * c + 4 * x, tile = 4 * c + (x >> 2), base = half * ROWS + (tile * 64 + (x & 3) * 16 + j) * 4;
    const f32x4 G1 = row4(&sG[0][D]), G2 = row4(&sG[1][D]);
    *reinterpret_cast<f32x4*>(cq + base) = half == 0 ? qj[c] * Gm[c] : qj[c] * Gm[c] * G1;
    const f32x4 P = half == 0 ? W[c] * G2 : W[c], own = bad ? f32x4{NAN, NAN, NAN, NAN} : P;
    // a row of lanes holds a token: turned, row r has channel 4 x + r of the wave's four tokens
    *reinterpret_cast<f32x4*>(cp + half * ROWS + (tile * 64 + (j >> 2) * 16 + 4 * (x & 3) + (j & 3)) * 4) = turn_rows(own);
    if (tid < 16) *reinterpret_cast<f32x4*>(cg + D) = G1 * G2;
  }
  if (w < 2) {                                               // A_21 and B_21: rows of the second tile against the keys of the first
    const float* rows = (w == 0 ? sk + ROWS : sq) + li * DK + 4 * g4;
    f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
    for (int c = 0; c < 4 * NS; c += 2) {
      a0 = mfma4(row4(rows + 16 * c), row4(sg + li * DK + 16 * c + 4 * g4), a0);
      a1 = mfma4(row4(rows + 16 * c + 16), row4(sg + li * DK + 16 * c + 16 + 4 * g4), a1);
    }
    a0 += a1;
    float* to = w == 0 ? sA[0] : cB + BT * BT;
#pragma unroll
    for (int e = 0; e < 4; ++e) to[(4 * g4 + e) * BT + li] = a0[e];
  }
  __syncthreads();
  // W and U, a wave a tile of 16 columns at a time: y1 = T_1 x1, y2 = T_2 (x2 - A_21 y1), with sums of 16 by themselves: begun at x2 each
  // would be rounded at its size
  const f32x4 T1 = row4(&sT[0][li * BT + 4 * g4]), T2 = row4(&sT[1][li * BT + 4 * g4]), X = -row4(&sA[0][li * BT + 4 * g4]);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int kt = w; kt < 4 * NS; kt += 8) {
    f32x4 x1, x2;
    const float G1 = sG[0][16 * kt + li];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x1[e] = sk[(4 * g4 + e) * DK + 16 * kt + li];
      x2[e] = sk[ROWS + (4 * g4 + e) * DK + 16 * kt + li] * G1;
    }
    // (with the factors the other way round a lane holds four channels of a token, as the rows stand in memory)
    float* to = ck + (kt * 64 + g4 * 16 + li) * 4;
    *reinterpret_cast<f32x4*>(to) = mfma4(x1, T1, zero);
    *reinterpret_cast<f32x4*>(to + ROWS) = mfma4(x2 + mfma4(X, mfma4(T1, x1, zero), zero), T2, zero);
  }
  bool odd = false;
  for (int vt = w; vt < vtiles; vt += 8) {
    if (vt != w) load_values(vt);
    f32x4 x1, x2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = 16 * vt + li < dv;
      x1[e] = in && 4 * g4 + e < n ? (float)vraw[0][e] : 0.f;
      x2[e] = in && BT + 4 * g4 + e < n ? (float)vraw[1][e] : 0.f;
      odd |= !isfinite(x1[e]) || !isfinite(x2[e]);           // (the walk makes up for what counts as 0 here)
      x1[e] = isfinite(x1[e]) ? x1[e] : 0.f;
      x2[e] = isfinite(x2[e]) ? x2[e] : 0.f;
    }
    const f32x4 y1 = mfma4(T1, x1, zero), y2 = mfma4(T2, x2 + mfma4(X, y1, zero), zero);
    *reinterpret_cast<f32x4*>(cU + (vt * 64 + lane) * 4) = y1;
    *reinterpret_cast<f32x4*>(cU + ((vtiles + vt) * 64 + lane) * 4) = y2;
  }
  odd = __any(odd);
  if (lane == 0) seen[((size_t)slot * H + hd) * SEEN + w] = odd;
}

// What is known of the state between two parts of a sequence of `blocks` blocks each, per (part, head): where the part leaves a state that
// it finds at 0 (the first part: at the one in front of it), 16 columns at a time in operand layout, and its product of transitions P,
// by which any other state in front of it goes on, as the left operand of the 16x16x4 products.  (The first part needs no P: the state in
// front of it stands there, since the last part may have written its own by the time the first one runs again.)
struct Parts {
  float* at;
  int blocks;
};
__host__ __device__ constexpr int part_floats(int dk, int dv) { return dk * (((dv + 15) & ~15) + (dk > dv ? dk : (dv + 15) & ~15)); }

// A block owns 16 value columns of one (sequence, head) and walks its blocks of tokens, a window between two barriers for each.  Four waves
// hold a quarter of the state's rows each, in registers in operand layout: they finish u from the shares of the key products, update
// their rows, leave these in LDS and form their shares of the next block's key products.  Four more, one on every SIMD beside them, take
// the state of the window before from LDS for the query products and finish the outputs of the block before that.  One wave alone
// on a SIMD leaves the float matrix unit idle in every barrier and round trip (3000 cycles a block for 1630 of products).
//
// Few long sequences leave most CUs idle behind that chain.  They are cut into parts that run side by side, in two launches: ENDS walks every
// part but a sequence's last without outputs (four waves), and beside its columns from a state of 0 - the recurrence is linear in the
// state - 16 columns of the unit matrix at a time without values, which become P.  PARTS then walks each part from the state in front of it,
// S <- P S + end over the parts before, and has the outputs.
template <typename T, int NS, int FORM>
__global__ __launch_bounds__(FORM == ENDS ? 256 : 512, FORM == WHOLE ? 2 : FORM == ENDS ? 3 : 4) void k_delta_walk(const float* __restrict__ ws, const unsigned* __restrict__ seen,
                                                       const T* __restrict__ v, int ldv, float* __restrict__ S,
                                                       float* __restrict__ out, int H, int dv, Pieces pc, Parts pt, SeqDesc d) {
  constexpr int DK = 64 * NS, ROWS = BT * DK, RING = FORM == WHOLE ? 2 : 1;
  __shared__ __attribute__((aligned(16))) f32x4 rk[2][4][2][64];     // shares of the key products, of the query products
  __shared__ __attribute__((aligned(16))) f32x4 rq[FORM == ENDS ? 1 : 2][4][2][64];
  __shared__ __attribute__((aligned(16))) f32x4 su[FORM == ENDS ? 1 : 2][2][64];        // u
  __shared__ __attribute__((aligned(16))) f32x4 ss[FORM == ENDS ? 1 : 2][4][NS][64];    // the state
  const int tid = threadIdx.x, vtiles = (dv + 15) / 16;
  int s, hd, slot, t0, t1, steps, part = 0, place = 0, tile = blockIdx.y;
  bool last = true;
  if constexpr (FORM == WHOLE) {
    s = blockIdx.x / H, hd = blockIdx.x % H;
    if (d.live && !d.live[s]) return;
    t0 = d.seq_off[s] + pc.first * LEN, t1 = d.seq_off[s + 1], steps = own_pieces<LEN>(d, pc, s, slot);
    if (steps <= 0) return;
  } else {
    // (a (part, head)'s columns, which read the same rows, are 8 apart: on one die)
    const int tiles = vtiles + (FORM == ENDS ? 4 * NS : 0), x = blockIdx.x / (8 * tiles) * 8 + blockIdx.x % 8;
    Part own;
    if (!find_part(d, pt.blocks * LEN, x / H, FORM == ENDS, own)) return;
    s = own.s, hd = x % H, part = own.idx, place = own.place, t0 = own.t0, t1 = own.t1, steps = (t1 - t0 + LEN - 1) / LEN;
    tile = blockIdx.x / 8 % tiles;
    slot = (t0 - part * pt.blocks * LEN) / LEN + s + part * pt.blocks;
    last = t1 == own.end;
    if (FORM == ENDS && part == 0 && tile >= vtiles) return;
  }
  const bool unit = FORM == ENDS && tile >= vtiles;         // columns of the unit matrix
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), w = wv & 3, lane = tid & 63, g = lane >> 4;
  const int col = unit ? dv : tile * 16 + (lane & 15);
  const bool colok = col < dv;
  // the places of the sequence's parts, and what this block's waves have in each
  const int PART = FORM == WHOLE ? 0 : part_floats(DK, dv), ENDF = FORM == WHOLE ? 0 : vtiles * 16 * DK;
  float* first = FORM == WHOLE ? nullptr : pt.at + ((size_t)place * H + hd) * PART;
  const size_t part_step = (size_t)H * PART;
  const unsigned own = (unsigned)(((FORM == WHOLE ? 0 : tile) * 4 * NS + NS * w) * 64 + lane) * 4;
  const int CELL = cell_floats(DK, dv);
  const float* cell = ws + ((size_t)slot * H + hd) * CELL;
  const size_t step = (size_t)H * CELL;
  const T* vp = v + (size_t)t0 * ldv + (size_t)hd * dv;
  const unsigned vcol = colok ? col : 0, rows = (NS * w * 64 + lane) * 4;
  // A value that is infinite or NaN: it counts as 0 in the products, its column of the state is NaN, and its column of the
  // outputs from its token on.  (A sequence without such values runs the loops that do not look at them.)
  auto number = [&](int i, int h, int e) {
    if (FORM == ENDS && unit) return true;
    const int tt = i * LEN + BT * h + 4 * g + e;
    return t0 + tt >= t1 || isfinite((float)vp[(size_t)min(tt, t1 - t0 - 1) * ldv + vcol]);
  };
  u32x4 any = {0u, 0u, 0u, 0u};
  for (int i = lane; i < 2 * steps; i += 64) any |= reinterpret_cast<const u32x4*>(seen)[(((size_t)slot + i / 2) * H + hd) * 2 + (i & 1)];
  const bool some = !unit && __any((any[0] | any[1]) | (any[2] | any[3]));
  const int half = w & 1;                                   // the tile whose outputs a wave finishes, every other block
  if (FORM == ENDS || wv < 4) {
    __builtin_amdgcn_s_setprio(3);                          // (the other wave's products fill the gaps)
    float* Sp = S + (((size_t)d.slots[s] * H + hd) * dv + (colok ? col : 0)) * DK + 16 * NS * w + 4 * g;
    const bool old = (pc.first > 0 || d.pos0[s] > 0) && colok;
    f32x4 St[NS];
    struct In {
      f32x4 k[2][NS], p[2][NS], g[NS], u[2];
    } in[RING];
    auto load_k = [&](int i, In& x) {
      const float* c0 = cell + (size_t)i * step;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < NS; ++c) x.k[h][c] = row4(c0 + h * ROWS + rows + c * 256);
    };
    auto load = [&](int i, In& x) {
      const float* c0 = cell + (size_t)i * step;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        x.u[h] = row4(c0 + 6 * ROWS + DK + 3 * BT * BT + ((h * vtiles + (unit ? 0 : tile)) * 64 + lane) * 4);
#pragma unroll
      for (int c = 0; c < NS; ++c) x.g[c] = row4(c0 + 6 * ROWS + 16 * (NS * w + c) + (unsigned)(4 * g));
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < NS; ++c) x.p[h][c] = row4(c0 + (4 + h) * ROWS + rows + c * 256);
    };
    auto keys = [&](int i, const In& x) {                   // shares of block i's key products, with the state in front of it
      f32x4 xk[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int c = 0; c < NS; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int h = 0; h < 2; ++h) xk[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[h][c][e], St[c][e], xk[h], 0, 0, 0);
#pragma unroll
      for (int h = 0; h < 2; ++h) rk[i & 1][w][h][lane] = xk[h];
    };
    // block i between its barrier and the next: u, the state behind it, the next block's key products.  An operand's place takes the one
    // two blocks later as soon as it is read
    auto window = [&](int i, In& x, In& next, auto odd) {
      f32x4 r[4][2], u[2];
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int h = 0; h < 2; ++h) r[a][h] = rk[i & 1][a][h][lane];
      if constexpr (RING == 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 own = FORM == ENDS && unit ? f32x4{0.f, 0.f, 0.f, 0.f} : x.u[h];   // (looked at in its turn)
        u[h] = own - ((r[0][h] + r[1][h]) + (r[2][h] + r[3][h]));
      }
      if constexpr (FORM != ENDS) su[i & 1][half][lane] = half ? u[1] : u[0];      // (two waves write the same)
      if constexpr (odd)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) u[h][e] = number(i, h, e) ? u[h][e] : NAN;
      f32x4 add[NS] = {};                                   // (added up by itself: fewer sums rounded at the state's size)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int c = 0; c < NS; ++c) add[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.p[h][c][e], u[h][e], add[c], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < NS; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) St[c][e] = fmaf(St[c][e], x.g[c][e], add[c][e]);
      load(min(i + RING, steps - 1), x);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (FORM != ENDS)
#pragma unroll
        for (int c = 0; c < NS; ++c) ss[(i + 1) & 1][w][c][lane] = St[c];
      keys(i + 1, next);                                    // (past the last block: nobody reads them)
      load_k(min(i + 1 + RING, steps - 1), next);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (RING == 2) {
      load_k(0, in[0]);
      load(0, in[0]);
      load_k(min(1, steps - 1), in[RING - 1]);
      load(min(1, steps - 1), in[RING - 1]);
    }
    if constexpr (FORM == ENDS) {
#pragma unroll
      for (int c = 0; c < NS; ++c) {
        St[c] = part == 0 && old ? row4(Sp + 16 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
        if (part == 0) *reinterpret_cast<f32x4*>(first + ENDF + own + c * 256) = St[c];
        if (unit)
#pragma unroll
          for (int e = 0; e < 4; ++e) St[c][e] = 16 * (NS * w + c) + 4 * g + e == 16 * (tile - vtiles) + (lane & 15) ? 1.f : 0.f;
      }
    } else if (FORM == PARTS && !(part == 0 && last)) {
#pragma unroll
      for (int c = 0; c < NS; ++c) St[c] = row4(first + (part == 0 ? ENDF : 0) + own + c * 256);
#pragma unroll 1
      for (int j = 1; j < part; ++j) {
        const float* f = first + j * part_step;
        f32x4 P[NS][4 * NS];
#pragma unroll
        for (int c = 0; c < NS; ++c)
#pragma unroll
          for (int k = 0; k < 4 * NS; ++k) P[c][k] = row4(f + ENDF + (unsigned)(((NS * w + c) * 4 * NS + k) * 64 + lane) * 4);
#pragma unroll
        for (int c = 0; c < NS; ++c) ss[j & 1][w][c][lane] = St[c];
        __syncthreads();
        f32x4 sum[NS] = {};
#pragma unroll
        for (int k = 0; k < 4 * NS; ++k) {
          const f32x4 x = ss[j & 1][k / NS][k % NS][lane];
#pragma unroll
          for (int c = 0; c < NS; ++c) sum[c] = mfma4(P[c][k], x, sum[c]);
        }
#pragma unroll
        for (int c = 0; c < NS; ++c) St[c] = row4(f + own + c * 256) + sum[c];
      }
    } else {
#pragma unroll
      for (int c = 0; c < NS; ++c) St[c] = old ? row4(Sp + 16 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (RING == 1) {
      load_k(0, in[0]);
      load(0, in[0]);
    }
    if constexpr (FORM == PARTS) __syncthreads();           // (the place of the first state is read)
    if constexpr (FORM != ENDS)
#pragma unroll
      for (int c = 0; c < NS; ++c) ss[0][w][c][lane] = St[c];
    keys(0, in[0]);
    load_k(min(RING, steps - 1), in[0]);
    auto walk = [&](auto odd) {
      int i = 0;
      for (; i + 2 <= steps; i += 2) {
        __syncthreads();
        window(i, in[0], in[RING - 1], odd);
        __syncthreads();
        window(i + 1, in[RING - 1], in[0], odd);
      }
      if (i < steps) {
        __syncthreads();
        window(i, in[0], in[RING - 1], odd);
      }
      __syncthreads();                                      // (the outputs of the last block)
    };
    if (some)
      walk(std::true_type{});
    else
      walk(std::false_type{});
    if constexpr (FORM == ENDS) {
      float* mine = first + part * part_step;
#pragma unroll
      for (int c = 0; c < NS; ++c) {
        if (!unit) *reinterpret_cast<f32x4*>(mine + own + c * 256) = St[c];
        // row 4 g + e, column (lane & 15) of its 16 x 16 as the left operand has them
        float* P = mine + ENDF + (((NS * w + c) * 4 * NS + tile - vtiles) * 64 + ((lane & 15) >> 2) * 16 + 4 * g) * 4 + (lane & 3);
        if (unit)
#pragma unroll
          for (int e = 0; e < 4; ++e) P[4 * e] = St[c][e];
      }
      return;
    }
    if (colok && last)
#pragma unroll
      for (int c = 0; c < NS; ++c) *reinterpret_cast<f32x4*>(Sp + 16 * c) = St[c];
    return;
  }
  if constexpr (FORM == PARTS) {
    for (int j = 1; j < part; ++j) __syncthreads();
    __syncthreads();
  }
  struct In {
    f32x4 q[2][NS], b[2];
  } in[RING];
  auto load = [&](int i, In& x) {
    const float* c0 = cell + (size_t)i * step;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int c = 0; c < NS; ++c) x.q[h][c] = row4(c0 + (2 + h) * ROWS + rows + c * 256);
      x.b[h] = row4(c0 + 6 * ROWS + DK + (half ? 1 + h : 0) * BT * BT + (lane & 15) * BT + 4 * g);
    }
  };
  f32x4 bo[2];                                              // B of the block before
  int oo[4];                                                // (a store that has no place goes past the end of its window and is dropped)
#pragma unroll
  for (int e = 0; e < 4; ++e) oo[e] = colok ? (((BT * half + 4 * g + e) * H + hd) * dv + col) * 4 : -4;
  auto outputs = [&](int i, auto odd) {
    const auto& r = rq[i & 1];
    const f32x4 u0 = su[i & 1][0][lane], u1 = su[i & 1][1][lane];
    f32x4 o = mfma4(bo[0], u0, f32x4{0.f, 0.f, 0.f, 0.f});
    if (half) o = mfma4(bo[1], u1, o);
    o += (r[0][half][lane] + r[1][half][lane]) + (r[2][half][lane] + r[3][half][lane]);
    if constexpr (odd) {
      int first = LEN;
#pragma unroll
      for (int h = 1; h >= 0; --h)
#pragma unroll
        for (int e = 3; e >= 0; --e) first = number(i, h, e) ? first : BT * h + 4 * g + e;
      first = min(first, __shfl_xor(first, 16, 64));
      first = min(first, __shfl_xor(first, 32, 64));
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = BT * half + 4 * g + e >= first ? NAN : o[e];
    }
    const int b0 = t0 + i * LEN;
    const auto win = __builtin_amdgcn_make_buffer_rsrc(out + (size_t)b0 * H * dv, 0, min(LEN, t1 - b0) * H * dv * 4, 0x00020000);
#pragma unroll
    for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[e]), win, oo[e], 0, 0);
  };
  auto window = [&](int i, In& x, auto odd) {
    f32x4 xq[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, St[NS];
#pragma unroll
    for (int c = 0; c < NS; ++c) St[c] = ss[i & 1][w][c][lane];
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h) xq[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[h][c][e], St[c][e], xq[h], 0, 0, 0);
#pragma unroll
    for (int h = 0; h < 2; ++h) rq[i & 1][w][h][lane] = xq[h];
    if (i > 0 && w >> 1 == (i & 1)) outputs(i - 1, odd);
#pragma unroll
    for (int h = 0; h < 2; ++h) bo[h] = x.b[h];
    load(min(i + RING, steps - 1), x);
    __builtin_amdgcn_sched_barrier(0);
  };
  load(0, in[0]);
  if constexpr (RING == 2) load(min(1, steps - 1), in[RING - 1]);
  auto walk = [&](auto odd) {
    int i = 0;
    for (; i + 2 <= steps; i += 2) {
      __syncthreads();
      window(i, in[0], odd);
      __syncthreads();
      window(i + 1, in[RING - 1], odd);
    }
    if (i < steps) {
      __syncthreads();
      window(i, in[0], odd);
    }
    __syncthreads();
    if (w >> 1 == (steps & 1)) outputs(steps - 1, odd);
  };
  if (some)
    walk(std::true_type{});
  else
    walk(std::false_type{});
}

// floats of a slot; 0.23 us a token at least in the token-by-token form
size_t slot_floats(int H, int dk, int dv) { return (size_t)H * (cell_floats(dk, dv) + SEEN); }
PiecePlan delta_plan(int T_, int B, int H, int dk, int dv, size_t most) {
  return plan_pieces(T_, B, LEN, slot_floats(H, dk, dv), most, 0.23f);
}

// Blocks of a part, 0: sequences in one piece.  A window takes 1.36 us alone on its CU, whatever the others do, so the longest sequence bounds
// a step that leaves CUs idle; in parts the windows of all of them count: 1.42 us a window of the outputs' walk where a CU has one block,
// 1.15 where it has two or more at once, 0.95 and 0.82 a window of the ends' (which bring 35 KB each, 7 to 10 TB/s out of the caches), 2 us
// for each part in front of the last one's state and 8 for the launch and what stands in front of the first windows (keys of 128; of 64
// three quarters).  The other sequences are taken to be of one length.
// Where there are others, a second estimate can object: as many as can be are of the longest's length, or all of them have the parts that their
// tokens make up; constants fitted to 930 timed calls of 1 to 64 heads and sequences with parts of up to nine lengths each (within 13 %).  Few long ones
// among short ones have more parts than the first one counts: 8 heads of 128 x 16, eight of 1134 tokens and 16 short ones 122 in one piece, 163 in parts of 8
// blocks.  Of 2450 calls 2080 ran in parts, 58 of them slower so, by up to a third; now 2010, 26 of them, by up to 18 %.
// us, in one piece -> in parts, 4 heads of 128 x 128: 1000 tokens 62 -> 47, 4093 197 -> 88, 9000 422 -> 170, 3000 + 1700 155 -> 103, 5000 and three
// of 40 240 -> 114 (400 33 -> 35, 4 x 2000 122 -> 121, 1000 + 700 + 500 + 600 + 800 67 -> 73: in one piece); 8 heads: 700 47 -> 43, 1000 61 -> 54, 1500 +
// 700 + 97 92 -> 86 (four parts, two and one; in parts of 8 / 10 / 14 / 16 / 18 / 24 blocks for 12 97 / 91 / 93 / 89 / 93 / 89), 4093 208 -> 136,
// 9000 445 -> 295, 3000 + 1700 167 -> 142 (4 x 2000 149 -> 206: in one piece).
int part_blocks(int T_, int B, int H, int dk, int dv, int longest) {
  const int tiles = (dv + 15) / 16, units = dk / 16, top = (longest + LEN - 1) / LEN;
  if (longest > T_ || top < 2 || (long)B * H * tiles > 256) return 0;
  const int rest = B > 1 ? ((T_ - longest) / (B - 1) + LEN - 1) / LEN : 0, alike = std::min(B, T_ / longest);
  const auto cus = [](float n) { return ceilf(n / 256.f); };
  const float scale = dk == 64 ? 0.75f : 1.f;
  struct Cost {
    float piece, window, parts, walk, end, more, prep;
  };
  constexpr Cost COST[2] = {{12.9f, 0.92f, 19.6f, 0.73f, 0.44f, 1.f, 3.3f}, {15.2f, 1.35f, 25.8f, 1.55f, 0.67f, 2.f, 6.4f}};
  const Cost& c = COST[dk / 128];
  const float prep = ((float)T_ / LEN + 0.5f * B) * H / 256 * (c.prep + 0.8f * dv / 64);
  float best = 0.92f * (1.36f * scale * top + 4.f);
  int blocks = 0;
  for (int parts = 2; parts <= 12; ++parts) {
    const int L = (top + parts - 1) / parts;
    if (L < 6) break;
    const int n = (top + L - 1) / L, m = (rest + L - 1) / L;
    const float walk = cus((float)(n + (B - 1) * m) * H * tiles);
    const float ends = cus(H * ((float)tiles * (n - 1 + (B - 1) * std::max(m - 1, 0)) + (float)units * (n - 2 + (B - 1) * std::max(m - 2, 0))));
    const float us = scale * (L * ((walk > 1.f ? 1.15f * walk : 1.42f) + (ends > 1.f ? 0.82f * ends : 0.95f)) + 2.f * (n - 2)) + 8.f;
    if (us >= best) continue;
    if (B > 1) {
      const auto takes = [&](float walked, float ended, float transitions) {
        const float w = walked * H * tiles / 256, e = H * (ended * tiles + transitions * units) / 256;
        return c.parts + prep + L * (c.walk * std::max(1.f, w) + c.end * std::max(1.f, e)) + c.more * (n - 2);
      };
      const float others = std::max((float)(T_ - longest) / (LEN * L) - 0.5f * (B - 1), 0.f);        // their ends
      if (std::max(takes(alike * n + B - alike, alike * (n - 1), alike * (n - 2)),
                   takes(n + others + B - 1, n - 1 + others, n - 2 + std::max(others - (B - 1), 0.f))) >= 0.99f * (c.piece + prep + c.window * top))
        continue;
    }
    best = us, blocks = L;
  }
  return blocks;
}
struct DeltaPlan {
  PiecePlan p;
  int blocks;            // of a part, 0: sequences in one piece
  size_t floats;
};
DeltaPlan plan_of(int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  DeltaPlan r = {delta_plan(T_, B, H, dk, dv, most), 0, 0};
  r.floats = r.p.slots * slot_floats(H, dk, dv);
  if (r.p.slots == 0 || r.p.count != 0) return r;
  if (const int blocks = part_blocks(T_, B, H, dk, dv, longest)) {      // (6 blocks or more of 65535: no more than MOST_PARTS)
    const size_t more = (size_t)T_ / (blocks * LEN) * H * part_floats(dk, dv);
    if (r.floats + more <= most) r.blocks = blocks, r.floats += more;
  }
  return r;
}

template <typename T, int NS>
void launch(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const float* g, const float* beta, float* S,
            float* out, float* ws, size_t most, int H, int G, int dv, int longest, const SeqDesc& d, hipStream_t st) {
  constexpr int DK = 64 * NS;
  const DeltaPlan plan = plan_of(d.Ttot, d.B, H, DK, dv, longest, most);
  unsigned* seen = reinterpret_cast<unsigned*>(ws + plan.p.slots * H * cell_floats(DK, dv));
  const Parts pt = {ws + plan.p.slots * slot_floats(H, DK, dv), plan.blocks};
  const unsigned tiles = (dv + 15) / 16;
  const unsigned all = plan.blocks > 0 ? d.Ttot / (plan.blocks * LEN) : 0, ends = (all * H + 7) / 8 * 8, parts = ((all + d.B) * H + 7) / 8 * 8;
  for (int w = 0; w < plan.p.windows; ++w) {
    const Pieces pc = {LEN, w * plan.p.count, plan.p.count};
    hipLaunchKernelGGL((k_delta_prep<T, NS>), dim3(H, (unsigned)plan.p.slots), dim3(512), 0, st, (const T*)q, ldq, (const T*)k, ldk,
                       (const T*)v, ldv, dv, g, beta, ws, seen, H, G, pc, d);
    if (plan.blocks == 0) {
      hipLaunchKernelGGL((k_delta_walk<T, NS, WHOLE>), dim3(d.B * H, tiles), dim3(512), 0, st, ws, seen, (const T*)v, ldv, S, out, H, dv,
                         pc, pt, d);
      continue;
    }
    hipLaunchKernelGGL((k_delta_walk<T, NS, ENDS>), dim3(ends * (tiles + 4 * NS)), dim3(256), 0, st, ws, seen, (const T*)v,
                       ldv, S, out, H, dv, pc, pt, d);
    hipLaunchKernelGGL((k_delta_walk<T, NS, PARTS>), dim3(parts * tiles), dim3(512), 0, st, ws, seen, (const T*)v, ldv, S,
                       out, H, dv, pc, pt, d);
  }
  LIPA_CHECK_LAUNCH();
}

}  // namespace

// Floats of workspace for at most `most` (longer steps run in windows), or 0 where blocks of 16 (seq_block.hip) are not slower or there is
// no room.  Two tiles between two barriers pay where one block of threads a CU walks a long sequence, and, with few columns, where the first
// kernel, whose blocks take all columns at once, is most of the work; with many columns blocks of 16 fit a CU twice.  us, 16 -> 32 tokens,
// heads of 128 x 128: 8 heads x 1000 tokens 75 -> 60, x 4000 262 -> 200, x 200 24.3 -> 24.1, 5 x 300 52 -> 52, 1500 + 700 + 97 112 -> 90, 4 x 2000
// (256 blocks of threads) 181 -> 147, 12 x 100 40 -> 44, 12 x 700 (768) 170 -> 164; 4 heads x 9000 540 -> 414, x 64 15.7 -> 17.5; 64 heads
// 2 x 1000 (1024) 336 -> 358, 4 x 256 203 -> 208.  Of 128 x 64: 32 heads 8 x 512 (1024) 285 -> 236, 16 heads 20 x 400 (1280) 288 -> 240; of
// 128 x 32, 8 x 512 103 -> 78; of 64 x 64, 4 x 600 (512) 86 -> 80, 40 x 320 (1280) 123 -> 122; of 64 x 128, 16 heads 16 x 512 (2048) 230 -> 238,
// 64 heads 4 x 300 136 -> 159.  Keys of 192 97 -> 95, of 256 146 -> 151.
// The first kernel's grid has 65535 slots at most.
size_t seq_delta_floats(int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  if (dk > 128 || T_ < 300l * B || (dv > 64 && (long)B * H * ((dv + 15) / 16) > 256)) return 0;
  const DeltaPlan plan = plan_of(T_, B, H, dk, dv, longest, most);
  return plan.p.slots > 65535 ? 0 : plan.floats;
}

// blocks of 32 tokens in a part of a sequence, 0: in one piece
int seq_delta_parts(int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  return plan_of(T_, B, H, dk, dv, longest, most).blocks;
}

void seq_delta(int code, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const float* g, const float* bpre, float* S,
               float* out, float* ws, size_t most, int H, int G, int dk, int dv, int longest, SeqDesc d, hipStream_t st) {
  SEQ_DISPATCH_T(code, {
    if (dk == 64)
      launch<T, 1>(q, ldq, k, ldk, v, ldv, g, bpre, S, out, ws, most, H, G, dv, longest, d, st);
    else
      launch<T, 2>(q, ldq, k, ldk, v, ldv, g, bpre, S, out, ws, most, H, G, dv, longest, d, st);
  });
}
