// Prompts through the recurrences whose decay differs per key channel - the gated delta rule and gated linear attention - in
// blocks of 16 tokens.  With G_t the product of the decays from the block's first token up to t (per key channel) and S the
// state in front of the block,
//   u_t = beta_t (v_t - (k_t G_t)^T S - sum_{j<t} A_tj u_j),   A_tj = sum_d k_td k_jd G_td / G_jd     (linear attention: u = v)
//   o_t = (q_t G_t)^T S + sum_{j<=t} B_tj u_j,                 B_tj = sum_d q_td k_jd G_td / G_jd
//   S  <- G_16 S + sum_j (k_j G_16 / G_j) u_j^T.
// A first kernel forms, for all blocks at once, everything that does not read the state: the scaled rows, B, and
// T = (I + beta A)^-1 beta, with which u = T (v - (k G)^T S).  The ratios G_t / G_j are running products of the decays
// themselves, never quotients, so a decay of 0 (or any other value) is what it is in the token-by-token scan.  The second
// kernel walks a sequence's blocks with the state in registers; all its products are float on the float matrix units
// (v_mfma_f32_16x16x4_f32), whose result layout is also its operand layout: the state, u and the outputs never move
// between lanes.
//
// Measured, token by token -> blocks: 12 sequences of 700 tokens, 8 delta heads of 128 x 128: 431 -> 163 us, of 200 tokens 124 -> 60; eight
// sequences of 512 tokens, 16 linear-attention heads of 64 x 128: 119 -> 71 us.
// Error against 64 bits as before (2.1e-7).  Ten inputs a lane two or three blocks ahead gave 2.0 -> 0.94 us a block of the longest
// sequence.  Long delta prompts that fill the chip at most once, or whose heads have 64 columns at most, run in blocks of 32 tokens
// (seq_delta.hip).
#include "seq_block.h"

#include <algorithm>
#include <type_traits>

using namespace lipa;

namespace {

// what the first kernel leaves per (block, head): [k G | q G | k G_16 / G] in operand order, G_16, T, B; and behind these, per
// (block, head) and of each of its four waves, whether a value of its tokens is infinite or NaN
__host__ __device__ constexpr int cell_floats(int dk) { return 3 * BT * dk + dk + 2 * BT * BT; }

struct DecayArgs {
  const float* g;           // [T, H * dk]: decays (delta rule) or their pre-activations (linear attention)
  const float* bias;        // linear attention: [H * dk]
  const float* beta;        // delta rule: [T, H] pre-activations
  float inv_tau, qscale;
};

// 256 threads: token j = tid / 16, and the four channels 4 x .. of every 64 (x = tid % 16).  A thread carries its token's key
// times the decays of the tokens behind it; at token s the 16 threads of a row sum k_s and q_s against it, and lane s keeps
// the sums.
template <typename T, int NS, bool DELTA>
__global__ __launch_bounds__(256) void k_block_prep(const T* __restrict__ q, int ldq, const T* __restrict__ k, int ldk,
                                                    const T* __restrict__ v, int ldv, int dv, DecayArgs a,
                                                    float* __restrict__ ws, unsigned* __restrict__ seen, int H, int G, Pieces pc,
                                                    SeqDesc d) {
  constexpr int DK = 64 * NS;
  __shared__ __attribute__((aligned(16))) float sg[BT * DK];
  __shared__ __attribute__((aligned(16))) float sk[BT * DK];
  __shared__ __attribute__((aligned(16))) float sq[BT * DK];
  __shared__ float sA[BT * BT];
  __shared__ float sb[BT];
  __shared__ int sbad[BT];
  const int slot = blockIdx.x, hd = blockIdx.y, tid = threadIdx.x;
  Piece blk;
  if (!find_piece<BT>(d, pc, slot, blk)) return;
  const int t0 = blk.t0, n = blk.n;
  const int j = tid >> 4, x = tid & 15, kh = hd / (H / G);
  const bool on = j < n;
  const size_t t = t0 + (on ? j : 0);
  f32x4 kj[NS], qj[NS], W[NS], Gm[NS];
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    const int D = 64 * c + 4 * x;
    f32x4 g = row4(a.g + (t * H + hd) * DK + D);
    kj[c] = row4(k + t * ldk + kh * DK + D);
    qj[c] = row4(q + t * ldq + kh * DK + D);
    if (!DELTA) {
      const f32x4 z = g + row4(a.bias + hd * DK + D);        // ln sigmoid(z) = min(z, 0) - ln(1 + e^-|z|)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        g[e] = __builtin_amdgcn_exp2f((fminf(z[e], 0.f) - log1p_exp_neg(fabsf(z[e]))) * (a.inv_tau * 1.4426950408889634f));
      qj[c] *= a.qscale;
    }
    if (!on) {                                               // past the end: tokens that change nothing
      kj[c] = qj[c] = f32x4{0.f, 0.f, 0.f, 0.f};
      g = f32x4{1.f, 1.f, 1.f, 1.f};
    }
    *reinterpret_cast<f32x4*>(sg + j * DK + D) = g;
    *reinterpret_cast<f32x4*>(sk + j * DK + D) = kj[c];
    *reinterpret_cast<f32x4*>(sq + j * DK + D) = qj[c];
    W[c] = kj[c];
    Gm[c] = f32x4{1.f, 1.f, 1.f, 1.f};
  }
  float vz = 0.f;
#pragma unroll 8
  for (int c = x; c < dv; c += 16) vz += 0.f * (float)v[t * ldv + (size_t)hd * dv + c];
  if (DELTA && tid < BT) sb[tid] = tid < n ? sigmoidf_(a.beta[(size_t)(t0 + tid) * H + hd]) : 0.f;
  __syncthreads();
  float ra = 0.f, rb = 0.f;                                  // A and B of (token x, token j)
#pragma unroll
  for (int s = 0; s < BT; ++s) {
    float pa = 0.f, pb = 0.f;
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      const int D = s * DK + 64 * c + 4 * x;
      const f32x4 g = row4(sg + D);
      if (s <= j)
        Gm[c] *= g;
      else
        W[c] *= g;
      const f32x4 qs = row4(sq + D);
#pragma unroll
      for (int e = 0; e < 4; ++e) pb += qs[e] * W[c][e];
      if (DELTA) {
        const f32x4 ks = row4(sk + D);
#pragma unroll
        for (int e = 0; e < 4; ++e) pa += ks[e] * W[c][e];
      }
    }
    pb = row16_sum(pb);
    if (DELTA) pa = row16_sum(pa);
    if (x == s) {
      rb = pb;
      ra = pa;
    }
  }
  // Delta rule: from the first token on whose key, decays or beta are no numbers everything is NaN.  In front of it T and B are 0
  // there, and 0 x NaN is NaN: such rows of k G and T are 0, and NaN stands in B's rows, which reach the outputs of these tokens,
  // and in the key that is written to the state.
  bool bad = false;
  if (DELTA) {
    float z = 0.f;
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) z += 0.f * (kj[c][e] * Gm[c][e]);
    bad = !(row16_sum(z) == 0.f && isfinite(sb[j]));
    if (x == 0) sbad[j] = bad ? j : BT;
  }
  float* cell = ws + ((size_t)slot * H + hd) * cell_floats(DK);
  const bool odd = __any(vz != 0.f);
  if ((tid & 63) == 0) seen[((size_t)slot * H + hd) * 4 + (tid >> 6)] = odd;
  float *ck = cell, *cq = cell + BT * DK, *cp = cell + 2 * BT * DK, *cg = cell + 3 * BT * DK, *cT = cg + DK, *cB = cT + BT * BT;
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    // operand order of the 16x16x4 products: [tile of 16 channels][4 channels][token][channel of the 4] for the rows, and
    // [tile][4 tokens][channel][token of the 4] for the keys that are written to the state
    const int tile = 4 * c + (x >> 2), base = (tile * 64 + (x & 3) * 16 + j) * 4;
    if (DELTA) *reinterpret_cast<f32x4*>(ck + base) = bad ? f32x4{0.f, 0.f, 0.f, 0.f} : kj[c] * Gm[c];
    *reinterpret_cast<f32x4*>(cq + base) = qj[c] * Gm[c];
#pragma unroll
    for (int e = 0; e < 4; ++e) cp[(tile * 64 + (j >> 2) * 16 + 4 * (x & 3) + e) * 4 + (j & 3)] = bad ? NAN : W[c][e];
    if (j == BT - 1) *reinterpret_cast<f32x4*>(cg + 64 * c + 4 * x) = Gm[c];
  }
  if (!DELTA) cB[x * BT + j] = x >= j ? rb : 0.f;
  if (DELTA) {
    sA[x * BT + j] = ra;
    __syncthreads();
    int first = sbad[x];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o, 16));
    cB[x * BT + j] = x >= first ? NAN : x >= j ? rb : 0.f;
    if (tid < BT) {                                          // column tid of (I + beta A)^-1 beta, row after row
      float r[BT];
#pragma unroll
      for (int s = 0; s < BT; ++s) {
        float acc = s == tid ? 1.f : 0.f;
#pragma unroll
        for (int i = 0; i < s; ++i) acc -= sA[s * BT + i] * r[i];
        r[s] = s >= first ? 0.f : sb[s] * acc;
        cT[s * BT + tid] = r[s];
      }
    }
  }
}

// A block owns 16 value columns of one (sequence, head); its four waves own a quarter of the key rows each, with the state in
// registers in operand layout.  Per 16 tokens a wave runs its share of the key products, the four shares meet in LDS (two
// buffers, one barrier), every wave finishes u for itself and updates its rows; the query products run under the LDS round trip
// and the waves take turns at summing them into outputs, one block of tokens later.  Bound by the chain of a block of tokens
// (key products, LDS round trip, u, update); what it reads is on its way two or three blocks ahead, since it comes from memory
// or another die's cache.
//
// Few long sequences of linear attention leave most CUs idle behind that chain: they run in parts side by side, in two launches.  ENDS
// walks every part but a sequence's last from a state of 0 (the first part: from the state in front of it), without queries, outputs or
// barriers, and leaves the state behind it and the product of its decays; PARTS walks each part from S <- decays x S + end over the
// parts before.  Per (part, head): 16 columns of the state at a time in operand layout, the state in front of the sequence (the last
// part may have written its own by the time the first one runs again), the decays.
struct Parts {
  float* at;
  int blocks;
};
__host__ __device__ constexpr int part_floats(int dk, int dv) { return 2 * dk * ((dv + 15) & ~15) + dk; }

template <typename T, int NS, bool DELTA, int FORM>
__global__ __launch_bounds__(256, NS > 2 ? 1 : 2) void k_block_scan(const float* __restrict__ ws, const unsigned* __restrict__ seen,
                                                                    const T* __restrict__ v, int ldv, float* __restrict__ S,
                                                                    float* __restrict__ out, int H, int dv, Pieces pc, Parts pt, SeqDesc d) {
  constexpr int DK = 64 * NS, CELL = cell_floats(DK), RING = NS == 1 ? 4 : 3;
  __shared__ __attribute__((aligned(16))) f32x4 red[FORM == ENDS ? 1 : 2][FORM == ENDS ? 1 : 4][2][64];
  const int tid = threadIdx.x, vtiles = (dv + 15) / 16;
  int s, hd, slot, t0, t1, steps, part = 0, place = 0, tile = blockIdx.y;
  bool last = true;
  if constexpr (FORM == WHOLE) {
    s = blockIdx.x / H, hd = blockIdx.x % H;
    if (d.live && !d.live[s]) return;
    t0 = d.seq_off[s] + pc.first * BT, t1 = d.seq_off[s + 1], steps = own_pieces<BT>(d, pc, s, slot);
    if (steps <= 0) return;
  } else {
    // (a (part, head)'s columns, which read the same rows, are 8 apart: on one die)
    const int x = blockIdx.x / (8 * vtiles) * 8 + blockIdx.x % 8;
    Part own;
    if (!find_part(d, pt.blocks * BT, x / H, FORM == ENDS, own)) return;
    s = own.s, hd = x % H, part = own.idx, place = own.place, t0 = own.t0, t1 = own.t1, steps = (t1 - t0 + BT - 1) / BT;
    tile = blockIdx.x / 8 % vtiles;
    slot = (t0 - part * pt.blocks * BT) / BT + s + part * pt.blocks;
    last = t1 == own.end;
  }
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, col = tile * 16 + (lane & 15);
  const bool colok = col < dv;
  const float* cell = ws + ((size_t)slot * H + hd) * CELL;
  const size_t step = (size_t)H * CELL;
  const T* vp = v + (size_t)t0 * ldv + (size_t)hd * dv;
  const unsigned vcol = colok ? col : 0, m = 3 * BT * DK + DK + (lane & 15) * BT + 4 * g;
  float* Sp = S + (((size_t)d.slots[s] * H + hd) * dv + (colok ? col : 0)) * DK + 16 * NS * w + 4 * g;
  f32x4 St[NS], Gs[NS];                           // the state; ENDS: the decays so far
  const bool old = (pc.first > 0 || d.pos0[s] > 0) && colok;
  const int ENDF = vtiles * 16 * DK;
  const size_t part_step = (size_t)H * part_floats(DK, dv);
  float* first = FORM == WHOLE ? nullptr : pt.at + ((size_t)place * H + hd) * part_floats(DK, dv);       // the sequence's first part's
  const unsigned own = (unsigned)((tile * 4 * NS + NS * w) * 64 + lane) * 4, rows = 16 * NS * w + 4 * g;
#pragma unroll
  for (int c = 0; c < NS; ++c) Gs[c] = f32x4{1.f, 1.f, 1.f, 1.f};
  if (FORM == PARTS && !(part == 0 && last)) {
#pragma unroll
    for (int c = 0; c < NS; ++c) St[c] = row4(first + (part == 0 ? ENDF : 0) + own + c * 256);
    for (int j = 1; j < part; ++j) {
      const float* f = first + j * part_step;
#pragma unroll
      for (int c = 0; c < NS; ++c) {
        const f32x4 D = row4(f + 2 * ENDF + 16 * c + rows), end = row4(f + own + c * 256);
#pragma unroll
        for (int e = 0; e < 4; ++e) St[c][e] = fmaf(D[e], St[c][e], end[e]);
      }
    }
  } else {
#pragma unroll
    for (int c = 0; c < NS; ++c) St[c] = part == 0 && old ? row4(Sp + 16 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (FORM == ENDS && part == 0)
#pragma unroll
    for (int c = 0; c < NS; ++c) *reinterpret_cast<f32x4*>(first + ENDF + own + c * 256) = St[c];
  struct In {
    f32x4 k[NS], q[NS], p[NS], g[NS], tm, bm;
    T v[4];
  } in[RING];
  auto load = [&](int i, In& x) {
    const float* c0 = cell + (size_t)i * step;
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      const unsigned o = ((NS * w + c) * 64 + lane) * 4;
      if (DELTA) x.k[c] = row4(c0 + o);
      if (FORM != ENDS) x.q[c] = row4(c0 + BT * DK + o);
      x.p[c] = row4(c0 + 2 * BT * DK + o);
      x.g[c] = row4(c0 + 3 * BT * DK + 16 * (NS * w + c) + (unsigned)(4 * g));
    }
    if (DELTA) x.tm = row4(c0 + m);
    if (FORM != ENDS) x.bm = row4(c0 + m + BT * BT);
    // (values are not looked at before their turn: that would wait for every load issued before them)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      x.v[e] = (vp + (size_t)i * BT * ldv)[(unsigned)min(4 * g + e, t1 - t0 - i * BT - 1) * (unsigned)ldv + vcol];
  };
  f32x4 uo, bo;                                   // u and B of the block of tokens before
  unsigned long long fo[4];                       // lanes whose value of token e of 4 there is a number
  // A value that is infinite or NaN: T and B are 0 in front of their diagonals, and 0 x inf is NaN, so it counts as 0 in the
  // products, its column of the state is NaN, and its column of the outputs from its token on.  (This costs a tenth of the time: a
  // sequence without such values runs the loop that does not look at them.)
  auto outputs = [&](int i, auto odd) {
    const auto& r = red[i & 1];
    f32x4 o = (r[0][1][lane] + r[1][1][lane]) + (r[2][1][lane] + r[3][1][lane]);
#pragma unroll
    for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(bo[e], uo[e], o, 0, 0, 0);
    if constexpr (odd) {
      int first = BT;
#pragma unroll
      for (int e = 3; e >= 0; --e) first = (fo[e] >> lane) & 1 ? first : 4 * g + e;
      first = min(first, __shfl_xor(first, 16, 64));
      first = min(first, __shfl_xor(first, 32, 64));
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = 4 * g + e >= first ? NAN : o[e];
    }
    // (a store that has no place goes past the end of its window and is dropped: with a branch around it the compiler waits for
    // every load in flight)
    const int b0 = t0 + i * BT;
    const auto win = __builtin_amdgcn_make_buffer_rsrc(out + (size_t)b0 * H * dv, 0, min(BT, t1 - b0) * H * dv * 4, 0x00020000);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[e]), win, colok ? (((4 * g + e) * H + hd) * dv + col) * 4 : -4, 0, 0);
  };
  auto run = [&](int i, const In& x, auto odd) {
    auto& r = red[i & 1];
    if (DELTA) {                                  // two chains of products: one alone waits for its own results
      f32x4 x0 = {0.f, 0.f, 0.f, 0.f}, x1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NS; ++c) {
        x0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[c][0], St[c][0], x0, 0, 0, 0);
        x1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[c][1], St[c][1], x1, 0, 0, 0);
        x0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[c][2], St[c][2], x0, 0, 0, 0);
        x1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[c][3], St[c][3], x1, 0, 0, 0);
      }
      r[w][0][lane] = x0 + x1;
    }
    f32x4 xq = {0.f, 0.f, 0.f, 0.f};
    if constexpr (FORM != ENDS) {
      __syncthreads();
#pragma unroll
      for (int c = 0; c < NS; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) xq = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[c][e], St[c][e], xq, 0, 0, 0);
    }
    f32x4 u;
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = t0 + i * BT + 4 * g + e < t1 ? (float)x.v[e] : 0.f;
    bool fin[4];
    if constexpr (odd)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        fin[e] = isfinite(u[e]);
        u[e] = fin[e] ? u[e] : 0.f;
      }
    if (DELTA) {
      const f32x4 e = u - ((r[0][0][lane] + r[1][0][lane]) + (r[2][0][lane] + r[3][0][lane]));
      u = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) u = __builtin_amdgcn_mfma_f32_16x16x4f32(x.tm[j], e[j], u, 0, 0, 0);
    }
    if constexpr (FORM != ENDS) r[w][1][lane] = xq;
    f32x4 us = u;
    if constexpr (odd)
#pragma unroll
      for (int e = 0; e < 4; ++e) us[e] = fin[e] ? u[e] : NAN;
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      St[c] *= x.g[c];
      if constexpr (FORM == ENDS) Gs[c] *= x.g[c];
#pragma unroll
      for (int e = 0; e < 4; ++e) St[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.p[c][e], us[e], St[c], 0, 0, 0);
    }
    if constexpr (FORM == ENDS) return;
    if (w == (i & 3) && i > 0) outputs(i - 1, odd);    // its query products were written in front of this barrier
    uo = u;
    bo = x.bm;
    if constexpr (odd)
#pragma unroll
      for (int e = 0; e < 4; ++e) fo[e] = __ballot(fin[e]);
  };
#pragma unroll
  for (int x = 0; x < RING - 1; ++x) load(min(x, steps - 1), in[x]);
  u32x4 any = {0u, 0u, 0u, 0u};
  for (int i = lane; i < steps; i += 64) any |= reinterpret_cast<const u32x4*>(seen)[((size_t)slot + i) * H + hd];
  if (__any((any[0] | any[1]) | (any[2] | any[3]))) {
#pragma unroll 1
    for (int i = 0; i < steps; ++i) {
      load(i, in[0]);
      run(i, in[0], std::true_type{});
    }
    if constexpr (FORM != ENDS) {
      __syncthreads();                            // the last query products stand
      if (w == (steps & 3)) outputs(steps - 1, std::true_type{});
    }
  } else {
    constexpr std::false_type odd{};
    int i = 0;
    for (; i + RING <= steps; i += RING) {
#pragma unroll
      for (int x = 0; x < RING; ++x) {
        load(min(i + x + RING - 1, steps - 1), in[(x + RING - 1) % RING]);
        run(i + x, in[x], odd);
      }
    }
#pragma unroll
    for (int x = 0; x < RING - 1; ++x)
      if (i + x < steps) run(i + x, in[x], odd);
    if constexpr (FORM != ENDS) {
      __syncthreads();
      if (w == (steps & 3)) outputs(steps - 1, odd);
    }
  }
  if constexpr (FORM == ENDS) {
    float* mine = first + part * part_step;
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      *reinterpret_cast<f32x4*>(mine + own + c * 256) = St[c];
      if (tile == 0 && (lane & 15) == 0) *reinterpret_cast<f32x4*>(mine + 2 * ENDF + 16 * c + rows) = Gs[c];
    }
    return;
  }
  if (colok && last)
#pragma unroll
    for (int c = 0; c < NS; ++c) *reinterpret_cast<f32x4*>(Sp + 16 * c) = St[c];
}

// floats of a slot; 0.23 us a token at least in the token-by-token form
size_t slot_floats(int H, int dk) { return (size_t)H * (cell_floats(dk) + 4); }

// Blocks of a part of linear attention, 0: sequences in one piece.  A block of tokens takes 0.49 us where a CU has one or two blocks of threads,
// whatever the others do; in parts the blocks of all of them count, twice: 0.28 us for each block of threads on a CU, at least as for 1.3,
// 0.6 for a part in front of the last one's state and 6 for the launch and the first blocks (keys of 64).  The other sequences are taken
// to be of one length.
// A second estimate can object.  It knows that keys of 192 and 256 leave one block of threads a CU, and that few long sequences among short ones have more parts:
// as many as can be are of the longest's length, or the others have the parts that their tokens make up.  Its constants are fitted to 1650 timed
// calls of 1 to 64 heads and sequences with parts of up to nine lengths each (within 17 %).  Of 3440 calls 2580 ran in parts, 93 of them slower so, by up to
// 36 % (keys of 192, 16 heads of 192 columns, one prompt of 1396 tokens 110 -> 147); now 2460, 31 of them, by up to 15 %.
// us, in one piece -> in parts, 8 heads of 64 x 128: 1000 tokens 40 -> 26, 4093 137 -> 68, 9000 288 -> 118, 3000 + 1700
// 107 -> 77, 5000 and three of 40 165 -> 76 (400 21 -> 20, 4 x 2000 86 -> 91, 10 x 700 74 -> 89: in one piece); 16 heads: 1000 45 -> 38, 4093
// 147 -> 100, 9000 312 -> 203, 5000 and three of 40 224 -> 127 (400 22 -> 25, 3000 + 1700 118 -> 113: in one piece).
int part_blocks(int T_, int B, int H, int dk, int dv, int longest) {
  const int top = (longest + BT - 1) / BT, rest = B > 1 ? ((T_ - longest) / (B - 1) + BT - 1) / BT : 0;
  if (longest <= 0 || longest > T_ || (long)B * H * ((dv + 15) / 16) > 1024) return 0;
  const float full = H * ((dv + 15) / 16) / 256.f, scale = (dk + 64) / 128.f;
  struct Cost {
    float launches, piece, shared, part, beside, prep, prep64;       // us: of a step; of a block in one piece, and for each on its CU beyond one; in parts
  };
  constexpr Cost COST[4] = {{10.3f, 0.43f, 0.09f, 0.64f, 0.215f, 1.45f, 0.6f},
                            {12.4f, 0.53f, 0.11f, 0.78f, 0.28f, 3.f, 0.95f},
                            {15.2f, 0.69f, 0.19f, 1.08f, 0.58f, 4.6f, 1.8f},
                            {15.6f, 0.98f, 0.36f, 1.4f, 0.74f, 8.f, 2.1f}};
  const Cost& c = COST[dk / 64 - 1];
  const float step = c.launches + ((float)T_ / BT + 0.5f * B) * H / 256 * (c.prep + c.prep64 * dv / 64);
  const float one = step + top * (c.piece + c.shared * std::max(0.f, B * full - 1.f));
  const int alike = std::min(B, T_ / longest);
  float best = 0.85f * 0.49f * scale * top;
  int blocks = 0;
  for (int parts = 2; parts <= 16; ++parts) {
    const int L = (top + parts - 1) / parts;
    if (L < 8) break;
    const int n = (top + L - 1) / L, m = (rest + L - 1) / L;
    const float walk = full * (n + (B - 1) * m), ends = full * (n - 1 + (B - 1) * std::max(m - 1, 0));
    const float us = scale * (0.28f * L * (std::max(walk, 1.3f) + std::max(ends, 1.3f)) + 0.6f * (n - 2)) + 6.f;
    if (us >= best) continue;
    const float others = std::max((float)(T_ - longest) / (BT * L) - 0.5f * (B - 1), 0.f);        // their ends
    const float walk2 = full * std::max((float)(alike * n + B - alike), n + others + B - 1), ends2 = full * std::max((float)(alike * (n - 1)), n - 1 + others);
    const float us2 = step + 5.5f + L * (c.part + c.beside * (std::max(0.f, walk2 - 1.f) + std::max(0.f, ends2 - 1.f))) + 0.25f * (n - 2);
    if (us2 < (dk <= 128 ? 0.97f : 0.94f) * one) best = us, blocks = L;
  }
  return blocks;
}

struct BlockPlan {
  PiecePlan p;
  int blocks;            // of a part, 0: sequences in one piece
  size_t floats;
};
BlockPlan block_plan(bool delta, int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  BlockPlan r = {plan_pieces(T_, B, BT, slot_floats(H, dk), most, 0.23f), 0, 0};
  r.floats = r.p.slots * slot_floats(H, dk);
  if (delta || r.p.slots == 0 || r.p.count != 0) return r;
  if (const int blocks = part_blocks(T_, B, H, dk, dv, longest)) {
    const size_t more = (size_t)T_ / (blocks * BT) * H * part_floats(dk, dv);
    // (16 parts of a sequence at most where none is longer than `longest`; a caller may have that wrong, and the estimates' constants are no bound)
    if (T_ / (blocks * BT) + B <= MOST_PARTS && r.floats + more <= most) r.blocks = blocks, r.floats += more;
  }
  return r;
}

template <typename T, int NS, bool DELTA>
void launch(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const DecayArgs& a, float* S, float* out,
            float* ws, size_t most, int H, int G, int dv, int longest, const SeqDesc& d, hipStream_t st) {
  constexpr int DK = 64 * NS;
  const BlockPlan plan = block_plan(DELTA, d.Ttot, d.B, H, DK, dv, longest, most);
  unsigned* seen = reinterpret_cast<unsigned*>(ws + plan.p.slots * H * cell_floats(DK));
  const Parts pt = {ws + plan.p.slots * slot_floats(H, DK), plan.blocks};
  const unsigned tiles = (dv + 15) / 16;
  for (int w = 0; w < plan.p.windows; ++w) {
    const Pieces pc = {BT, w * plan.p.count, plan.p.count};
    hipLaunchKernelGGL((k_block_prep<T, NS, DELTA>), dim3((unsigned)plan.p.slots, H), dim3(256), 0, st, (const T*)q, ldq, (const T*)k,
                       ldk, (const T*)v, ldv, dv, a, ws, seen, H, G, pc, d);
    if constexpr (!DELTA)
      if (plan.blocks > 0) {
        const unsigned all = d.Ttot / (plan.blocks * BT), ends = (all * H + 7) / 8 * 8, parts = ((all + d.B) * H + 7) / 8 * 8;
        hipLaunchKernelGGL((k_block_scan<T, NS, DELTA, ENDS>), dim3(ends * tiles), dim3(256), 0, st, ws, seen, (const T*)v, ldv, S, out, H,
                           dv, pc, pt, d);
        hipLaunchKernelGGL((k_block_scan<T, NS, DELTA, PARTS>), dim3(parts * tiles), dim3(256), 0, st, ws, seen, (const T*)v, ldv, S, out,
                           H, dv, pc, pt, d);
        continue;
      }
    hipLaunchKernelGGL((k_block_scan<T, NS, DELTA, WHOLE>), dim3(d.B * H, tiles), dim3(256), 0, st, ws, seen, (const T*)v, ldv, S, out, H,
                       dv, pc, pt, d);
  }
  LIPA_CHECK_LAUNCH();
}

template <bool DELTA>
void dispatch(int code, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const DecayArgs& a, float* S,
              float* out, float* ws, size_t most, int H, int G, int dk, int dv, int longest, const SeqDesc& d, hipStream_t st) {
  SEQ_DISPATCH_T(code, {
    switch (dk / 64) {
      case 1: launch<T, 1, DELTA>(q, ldq, k, ldk, v, ldv, a, S, out, ws, most, H, G, dv, longest, d, st); break;
      case 2: launch<T, 2, DELTA>(q, ldq, k, ldk, v, ldv, a, S, out, ws, most, H, G, dv, longest, d, st); break;
      case 3: launch<T, 3, DELTA>(q, ldq, k, ldk, v, ldv, a, S, out, ws, most, H, G, dv, longest, d, st); break;
      default: launch<T, 4, DELTA>(q, ldq, k, ldk, v, ldv, a, S, out, ws, most, H, G, dv, longest, d, st); break;
    }
  });
}

}  // namespace

size_t seq_delta_floats(int, int, int, int, int, int, size_t);
void seq_delta(int, const void*, int, const void*, int, const void*, int, const float*, const float*, float*, float*, float*, size_t,
               int, int, int, int, int, SeqDesc, hipStream_t);

// Floats of workspace of the blocked form, or 0 where the token-by-token scan is the one to run: key sizes that are no multiple
// of 64 or above 256, rows that vector loads of four channels cannot take, and steps of few tokens a sequence.  At most `most`: longer
// steps run in windows.
size_t seq_block_floats(int code, bool delta, const void* q, int ldq, const void* k, int ldk, const void* g, const void* bias,
                        const void* S, int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  const int bytes = code == 0 ? 8 : 16;
  const auto fits = [](const void* p, int ld, int b) { return ld % 4 == 0 && ((uintptr_t)p & (b - 1)) == 0; };
  if (dk % 64 != 0 || dk > 256 || !fits(q, ldq, bytes) || !fits(k, ldk, bytes) || !fits(g, 4, 16) || !fits(bias, 4, 16) ||
      !fits(S, 4, 16) || B == 0)
    return 0;
  // Two launches and a block's chain of 0.5 to 0.9 us per 16 tokens, against 0.23 (linear attention) and 0.39 us a token; with
  // many (sequence, head, 16 columns) to run at once both are bound by issue, and linear attention's token form is then the
  // cheaper one.  us, tokens -> blocks, heads of 128 x 128 (delta) and 64 x 128: 64 delta heads (512 blocks) at 32 tokens 19 -> 16,
  // at 512 201 -> 83; 384 heads at 48 tokens 69 -> 73, at 64 88 -> 85, at 256 318 -> 290.  Linear attention: 64 heads at 32
  // tokens 11 -> 12, at 48 15 -> 12, at 512 119 -> 44; 128 heads at 48 16 -> 17, at 64 20 -> 19; 384 heads at 256 100 -> 120.
  // Many (sequence, head) pairs of few columns, or of keys of 64, leave the token form nothing to wait for, at any length: times its
  // time, delta, 1024 pairs of 64 x 64 2.0, of 128 x 32 1.1, 4096 of 128 x 64 1.1, 256 of 64 x 256 1.2 (of 64 x 128 0.95 from 96 tokens on,
  // of 128 x 32 1.2 at 64, 0.7 at 128); linear attention, 256 of 128 x 64 1.06, of 256 x 32 1.15 (of 64 x 32 1.07 at 64, 0.91 at 128).
  const long pairs = (long)B * H, blocks = pairs * ((dv + 15) / 16), never = 1l << 40;
  long least;
  if (delta) {
    least = pairs < 128 && blocks <= 1024 ? 32 : 64;
    if (pairs >= 256 && dv <= 64) least = dv <= 32 ? 128 : 96;
    if (dk == 64 && blocks > 1024) least = 96;
    if ((dk == 64 && (pairs > 512 || blocks >= 4096)) || (dv <= 32 && pairs >= 1024) || (dv <= 64 && pairs >= 4096)) least = never;
  } else if (pairs >= 256) {
    least = blocks <= 512 && dk <= 192 ? 128 : never;
  } else {
    least = blocks > 1536 ? never : blocks > 512 || dk == 64 ? 64 : 40;
  }
  if (T_ < least * B) return 0;
  if (const size_t n = delta ? seq_delta_floats(T_, B, H, dk, dv, longest, most) : 0) return n;
  return block_plan(delta, T_, B, H, dk, dv, longest, most).floats;
}

// blocks of 16 tokens in a part of a sequence of linear attention, 0: in one piece
int seq_gla_parts(int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  return block_plan(false, T_, B, H, dk, dv, longest, most).blocks;
}

void seq_block_delta(int code, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const float* g,
                     const float* bpre, float* S, float* out, float* ws, size_t most, int H, int G, int dk, int dv,
                     int longest, SeqDesc d, hipStream_t st) {
  if (seq_delta_floats(d.Ttot, d.B, H, dk, dv, longest, most) > 0) {
    seq_delta(code, q, ldq, k, ldk, v, ldv, g, bpre, S, out, ws, most, H, G, dk, dv, longest, d, st);
    return;
  }
  const DecayArgs a = {g, nullptr, bpre, 1.f, 1.f};
  dispatch<true>(code, q, ldq, k, ldk, v, ldv, a, S, out, ws, most, H, G, dk, dv, longest, d, st);
}

void seq_block_gla(int code, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const float* z,
                   const float* zb, float inv_tau, float qscale, float* S, float* out, float* ws, size_t most, int H, int dk,
                   int dv, int longest, SeqDesc d, hipStream_t st) {
  const DecayArgs a = {z, zb, nullptr, inv_tau, qscale};
  dispatch<false>(code, q, ldq, k, ldk, v, ldv, a, S, out, ws, most, H, H, dk, dv, longest, d, st);
}
