// Prompts through the recurrences whose decay is one scalar per (token, head), a block of threads per (sequence, head, 16 to 64 value columns)
// that walks the sequence's tokens and never lets go of the state.  The sums are those of seq_chunk.hip over pieces of 64 tokens: with F_t the
// log decay summed from the piece's first token, a_j = i_j - F_j the log weight of a key and b_i what a query adds to it,
//   o_i = e^{m + b_i} S^T q_i + sum_{j <= i} e^{a_j + b_i} c_j (q_i . k_j) v_j,      S <- e^{m + b_end} S + sum_j e^{a_j + b_end} c_j k_j v_j^T
// (state space: a = -F, b = F, m = 0; mLSTM: m the unit that S is counted in, b_i = -max(m, a_1 .. a_i)).
//
// A first, small kernel takes the gates of all pieces at once: their sums are in 64 bits, which would be most of a piece's time here.
// The second takes two pieces a turn.  The state stays in float accumulators; the products with queries read it from LDS as three bf16
// parts (see split3), as they do the weighted values of its update and the scores.  Nothing of a turn waits for the state but two fused
// multiply-adds, their split and the products with the queries, which stand behind a barrier while the next turn's tokens, loaded since the
// turn's start, take the places of this turn's.
//
// Measured, chunks with the states in memory (seq_chunk.hip) -> here: mLSTM, 8 prompts of 333 to 1024 tokens, 8 heads of 128 x 192: 77.9 -> 50.6 us,
// error against 64 bits 1.9 -> 1.8e-7; more shapes at walk_tiles.  Of a turn's 10 000 cycles there (48 columns) the query waves work 6 500
// (scores 900, their split and products with values 2 000, products with the state 2 400) and the state waves 9 000 (splits and products
// 4 500, staging 3 100), both on one SIMD: vector issue, three parts of everything that is float, then LDS.  What it took from 72: two kinds of
// waves, so that a scores' keys serve two tiles and a state's products two (59); loads in parts between the steps instead of all at a turn's start,
// where a wave stands still for 2 500 cycles until the address unit has them (52); gates as whole rows, 16 bytes a load (50.6).  Queries through
// LDS as whole rows: the same.
#include "seq_gates.h"

#include <algorithm>
#include <type_traits>

using namespace lipa;

int seq_run_chunks(int, int, int, int);
long seq_chunk_least(int, int, int, int);

namespace {

constexpr int PT = 64;                  // tokens of a piece
constexpr int TURN = 2 * PT;            // tokens of a turn

struct WalkWs {                         // what the first kernel leaves, per piece and head
  double *loc, *m0;                     // [slot, H, 2]: log decay of the piece, largest a; [sequence, H]: log of the state's unit in front
  float* tab;                           // [slot, H, PT, 8]: see below
};
// A token's row of the table.  A double is a float and what that leaves (A, B, F); W is the weight of a token in the piece's own contribution to the
// state, E what a query's b adds to that of the first of its 16.  The mLSTM's are against the largest a alone: what the state's unit adds is one
// factor for a query, or for the whole contribution.
enum { A_HI, A_LO, W_, E_, C_, EST_, B_HI = 4, B_LO, F_HI, F_LO };

template <bool MLSTM>
__global__ __launch_bounds__(256) void k_walk_gates(GateArgs g, WalkWs ws, const float* __restrict__ M, int H, Pieces pc, SeqDesc d) {
  const int slot = blockIdx.x, hd = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  Piece c;
  if (hd >= H || !find_piece<PT>(d, pc, slot, c)) return;
  const bool on = lane < c.n;
  const size_t t = c.t0 + min(lane, c.n - 1), cell = (size_t)slot * H + hd;
  double l, ig = 0.0;
  float dt = 0.f;
  if (MLSTM) {
    const float i = g.cap * tanhf((g.ipre[t * H + hd] + g.ib[hd]) / g.cap);
    const float f = logsigmoidf_(g.cap * tanhf((g.fpre[t * H + hd] + g.fb[hd]) / g.cap));
    ig = on ? (double)i * LOG2E : -(double)INFINITY;
    l = on ? (double)f * LOG2E : 0.0;
  } else {
    dt = softplusf_((float)g.dt[t * g.lddt + hd] + g.dt_bias[hd]);
    l = on ? (double)(-expf(g.a_log[hd]) * dt) * LOG2E : 0.0;
    // a token that forgets everything (down to -inf) counts as 2^-512, which is 0 in every float it meets: the sums behind it keep
    // their bits.  (The mLSTM weighs its inputs against the log decays: those stay as they are, and above -cap - 1.)
    l = l < -512.0 ? -512.0 : l;
  }
  const double F = scan_lanes(l, 0.0, [](double a, double b) { return a + b; }), a = ig - F;
  const double top = MLSTM ? scan_lanes(a, -(double)INFINITY, [](double x, double y) { return fmax(x, y); }) : 0.0;
  const double b = MLSTM ? -top : F, end = MLSTM ? -last_lane_d(top) : last_lane_d(F);
  if (lane == 63) {
    ws.loc[2 * cell] = F;
    ws.loc[2 * cell + 1] = top;
  }
  if (lane == 0 && c.idx == pc.first) {
    const bool old = pc.first > 0 || c.pos0 > 0;
    ws.m0[(size_t)c.s * H + hd] = MLSTM && old ? (double)M[(size_t)d.slots[c.s] * H + hd] * LOG2E : 0.0;
  }
  const long long bits = __double_as_longlong(b);
  const double b0 = __longlong_as_double(((long long)__shfl((int)(bits >> 32), lane & 48, 64) << 32) | (unsigned)__shfl((int)bits, lane & 48, 64));
  const float wt = exp2f((float)(a + end));
  float row[8];
  const auto two = [&](int i, double x) {
    row[i] = (float)x;
    row[i + 1] = on ? (float)(x - (double)row[i]) : 0.f;
  };
  two(A_HI, a);
  row[W_] = !on ? 0.f : MLSTM ? wt : wt * dt;
  row[E_] = exp2f((float)(b - b0));
  if (MLSTM) {
    two(B_HI, b);
    two(F_HI, F);
  } else {
    row[C_] = on ? dt : 0.f;
    row[EST_] = exp2f((float)F);
    row[6] = row[7] = 0.f;
  }
  f32x4* tab = reinterpret_cast<f32x4*>(ws.tab + (cell * PT + lane) * 8);
  tab[0] = f32x4{row[0], row[1], row[2], row[3]};
  tab[1] = f32x4{row[4], row[5], row[6], row[7]};
}

// Where the 16-byte piece x8 of row r stands in rows of COLS bf16 (64 or 128): operand reads take 16 rows at one piece, transposed reads 8 rows
// at two neighbouring pieces (a multiple of two, and the next); both then meet every bank once.
template <int COLS>
__device__ __forceinline__ int row_piece(int r, int x8) {
  if (COLS == 128) return x8 ^ (((r & 7) << 1) | ((r >> 3) & 1));
  const int u = r >> 1;
  return x8 ^ (((u & 3) << 1) | ((u >> 2) & 1));
}

__device__ __forceinline__ f32x4 mfma32(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 join(const bf16x4& a, const bf16x4& b) { return bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}; }
__device__ __forceinline__ float quad_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));
  return v;
}
__device__ __forceinline__ f32x4 at4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ bf16x8 at8(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

// Products of 16 x 16 x 32: lane (li, g) holds row or column li at k 8 g .. 8 g + 7 of an operand, and rows 4 g .. 4 g + 3 of column li of a
// result.  Sums over tokens take them as the results of a product of keys have them: 4 g .. 4 g + 3 of one tile, then of the next.
// Four waves own the queries, two tiles of 16 each (the first and last or the middle two of a piece: five tiles of scores), four the
// state, and stage the tokens; a SIMD has one of each.
template <int NK, int NT, bool MLSTM>
__global__ __launch_bounds__(512, 2) void k_walk(const bf16* __restrict__ q, int ldq, const bf16* __restrict__ k, int ldk,
                                                 const bf16* __restrict__ v, int ldv, float qscale, const float* __restrict__ dskip, WalkWs ws,
                                                 float* __restrict__ S, float* __restrict__ N, float* __restrict__ M, float* __restrict__ out,
                                                 float* __restrict__ den, float* __restrict__ efl, int H, int G, int dv, Pieces pc, SeqDesc d) {
  constexpr int DK = 32 * NK;
  constexpr int NR = NK / 2;                                // tiles of 16 rows of the state a wave
  static_assert(NK % 2 == 0, "key channels");
  __shared__ __attribute__((aligned(16))) bf16 sk[TURN * DK];                     // keys [token][dk]
  __shared__ __attribute__((aligned(16))) bf16 sv[NT][TURN][16];                  // values, those that are no numbers as 0
  __shared__ __attribute__((aligned(16))) bf16 sw[3][NT][TURN][16];               // weighted values for the state
  __shared__ __attribute__((aligned(16))) bf16 ss[2][3][NT][16 * DK];             // the state in front of the turn's pieces [column][dk]
  __shared__ __attribute__((aligned(16))) bf16 sn[MLSTM ? 2 : 1][MLSTM ? 3 * DK : 8];     // the normaliser's three parts
  __shared__ __attribute__((aligned(16))) bf16 sw3[MLSTM ? 3 : 1][MLSTM ? TURN : 8];      // the weights' three parts
  __shared__ __attribute__((aligned(16))) float sah[TURN], sal[TURN], sbh[TURN], sbl[TURN], seq[TURN], sest[TURN], sfc[TURN];
  __shared__ __attribute__((aligned(16))) float swk[4][64];              // a query tile's keys in front of it: 16 of the first, then the second's
  __shared__ int sbad[2][2][16 * NT];                       // per turn (two in turns), piece and column: first token whose value is no number
  const int s = blockIdx.x / H, hd = blockIdx.x % H, cb = blockIdx.y * 16 * NT, tid = threadIdx.x;
  if (d.live && !d.live[s]) return;
  int slot;
  const int np = own_pieces<PT>(d, pc, s, slot);
  if (np <= 0) return;
  const int t0 = d.seq_off[s] + pc.first * PT, n = min(d.seq_off[s + 1] - t0, np * PT), turns = (n + TURN - 1) / TURN;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, lane = tid & 63, li = lane & 15, g = lane >> 4, kh = hd / (H / G);

  const auto state_waves = [&](auto has_norm) {             // the state, and what stands in LDS
    constexpr bool norm = decltype(has_norm)::value;        // (known to the compiler: no branch between a product and what reads it)
    const int st = tid & 255, r = st >> 1, c8 = 8 * (st & 1), u = r >> 6;      // the token and columns of each tile that it stages
    const bool old = pc.first > 0 || d.pos0[s] > 0;
    const size_t hb = (size_t)d.slots[s] * H + hd;
    const bf16 *kp = k + (size_t)t0 * ldk + kh * DK, *vp = v + (size_t)t0 * ldv + (size_t)hd * dv;
    bf16x8 rk[2 * NK];
    bf16x4 rv[NT][2];
    float rtab[8];
    double rF[2], rtop[2];
    int apart;                                              // 0, which the compiler does not see: scalar loads would end every wait for LDS behind them
    asm volatile("v_mov_b32 %0, 0" : "=v"(apart));
    // A wave stands still until the address unit has taken its loads: a part of them at a time, between the turn's steps
    const auto load_keys = [&](int c, auto part) {
      constexpr int P = decltype(part)::value;
      const int tb = c * TURN, left = n - tb;
#pragma unroll
      for (int i = P * NK / 2; i < (P + 1) * NK / 2; ++i) {
        const int e = st + 256 * i, row = e / (DK / 8), x8 = e % (DK / 8);
        rk[i] = at8(kp + (size_t)(tb + min(row, left - 1)) * ldk + 8 * x8);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    const auto load_rest = [&](int c) {
      const int tb = c * TURN, left = n - tb;
      const bf16* vr = vp + (size_t)(tb + min(r, left - 1)) * ldv;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) rv[t][h] = *reinterpret_cast<const bf16x4*>(vr + min(cb + 16 * t + c8 + 4 * h, dv - 4));
      const float* tp = ws.tab + (((size_t)(slot + min(2 * c + u, np - 1)) * H + hd) * PT + (r & (PT - 1))) * 8;
      const f32x4 ta = at4(tp), tb4 = at4(tp + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        rtab[i] = ta[i];
        rtab[4 + i] = tb4[i];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const double2 l = *reinterpret_cast<const double2*>(ws.loc + 2 * ((size_t)(slot + min(2 * c + i, np - 1)) * H + hd + apart));
        rF[i] = l.x;
        rtop[i] = l.y;
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    double m = ws.m0[(size_t)s * H + hd];                   // unit of the state in front of the turn that is staged next
    float dec[2], own[2];                                   // of the turn that stands in LDS: factors of the state and of a piece's contribution
    const auto stage = [&](int c) {
      const int left = n - c * TURN;
      const bool on = r < left, both = left > PT;
      float bh, bl, est, f = 1.f;
      if (MLSTM) {
        const double e0 = fmax(m, rtop[0]), m1 = rF[0] + e0, e1 = fmax(m1, rtop[1]), mu = u ? m1 : m;
        dec[0] = exp2f((float)(m - e0));
        own[0] = exp2f((float)(rtop[0] - e0));
        dec[1] = exp2f((float)(m1 - e1));
        own[1] = exp2f((float)(rtop[1] - e1));
        m = both ? rF[1] + e1 : m1;
        bh = rtab[B_HI];
        bl = rtab[B_LO];
        const double b = (double)bh + (double)bl;
        const float over = (float)(mu + b);                 // the state's unit over the largest a
        est = exp2f(fminf(over, 0.f));
        f = exp2f(fminf(-over, 0.f));
        if (norm && (st & 1) == 0 && on)
          efl[(size_t)(t0 + c * TURN + r) * H + hd] = exp2f((float)(fmin(b, -mu) - ((double)rtab[F_HI] + (double)rtab[F_LO])));
      } else {
        dec[0] = exp2f((float)rF[0]);
        dec[1] = exp2f((float)rF[1]);
        bh = -rtab[A_HI];
        bl = -rtab[A_LO];
        est = rtab[EST_];
      }
      if ((st & 1) == 0) {
        sah[r] = rtab[A_HI];
        sal[r] = rtab[A_LO];
        sbh[r] = bh;
        sbl[r] = bl;
        seq[r] = rtab[E_] * f;
        sest[r] = est;
        sfc[r] = MLSTM ? f : rtab[C_];
        if constexpr (norm) {
          const Split z = split3(on ? rtab[W_] : 0.f, 0.f);
          sw3[0][r] = __builtin_bit_cast(bf16, (unsigned short)z.h);
          sw3[MLSTM ? 1 : 0][r] = __builtin_bit_cast(bf16, (unsigned short)z.m);
          sw3[MLSTM ? 2 : 0][r] = __builtin_bit_cast(bf16, (unsigned short)z.l);
        }
      }
      if (left < TURN)
#pragma unroll
        for (int i = 0; i < 2 * NK; ++i) rk[i] = (st + 256 * i) / (DK / 8) < left ? rk[i] : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 2 * NK; ++i) {
        const int e = st + 256 * i, row = e / (DK / 8), x8 = e % (DK / 8);
        *reinterpret_cast<bf16x8*>(sk + row * DK + 8 * row_piece<DK>(row, x8)) = rk[i];
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        // A masked score is a 0 that multiplies a later token's value: an infinite or NaN value would reach the queries in front of it.  It
        // counts as 0 in these products, and its column is NaN from its token on.  (Tokens past the end repeat the last one.)
        if (!on) rv[t][0] = rv[t][1] = bf16x4{0, 0, 0, 0};
        u32x4 o[3];
        unsigned bad = 0u;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const bf16x4 x = rv[t][h >> 1];
          const unsigned bits = __builtin_bit_cast(u32x2, x)[h & 1];
          const Split z = split3(rtab[W_] * (float)x[2 * (h & 1)], rtab[W_] * (float)x[2 * (h & 1) + 1]);
          o[0][h] = z.h;
          o[1][h] = z.m;
          o[2][h] = z.l;
          bad |= (bits & 0x7f807f80u) + 0x00800080u;
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(&sw[p][t][r][c8]) = o[p];
        if (bad & 0x80008000u)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (!isfinite((float)rv[t][e >> 2][e & 3])) {
              rv[t][e >> 2][e & 3] = (bf16)0.f;
              atomicMin(&sbad[c & 1][u][16 * t + c8 + e], r & (PT - 1));
            }
        *reinterpret_cast<bf16x8*>(&sv[t][r][c8]) = join(rv[t][0], rv[t][1]);
      }
    };
    load_keys(0, std::integral_constant<int, 0>{});
    load_keys(0, std::integral_constant<int, 1>{});
    load_keys(0, std::integral_constant<int, 2>{});
    load_keys(0, std::integral_constant<int, 3>{});
    load_rest(0);
    for (int i = st; i < 2 * 2 * 16 * NT; i += 256) (&sbad[0][0][0])[i] = PT;
    const int row0 = 16 * NR * w + 4 * g;                   // the lane's first row of the state
    f32x4 St[NR][NT], Nt[NR];
#pragma unroll
    for (int a = 0; a < NR; ++a) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int col = cb + 16 * t + li;
        St[a][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (old && col < dv) St[a][t] = at4(S + (hb * dv + col) * DK + row0 + 16 * a);
      }
      Nt[a] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (norm && old && li == 0) Nt[a] = at4(N + hb * DK + row0 + 16 * a);
    }
    const auto put_state = [&](int b) {                     // the state's parts to where the products with queries read them
#pragma unroll
      for (int a = 0; a < NR; ++a) {
        const int at = li * DK + 8 * row_piece<DK>(li, 2 * (NR * w + a) + (g >> 1)) + 4 * (g & 1);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const Split x = split3(St[a][t][0], St[a][t][1]), y = split3(St[a][t][2], St[a][t][3]);
          *reinterpret_cast<u32x2*>(&ss[b][0][t][at]) = u32x2{x.h, y.h};
          *reinterpret_cast<u32x2*>(&ss[b][1][t][at]) = u32x2{x.m, y.m};
          *reinterpret_cast<u32x2*>(&ss[b][2][t][at]) = u32x2{x.l, y.l};
        }
        if constexpr (norm) {                                         // (the parts' sums stand in three lanes)
          f32x4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = quad_sum(Nt[a][e]);
          const Split y = split3(x[0], x[1]), z = split3(x[2], x[3]);
          const u32x2 o = li == 0 ? u32x2{y.h, z.h} : li == 1 ? u32x2{y.m, z.m} : u32x2{y.l, z.l};
          if (li < 3) *reinterpret_cast<u32x2*>(&sn[b][li * DK + row0 + 16 * a]) = o;
        }
      }
    };
    const auto update = [&](int b) {                        // the state behind piece b of the turn
      f32x4 add[NR][NT] = {}, nadd[NR] = {};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int tok = PT * b + 32 * ks + 4 * g + (li >> 2);
        bf16x8 a[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const auto keys = [&](int row) {
            return read_tr(sk + row * DK + 8 * row_piece<DK>(row, 2 * (NR * w + i) + ((li >> 1) & 1)) + 4 * (li & 1));
          };
          a[i] = join(keys(tok), keys(tok + 16));
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int p = 2; p >= 0; --p) {
            const bf16x8 x = join(read_tr(&sw[p][t][tok][4 * (li & 3)]), read_tr(&sw[p][t][tok + 16][4 * (li & 3)]));
#pragma unroll
            for (int i = 0; i < NR; ++i) add[i][t] = mfma32(a[i], x, add[i][t]);
          }
        if constexpr (norm) {
          const bf16* p = &sw3[MLSTM ? min(li, 2) : 0][PT * b + 32 * ks + 4 * g];
          bf16x8 x = join(*reinterpret_cast<const bf16x4*>(p), *reinterpret_cast<const bf16x4*>(p + 16));
          if (li > 2) x = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
          for (int i = 0; i < NR; ++i) nadd[i] = mfma32(a[i], x, nadd[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int t = 0; t < NT; ++t) St[i][t][e] = fmaf(St[i][t][e], dec[b], MLSTM ? own[b] * add[i][t][e] : add[i][t][e]);
          if (norm) Nt[i][e] = fmaf(Nt[i][e], dec[b], own[b] * nadd[i][e]);
        }
    };
    __syncthreads();                                        // sbad
    stage(0);
    __syncthreads();
    for (int c = 0; c < turns; ++c) {
      const bool more = c + 1 < turns;
      const int next = min(c + 1, turns - 1);               // (behind the last turn: the same again, for nobody)
      load_keys(next, std::integral_constant<int, 0>{});
      put_state(0);
      load_keys(next, std::integral_constant<int, 1>{});
      update(0);
      load_keys(next, std::integral_constant<int, 2>{});
      if (n - c * TURN > PT) {
        put_state(1);
        load_keys(next, std::integral_constant<int, 3>{});
        update(1);
      } else {
        load_keys(next, std::integral_constant<int, 3>{});
      }
      load_rest(next);
      for (int i = st; i < 2 * 16 * NT; i += 256) (&sbad[(c + 1) & 1][0][0])[i] = PT;
      __syncthreads();
      if (more) stage(c + 1);
      __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < NR; ++a) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int col = cb + 16 * t + li;
        if (col < dv) *reinterpret_cast<f32x4*>(S + (hb * dv + col) * DK + row0 + 16 * a) = St[a][t];
      }
      if constexpr (norm) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = quad_sum(Nt[a][e]);
        if (li == 0) *reinterpret_cast<f32x4*>(N + hb * DK + row0 + 16 * a) = x;
      }
    }
    if (norm && st == 0) M[hb] = (float)(m * 0.69314718055994530942);
  };
  if (__builtin_amdgcn_readfirstlane(tid >> 6) >= 4) {
    if constexpr (MLSTM)
      if (cb == 0) return state_waves(std::true_type{});
    return state_waves(std::false_type{});
  }

  // queries: tiles `first` and 3 - first of piece u
  const int u = w >> 1;
  const bf16* qp = q + (size_t)t0 * ldq + kh * DK + 8 * g;
  f32x4 skips, zero = {0.f, 0.f, 0.f, 0.f};
  const float skip = MLSTM ? 0.f : dskip[hd];
#pragma unroll
  for (int e = 0; e < 4; ++e) skips[e] = 4 * g + e == li ? skip : 0.f;
  const auto walk = [&](auto first, auto has_norm) {
    constexpr int T0 = decltype(first)::value, TL[2] = {T0, 3 - T0};      // tiles of the piece
    constexpr bool norm = decltype(has_norm)::value;
    bf16x8 qf[2][NK];
    const auto load = [&](int c, int i) {                   // a part of the turn's queries: where they go, none is needed any more
      const int tb = c * TURN, left = n - tb;
#pragma unroll
      for (int x = 0; x < 2; ++x) qf[x][i] = at8(qp + (size_t)(tb + min(PT * u + 16 * TL[x] + li, left - 1)) * ldq + 32 * i);
    };
#pragma unroll
    for (int i = 0; i < NK; ++i) load(0, i);
    __syncthreads();
    __syncthreads();
    for (int c = 0; c < turns; ++c) {
      const int tb = c * TURN, left = n - tb;
      const bool work = PT * u < left;
      f32x4 acc[2][NT], est[2], rs[2] = {};
      if (work) {
        const float *ah = sah + PT * u, *al = sal + PT * u, *bh = sbh + PT * u, *bl = sbl + PT * u, *eq = seq + PT * u, *fc = sfc + PT * u;
        // e^{a_j + b_i} = e^{a_j + b of the tile's first} e^{b_i - that b} for the keys in front of the tile: neither factor is above 1 (but
        // for c), and one exponential serves a key; only the 16 x 16 scores on the diagonal take one each
        const float kh_ = ah[lane], kl_ = al[lane], kc = MLSTM ? 1.f : fc[lane];
        f32x4 y[2][4];                                      // scores, a lane one query's
#pragma unroll
        for (int kt = 0; kt <= TL[1]; ++kt) {
          const bf16* row = sk + (PT * u + 16 * kt + li) * DK;
          y[0][kt] = y[1][kt] = zero;
#pragma unroll
          for (int i = 0; i < NK; ++i) {
            const bf16x8 x = at8(row + 8 * row_piece<DK>(li, 4 * i + g));
            if (kt <= TL[0]) y[0][kt] = mfma32(x, qf[0][i], y[0][kt]);
            y[1][kt] = mfma32(x, qf[1][i], y[1][kt]);
          }
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
          if (TL[x] > 0) {
            const float e = __builtin_amdgcn_exp2f((bh[16 * TL[x]] + kh_) + (bl[16 * TL[x]] + kl_));
            if (lane < 16 * TL[x]) swk[w][16 * x + lane] = MLSTM ? e : e * kc;
          }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          est[x] = at4(sest + PT * u + 16 * TL[x] + 4 * g);
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[x][t] = zero;
        }
        float rsum[2] = {0.f, 0.f};
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          u32x4 pw[2][3];
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            if (2 * pr > TL[x]) continue;
            const float qe = eq[16 * TL[x] + li];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int kt = 2 * pr + h;
              f32x4 z = zero;
              if (kt < TL[x]) {
                const f32x4 wk = at4(&swk[w][16 * x + 16 * kt + 4 * g]);
#pragma unroll
                for (int e = 0; e < 4; ++e) z[e] = y[x][kt][e] * (wk[e] * qe);
              } else if (kt == TL[x]) {
                const f32x4 a = at4(ah + 16 * kt + 4 * g), b = at4(al + 16 * kt + 4 * g);
                const float qh = bh[16 * kt + li], ql = bl[16 * kt + li];
                f32x4 cw;
                if (MLSTM)
                  cw[0] = cw[1] = cw[2] = cw[3] = fc[16 * kt + li];
                else
                  cw = at4(fc + 16 * kt + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const float p = y[x][kt][e] * __builtin_amdgcn_exp2f((qh + a[e]) + (ql + b[e]));
                  z[e] = 4 * g + e <= li ? (MLSTM ? p * cw[e] : fmaf(p, cw[e], skips[e])) : 0.f;
                }
              }
              if (MLSTM) rsum[x] += (z[0] + z[1]) + (z[2] + z[3]);
              const Split lo = split3(z[0], z[1]), hi = split3(z[2], z[3]);
              pw[x][0][2 * h] = lo.h;
              pw[x][1][2 * h] = lo.m;
              pw[x][2][2 * h] = lo.l;
              pw[x][0][2 * h + 1] = hi.h;
              pw[x][1][2 * h + 1] = hi.m;
              pw[x][2][2 * h + 1] = hi.l;
            }
          }
          const int tok = PT * u + 32 * pr + 4 * g + (li >> 2);
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const bf16x8 b = join(read_tr(&sv[t][tok][4 * (li & 3)]), read_tr(&sv[t][tok + 16][4 * (li & 3)]));
#pragma unroll
            for (int p = 2; p >= 0; --p)
#pragma unroll
              for (int x = 0; x < 2; ++x)
                if (2 * pr <= TL[x]) acc[x][t] = mfma32(__builtin_bit_cast(bf16x8, pw[x][p]), b, acc[x][t]);
          }
        }
        if constexpr (norm) {
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            rsum[x] += __shfl_xor(rsum[x], 16, 64);
            rsum[x] += __shfl_xor(rsum[x], 32, 64);
            if (g == 0) swk[w][16 * x + li] = rsum[x];
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
          for (int x = 0; x < 2; ++x) rs[x] = at4(&swk[w][16 * x + 4 * g]);
        }
      }
      __syncthreads();
      if (work) {
        f32x4 o[2][NT], xn[2] = {};
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int t = 0; t < NT; ++t) o[x][t] = zero;
#pragma unroll
        for (int i = 0; i < NK; ++i) {
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int p = 2; p >= 0; --p) {
              const bf16x8 b = at8(&ss[u][p][t][li * DK + 8 * row_piece<DK>(li, 4 * i + g)]);
#pragma unroll
              for (int x = 0; x < 2; ++x) o[x][t] = mfma32(qf[x][i], b, o[x][t]);
            }
          if constexpr (norm) {
            bf16x8 b = at8(&sn[MLSTM ? u : 0][min(li, 2) * DK + 32 * i + 8 * g]);
            if (li > 2) b = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int x = 0; x < 2; ++x) xn[x] = mfma32(qf[x][i], b, xn[x]);
          }
          load(min(c + 1, turns - 1), i);
          __builtin_amdgcn_sched_barrier(0);
        }
        // (a store that has no place goes past the end of its window and is dropped)
        const auto win = __builtin_amdgcn_make_buffer_rsrc(out + ((size_t)(t0 + tb) * H + hd) * dv, 0, ((min(left, TURN) - 1) * H + 1) * dv * 4, 0x00020000);
        int bad[NT], first_bad = PT;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          bad[t] = sbad[c & 1][u][16 * t + li];
          first_bad = min(first_bad, bad[t]);
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              o[x][t][e] = fmaf(est[x][e], o[x][t][e], acc[x][t][e]);
              if (MLSTM) o[x][t][e] *= qscale;
            }
        }
        if (__any(first_bad < PT))
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
              for (int e = 0; e < 4; ++e) o[x][t][e] = 16 * TL[x] + 4 * g + e >= bad[t] ? NAN : o[x][t][e];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int col = cb + 16 * t + li;
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const unsigned at = col < dv ? ((unsigned)((PT * u + 16 * TL[x] + 4 * g) * H) * dv + col) * 4 : 0x80000000u;
#pragma unroll
            for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[x][t][e]), win, at + (unsigned)(e * H) * dv * 4, 0, 2);
          }
        }
        if constexpr (norm)
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float z = quad_sum(xn[x][e]);
              const int i = PT * u + 16 * TL[x] + 4 * g + e;
              if (li == 0 && i < left) den[(size_t)(t0 + tb + i) * H + hd] = qscale * fmaf(est[x][e], z, rs[x][e]);
            }
      }
      __syncthreads();
    }
  };
  const auto walk_tiles = [&](auto has_norm) {
    if (w & 1)
      walk(std::integral_constant<int, 1>{}, has_norm);
    else
      walk(std::integral_constant<int, 0>{}, has_norm);
  };
  if constexpr (MLSTM)
    if (cb == 0) return walk_tiles(std::true_type{});
  walk_tiles(std::false_type{});
}

// Where the tables of `cells` (piece, head) stand, in floats.  The rows of 32 bytes come first: 16-byte loads and stores take them, and behind the
// doubles of an odd number of cells they would be 8 bytes off.
struct WalkPlaces {
  size_t tab, loc, m0, end;
};
WalkPlaces walk_places(size_t cells) {
  const size_t loc = cells * 8 * PT, m0 = loc + 4 * cells;
  return {0, loc, m0, m0 + 2 * cells};
}
// floats of a piece's slot; 0.4 us a token in the token-by-token form
size_t slot_floats(int H) { return walk_places(H).end; }
PiecePlan walk_plan(int T_, int B, int H, size_t most) { return plan_pieces(T_, B, PT, slot_floats(H), most, 0.4f); }

// Tiles of 16 columns a block, or 0 where the states in chunks (seq_chunk.hip) are ahead or the sizes have no form here.  Two estimates have to agree:
//  * a block takes `turn` us for 128 tokens and 3 around them, one runs on a CU, and the longest sequence's have to follow each other beside the
//    rounds of all blocks; the chunks' three launches go by their blocks of 128 tokens and 64 columns alone;
//  * the longest sequence's last block may be in the last round, so its turns beyond the mean stand behind all rounds, where there is more than one; a
//    turn is a seventh shorter where most CUs are idle; the chunks go by their blocks, the columns that these have, and the longest sequence's chunks in
//    their second launch, in runs.
// The first alone walks one or a few long prompts among short ones where that takes up to twice as long (mLSTM, 8 heads of 64 x 160, six of 2517 tokens
// and 14 short ones 110 in chunks, 160 here).  The second is fitted to the chunks and every width of a block on 3600 calls, 1 to 64 heads, 1 to
// 64 sequences, all of one length, ragged, or one or a few long ones among short ones in any place: chunks within 10 %, blocks of one round within
// 6.  It does not know which place that is, nor how many heads share keys, so it only has to be within 5 % of agreeing (state space, where heads do, 10).  Of 6370
// calls the first one walks 3770, 156 of them slower so; both together 3490, 29 of them slower, by 2 to 25 %.
// Prompts that no chunks are there for (seq_walk_short) ask the first one alone.
// Chunks -> here, us: mLSTM, 8 heads of 128 x 192: 80 tokens 21 -> 11, 512 28 -> 21, 2 x 512 31 -> 22, 8 x 1024 89 -> 52, 48 x 128 99 -> 67, but one
// prompt of 2048 44 -> 58; of 64 x 96: 8 x 512 32 -> 21, 12 x 700 47 -> 32, one of 2048 32 -> 43; state space, 64 heads of 128 x 64: 512 34 -> 19, 4 x 512 63 ->
// 45, 8 x 1024 172 -> 143, 2 x 4096 162 -> 129, one of 4093 91 -> 92; 32 heads: 1000 33 -> 27, 12 x 700 108 -> 83, one of 4093 61 -> 89.  More
// columns a block: fewer blocks for the scores and splits, but longer turns (8 x 1024 of 128 x 192 with 16 / 32 / 48 columns 78 / 70 / 52, one prompt
// of 512 21 / 25 / 29; 8 x 512 of 64 x 96 25 / 21 / 24).
int walk_tiles(bool mlstm, int T_, int B, int H, int dk, int dv, int longest, float* takes = nullptr) {
  if ((dk != 64 && dk != 128) || B == 0) return 0;
  constexpr float TURN_US[2][4] = {{2.1f, 2.9f, 3.5f, 4.4f}, {2.8f, 3.8f, 4.9f, 0.f}};
  struct Cost {
    float turn[4], launches, block, column, head;
  };
  constexpr Cost COST[2][2] = {{{{1.97f, 2.95f, 3.74f, 4.67f}, 17.f, 0.0135f, 0.011f, 0.003f}, {{2.77f, 3.94f, 5.02f, 0.f}, 20.f, 0.023f, 0.017f, 0.002f}},
                               {{{2.51f, 3.38f, 3.9f, 4.8f}, 18.5f, 0.014f, 0.0125f, 0.007f}, {{3.31f, 4.37f, 5.3f, 0.f}, 22.f, 0.02f, 0.024f, 0.009f}}};
  const Cost& cost = COST[mlstm][dk / 128];
  const long pairs = (long)B * H, tiles = (dv + 15) / 16;
  if (longest <= 0 || longest > T_) longest = T_ - (B - 1);                    // (not known: all but a token of each other sequence)
  const bool chunked = T_ >= seq_chunk_least(B, H, dk, dv) * B;
  const long most = (longest + TURN - 1) / TURN, mean = (T_ / B + TURN - 1) / TURN;
  const float cells = ((float)T_ / 128 + 0.5f * B) * H, blocks64 = (dv + 63) / 64;
  const float chunks = 18.f + (dk == 64 ? 0.03f : 0.04f) * cells * blocks64;
  const int run = seq_run_chunks(T_, B, H, dv);
  const float chunks2 = (cost.launches + 0.55f / run * longest / 128 + cells * (cost.block * blocks64 + cost.column * dv / 64 + cost.head)) *
                        (run == 4 ? 0.92f : 1.f);
  const float most2 = 0.5f * ((longest + PT - 1) / PT), mean2 = std::min(most2, (float)T_ / B / TURN + 0.25f);
  float best = 3.f;
  int nt = 0;
  for (int t = 1; t <= (dk == 64 ? 4 : 3) && t <= tiles; ++t) {
    const long blocks = pairs * ((tiles + t - 1) / t), rounds = (blocks + 255) / 256;
    const float turn = TURN_US[dk / 128][t - 1], us = 6.f + std::max(3.f + most * turn, rounds * (3.f + mean * turn));
    float score = us / chunks;
    if (score >= 0.97f) continue;
    if (chunked) {
      const float turn2 = cost.turn[t - 1] * (0.87f + 0.13f * std::min(1.f, blocks / 256.f));
      const float late = ((mlstm ? 9.7f : 8.6f) + turn2 * (most2 + 0.25f) + (float)(rounds - 1) * (3.f + turn2 * (mean2 + 0.25f))) / chunks2;
      if (late >= (mlstm ? 1.05f : 1.1f)) continue;
      score += late;
    }
    if (score < best) {
      best = score;
      nt = t;
      if (takes != nullptr) *takes = us;
    }
  }
  return nt;
}

template <int NK, int NT, bool MLSTM>
void launch(const bf16* q, int ldq, const bf16* k, int ldk, const bf16* v, int ldv, const GateArgs& ga, float* S, float* N, float* M,
            float* out, float* den, float* efl, float* ws, size_t most, int H, int G, int dv, const SeqDesc& d, hipStream_t st) {
  const PiecePlan plan = walk_plan(d.Ttot, d.B, H, most);
  const WalkPlaces at = walk_places(plan.slots * H);
  const WalkWs w = {reinterpret_cast<double*>(ws + at.loc), reinterpret_cast<double*>(ws + at.m0), ws + at.tab};
  for (int i = 0; i < plan.windows; ++i) {
    const Pieces pc = {PT, i * plan.count, plan.count};
    hipLaunchKernelGGL((k_walk_gates<MLSTM>), dim3((unsigned)plan.slots, (H + 3) / 4), dim3(256), 0, st, ga, w, M, H, pc, d);
    hipLaunchKernelGGL((k_walk<NK, NT, MLSTM>), dim3(d.B * H, (dv + 16 * NT - 1) / (16 * NT)), dim3(512), 0, st, q, ldq, k, ldk, v, ldv, ga.qscale,
                       ga.dskip, w, S, N, M, out, den, efl, H, G, dv, pc, d);
  }
  LIPA_CHECK_LAUNCH();
}

template <bool MLSTM>
void dispatch(const bf16* q, int ldq, const bf16* k, int ldk, const bf16* v, int ldv, const GateArgs& ga, float* S, float* N, float* M,
              float* out, float* den, float* efl, float* ws, size_t most, int H, int G, int dk, int dv, int longest, const SeqDesc& d, hipStream_t st) {
#define WALK(NK_, NT_) \
  return launch<NK_, NT_, MLSTM>(q, ldq, k, ldk, v, ldv, ga, S, N, M, out, den, efl, ws, most, H, G, dv, d, st)
  const int nt = walk_tiles(MLSTM, d.Ttot, d.B, H, dk, dv, longest);
  if (dk == 64) {
    if (nt == 1) WALK(2, 1);
    if (nt == 2) WALK(2, 2);
    if (nt == 3) WALK(2, 3);
    WALK(2, 4);
  }
  if (nt == 1) WALK(4, 1);
  if (nt == 2) WALK(4, 2);
  WALK(4, 3);
#undef WALK
}

}  // namespace

// the same, for checks: the three tables' places and the end
void seq_walk_places(size_t cells, size_t* at) {
  const WalkPlaces p = walk_places(cells);
  at[0] = p.tab, at[1] = p.loc, at[2] = p.m0, at[3] = p.end;
}

int seq_walk_tiles(bool mlstm, int T_, int B, int H, int dk, int dv, int longest) { return walk_tiles(mlstm, T_, B, H, dk, dv, longest); }

// Whether an mLSTM's prompts too short for chunks walk their tokens here and not one by one (lengths that are known).  That form takes 7 us and 0.38 a
// token of the longest sequence (keys of 64: 5.5 and 0.3), or 0.14 ps a token, key channel and column where they fill the chip.  us, token by token ->
// here: 8 heads of 128 x 192, one prompt of 12 / 16 / 20 / 32 / 63 tokens 13 (not taken), 13 -> 13, 17 -> 13, 20 -> 13, 34 -> 13, 8 of 20 / 40 / 63 19 -> 14, 27 -> 14, 37 ->
// 15, 12 of 20 / 63 21 (not taken), 44 -> 21, 32 of 63 113 -> 36; of 64 x 96, 8 of 24 / 63 16 -> 13, 31 -> 13; 32 heads of 64 x 96, 32 prompts of 24 41 (53 here:
// not taken).  Error against 64 bits of 20 to 63 tokens 1.6 to 2.6e-7 -> 0.9 to 1.4e-7.  (The state space would gain as much, 13 -> 11 us at 20 tokens, 30 -> 11 at
// 63, but its outputs' error is 0.4e-7 token by token and 0.6 here.)
bool seq_walk_short(int T_, int B, int H, int dk, int dv, int longest) {
  float us = 0.f;
  if (longest <= 0 || longest > T_ || walk_tiles(true, T_, B, H, dk, dv, longest, &us) == 0) return false;
  const float full = 0.14e-6f * ((float)B * H * dv * dk) * T_ / B, chain = (dk == 64 ? 0.3f : 0.38f) * longest;
  return us < 0.97f * ((dk == 64 ? 5.5f : 7.f) + std::max(chain, full));
}

// Floats of workspace for at most `most` (longer steps run in windows), or 0 where the state in chunks (seq_chunk.hip) is to run.  longest: tokens of
// the longest sequence, 0 where the caller does not know.
size_t seq_walk_floats(bool mlstm, int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  if (walk_tiles(mlstm, T_, B, H, dk, dv, longest) == 0) return 0;
  return walk_plan(T_, B, H, most).slots * slot_floats(H);
}

void seq_walk(bool mlstm, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const GateArgs& ga, float* S, float* N,
              float* M, float* out, float* den, float* efl, float* ws, size_t most, int H, int G, int dk, int dv, int longest, const SeqDesc& d,
              hipStream_t st) {
  (mlstm ? dispatch<true> : dispatch<false>)((const bf16*)q, ldq, (const bf16*)k, ldk, (const bf16*)v, ldv, ga, S, N, M, out, den, efl, ws, most,
                                             H, G, dk, dv, longest, d, st);
}
