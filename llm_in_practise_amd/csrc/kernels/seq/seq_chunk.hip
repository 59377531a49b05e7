// Prompts through the recurrences whose decay is one scalar per (token, head) - the state-space-duality form and the
// mLSTM - chunk by chunk instead of token by token.  With F_t the log decay summed from the chunk's first token,
//   o_t = e^{F_t} S_prev^T q_t + sum_{j <= t} e^{F_t - F_j} c_j (q_t . k_j) v_j,
//   S_end = e^{F_C} S_prev + sum_j e^{F_C - F_j} c_j k_j v_j^T,
// which is matrix products over a chunk of CK tokens.  Three kernels: (1) every run of one, two or four chunks' own contribution to the
// state, all runs at once, and what stands in front of the run's later chunks; (2) the states in front of the runs, an element-wise
// walk over a sequence's runs that leaves them where the contributions stood; (3) the outputs, all chunks at once.
//
// What is float in the token-by-token scans stays float here.  q, k and v are bf16, so q.k runs on the bf16 matrix units
// exactly (float sums).  A float factor of a product (decayed scores, weighted values, the state) is the sum of three bf16
// numbers, which hold its 24 bits: three products with float sums, at five times the rate of the float matrix units.  Log
// decays are summed in 64 bits and kept as two floats, so that the difference of two large sums is exact.
//
// Measured, token by token -> chunks: state space, one prompt of 4093 tokens, 64 heads of 128 x 64: 2350 -> 92 us (state 32, walk 9,
// outputs 50); mLSTM, 8 prompts of 333 to 1024 tokens, 8 heads of 128 x 192: 649 -> 80 us (25, 11, 43;
// they now walk in 50, seq_walk.hip).  Error against 64 bits
// 1.6e-7 -> 0.9e-7 and 4.4e-7 -> 1.9e-7: fewer roundings stand between a token and the outputs far behind it.
// The first case reads and writes 335 MB, 235 of them states and outputs, of which a copy moves 5 TB/s.  With every chunk's contribution
// walked by itself (69 MB of states out, in, out and in), operands of the outputs loaded from memory rows as they are needed, an
// exponential for each score and splits by rounding it took 150 us (46, 25, 80).
#include "seq_gates.h"

#include <algorithm>
#include <type_traits>

using namespace lipa;

size_t seq_walk_floats(bool, int, int, int, int, int, int, size_t);
bool seq_walk_short(int, int, int, int, int, int);
void seq_walk(bool, const void*, int, const void*, int, const void*, int, const GateArgs&, float*, float*, float*, float*, float*, float*, float*, size_t,
              int, int, int, int, int, const SeqDesc&, hipStream_t);

namespace {

constexpr int CK = 128;                 // tokens of a chunk (4 waves x 32 queries)

struct Gate {                           // of a wave's lane: tokens 2 * lane and 2 * lane + 1, in powers of two
  double F0, F1, Fc;                    // log decays from the chunk's start, and of the whole chunk
  double a0, a1;                        // log of the input weight against the chunk's start: i - F (state space: -F)
  float c0, c1;                         // factor of the input that is not in the logarithm (state space: dt)
};

struct GateIn {                         // a lane's two tokens as they stand in memory
  float i[2], f[2];
};
template <bool MLSTM>
__device__ __forceinline__ GateIn gate_in(const GateArgs& g, const Piece& c, int hd, int lane) {
  GateIn r;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const size_t t = c.t0 + min(2 * lane + e, c.n - 1);
    r.i[e] = MLSTM ? g.ipre[t * g.H + hd] : (float)g.dt[t * g.lddt + hd];
    r.f[e] = MLSTM ? g.fpre[t * g.H + hd] : 0.f;
  }
  return r;
}

template <bool MLSTM>
__device__ __forceinline__ Gate gates(const GateArgs& g, const GateIn& in, const Piece& c, int hd, int lane) {
  Gate r;
  double l[2], ig[2] = {0.0, 0.0};
  float w[2] = {0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int j = 2 * lane + e;
    const bool on = j < c.n;
    if (MLSTM) {
      const float i = g.cap * tanhf((in.i[e] + g.ib[hd]) / g.cap);
      const float f = logsigmoidf_(g.cap * tanhf((in.f[e] + g.fb[hd]) / g.cap));
      ig[e] = on ? (double)i * LOG2E : -(double)INFINITY;
      l[e] = on ? (double)f * LOG2E : 0.0;
      w[e] = on ? 1.f : 0.f;
    } else {
      const float dt = softplusf_(in.i[e] + g.dt_bias[hd]);
      l[e] = on ? (double)(-expf(g.a_log[hd]) * dt) * LOG2E : 0.0;
      w[e] = on ? dt : 0.f;
    }
  }
  // state space: a token that forgets everything (down to -inf) counts as 2^-512, which is 0 in every float it meets: the sums
  // behind it keep their bits.  (The mLSTM weighs its inputs against the log decays: those stay as they are, and above -cap - 1.)
  if (!MLSTM)
#pragma unroll
    for (int e = 0; e < 2; ++e) l[e] = l[e] < -512.0 ? -512.0 : l[e];
  const double sum = scan_lanes(l[0] + l[1], 0.0, [](double a, double b) { return a + b; });
  r.F1 = sum;
  const double before = shfl_up_d(sum, 1);
  r.F0 = l[1] == l[1] ? sum - l[1] : lane ? before + l[0] : l[0];      // (a NaN decay starts at its own token)
  r.Fc = last_lane_d(sum);
  r.a0 = ig[0] - r.F0;
  r.a1 = ig[1] - r.F1;
  r.c0 = w[0];
  r.c1 = w[1];
  return r;
}

// the running maximum of a over a chunk's tokens, up to and including this lane's two
__device__ __forceinline__ void running_max(const Gate& g, int lane, double& m0, double& m1) {
  const double top = scan_lanes(fmax(g.a0, g.a1), -(double)INFINITY, [](double a, double b) { return fmax(a, b); });
  m1 = top;
  const double before = shfl_up_d(top, 1);
  m0 = lane ? fmax(before, g.a0) : g.a0;
}

__device__ __forceinline__ int c_row(int i, int half) { return (i & 3) + 8 * (i >> 2) + 4 * half; }   // 32x32 tile: row of register i

// What the kernels leave for each other, per run of `sc` chunks of a sequence (a piece) and head, and per chunk of it.
struct Ws {
  double* sup;       // [slot, H, 3]: log decay of the run, log of the unit that E is counted in, log of the unit in front of the run
  double* loc;       // [chunk, H, 2]: log decay from the run's start to the chunk, log of the unit that U is counted in
  float* tab;        // [chunk, H, 3 or 6, CK]: the tokens' gates, a float and what it leaves: a; (input factor | F, running maximum of a)
  float *E, *NE;     // [slot, H, dv, dk], [slot, H, dk]: the run's contribution to the state, later the state in front of the run
  float *U, *NU;     // [slot, sc - 1, H, ..]: what the run's chunks in front of the second, third .. contribute
  int sc;
};

// Where the 16-byte piece x8 of row r stands in an unpadded row of COLS bf16.  Transposed reads take four rows by two blocks of 16
// columns at a time, operand reads 16 rows of one piece: both then meet every bank once.
template <int COLS>
__device__ __forceinline__ int tr_piece(int r, int x8) {
  return COLS % 128 == 0 ? x8 ^ ((r & 3) << 2) : COLS % 128 == 64 ? x8 ^ ((r & 2) << 1) : x8;
}
template <int COLS>
__device__ __forceinline__ int op_piece(int r, int x8) {
  return x8 ^ (COLS % 128 == 0 ? r & 15 : COLS % 128 == 64 ? (r >> 1) & 7 : (r >> 2) & 3);
}

// (1) A run's contribution to the state, E[slot, head, dv, dk] = sum_j w_j v_j k_j^T with w_j = e^{F_end - F_j} c_j (mLSTM: against the
// largest), for 64 value columns, and on the way what stands in front of its second, third .. chunk.  A wave works out the gates of
// one chunk, all at once; then 64 tokens at a time go through LDS as they stand in memory, and the products, which sum over tokens,
// read them transposed.  The next 64 tokens' loads are on their way under the products.
template <int NK, bool MLSTM>
__global__ __launch_bounds__(256, 3) void k_chunk_state(const bf16* __restrict__ k, int ldk, const bf16* __restrict__ v,
                                                        int ldv, GateArgs ga, Ws ws, int H, int G, int dv, Pieces pc, SeqDesc d) {
  constexpr int DK = 32 * NK, TILES = (NK + 1) / 2, TAB = MLSTM ? 6 : 3;
  __shared__ __attribute__((aligned(16))) bf16 sk[64 * DK];              // [token][dk]
  __shared__ __attribute__((aligned(16))) bf16 sv[3 * 64 * 64];          // [part][token][dv]
  __shared__ float sw[4 * CK], sscale[4];
  __shared__ double sF[4], sTop[4];
  Piece c;
  const int slot = blockIdx.x, hd = blockIdx.y, cb = blockIdx.z * 64, tid = threadIdx.x;
  if (!find_piece<0>(d, pc, slot, c)) return;
  c.t0 = __builtin_amdgcn_readfirstlane(c.t0);
  c.n = __builtin_amdgcn_readfirstlane(c.n);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, g = lane >> 4, kh = hd / (H / G);
  const int l32 = lane & 31, half = lane >> 5, chunks = (c.n + CK - 1) / CK;
  const size_t cell = (size_t)slot * H + hd;
  const bf16* kp = k + (size_t)c.t0 * ldk + kh * DK;
  const bf16* vp = v + (size_t)c.t0 * ldv + (size_t)hd * dv + cb;
  Piece own = {c.s, 0, c.t0 + min(w, chunks - 1) * CK, 0, 0};
  own.n = min(CK, c.t0 + c.n - own.t0);
  const GateIn gi = gate_in<MLSTM>(ga, own, hd, lane);
  bf16x8 rk[NK];
  bf16x4 rv[2][2];
  auto load = [&](int j0) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int e = tid + 256 * i, r = min(j0 + e / (DK / 8), c.n - 1), x8 = e % (DK / 8);
      rk[i] = *reinterpret_cast<const bf16x8*>(kp + (unsigned)(r * ldk + 8 * x8));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {             // (columns past the last give columns past the last)
        const int e = tid + 256 * i, r = min(j0 + (e >> 3), c.n - 1), col = min(8 * (e & 7) + 4 * h, dv - cb - 4);
        rv[i][h] = *reinterpret_cast<const bf16x4*>(vp + (unsigned)(r * ldv + col));
      }
  };
  load(0);
  if (w < chunks) {
    const Gate gt = gates<MLSTM>(ga, gi, own, hd, lane);
    double m0 = 0.0, m1 = 0.0;
    if (MLSTM) running_max(gt, lane, m0, m1);
    if (lane == 0) sF[w] = gt.Fc;
    if (lane == 63) sTop[w] = m1;
    __syncthreads();
    double F = 0.0, m = -(double)INFINITY;           // log decay and unit in front of the wave's chunk
    for (int i = 0; i < w; ++i) {
      F += sF[i];
      m = fmax(m + sF[i], sF[i] + sTop[i]);
    }
    const double mn = fmax(m + gt.Fc, gt.Fc + m1);   // (of lane 63)
    const double unit = MLSTM ? last_lane_d(mn) : 0.0;
    const int j = 2 * lane;
    sw[CK * w + j] = j < own.n ? exp2f((float)(gt.a0 + (gt.Fc - unit))) * gt.c0 : 0.f;
    sw[CK * w + j + 1] = j + 1 < own.n ? exp2f((float)(gt.a1 + (gt.Fc - unit))) * gt.c1 : 0.f;
    if (lane == 0) sscale[w] = MLSTM ? exp2f((float)(m + gt.Fc - unit)) : exp2f((float)gt.Fc);
    if (cb == 0) {
      const size_t cc = ((size_t)slot * ws.sc + w) * H + hd;
      if (lane == 0) {
        ws.loc[2 * cc] = F;
        ws.loc[2 * cc + 1] = m;
        if (w == chunks - 1) {
          ws.sup[3 * cell] = F + gt.Fc;
          ws.sup[3 * cell + 1] = unit;
        }
      }
      float* tab = ws.tab + cc * TAB * CK + j;
      const auto two = [&](int i, double x0, double x1) {       // a double as a float and what that leaves
        const float h0 = (float)x0, h1 = (float)x1;
        *reinterpret_cast<float2*>(tab + i * CK) = float2{h0, h1};
        *reinterpret_cast<float2*>(tab + (i + 1) * CK) =
            float2{j < own.n ? (float)(x0 - (double)h0) : 0.f, j + 1 < own.n ? (float)(x1 - (double)h1) : 0.f};
      };
      two(0, gt.a0, gt.a1);
      if (MLSTM) {
        two(2, gt.F0, gt.F1);
        two(4, m0, m1);
      } else {
        *reinterpret_cast<float2*>(tab + 2 * CK) = float2{gt.c0, gt.c1};
      }
    }
  } else {
    __syncthreads();
  }
  f32x16 acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  // the normaliser (the column whose value is always 1): two key channels per thread, a part of the tokens
  constexpr int PARTS = NK == 3 ? 4 : 16 / NK, TOK = 64 / PARTS;
  const int nc = tid % (DK / 2), part = tid / (DK / 2);
  const bool norm = MLSTM && cb == 0;
  float n0 = 0.f, n1 = 0.f;
  // (what has no place goes past the end of its window and is dropped)
  const int left = max(min(dv - cb - (w & 1) * 32, 32), 0);
  auto store = [&](float* to) {
    const auto win = __builtin_amdgcn_make_buffer_rsrc(to + (size_t)(cb + (w & 1) * 32) * DK, 0, left * DK * 4, 0x00020000);
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const int kt = (w >> 1) + 2 * t;
      const unsigned at = kt < NK ? (4 * half * DK + kt * 32 + l32) * 4 : 0x80000000u;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[t][i]), win, at + c_row(i, 0) * DK * 4, 0, 0);
    }
  };
  auto store_norm = [&](float* to) {
    float* sn = reinterpret_cast<float*>(sv);         // (the last products' reads are past a barrier)
    if (part < PARTS) *reinterpret_cast<float2*>(sn + part * DK + 2 * nc) = float2{n0, n1};
    __syncthreads();
    if (tid < DK) {
      float t = sn[tid];
#pragma unroll
      for (int q = 1; q < PARTS; ++q) t += sn[tid + q * DK];
      to[tid] = t;
    }
  };
  for (int j0 = 0; j0 < c.n; j0 += 64) {
    __syncthreads();                           // the last turn's reads are done; the weights stand
    const int ci = j0 / CK;
    if (norm && j0 % CK == 0 && ci > 0) {
      store_norm(ws.NU + (((size_t)slot * (ws.sc - 1) + ci - 1) * H + hd) * DK);
      __syncthreads();
      n0 *= sscale[ci];
      n1 *= sscale[ci];
    }
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int e = tid + 256 * i, r = e / (DK / 8), x8 = e % (DK / 8);
      *reinterpret_cast<bf16x8*>(sk + r * DK + 8 * tr_piece<DK>(r, x8)) = j0 + r < c.n ? rk[i] : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int e = tid + 256 * i, r = e >> 3, x8 = e & 7;
      const float wt = sw[j0 + r];
      const bool on = j0 + r < c.n;            // (tokens past the end repeat the last: an infinite one times 0 would be no number)
      u32x4 o[3];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const bf16x4 y = rv[i][x >> 1];
        const float y0 = wt * (float)y[2 * (x & 1)], y1 = wt * (float)y[2 * (x & 1) + 1];
        const Split z = split3(on ? y0 : 0.f, on ? y1 : 0.f);
        o[0][x] = z.h;
        o[1][x] = z.m;
        o[2][x] = z.l;
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(sv + (q * 64 + r) * 64 + 8 * tr_piece<64>(r, x8)) = o[q];
    }
    if (j0 % CK == 0 && ci > 0) {              // (in front of the loads: a wait for those then waits for nothing younger)
      store(ws.U + (((size_t)slot * (ws.sc - 1) + ci - 1) * H + hd) * dv * DK);
      const float f = sscale[ci];
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] *= f;
    }
    load(j0 + 64);                             // (past the end: its last token again)
    __syncthreads();
    // operand rows are columns here: lanes 16 g .. read the tokens of half g / 2 in columns 16 (g % 2) .., four tokens a read
    const int row = 8 * (g >> 1) + (li >> 2);
    const auto operand = [&](const bf16* base, auto cols, int r, int tile) {
      constexpr int COLS = decltype(cols)::value;
      const int x8 = 4 * tile + 2 * (g & 1) + ((li >> 1) & 1);
      const bf16x4 lo = read_tr(base + r * COLS + 8 * tr_piece<COLS>(r, x8) + 4 * (li & 1)),
                   hi = read_tr(base + (r + 4) * COLS + 8 * tr_piece<COLS>(r + 4, x8) + 4 * (li & 1));
      return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    if (cb + (w & 1) * 32 < dv) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        bf16x8 a[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) a[q] = operand(sv + q * 64 * 64, std::integral_constant<int, 64>{}, 16 * ks + row, w & 1);
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
          const int kt = (w >> 1) + 2 * t;
          if (kt < NK) {
            const bf16x8 b = operand(sk, std::integral_constant<int, DK>{}, 16 * ks + row, kt);
#pragma unroll
            for (int q = 2; q >= 0; --q) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[q], b, acc[t], 0, 0, 0);
          }
        }
      }
    }
    if (norm && part < PARTS) {
#pragma unroll
      for (int i = 0; i < TOK; ++i) {
        const int r = part * TOK + i;
        const bf16x2 kk = *reinterpret_cast<const bf16x2*>(sk + r * DK + 8 * tr_piece<DK>(r, nc >> 2) + 2 * (nc & 3));
        n0 += sw[j0 + r] * (float)kk[0];
        n1 += sw[j0 + r] * (float)kk[1];
      }
    }
  }
  store(ws.E + cell * dv * DK);
  if (norm) {
    __syncthreads();
    store_norm(ws.NE + cell * DK);
  }
}

// (2) A sequence's runs in order, four state elements per thread: the state in front of a run replaces the run's
// contribution, the state behind the last one goes to its slot.  Bound by memory: every contribution is read and written once.
template <bool MLSTM>
__global__ __launch_bounds__(256) void k_chunk_walk(Ws ws, float* __restrict__ S, float* __restrict__ N,
                                                    const float* __restrict__ M, int H, int dk, int dv, int nb, Pieces pc,
                                                    SeqDesc d) {
  const int s = blockIdx.x / H, hd = blockIdx.x % H, tid = threadIdx.x;
  if (d.live && !d.live[s]) return;
  const bool norm = MLSTM && (int)blockIdx.y == nb;        // the last block walks the normaliser
  int first;
  const int n = own_pieces<0>(d, pc, s, first);
  const int size = norm ? dk : dv * dk, e = (norm ? 0 : (int)blockIdx.y * 1024) + 4 * tid;
  const size_t hbase = (size_t)d.slots[s] * H + hd, step = (size_t)H * size;
  float* st = (norm ? N : S) + hbase * size + e;
  float* u = (norm ? ws.NE : ws.E) + ((size_t)first * H + hd) * size + e;
  double* mt = ws.sup + 3 * ((size_t)first * H + hd);
  const bool on = e < size, old = pc.first > 0 || d.pos0[s] > 0;
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  if (on && old) x = *reinterpret_cast<const f32x4*>(st);
  double m = MLSTM && old ? (double)M[hbase] * LOG2E : 0.0;
  constexpr int AHEAD = 4;                                  // contributions in flight
  f32x4 f[AHEAD];
  double fd[AHEAD], fl[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (i < n) {
      if (on) f[i] = *reinterpret_cast<const f32x4*>(u + i * step);
      fd[i] = mt[3 * (size_t)i * H];
      fl[i] = mt[3 * (size_t)i * H + 1];
    }
  for (int c0 = 0; c0 < n; c0 += AHEAD) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int c = c0 + i;
      if (c < n) {
        const f32x4 add = f[i];
        const double dec = fd[i], unit = fl[i];
        if (c + AHEAD < n) {
          if (on) f[i] = *reinterpret_cast<const f32x4*>(u + (c + AHEAD) * step);
          fd[i] = mt[3 * (size_t)(c + AHEAD) * H];
          fl[i] = mt[3 * (size_t)(c + AHEAD) * H + 1];
        }
        if (on) *reinterpret_cast<f32x4*>(u + c * step) = x;
        float a, b = 1.f;
        if (MLSTM) {
          if (norm && tid == 0) mt[3 * (size_t)c * H + 2] = m;
          const double mn = fmax(m + dec, unit);
          a = exp2f((float)(m + dec - mn));
          b = exp2f((float)(unit - mn));
          m = mn;
        } else {
          a = exp2f((float)dec);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = a * x[j] + (MLSTM ? b * add[j] : add[j]);
      }
    }
  }
  if (on && n > 0) *reinterpret_cast<f32x4*>(st) = x;
}

// (3) Outputs of a chunk and head in 64 value columns: a wave owns 32 queries.  First queries . state, the state in front of the chunk
// put together from the run's and the chunk's part and split into LDS once for the block; then its scores against the chunk's keys, 32
// keys at a time, as three bf16 parts . values.  Scores are computed transposed (a lane owns one query), which is the operand layout
// of the second product; its keys then come in the order of the score registers.
// With R the decay at the wave's first query, e^{F_i - F_j} = e^{F_i - R} e^{R - F_j} for a key in front of that query: neither factor
// is above 1, the second is one number per key, and the first scales sums (of the state's part too).  Only the 32 x 32 scores on the
// diagonal take an exponential each.
template <int NK, bool MLSTM>
__global__ __launch_bounds__(256, 3) void k_chunk_out(const bf16* __restrict__ q, int ldq, const bf16* __restrict__ k, int ldk,
                                                      const bf16* __restrict__ v, int ldv, GateArgs ga, Ws ws,
                                                      float* __restrict__ M, float* __restrict__ out, float* __restrict__ den,
                                                      float* __restrict__ efl, int H, int G, int dv, Pieces pc, SeqDesc d) {
  constexpr int DK = 32 * NK, TAB = MLSTM ? 6 : 3;
  constexpr int HW = NK % 2 ? 32 : 64, NL = HW / 16;                     // key channels of a piece of the state, its loads a thread
  constexpr int KV = CK * DK + CK * 64, ST = 3 * 64 * HW;
  __shared__ __attribute__((aligned(16))) bf16 buf[KV > ST ? KV : ST];   // queries [token][dk]; state [part][dv][HW]; keys [token][dk], values
  bf16* const sv = buf + CK * DK;                                        // [token][dv]
  __shared__ __attribute__((aligned(16))) float sah[CK], sal[CK], sbh[CK], sbl[CK], sx[CK], swk[192];
  __shared__ int sbad[64];                                 // per column the first token whose value is no number
  static_assert(DK <= CK, "sx holds a normaliser");
  Piece c;
  const int slot = blockIdx.x / ws.sc, ci = blockIdx.x % ws.sc, hd = blockIdx.y, cb = blockIdx.z * 64, tid = threadIdx.x;
  if (!find_piece<0>(d, pc, slot, c)) return;
  const int t0 = __builtin_amdgcn_readfirstlane(c.t0 + ci * CK), n = __builtin_amdgcn_readfirstlane(min(CK, c.n - ci * CK));
  if (n <= 0) return;
  // Wave 3 has four times the scores of wave 0, and a block's waves go to the SIMDs in order: neighbours on a CU take turns.
  const unsigned id = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const int w = __builtin_amdgcn_readfirstlane(((tid >> 6) + (id >> 8)) & 3), lane = tid & 63, l32 = lane & 31, half = lane >> 5, kh = hd / (H / G);
  const size_t cell = (size_t)slot * H + hd, cc = (size_t)blockIdx.x * H + hd, cu = ((size_t)slot * (ws.sc - 1) + ci - 1) * H + hd;
  const bool run = c.idx > 0 || c.pos0 > 0, old = run || ci > 0;    // is there a state in front of the run; of the chunk
  float tv[TAB];
  const float* tab = ws.tab + cc * TAB * CK + (tid & (CK - 1));
#pragma unroll
  for (int i = 0; i < TAB; ++i) tv[i] = tab[i * CK];
  const double floc = ws.loc[2 * cc], mloc = ws.loc[2 * cc + 1], msup = MLSTM ? ws.sup[3 * cell + 2] + floc : floc;
  // Rows of 16-byte pieces side by side: an operand's own load would touch 32 rows of memory.  All loads first.
  constexpr int PER = 2 * NK;
  const bf16 *qp = q + (size_t)t0 * ldq + kh * DK, *kp = k + (size_t)t0 * ldk + kh * DK, *vp = v + (size_t)t0 * ldv + (size_t)hd * dv + cb;
  bf16x8 rq[PER], rk[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i, r = min(32 * w + e / (DK / 8), n - 1), x8 = e % (DK / 8);
    rq[i] = *reinterpret_cast<const bf16x8*>(qp + (unsigned)(r * ldq + 8 * x8));
  }
  f32x4 re[NL], ru[NL];
  const float *ep = ws.E + (cell * dv + cb) * DK, *up = ws.U + (cu * dv + cb) * DK;
  auto load = [&](int h) {                                 // HW key channels of the state's two parts
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = tid + 256 * i, r = min(e / (HW / 4), dv - cb - 1), x4 = e % (HW / 4);
      const unsigned at = r * DK + h * HW + 4 * x4;
      re[i] = *reinterpret_cast<const f32x4*>(ep + at);     // (zeros in front of a fresh sequence's first run)
      if (ci > 0) ru[i] = *reinterpret_cast<const f32x4*>(up + at);
    }
  };
  if (old) load(0);
  bf16x4 rv[4][2];
  const int v8 = tid & 7, vr = tid >> 3;                   // a thread's columns and first token of 32 at a time
  auto load_kv = [&] {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 256 * i, r = min(e / (DK / 8), n - 1), x8 = e % (DK / 8);
      rk[i] = *reinterpret_cast<const bf16x8*>(kp + (unsigned)(r * ldk + 8 * x8));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int x = 0; x < 2; ++x)
        rv[i][x] = *reinterpret_cast<const bf16x4*>(vp + (unsigned)(min(32 * i + vr, n - 1) * ldv + min(8 * v8 + 4 * x, dv - cb - 4)));
  };
  // the state in front of the chunk is fu U + fe E
  const double mp = fmax(mloc, msup);
  const float fe = !MLSTM ? exp2f((float)msup) : msup == mp ? 1.f : exp2f((float)(msup - mp));
  const float fu = !MLSTM || mloc == mp ? 1.f : exp2f((float)(mloc - mp));
  if (tid < CK) {
    sah[tid] = tv[0];
    sal[tid] = tv[1];
    if (MLSTM) {
      const double F = (double)tv[TAB - 4] + (double)tv[TAB - 3], m = fmax((double)tv[TAB - 2] + (double)tv[TAB - 1], mp);
      const float h = (float)-m;
      sbh[tid] = h;
      sbl[tid] = (float)(-m - (double)h);
      if (cb == 0 && tid < n) {
        efl[(size_t)(t0 + tid) * H + hd] = exp2f((float)(-(F + m)));
        // behind the last chunk, here or at all
        if (tid == n - 1 && (t0 + n == d.seq_off[c.s + 1] || (pc.count > 0 && c.idx == pc.first + pc.count - 1 && t0 + n == c.t0 + c.n)))
          M[(size_t)d.slots[c.s] * H + hd] = (float)((F + m) * 0.69314718055994530942);
      }
    } else {
      sbh[tid] = -tv[0];
      sbl[tid] = -tv[1];
      sx[tid] = tv[2];
    }
  } else if (MLSTM && tid - CK < DK) {
    const int r = tid - CK;
    sx[r] = (run ? fe * ws.NE[cell * DK + r] : 0.f) + (ci > 0 ? fu * ws.NU[cu * DK + r] : 0.f);
  }
  if (tid < 64) sbad[tid] = CK;
  const bool work = 32 * w < n;
  const int qi = 32 * w + l32;                              // this lane's query
  bf16x8 qf[2 * NK];
#pragma unroll
  for (int i = 0; i < PER; ++i) {                           // (each wave its own 32 rows)
    const int e = lane + 64 * i, r = e / (DK / 8), x8 = e % (DK / 8);
    *reinterpret_cast<bf16x8*>(buf + (32 * w + r) * DK + 8 * op_piece<DK>(r, x8)) = rq[i];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int s = 0; s < 2 * NK; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(buf + qi * DK + 8 * op_piece<DK>(l32, 2 * s + half));
  __syncthreads();
  const float rh = sbh[32 * w], rl = sbl[32 * w];
  f32x16 acc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  const bool two = cb + 32 < dv;
  const float est = MLSTM ? exp2f((float)(mp + (double)rh + (double)rl)) : exp2f(rh + rl);   // factor of the state at the wave's first query
  if (old) {
#pragma unroll
    for (int h = 0; h < DK / HW; ++h) {
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int e = tid + 256 * i, r = e / (HW / 4), x4 = e % (HW / 4);
        f32x4 x;
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = ci > 0 ? fe * re[i][t] + fu * ru[i][t] : fe * re[i][t];
        const Split a = split3(x[0], x[1]), b = split3(x[2], x[3]);
        bf16* row = buf + r * HW + 8 * op_piece<HW>(r, x4 >> 1) + 4 * (x4 & 1);
        *reinterpret_cast<u32x2*>(row) = u32x2{a.h, b.h};
        *reinterpret_cast<u32x2*>(row + 64 * HW) = u32x2{a.m, b.m};
        *reinterpret_cast<u32x2*>(row + 2 * 64 * HW) = u32x2{a.l, b.l};
      }
      if (h + 1 < DK / HW)
        load(h + 1);
      else
        load_kv();
      __syncthreads();
      if (work)
#pragma unroll
        for (int s = 0; s < HW / 16; ++s)
#pragma unroll
          for (int p = 2; p >= 0; --p) {
            const bf16* bp = buf + (p * 64 + l32) * HW + 8 * op_piece<HW>(l32, 2 * s + half);
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[h * (HW / 16) + s], *reinterpret_cast<const bf16x8*>(bp), acc[0], 0, 0, 0);
            if (two)
              acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[h * (HW / 16) + s], *reinterpret_cast<const bf16x8*>(bp + 32 * HW), acc[1], 0, 0, 0);
          }
      __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][i] *= est;
  } else {
    load_kv();
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = tid + 256 * i, r = e / (DK / 8), x8 = e % (DK / 8);
    *reinterpret_cast<bf16x8*>(buf + r * DK + 8 * op_piece<DK>(r, x8)) = rk[i];
  }
  // A masked score is a 0 that multiplies a later token's value: an infinite or NaN value would reach the queries in front of
  // it.  It counts as 0 in the products, and its column is NaN from its token on.
  unsigned m2 = 0u;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const u32x2 u = __builtin_bit_cast(u32x2, rv[i][x]);
      m2 |= ((u[0] & 0x7f807f80u) + 0x00800080u) | ((u[1] & 0x7f807f80u) + 0x00800080u);      // bit 15 of a half: its exponent is all ones
    }
  if (m2 & 0x80008000u)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int x = 0; x < 8; ++x)
        if (!isfinite((float)rv[i][x >> 2][x & 3])) {
          rv[i][x >> 2][x & 3] = (bf16)0.f;
          atomicMin(sbad + 8 * v8 + x, 32 * i + vr);
        }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 32 * i + vr;
    *reinterpret_cast<bf16x8*>(sv + r * 64 + 8 * tr_piece<64>(r, v8)) =
        bf16x8{rv[i][0][0], rv[i][0][1], rv[i][0][2], rv[i][0][3], rv[i][1][0], rv[i][1][1], rv[i][1][2], rv[i][1][3]};
  }
  __syncthreads();
  if (!work) return;
  const float bh = sbh[qi], bl = sbl[qi];
  float* const wk = swk + 16 * w * (w - 1);                  // 0, 32, 64, 96 numbers
  float rsum = 0.f, roff = 0.f;
  for (int j = lane; j < 32 * w; j += 64) {
    const float e = __builtin_amdgcn_exp2f((rh + sah[j]) + (rl + sal[j]));
    wk[j] = MLSTM ? e : e * sx[j];
  }
  const float eq = __builtin_amdgcn_exp2f((bh - rh) + (bl - rl));         // of this lane's query against the first
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (half == 0) sbh[qi] = eq;                              // (no other wave reads its queries' decays)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  unsigned pw[2][3][4];
  const auto scores = [&](int kt) {
    f32x16 p;
#pragma unroll
    for (int i = 0; i < 16; ++i) p[i] = 0.f;
#pragma unroll
    for (int s = 0; s < 2 * NK; ++s)
      p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          *reinterpret_cast<const bf16x8*>(buf + (32 * kt + l32) * DK + 8 * op_piece<DK>(l32, 2 * s + half)), qf[s], p, 0, 0, 0);
    return p;
  };
  const auto keep = [&](int g4, const f32x4& y) {           // the scores of registers 4 g4 ..
    const Split a = split3(y[0], y[1]), b = split3(y[2], y[3]);
    const int i = 2 * (g4 & 1);
    pw[g4 >> 1][0][i] = a.h;
    pw[g4 >> 1][1][i] = a.m;
    pw[g4 >> 1][2][i] = a.l;
    pw[g4 >> 1][0][i + 1] = b.h;
    pw[g4 >> 1][1][i + 1] = b.m;
    pw[g4 >> 1][2][i + 1] = b.l;
  };
  const int li = lane & 15, g2 = (lane >> 4) & 1;
  const auto values = [&](int kt) {                         // the operand's tokens are in the order of the score registers
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (t == 0 || two) {
          const int r = 32 * kt + 16 * ks + 4 * half + (li >> 2), x8 = 4 * t + 2 * g2 + ((li >> 1) & 1);
          const bf16x4 b0 = read_tr(sv + r * 64 + 8 * tr_piece<64>(r, x8) + 4 * (li & 1)),
                       b1 = read_tr(sv + (r + 8) * 64 + 8 * tr_piece<64>(r + 8, x8) + 4 * (li & 1));
          const bf16x8 b = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
#pragma unroll
          for (int part = 2; part >= 0; --part)
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8, u32x4{pw[ks][part][0], pw[ks][part][1], pw[ks][part][2], pw[ks][part][3]}), b, acc[t], 0, 0, 0);
        }
  };
  for (int kt = 0; kt < w; ++kt) {
    const f32x16 p = scores(kt);
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      f32x4 y = *reinterpret_cast<const f32x4*>(wk + 32 * kt + 8 * g4 + 4 * half);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        y[x] *= p[4 * g4 + x];
        if (MLSTM) roff += y[x];
      }
      keep(g4, y);
    }
    values(kt);
  }
  {
    const f32x16 p = scores(w);
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int j0 = 8 * g4 + 4 * half;
      const f32x4 ah = *reinterpret_cast<const f32x4*>(sah + 32 * w + j0), al = *reinterpret_cast<const f32x4*>(sal + 32 * w + j0),
                  cw = *reinterpret_cast<const f32x4*>(sx + 32 * w + j0), e = *reinterpret_cast<const f32x4*>(sbh + 32 * w + j0);
      f32x4 y;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        y[x] = p[4 * g4 + x] * __builtin_amdgcn_exp2f((bh + ah[x]) + (bl + al[x]));
        if (!MLSTM) y[x] *= cw[x];
        y[x] = j0 + x <= l32 ? y[x] : 0.f;
        if (MLSTM) rsum += y[x];
        acc[0][4 * g4 + x] *= e[x];                         // rows 8 g4 + 4 half + x, against their wave's first
        acc[1][4 * g4 + x] *= e[x];
      }
      keep(g4, y);
    }
    values(w);
  }
  if (MLSTM && cb == 0) {
    float dot = 0.f;
#pragma unroll
    for (int s = 0; s < 2 * NK; ++s)
#pragma unroll
      for (int x = 0; x < 8; ++x) dot += (float)qf[s][x] * sx[16 * s + 8 * half + x];
    float t = rsum + eq * (roff + est * dot);
    t += __shfl_xor(t, 32, 64);
    if (half == 0 && qi < n) den[(size_t)(t0 + qi) * H + hd] = t * ga.qscale;
  }
  const float skip = MLSTM ? 0.f : ga.dskip[hd];
  // (a store that has no place goes past the end of its window and is dropped.  The outputs leave nothing in the caches, which hold the states that
  // other blocks are about to read: state space, 4093 tokens 93.4 -> 91.8 us, 8 prompts of 333 to 1024 169.7 -> 159; mLSTM, the same 82.1 -> 80.1.
  // (Calls on the same inputs, which then stay in the last cache; on inputs from memory 4093 tokens take 109 to 117 and the mLSTM 98, as before.)  The
  // states, just written, as loads that leave nothing: 99.5 and 165.)
  const auto win = __builtin_amdgcn_make_buffer_rsrc(out + ((size_t)t0 * H + hd) * dv, 0, ((n - 1) * H + 1) * dv * 4, 0x00020000);
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int col = 32 * t + l32, first = sbad[col];
    if (__any(first < CK))
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][i] = 32 * w + c_row(i, half) >= first ? NAN : acc[t][i];
    const unsigned at = cb + col < dv ? ((unsigned)((32 * w + 4 * half) * H) * dv + cb + col) * 4 : 0x80000000u;
    const bf16* own = sv + (32 * w + 4 * half) * 64 + (col & 7);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float y = acc[t][i];
      if (MLSTM)
        y *= ga.qscale;
      else
        y += skip * (float)own[c_row(i, 0) * 64 + 8 * tr_piece<64>(c_row(i, 0), col >> 3)];
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), win, at + (unsigned)(c_row(i, 0) * H) * dv * 4, 0, 2);
    }
  }
}

// Chunks of a run.  Longer runs pass less of the state through memory, but are fewer and take their chunks one after another, so there
// have to be enough of them.  us at 1 / 2 / 4 chunks (state space, 64 heads of 128 x 64; mLSTM, 8 heads of 128 x 192): one prompt of 4093
// tokens 110 / 101 / 95, twelve of 700 243 / 234 / 243, one of 1000 42 / 42 / 47; one of 9000 134 / 112 / 103, eight of 333 to 1024 89 / 82 /
// 87, one of 3000 54 / 52 / 55, one of 700 31 / 34 / 44.
int run_chunks(int T_, int B, int H, int dv) {
  const long blocks = (long)((T_ + CK - 1) / CK) * H * ((dv + 63) / 64), mean = T_ / B;
  return blocks >= 1536 && mean >= 8 * CK ? 4 : blocks >= 512 && mean >= 3 * CK ? 2 : 1;
}
// floats of a run's slot; 0.4 us a token in the token-by-token form
size_t run_floats(int sc, int H, int dk, int dv) { return (size_t)H * (6 + sc * (4 + 6 * CK + (size_t)dk * (dv + 1))); }
PiecePlan run_plan(int T_, int B, int H, int dk, int dv, int sc, size_t most) {
  return plan_pieces(T_, B, CK * sc, run_floats(sc, H, dk, dv), most < 4 ? 0 : most - 4, 0.4f);      // (4 for the tables' alignment)
}

template <int NK, bool MLSTM>
void chunk_launch(const bf16* q, int ldq, const bf16* k, int ldk, const bf16* v, int ldv, const GateArgs& ga, float* S, float* N,
                  float* M, float* out, float* den, float* efl, float* ws, size_t most, int H, int G, int dv, SeqDesc d,
                  hipStream_t st) {
  const int sc = run_chunks(d.Ttot, d.B, H, dv), dk = 32 * NK;
  const PiecePlan plan = run_plan(d.Ttot, d.B, H, dk, dv, sc, most);
  const size_t cells = plan.slots * H, state = (size_t)dv * dk;
  Ws w_;
  w_.sc = sc;
  w_.sup = reinterpret_cast<double*>(ws);
  w_.loc = w_.sup + 3 * cells;
  w_.tab = reinterpret_cast<float*>(w_.loc + 2 * cells * sc);
  w_.tab += (4 - ((w_.tab - ws) & 3)) & 3;
  w_.E = w_.tab + cells * sc * (MLSTM ? 6 : 3) * CK;
  w_.U = w_.E + cells * state;
  w_.NE = w_.U + cells * (sc - 1) * state;
  w_.NU = w_.NE + cells * dk;
  const int nb = (int)((state + 1023) / 1024), cols = (dv + 63) / 64;
  for (int w = 0; w < plan.windows; ++w) {
    const Pieces pc = {CK * sc, w * plan.count, plan.count};
    hipLaunchKernelGGL((k_chunk_state<NK, MLSTM>), dim3((unsigned)plan.slots, H, cols), dim3(256), 0, st, k, ldk, v, ldv, ga, w_, H, G,
                       dv, pc, d);
    hipLaunchKernelGGL((k_chunk_walk<MLSTM>), dim3(d.B * H, nb + (MLSTM ? 1 : 0)), dim3(256), 0, st, w_, S, N, M, H, dk, dv, nb, pc,
                       d);
    hipLaunchKernelGGL((k_chunk_out<NK, MLSTM>), dim3((unsigned)(plan.slots * sc), H, cols), dim3(256), 0, st, q, ldq, k, ldk, v, ldv,
                       ga, w_, M, out, den, efl, H, G, dv, pc, d);
  }
  LIPA_CHECK_LAUNCH();
}

template <bool MLSTM>
void chunk_dispatch(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const GateArgs& ga, float* S, float* N,
                    float* M, float* out, float* den, float* efl, float* ws, size_t most, int H, int G, int dk, int dv,
                    int longest, SeqDesc d, hipStream_t st) {
  if (seq_walk_floats(MLSTM, d.Ttot, d.B, H, dk, dv, longest, most) > 0)
    return seq_walk(MLSTM, q, ldq, k, ldk, v, ldv, ga, S, N, M, out, den, efl, ws, most, H, G, dk, dv, longest, d, st);
#define CHUNK(NK_)                                                                                                          \
  chunk_launch<NK_, MLSTM>((const bf16*)q, ldq, (const bf16*)k, ldk, (const bf16*)v, ldv, ga, S, N, M, out, den, efl, ws, \
                           most, H, G, dv, d, st)
  switch (dk / 32) {
    case 1: CHUNK(1); break;
    case 2: CHUNK(2); break;
    case 3: CHUNK(3); break;
    default: CHUNK(4); break;
  }
#undef CHUNK
}

}  // namespace

int seq_run_chunks(int T_, int B, int H, int dv) { return run_chunks(T_, B, H, dv); }

// Tokens a sequence from which on prompts run in chunks.
// Three launches and a chunk of padding against 0.4 us a token (two heads a CU) in the token-by-token form: 64 tokens a
// sequence are 21 / 32 / 96 us here and 30 / 36 / 148 us there (state space, 32 heads, 1 / 8 / 48 sequences), 48 are 21 / 32 / 94
// and 24 / 29 / 118 us; mLSTM (8 heads of 128 x 192) at 64: 26 / 34 / 68 against 31 / 36 / 159 us.  The outputs walk the columns 32 at a
// time, one after another: 512 of them 43 against 26 us at 64 tokens, even at 128 to 160.  Where (sequence, head) pairs fill the chip,
// the padding counts, and with small keys the token form is the cheaper one for longer: 1024 pairs of 64 x 64 take 1.3 times its time at
// 64 to 128 tokens, 0.94 at 192; 1024 of 32 x 128 1.2 at 192, 1.08 at 256, 0.92 at 512; 1024 of 128 x 64 are ahead from 64 on.
long seq_chunk_least(int B, int H, int dk, int dv) {
  const long pairs = (long)B * H;
  long least = std::max(64, std::min(dv * 5 / 12, 192));
  if (pairs >= 256 && dk <= 64 && dv >= 128) least = std::max(least, 96l);
  if (pairs >= 1024 && (dk <= 64 || dv <= 32)) least = 192;
  if (pairs * dv >= 1l << 17 && dk <= 32) least = 256;
  return least;
}

// Floats of workspace of the chunked form, or 0 where the token-by-token scan is the one to run: float activations, key sizes
// that are no multiple of 32 or above 128, rows that 16-byte (q, k, the states S and N) or 8-byte (v) loads cannot take, and steps of
// few tokens a sequence.  At most `most`: longer steps run in windows.
size_t seq_chunk_floats(int code, bool mlstm, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const void* S,
                        const void* N, int T_, int B, int H, int dk, int dv, int longest, size_t most) {
  const auto fits = [](const void* p, int ld, int n) { return ld % n == 0 && ((uintptr_t)p & (2 * n - 1)) == 0; };
  if (code != 0 || dk % 32 != 0 || dk > 128 || dv % 4 != 0 || (long)H * dv >= 1l << 22 || std::max({ldq, ldk, ldv}) >= 1 << 22 ||
      !fits(q, ldq, 8) || !fits(k, ldk, 8) || !fits(v, ldv, 4) ||
      !fits(S, 8, 8) || !fits(N, 8, 8))
    return 0;
  if (B == 0) return 0;
  if (T_ < seq_chunk_least(B, H, dk, dv) * B)
    return mlstm && seq_walk_short(T_, B, H, dk, dv, longest) ? seq_walk_floats(true, T_, B, H, dk, dv, longest, most) : 0;
  if (const size_t n = seq_walk_floats(mlstm, T_, B, H, dk, dv, longest, most)) return n;      // (the state never leaves its block)
  const int sc = run_chunks(T_, B, H, dv);
  const size_t slots = run_plan(T_, B, H, dk, dv, sc, most).slots;
  return slots == 0 ? 0 : slots * run_floats(sc, H, dk, dv) + 4;
}

void seq_chunk_ssd(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const void* dt, int lddt,
                   const float* dt_bias, const float* a_log, const float* dskip, float* S, float* out, float* ws, size_t most,
                   int H, int G, int dk, int dv, int longest, SeqDesc d, hipStream_t st) {
  const GateArgs ga = {(const bf16*)dt, lddt, dt_bias, a_log, dskip, nullptr, nullptr, nullptr, nullptr, 1.f, 1.f, H};
  chunk_dispatch<false>(q, ldq, k, ldk, v, ldv, ga, S, nullptr, nullptr, out, nullptr, nullptr, ws, most, H, G, dk, dv, longest, d, st);
}

void seq_chunk_mlstm(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const float* ipre, const float* fpre,
                     const float* ib, const float* fb, float cap, float qscale, float* S, float* N, float* M, float* out,
                     float* den, float* efl, float* ws, size_t most, int H, int dk, int dv, int longest, SeqDesc d, hipStream_t st) {
  const GateArgs ga = {nullptr, 0, nullptr, nullptr, nullptr, ipre, fpre, ib, fb, cap, qscale, H};
  chunk_dispatch<true>(q, ldq, k, ldk, v, ldv, ga, S, N, M, out, den, efl, ws, most, H, H, dk, dv, longest, d, st);
}
