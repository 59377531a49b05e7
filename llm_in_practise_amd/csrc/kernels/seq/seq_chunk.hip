// Prompts through the recurrences whose decay is one scalar per (token, head) - the state-space-duality form and the
// mLSTM - chunk by chunk instead of token by token.  With F_t the log decay summed from the chunk's first token,
//   o_t = e^{F_t} S_prev^T q_t + sum_{j <= t} e^{F_t - F_j} c_j (q_t . k_j) v_j,
//   S_end = e^{F_C} S_prev + sum_j e^{F_C - F_j} c_j k_j v_j^T,
// which is matrix products over a chunk of CK tokens.  Three kernels: (1) every chunk's own contribution to the state, all
// chunks at once; (2) the states in front of the chunks, an element-wise walk over a sequence's chunks that leaves them where
// the contributions stood; (3) the outputs, all chunks at once.
//
// What is float in the token-by-token scans stays float here.  q, k and v are bf16, so q.k runs on the bf16 matrix units
// exactly (float sums).  A float factor of a product (decayed scores, weighted values, the state) is the sum of three bf16
// numbers, which hold its 24 bits: three products with float sums, at five times the rate of the float matrix units.  Log
// decays are summed in 64 bits and kept as two floats, so that the difference of two large sums is exact.
//
// Measured, token by token -> chunks: state space, one prompt of 4093 tokens, 64 heads of 128 x 64: 2350 -> 151 us (state 46,
// walk 25, outputs 80); mLSTM, 8 prompts of 333 to 1024 tokens, 8 heads of 128 x 192: 649 -> 94 us (36, 17, 41; under the profiler 39, 18,
// 41).  Error against 64 bits 1.6e-7 -> 0.8e-7 and 4.4e-7 -> 1.9e-7: fewer roundings stand between a token and the outputs far behind it.
// Chunks of 128 tokens: the states of a step pass through memory once per chunk (69 MB of the first case, three times), and a
// chunk's scores grow with its square.
#include "seq_common.h"

#include <algorithm>

using namespace lipa;

namespace {

constexpr int CK = 128;                 // tokens of a chunk (4 waves x 32 queries)
constexpr int KP = 64 + 8;              // row of 64 staged tokens, padded: 16-byte reads of 16 rows hit all banks
constexpr int VP = CK + 4;              // row of a chunk's tokens, padded: 8-byte reads of 32 rows hit all banks
constexpr double LOG2E = 1.4426950408889634074;

// x = hi + mid + lo in bf16 to float accuracy (an infinity stays one)
__device__ __forceinline__ void split3(float x, bf16& h, bf16& m, bf16& l) {
  h = (bf16)x;
  const float r = fabsf(x) < 3.38e38f ? x - (float)h : 0.f;
  m = (bf16)r;
  l = (bf16)(r - (float)m);
}

__device__ __forceinline__ double shfl_up_d(double v, int o) {
  const long long b = __double_as_longlong(v);
  const int lo = __shfl_up((int)b, o, 64), hi = __shfl_up((int)(b >> 32), o, 64);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double last_lane_d(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __shfl((int)b, 63, 64), hi = __shfl((int)(b >> 32), 63, 64);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

struct GateArgs {
  // state space: dt (bf16, row stride lddt), per head bias and log rate
  const bf16* dt;
  int lddt;
  const float *dt_bias, *a_log, *dskip;
  // mLSTM: gate pre-activations [T, H], per head biases, cap
  const float *ipre, *fpre, *ib, *fb;
  float cap, qscale;
  int H;
};

struct Gate {                           // of a wave's lane: tokens 2 * lane and 2 * lane + 1, in powers of two
  double F0, F1, Fc;                    // log decays from the chunk's start, and of the whole chunk
  double a0, a1;                        // log of the input weight against the chunk's start: i - F (state space: -F)
  float c0, c1;                         // factor of the input that is not in the logarithm (state space: dt)
};

template <bool MLSTM>
__device__ __forceinline__ Gate gates(const GateArgs& g, const Piece& c, int hd, int lane) {
  Gate r;
  double l[2], ig[2] = {0.0, 0.0};
  float w[2] = {0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int j = 2 * lane + e;
    const bool on = j < c.n;
    const size_t t = c.t0 + (on ? j : 0);
    if (MLSTM) {
      const float i = g.cap * tanhf((g.ipre[t * g.H + hd] + g.ib[hd]) / g.cap);
      const float f = logsigmoidf_(g.cap * tanhf((g.fpre[t * g.H + hd] + g.fb[hd]) / g.cap));
      ig[e] = on ? (double)i * LOG2E : -(double)INFINITY;
      l[e] = on ? (double)f * LOG2E : 0.0;
      w[e] = on ? 1.f : 0.f;
    } else {
      const float dt = softplusf_((float)g.dt[t * g.lddt + hd] + g.dt_bias[hd]);
      l[e] = on ? (double)(-expf(g.a_log[hd]) * dt) * LOG2E : 0.0;
      w[e] = on ? dt : 0.f;
    }
  }
  // state space: a token that forgets everything (down to -inf) counts as 2^-512, which is 0 in every float it meets: the sums
  // behind it keep their bits.  (The mLSTM weighs its inputs against the log decays: those stay as they are, and above -cap - 1.)
  if (!MLSTM)
#pragma unroll
    for (int e = 0; e < 2; ++e) l[e] = l[e] < -512.0 ? -512.0 : l[e];
  double sum = l[0] + l[1];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double t = shfl_up_d(sum, o);
    if (lane >= o) sum += t;
  }
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
  double top = fmax(g.a0, g.a1);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double t = shfl_up_d(top, o);
    if (lane >= o) top = fmax(top, t);
  }
  m1 = top;
  const double before = shfl_up_d(top, 1);
  m0 = lane ? fmax(before, g.a0) : g.a0;
}

// Four tokens x four columns of a row-major bf16 matrix, transposed: out[e] holds column e's four tokens (0 past the end).
__device__ __forceinline__ void load_4x4(const bf16* __restrict__ p, size_t ld, int tokens, bool on, bf16x4 (&out)[4]) {
  bf16x4 r[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    r[t] = bf16x4{(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
    if (on && t < tokens) r[t] = *reinterpret_cast<const bf16x4*>(p + t * ld);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = bf16x4{r[0][e], r[1][e], r[2][e], r[3][e]};
}

__device__ __forceinline__ int c_row(int i, int half) { return (i & 3) + 8 * (i >> 2) + 4 * half; }   // 32x32 tile: row of register i

// (1) U[slot, head, dv, dk] = sum_j w_j v_j k_j^T over a chunk, w_j = e^{F_C - F_j} c_j (mLSTM: against the chunk's largest),
// for 64 value columns.  Bound by latency: a wave of a SIMD's three waits in turn for the gates, k and v, and the LDS, so the loads
// stand before the gates and the second half's before the first half's products (56 -> 45 us for 4093 tokens of 64 heads, with
// the registers held to three workgroups a CU; 40 -> 38 for the mLSTM's).
template <int NK, bool MLSTM>
__global__ __launch_bounds__(256, 3) void k_chunk_state(const bf16* __restrict__ k, int ldk, const bf16* __restrict__ v,
                                                     int ldv, GateArgs ga, float* __restrict__ U, float* __restrict__ NU,
                                                     double* __restrict__ meta, int H, int G, int dv, Pieces pc, SeqDesc d) {
  constexpr int DK = 32 * NK;
  __shared__ __attribute__((aligned(16))) bf16 sk[DK * KP];              // [dk][token]
  __shared__ __attribute__((aligned(16))) bf16 sv[3 * 64 * KP];          // [part][dv][token]
  __shared__ float sw[CK];
  __shared__ float sn[256];
  Piece c;
  const int slot = blockIdx.x, hd = blockIdx.y, cb = blockIdx.z * 64, tid = threadIdx.x;
  if (!find_piece<CK>(d, pc, slot, c)) return;
  const int w = tid >> 6, lane = tid & 63, l32 = lane & 31, half = lane >> 5, kh = hd / (H / G);
  const size_t cell = (size_t)slot * H + hd;
  const bf16* kp = k + (size_t)c.t0 * ldk + kh * DK;
  const bf16* vp = v + (size_t)c.t0 * ldv + (size_t)hd * dv + cb;
  constexpr int KL = (DK / 4 * 16 + 255) / 256;
  bf16x4 rk[KL][4], rv[4];
  const int c4 = tid & 15, vt = tid >> 4;
  auto load = [&](int j0) {                    // (the second half over the products of the first)
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const int e = tid + 256 * i, d4 = e % (DK / 4), t4 = j0 + 4 * (e / (DK / 4));
      load_4x4(kp + (size_t)t4 * ldk + 4 * d4, ldk, c.n - t4, e < DK / 4 * 16, rk[i]);
    }
    load_4x4(vp + (size_t)(j0 + 4 * vt) * ldv + 4 * c4, ldv, c.n - j0 - 4 * vt, cb + 4 * c4 < dv, rv);
  };
  load(0);
  if (w == 0) {
    const Gate g = gates<MLSTM>(ga, c, hd, lane);
    double top = 0.0, add = g.Fc;
    if (MLSTM) {
      double m0, m1;
      running_max(g, lane, m0, m1);
      top = last_lane_d(m1);
      add = -top;
    }
    sw[2 * lane] = 2 * lane < c.n ? exp2f((float)(g.a0 + add)) * g.c0 : 0.f;
    sw[2 * lane + 1] = 2 * lane + 1 < c.n ? exp2f((float)(g.a1 + add)) * g.c1 : 0.f;
    if (lane == 0 && cb == 0) {
      meta[3 * cell] = g.Fc;
      meta[3 * cell + 1] = g.Fc + top;         // log of the unit that U is counted in
    }
  }
  f32x16 acc[(NK + 1) / 2];
#pragma unroll
  for (int t = 0; t < (NK + 1) / 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  float nsum = 0.f;
  for (int j0 = 0; j0 < c.n; j0 += 64) {
    __syncthreads();                           // the last turn's reads are done; the weights stand
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const int e = tid + 256 * i, d4 = e % (DK / 4), t4 = e / (DK / 4);
      if (e < DK / 4 * 16)
#pragma unroll
        for (int x = 0; x < 4; ++x) *reinterpret_cast<bf16x4*>(sk + (4 * d4 + x) * KP + 4 * t4) = rk[i][x];
    }
    const f32x4 wt = *reinterpret_cast<const f32x4*>(sw + j0 + 4 * vt);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      bf16x4 h, m, l;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        bf16 a, b, e;
        split3(wt[t] * (float)rv[x][t], a, b, e);
        h[t] = a;
        m[t] = b;
        l[t] = e;
      }
      bf16* row = sv + (4 * c4 + x) * KP + 4 * vt;
      *reinterpret_cast<bf16x4*>(row) = h;
      *reinterpret_cast<bf16x4*>(row + 64 * KP) = m;
      *reinterpret_cast<bf16x4*>(row + 2 * 64 * KP) = l;
    }
    if (j0 + 64 < c.n) load(j0 + 64);
    __syncthreads();
    const int vrow = (w & 1) * 32 + l32;
    if (cb + (w & 1) * 32 < dv) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16* ap = sv + vrow * KP + 16 * ks + 8 * half;
        const bf16x8 ah = *reinterpret_cast<const bf16x8*>(ap), am = *reinterpret_cast<const bf16x8*>(ap + 64 * KP),
                     al = *reinterpret_cast<const bf16x8*>(ap + 2 * 64 * KP);
#pragma unroll
        for (int t = 0; t < (NK + 1) / 2; ++t) {
          const int kt = (w >> 1) + 2 * t;
          if (kt < NK) {
            const bf16x8 b = *reinterpret_cast<const bf16x8*>(sk + (kt * 32 + l32) * KP + 16 * ks + 8 * half);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, b, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, b, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, b, acc[t], 0, 0, 0);
          }
        }
      }
    }
    if (MLSTM && cb == 0) {                    // the normaliser: the column whose value is always 1
      constexpr int PARTS = 256 / DK;
      const int r = tid % DK, part = tid / DK;
      if (part < PARTS)
        for (int j = part * 8; j < 64; j += 8 * PARTS) {
          const bf16x8 kk = *reinterpret_cast<const bf16x8*>(sk + r * KP + j);
#pragma unroll
          for (int x = 0; x < 8; ++x) nsum += sw[j0 + j + x] * (float)kk[x];
        }
    }
  }
  if (cb + (w & 1) * 32 < dv) {
#pragma unroll
    for (int t = 0; t < (NK + 1) / 2; ++t) {
      const int kt = (w >> 1) + 2 * t;
      if (kt < NK)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int col = cb + (w & 1) * 32 + c_row(i, half);
          if (col < dv) U[(cell * dv + col) * DK + kt * 32 + l32] = acc[t][i];
        }
    }
  }
  if (MLSTM && cb == 0) {
    constexpr int PARTS = 256 / DK;
    sn[tid] = nsum;
    __syncthreads();
    if (tid < DK) {
      float t = sn[tid];
#pragma unroll
      for (int p = 1; p < PARTS; ++p) t += sn[tid + p * DK];
      NU[cell * DK + tid] = t;
    }
  }
}

// (2) A sequence's chunks in order, four state elements per thread: the state in front of a chunk replaces the chunk's
// contribution, the state behind the last one goes to its slot.  Bound by memory: every contribution is read and written once.
template <bool MLSTM>
__global__ __launch_bounds__(256) void k_chunk_walk(float* __restrict__ U, float* __restrict__ NU, double* __restrict__ meta,
                                                    float* __restrict__ S, float* __restrict__ N,
                                                    const float* __restrict__ M, int H, int dk, int dv, int nb, Pieces pc,
                                                    SeqDesc d) {
  const int s = blockIdx.x / H, hd = blockIdx.x % H, tid = threadIdx.x;
  if (d.live && !d.live[s]) return;
  const bool norm = MLSTM && (int)blockIdx.y == nb;        // the last block walks the normaliser
  int first;
  const int n = own_pieces<CK>(d, pc, s, first);
  const int size = norm ? dk : dv * dk, e = (norm ? 0 : (int)blockIdx.y * 1024) + 4 * tid;
  const size_t hbase = (size_t)d.slots[s] * H + hd, step = (size_t)H * size;
  float* st = (norm ? N : S) + hbase * size + e;
  float* u = (norm ? NU : U) + ((size_t)first * H + hd) * size + e;
  double* mt = meta + 3 * ((size_t)first * H + hd);
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

// (3) Outputs of a chunk and head: a wave owns 32 queries, keeps their decayed scores against the chunk's keys as three bf16
// parts in registers, and walks the value columns 32 at a time: scores . values, and queries . state with the state split into
// LDS once for the block.  Scores are computed transposed (a lane owns one query), which is the operand layout of the second
// product; its keys then come in the order of the score registers.
template <int NK, bool MLSTM>
__global__ __launch_bounds__(256, 2) void k_chunk_out(const bf16* __restrict__ q, int ldq, const bf16* __restrict__ k, int ldk,
                                                      const bf16* __restrict__ v, int ldv, GateArgs ga,
                                                      const float* __restrict__ U, const float* __restrict__ NU,
                                                      const double* __restrict__ meta, float* __restrict__ M,
                                                      float* __restrict__ out, float* __restrict__ den,
                                                      float* __restrict__ efl, int H, int G, int dv, Pieces pc, SeqDesc d) {
  constexpr int DK = 32 * NK, SP = DK + 8;
  __shared__ __attribute__((aligned(16))) bf16 ss[3 * 32 * SP];          // state: [part][dv][dk]
  __shared__ __attribute__((aligned(16))) bf16 sv[32 * VP];              // values: [dv][token]
  __shared__ __attribute__((aligned(16))) float sah[CK], sal[CK], sc[CK], sbh[CK], sbl[CK], sx[CK];
  __shared__ float sN[DK];
  __shared__ int sbad[2][32];                              // per column the first token whose value is no number
  Piece c;
  const int slot = blockIdx.x, hd = blockIdx.y, tid = threadIdx.x;
  if (!find_piece<CK>(d, pc, slot, c)) return;
  const int w = tid >> 6, lane = tid & 63, l32 = lane & 31, half = lane >> 5, kh = hd / (H / G);
  const size_t cell = (size_t)slot * H + hd;
  const bool old = c.idx > 0 || d.pos0[c.s] > 0;           // is there a state in front of the chunk
  if (w == 0) {
    const Gate g = gates<MLSTM>(ga, c, hd, lane);
    double b0 = g.F0, b1 = g.F1, x0 = g.F0, x1 = g.F1;
    if (MLSTM) {
      const double mp = meta[3 * cell + 2];
      double m0, m1;
      running_max(g, lane, m0, m1);
      m0 = fmax(m0, mp);
      m1 = fmax(m1, mp);
      b0 = -m0;
      b1 = -m1;
      x0 = mp - m0;
      x1 = mp - m1;
      if (2 * lane < c.n) efl[(size_t)(c.t0 + 2 * lane) * H + hd] = exp2f((float)(-(g.F0 + m0)));
      if (2 * lane + 1 < c.n) efl[(size_t)(c.t0 + 2 * lane + 1) * H + hd] = exp2f((float)(-(g.F1 + m1)));
      // behind the last chunk, here or at all (tokens past its end change nothing)
      if (lane == 63 && (c.t0 + c.n == d.seq_off[c.s + 1] || (pc.count > 0 && c.idx == pc.first + pc.count - 1)))
        M[(size_t)d.slots[c.s] * H + hd] = (float)((g.F1 + m1) * 0.69314718055994530942);
    }
    const float ah0 = (float)g.a0, ah1 = (float)g.a1, bh0 = (float)b0, bh1 = (float)b1;
    const int j = 2 * lane;
    sah[j] = ah0;
    sah[j + 1] = ah1;
    sal[j] = j < c.n ? (float)(g.a0 - (double)ah0) : 0.f;
    sal[j + 1] = j + 1 < c.n ? (float)(g.a1 - (double)ah1) : 0.f;
    sc[j] = g.c0;
    sc[j + 1] = g.c1;
    sbh[j] = bh0;
    sbh[j + 1] = bh1;
    sbl[j] = (float)(b0 - (double)bh0);
    sbl[j + 1] = (float)(b1 - (double)bh1);
    sx[j] = exp2f((float)x0);
    sx[j + 1] = exp2f((float)x1);
  }
  if (tid < 64) sbad[tid >> 5][tid & 31] = CK;
  if (MLSTM && tid >= 256 - DK) sN[tid - (256 - DK)] = old ? NU[cell * DK + tid - (256 - DK)] : 0.f;
  const bool work = 32 * w < c.n;
  const int qi = 32 * w + l32;                              // this lane's query
  bf16x8 qf[2 * NK], pf[4][2][3];
  if (work) {
    const bf16* qp = q + (size_t)(c.t0 + min(qi, c.n - 1)) * ldq + kh * DK + 8 * half;
#pragma unroll
    for (int s = 0; s < 2 * NK; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
  }
  __syncthreads();
  if (work) {
    const float bh = sbh[qi], bl = sbl[qi];
    float rsum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
      if (kt <= w) {
        const bf16* kp = k + (size_t)(c.t0 + min(32 * kt + l32, c.n - 1)) * ldk + kh * DK + 8 * half;
        bf16x8 kf[2 * NK];
#pragma unroll
        for (int s = 0; s < 2 * NK; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(kp + 16 * s);
        f32x16 p;
#pragma unroll
        for (int i = 0; i < 16; ++i) p[i] = 0.f;
#pragma unroll
        for (int s = 0; s < 2 * NK; ++s) p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qf[s], p, 0, 0, 0);
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const int j0 = 32 * kt + 8 * g4 + 4 * half;
          const f32x4 ah = *reinterpret_cast<const f32x4*>(sah + j0), al = *reinterpret_cast<const f32x4*>(sal + j0),
                      cw = *reinterpret_cast<const f32x4*>(sc + j0);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            float y = p[4 * g4 + x] * __builtin_amdgcn_exp2f((bh + ah[x]) + (bl + al[x]));
            if (!MLSTM) y *= cw[x];
            y = j0 + x <= qi ? y : 0.f;
            if (MLSTM) rsum += y;
            bf16 a, b, e;
            split3(y, a, b, e);
            const int i = 4 * g4 + x;
            pf[kt][i >> 3][0][i & 7] = a;
            pf[kt][i >> 3][1][i & 7] = b;
            pf[kt][i >> 3][2][i & 7] = e;
          }
        }
      }
    if (MLSTM) {
      float dot = 0.f;
#pragma unroll
      for (int s = 0; s < 2 * NK; ++s)
#pragma unroll
        for (int x = 0; x < 8; ++x) dot += (float)qf[s][x] * sN[16 * s + 8 * half + x];
      float t = rsum + sx[qi] * dot;
      t += __shfl_xor(t, 32, 64);
      if (half == 0 && qi < c.n) den[(size_t)(c.t0 + qi) * H + hd] = t * ga.qscale;
    }
  }
  const float skip = MLSTM ? 0.f : ga.dskip[hd];
  const bf16* vp = v + (size_t)c.t0 * ldv + (size_t)hd * dv;
  const float* up = U + cell * dv * DK;
  for (int cb = 0; cb < dv; cb += 32) {
    bf16x4 rv[4];
    const int c4 = tid & 7, vt = tid >> 3;
    load_4x4(vp + (size_t)(4 * vt) * ldv + cb + 4 * c4, ldv, c.n - 4 * vt, cb + 4 * c4 < dv, rv);
    f32x4 ru[NK];
    if (old) {
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        const int e = tid + 256 * i, r = e / (DK / 4), x4 = e % (DK / 4);
        ru[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (cb + r < dv) ru[i] = *reinterpret_cast<const f32x4*>(up + (size_t)(cb + r) * DK + 4 * x4);
      }
    }
    if (cb) __syncthreads();                                // the last columns' reads are done
    // A masked score is a 0 that multiplies a later token's value: an infinite or NaN value would reach the queries in front of
    // it.  It counts as 0 in the products, and its column is NaN from its token on.
    int* const bad = sbad[(cb >> 5) & 1];
    unsigned m[2] = {0u, 0u};
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const u32x2 u = __builtin_bit_cast(u32x2, rv[x]);
      m[0] |= (u[0] & 0x7f807f80u) + 0x00800080u;           // bit 15 of a half: its exponent is all ones
      m[1] |= (u[1] & 0x7f807f80u) + 0x00800080u;
    }
    if ((m[0] | m[1]) & 0x80008000u)
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (!isfinite((float)rv[x][t])) {
            rv[x][t] = (bf16)0.f;
            atomicMin(bad + 4 * c4 + x, 4 * vt + t);
          }
#pragma unroll
    for (int x = 0; x < 4; ++x) *reinterpret_cast<bf16x4*>(sv + (4 * c4 + x) * VP + 4 * vt) = rv[x];
    if (old) {
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        const int e = tid + 256 * i, r = e / (DK / 4), x4 = e % (DK / 4);
        bf16x4 h, m, l;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          bf16 a, b, g;
          split3(ru[i][t], a, b, g);
          h[t] = a;
          m[t] = b;
          l[t] = g;
        }
        bf16* row = ss + r * SP + 4 * x4;
        *reinterpret_cast<bf16x4*>(row) = h;
        *reinterpret_cast<bf16x4*>(row + 32 * SP) = m;
        *reinterpret_cast<bf16x4*>(row + 2 * 32 * SP) = l;
      }
    }
    __syncthreads();
    if (!work) continue;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if (old) {
#pragma unroll
      for (int s = 0; s < 2 * NK; ++s) {
        const bf16* bp = ss + l32 * SP + 16 * s + 8 * half;
#pragma unroll
        for (int part = 2; part >= 0; --part)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[s], *reinterpret_cast<const bf16x8*>(bp + part * 32 * SP), acc, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] *= sx[32 * w + c_row(i, half)];
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
      if (kt <= w) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const bf16* bp = sv + l32 * VP + 32 * kt + 16 * ks + 4 * half;
          const bf16x4 b0 = *reinterpret_cast<const bf16x4*>(bp), b1 = *reinterpret_cast<const bf16x4*>(bp + 8);
          const bf16x8 b = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
#pragma unroll
          for (int part = 2; part >= 0; --part) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pf[kt][ks][part], b, acc, 0, 0, 0);
        }
      }
    if (tid < 32) sbad[(~cb >> 5) & 1][tid] = CK;           // (for the next columns; this one's last readers are past a barrier)
    const int col = cb + l32;
    const int first = bad[l32];
    if (col < dv) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int r = 32 * w + c_row(i, half);
        if (r < c.n) {
          const float y = MLSTM ? acc[i] * ga.qscale : acc[i] + skip * (float)sv[l32 * VP + r];
          out[((size_t)(c.t0 + r) * H + hd) * dv + col] = r >= first ? NAN : y;
        }
      }
    }
  }
}

// floats of a slot; 0.4 us a token in the token-by-token form
size_t chunk_floats(int H, int dk, int dv) { return (size_t)H * (6 + (size_t)dk * (dv + 1)); }
PiecePlan chunk_plan(int T_, int B, int H, int dk, int dv, size_t most) {
  return plan_pieces(T_, B, CK, chunk_floats(H, dk, dv), most, 0.4f);
}

template <int NK, bool MLSTM>
void chunk_launch(const bf16* q, int ldq, const bf16* k, int ldk, const bf16* v, int ldv, const GateArgs& ga, float* S, float* N,
                  float* M, float* out, float* den, float* efl, float* ws, size_t most, int H, int G, int dv, SeqDesc d,
                  hipStream_t st) {
  const PiecePlan plan = chunk_plan(d.Ttot, d.B, H, 32 * NK, dv, most);
  const size_t ns = plan.slots, cells = ns * H;
  double* meta = reinterpret_cast<double*>(ws);
  float* U = ws + 6 * cells + (6 * cells & 3);
  float* NU = U + cells * dv * 32 * NK;
  const int nb = (dv * 32 * NK + 1023) / 1024;
  for (int w = 0; w < plan.windows; ++w) {
    const Pieces pc = {CK, w * plan.count, plan.count};
    hipLaunchKernelGGL((k_chunk_state<NK, MLSTM>), dim3((unsigned)ns, H, (dv + 63) / 64), dim3(256), 0, st, k, ldk, v, ldv, ga, U,
                       NU, meta, H, G, dv, pc, d);
    hipLaunchKernelGGL((k_chunk_walk<MLSTM>), dim3(d.B * H, nb + (MLSTM ? 1 : 0)), dim3(256), 0, st, U, NU, meta, S, N, M, H,
                       32 * NK, dv, nb, pc, d);
    hipLaunchKernelGGL((k_chunk_out<NK, MLSTM>), dim3((unsigned)ns, H), dim3(256), 0, st, q, ldq, k, ldk, v, ldv, ga, U, NU, meta,
                       M, out, den, efl, H, G, dv, pc, d);
  }
  LIPA_CHECK_LAUNCH();
}

template <bool MLSTM>
void chunk_dispatch(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const GateArgs& ga, float* S, float* N,
                    float* M, float* out, float* den, float* efl, float* ws, size_t most, int H, int G, int dk, int dv,
                    SeqDesc d, hipStream_t st) {
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

// Floats of workspace of the chunked form, or 0 where the token-by-token scan is the one to run: float activations, key sizes
// that are no multiple of 32 or above 128, rows that 16-byte (q, k, the states S and N) or 8-byte (v) loads cannot take, and steps of
// few tokens a sequence.  At most `most`: longer steps run in windows.
size_t seq_chunk_floats(int code, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const void* S,
                        const void* N, int T_, int B, int H, int dk, int dv, size_t most) {
  const auto fits = [](const void* p, int ld, int n) { return ld % n == 0 && ((uintptr_t)p & (2 * n - 1)) == 0; };
  if (code != 0 || dk % 32 != 0 || dk > 128 || dv % 4 != 0 || !fits(q, ldq, 8) || !fits(k, ldk, 8) || !fits(v, ldv, 4) ||
      !fits(S, 8, 8) || !fits(N, 8, 8))
    return 0;
  // Three launches and a chunk of padding against 0.4 us a token (two heads a CU) in the token-by-token form: 64 tokens a
  // sequence are 21 / 32 / 96 us here and 30 / 36 / 148 us there (state space, 32 heads, 1 / 8 / 48 sequences), 48 are 21 / 32 / 94
  // and 24 / 29 / 118 us; mLSTM (8 heads of 128 x 192) at 64: 26 / 34 / 68 against 31 / 36 / 159 us.  The outputs walk the columns 32 at a
  // time, one after another: 512 of them 43 against 26 us at 64 tokens, even at 128 to 160.  Where (sequence, head) pairs fill the chip,
  // the padding counts, and with small keys the token form is the cheaper one for longer: 1024 pairs of 64 x 64 take 1.3 times its time at
  // 64 to 128 tokens, 0.94 at 192; 1024 of 32 x 128 1.2 at 192, 1.08 at 256, 0.92 at 512; 1024 of 128 x 64 are ahead from 64 on.
  const long pairs = (long)B * H;
  long least = std::max(64, std::min(dv * 5 / 12, 192));
  if (pairs >= 256 && dk <= 64 && dv >= 128) least = std::max(least, 96l);
  if (pairs >= 1024 && (dk <= 64 || dv <= 32)) least = 192;
  if (pairs * dv >= 1l << 17 && dk <= 32) least = 256;
  if (B == 0 || T_ < least * B) return 0;
  const size_t slots = chunk_plan(T_, B, H, dk, dv, most).slots;
  return slots == 0 ? 0 : slots * chunk_floats(H, dk, dv) + 4;
}

void seq_chunk_ssd(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const void* dt, int lddt,
                   const float* dt_bias, const float* a_log, const float* dskip, float* S, float* out, float* ws, size_t most,
                   int H, int G, int dk, int dv, SeqDesc d, hipStream_t st) {
  const GateArgs ga = {(const bf16*)dt, lddt, dt_bias, a_log, dskip, nullptr, nullptr, nullptr, nullptr, 1.f, 1.f, H};
  chunk_dispatch<false>(q, ldq, k, ldk, v, ldv, ga, S, nullptr, nullptr, out, nullptr, nullptr, ws, most, H, G, dk, dv, d,
                        st);
}

void seq_chunk_mlstm(const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const float* ipre, const float* fpre,
                     const float* ib, const float* fb, float cap, float qscale, float* S, float* N, float* M, float* out,
                     float* den, float* efl, float* ws, size_t most, int H, int dk, int dv, SeqDesc d, hipStream_t st) {
  const GateArgs ga = {nullptr, 0, nullptr, nullptr, nullptr, ipre, fpre, ib, fb, cap, qscale, H};
  chunk_dispatch<true>(q, ldq, k, ldk, v, ldv, ga, S, N, M, out, den, efl, ws, most, H, H, dk, dv, d, st);
}
