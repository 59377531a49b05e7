// Recurrences whose decay differs per state row: the selective state space with a step size per channel and a decay per
// (channel, state), and gated linear attention with a data-dependent decay per key channel.  Packed variable-length
// sequences, float state per slot; one token is the decode step.  Like the scans of seq_scan.hip these walk the tokens
// of a step in order with the state in registers and stage 16 tokens at a time through LDS; here a lane owns a small
// TILE of the state (rows x columns), so that a row vector read from LDS serves several columns and a column value
// several rows: the reads, not the arithmetic, bound a scan whose lanes own one column each.
#include "seq_common.h"

#include <algorithm>
#include <cfloat>
#include <utility>

using namespace lipa;

namespace {

constexpr int CT = 16;      // tokens staged per chunk

__device__ __forceinline__ float softplus_fast(float x) { return fmaxf(x, 0.f) + log1p_exp_neg(fabsf(x)); }
__device__ __forceinline__ float silu_fast(float z) {
  return z * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(z * -1.4426950408889634f));
}

// Lane layout of a wave: R lanes (4, 8 or 16) share a column; they differ in lane bits 4 and 5 (the wave's rows of 16
// lanes) and, above four, in bits 0 and 1.  The other bits tell the wave's 64 / R column groups apart.
template <int R>
__device__ __forceinline__ int lane_part(int lane) {
  return (lane >> 4) | (R >= 8 ? (lane & 1) << 2 : 0) | (R >= 16 ? (lane & 2) << 2 : 0);
}
template <int R>
__device__ __forceinline__ int lane_group(int lane) {
  return R == 4 ? lane & 15 : R == 8 ? (lane & 15) >> 1 : (lane & 15) >> 2;
}
// Four values summed over a column's R lanes at once: after exchanging halves of the wave and rows of 16 lanes, row i of
// the wave holds value i (in all lanes of its group): two exchanges and an exchange of sums instead of four butterflies.
__device__ __forceinline__ float dpp_quad_add(float v, int which) {
  const int o = which == 0 ? __builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true)     // quad_perm [1, 0, 3, 2]
                           : __builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true);    // quad_perm [2, 3, 0, 1]
  return v + __int_as_float(o);
}
template <int R>
__device__ __forceinline__ float sum_four(float v0, float v1, float v2, float v3) {
  float v = swap16_add(swap32_add(v0, v2), swap32_add(v1, v3));
  if (R >= 8) v = dpp_quad_add(v, 0);
  if (R >= 16) v = dpp_quad_add(v, 1);
  return v;
}

// NR contiguous entries of a state row of `len`, starting at i0 (past the row's end: 0); 16-byte accesses where they fit
template <int NR>
__device__ __forceinline__ void load_state(const float* p, int i0, int len, bool on, float (&r)[NR]) {
#pragma unroll
  for (int i4 = 0; i4 < NR / 4; ++i4) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    const int i = i0 + 4 * i4;
    if (on && (len & 3) == 0) {
      if (i < len) v = *reinterpret_cast<const f32x4*>(p + i);
    } else if (on) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j < len) v[j] = p[i + j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) r[4 * i4 + j] = v[j];
  }
}
template <int NR>
__device__ __forceinline__ void store_state(float* p, int i0, int len, const float (&r)[NR]) {
#pragma unroll
  for (int i4 = 0; i4 < NR / 4; ++i4) {
    const int i = i0 + 4 * i4;
    if ((len & 3) == 0) {
      if (i < len) *reinterpret_cast<f32x4*>(p + i) = f32x4{r[4 * i4], r[4 * i4 + 1], r[4 * i4 + 2], r[4 * i4 + 3]};
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j < len) p[i + j] = r[4 * i4 + j];
    }
  }
}

// ------------------------------------------------------------------------------------------------ selective scan
// dt = softplus(dt_pre + bias);  S[c, n] <- exp(-dt_c e^{A_log[c, n]}) S[c, n] + dt_c x_c B_n;
// y_c = sum_n S[c, n] C_n + D_c x_c;  out = scale * y * silu(z).
// A lane owns NS states of CH = 2 channels; R >= N / NS lanes share those channels, a block of 256 threads owns
// NC = 256 / R * CH channels of one sequence.  dt and dt x of the chunk go through LDS, a thread keeps the x and z it
// fetched for the read-out of the same (token, channel) pairs.  Two tokens per turn: their four read-outs are summed over
// the lanes together, and the next pair's inputs are read while the current pair is computed.
//
// One prompt keeps C / NC blocks busy for as long as it has tokens (0.23 us each), so a step whose sequences do not fill the
// chip is cut over time (k_selective_walk and the two cut modes): every segment of 32 or 64 tokens first runs from a zero state for
// the state it leaves and the sum of its step sizes (its decay is e^{A sum dt}), a walk over a sequence's segments turns those
// into the states in front of the segments, and every segment then runs from its own.  One prompt of 4096 tokens, 2048
// channels of 16 states: 886 -> 103 us (37 for what segments leave, 27, 48 under a profiler: bound by one half-rate exponential per
// channel, state and token in either pass).  Steps that a state per lane serves better (k_selective_row) go there.
constexpr int CH = 2;
enum { WHOLE, LEAVES, FROM };       // a sequence; a segment from zero (state and step sizes); a segment from the state before it

template <typename T, int NS, int R, int MODE>
__global__ __launch_bounds__(256) void k_selective_scan(const T* __restrict__ x, int ldx, const float* __restrict__ dtp,
                                                        const float* __restrict__ dtb, const T* __restrict__ bm, int ldb,
                                                        const T* __restrict__ cm, int ldc, const float* __restrict__ a_log,
                                                        const float* __restrict__ dskip, const T* __restrict__ z, int ldz,
                                                        float* __restrict__ S, T* __restrict__ out, int ldo, float scale,
                                                        int C, int N, float* __restrict__ ws, float* __restrict__ wdt,
                                                        Pieces pc, SeqDesc d) {
  constexpr int NC = 256 / R * CH, PER = CT * NC / 256, NP = NS * R, PB = (CT * NP + 255) / 256;
  __shared__ __attribute__((aligned(16))) float sdt[CT * NC];
  __shared__ __attribute__((aligned(16))) float sdx[CT * NC];     // dt x
  __shared__ __attribute__((aligned(16))) float sy[CT * NC];      // the tokens' read-outs
  __shared__ __attribute__((aligned(16))) float sB[CT * NP];
  __shared__ __attribute__((aligned(16))) float sC[CT * NP];
  const int tid = threadIdx.x;
  const int lane = tid & 63, grp = (tid >> 6) * (64 / R) + lane_group<R>(lane), row = lane >> 4;
  const int cb = blockIdx.y * NC, c0 = cb + grp * CH, n0 = lane_part<R>(lane) * NS;
  Piece seg = {(int)blockIdx.x, 0, 0, 0};
  if (MODE != WHOLE && !find_piece<0>(d, pc, blockIdx.x, seg)) return;
  const int s = seg.s;
  if (d.live && !d.live[s]) return;
  const int end = d.seq_off[s + 1], t0 = MODE == WHOLE ? d.seq_off[s] : seg.t0, t1 = MODE == WHOLE ? end : t0 + seg.n;
  const bool last = t1 == end || (pc.count > 0 && seg.idx == pc.first + pc.count - 1);     // of the sequence, or of it here
  if (MODE == LEAVES && last) return;                 // (nothing that a leaving state would serve stands behind it)
  const int p0 = d.pos0[s], slot = d.slots[s];
  float Sr[CH][NS], A[CH][NS], sum[CH] = {0.f, 0.f};
#pragma unroll
  for (int h = 0; h < CH; ++h) {
    const bool ok = c0 + h < C;
    const size_t ch = ok ? c0 + h : 0;
    load_state<NS>(a_log + ch * N, n0, N, ok, A[h]);
    if (MODE == FROM)
      load_state<NS>(ws + ((size_t)blockIdx.x * C + ch) * N, n0, N, ok, Sr[h]);
    else
      load_state<NS>(S + ((size_t)slot * C + ch) * N, n0, N, MODE == WHOLE && ok && p0 > 0, Sr[h]);
#pragma unroll
    for (int i = 0; i < NS; ++i) A[h][i] = -expf(A[h][i]) * 1.4426950408889634f;    // decays as powers of two
  }
  // A chunk's inputs are fetched without branches (addresses clamped to the step's last token and the last channel, values
  // past them dropped when they are staged), so that all of a thread's loads are in flight together; a thread's channel
  // is the same for all of its tokens.
  static_assert(256 % NC == 0 && 256 % NP == 0, "a thread keeps its column");
  const int fc = cb + tid % NC, ft = tid / NC, fcc = min(fc, C - 1), br = tid % NP, bt = tid / NP, brc = min(br, N - 1);
  const float bias = dtb[fcc], skip = dskip[fcc];
  T fx[PER], fz[PER], gx[PER], gz[PER], fB[PB], fC[PB];
  float fd[PER];
  auto fetch = [&](int tb) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const size_t t = min(tb + ft + 256 / NC * i, t1 - 1);
      fx[i] = x[t * ldx + fcc];
      if (MODE != LEAVES) fz[i] = z[t * ldz + fcc];
      fd[i] = dtp[t * C + fcc];
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const size_t t = min(tb + bt + 256 / NP * i, t1 - 1);
      fB[i] = bm[t * ldb + brc];
      if (MODE != LEAVES) fC[i] = cm[t * ldc + brc];
    }
  };
  if (t0 < t1) fetch(t0);
  for (int tb = t0; tb < t1; tb += CT) {
    const int n = min(CT, t1 - tb);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const float dt = softplus_fast(fd[i] + bias);
      sdt[tid + 256 * i] = dt;
      sdx[tid + 256 * i] = dt * (float)fx[i];
      if (MODE != LEAVES) {
        gx[i] = fx[i];
        gz[i] = fz[i];
      }
    }
#pragma unroll
    for (int i = 0; i < PB; ++i)
      if (CT * NP >= 256 || tid < CT * NP) {
        sB[tid + 256 * i] = br < N ? (float)fB[i] : 0.f;          // a padded state never leaves zero
        if (MODE != LEAVES) sC[tid + 256 * i] = br < N ? (float)fC[i] : 0.f;
      }
    __syncthreads();
    if (tb + CT < t1) fetch(tb + CT);
    struct In {
      f32x4 B[NS / 4], C[NS / 4];
      float dt[CH], dx[CH];
    };
    auto load = [&](int tt, In& in) {
#pragma unroll
      for (int i4 = 0; i4 < NS / 4; ++i4) {
        in.B[i4] = *reinterpret_cast<const f32x4*>(sB + tt * NP + n0 + 4 * i4);
        if (MODE != LEAVES) in.C[i4] = *reinterpret_cast<const f32x4*>(sC + tt * NP + n0 + 4 * i4);
      }
#pragma unroll
      for (int h = 0; h < CH; ++h) {
        in.dt[h] = sdt[tt * NC + grp * CH + h];
        in.dx[h] = sdx[tt * NC + grp * CH + h];
      }
    };
    auto step = [&](const In& in, float (&y)[CH]) {
#pragma unroll
      for (int h = 0; h < CH; ++h) {
        float p[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NS; ++i) {
          Sr[h][i] = __builtin_amdgcn_exp2f(in.dt[h] * A[h][i]) * Sr[h][i] + in.dx[h] * in.B[i >> 2][i & 3];
          if (MODE != LEAVES) p[i & 1] += Sr[h][i] * in.C[i >> 2][i & 3];
        }
        if (MODE == LEAVES)
          sum[h] += in.dt[h];
        else
          y[h] = p[0] + p[1];
      }
    };
    In a0, a1;
    float ya[CH], yb[CH] = {0.f, 0.f};
    load(0, a0);
    int tt = 0;
    for (; tt + 1 < n; tt += 2) {
      load(tt + 1, a1);
      step(a0, ya);
      load(min(tt + 2, n - 1), a0);
      step(a1, yb);
      if (MODE == LEAVES) continue;
      const float v = sum_four<R>(ya[0], ya[1], yb[0], yb[1]);     // row i of the wave: token tt + i / 2, channel i % 2
      if (R == 4 || (lane & (R == 8 ? 1 : 3)) == 0) sy[(tt + (row >> 1)) * NC + grp * CH + (row & 1)] = v;
    }
    if (tt < n) {
      step(a0, ya);
      const float v = MODE == LEAVES ? 0.f : sum_four<R>(ya[0], ya[1], yb[0], yb[1]);
      if (MODE != LEAVES && (R == 4 || (lane & (R == 8 ? 1 : 3)) == 0) && row < 2) sy[tt * NC + grp * CH + row] = v;
    }
    if (MODE == LEAVES) continue;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int tt = ft + 256 / NC * i;
      if (tt < n && fc < C) {
        const float v = (sy[tid + 256 * i] + skip * (float)gx[i]) * silu_fast((float)gz[i]) * scale;
        out[(size_t)(tb + tt) * ldo + fc] = (T)v;
      }
    }
  }
#pragma unroll
  for (int h = 0; h < CH; ++h)
    if (c0 + h < C) {
      if (MODE == LEAVES) {
        store_state<NS>(ws + ((size_t)blockIdx.x * C + c0 + h) * N, n0, N, Sr[h]);
        if (n0 == 0) wdt[(size_t)blockIdx.x * C + c0 + h] = sum[h];
      } else if (MODE == WHOLE || last) {
        store_state<NS>(S + ((size_t)slot * C + c0 + h) * N, n0, N, Sr[h]);
      }
    }
}

// ------------------------------------------------------------------------------- selective scan, one state per lane
// Prompts whose sequences do not fill the chip: a lane owns ONE state, a row of 16 lanes a channel, so that two sequences of 4096 channels
// of 16 states are two waves on every SIMD where the tiles of k_selective_scan are half a wave, and nothing has to be cut over time, which
// takes every exponential twice.  64 tokens are staged at once: a thread fetches four tokens of one channel (and of one column of B and C) in
// rows of 16, finishes their dt and dt x and leaves them transposed in LDS.  In the scan lane t of a row holds dt and dt x of token t of 16 and
// hands them to the row with the multiplication that reads them (row_newbcast); a lane's 16 read-outs are summed over the row in
// halves (15 adds for 16 sums), which leaves lane t with token t, in the place of its dt.
// Bound by issue: a half-rate exponential and four instructions a token and state, three for the sums, three for the staging.  Two
// prompts of 2048 and 1337 tokens, 4096 channels of 16: 129 -> 84 us (33 ns a token with one wave on a SIMD, 19 a wave with many).  With x, z
// and dt fetched where they are needed (16 rows a load) the address units were busy for 80% of 123 us.
constexpr int RT = 64, RLD = RT + 4, DLD = RT + 20;      // tokens staged at once; rows of B and C, of dt and dt x in LDS (for the banks)

template <int L>
__device__ __forceinline__ float row_lane(float v) {       // lane L of every row, in all lanes of the row
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + L, 0xF, 0xF, true));
}
// lanes where `hi` keep b and give a away, the others keep a and give b; the partner is the lane that CTRL names
template <int CTRL>
__device__ __forceinline__ float half_sum(float a, float b, bool hi) {
  return (hi ? b : a) + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(hi ? a : b), CTRL, 0xF, 0xF, true));
}
// the bits of a T through a bounds-checked window
template <typename T>
struct Raw {
  using type = unsigned short;
  template <typename W>
  static __device__ __forceinline__ type load(W w, unsigned o) { return __builtin_amdgcn_raw_buffer_load_b16(w, o, 0, 0); }
  static __device__ __forceinline__ float value(type v) { return __uint_as_float((unsigned)v << 16); }
  template <typename W>
  static __device__ __forceinline__ void store(W w, unsigned o, float v) {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (T)v), w, o, 0, 0);
  }
};
template <>
struct Raw<float> {
  using type = unsigned;
  template <typename W>
  static __device__ __forceinline__ type load(W w, unsigned o) { return __builtin_amdgcn_raw_buffer_load_b32(w, o, 0, 0); }
  static __device__ __forceinline__ float value(type v) { return __uint_as_float(v); }
  template <typename W>
  static __device__ __forceinline__ void store(W w, unsigned o, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), w, o, 0, 0);
  }
};
__device__ __forceinline__ auto window(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// the decays and inputs of 16 tokens, for one state
template <int... I>
__device__ __forceinline__ void row_tokens(std::integer_sequence<int, I...>, float dt, float dx, float A, const float* b,
                                           float (&e)[16], float (&in)[16]) {
  ((e[I] = __builtin_amdgcn_exp2f(row_lane<I>(dt) * A), in[I] = row_lane<I>(dx) * b[I]), ...);
}

template <typename T>
__global__ __launch_bounds__(256) void k_selective_row(const T* __restrict__ x, int ldx, const float* __restrict__ dtp,
                                                       const float* __restrict__ dtb, const T* __restrict__ bm, int ldb,
                                                       const T* __restrict__ cm, int ldc, const float* __restrict__ a_log,
                                                       const float* __restrict__ dskip, const T* __restrict__ z, int ldz,
                                                       float* __restrict__ S, T* __restrict__ out, int ldo, float scale, int C,
                                                       int N, SeqDesc d) {
  __shared__ __attribute__((aligned(16))) float sB[16 * RLD];
  __shared__ __attribute__((aligned(16))) float sC[16 * RLD];
  __shared__ float sdt[16 * DLD];                                 // [channel][token]: dt, then the read-out that takes its place
  __shared__ float sdx[16 * DLD];                                 // dt x
  const int s = blockIdx.y, tid = threadIdx.x, lane = tid & 15, row = tid >> 4;
  if (d.live && !d.live[s]) return;
  // consecutive channels on the same die: a line of x, z or dt is read by up to four blocks
  const int groups = gridDim.x, cg = groups % 8 == 0 ? (blockIdx.x & 7) * (groups >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int t0 = d.seq_off[s], t1 = d.seq_off[s + 1];
  // in the scan a thread is a state of channel `row`, everywhere else channel `lane` of token `row` of 16
  const int c = cg * 16 + row, fc = cg * 16 + lane, ch = min(c, C - 1), fch = min(fc, C - 1);
  const bool own = c < C && lane < N;
  float* Sp = S + ((size_t)d.slots[s] * C + ch) * N + lane;
  float st = own && d.pos0[s] > 0 ? *Sp : 0.f;
  float A = -expf(own ? a_log[(size_t)ch * N + lane] : 0.f) * 1.4426950408889634f;      // decays as powers of two
  A = A < -FLT_MAX ? -FLT_MAX : A;                                // (past a sequence's end it meets steps of 0)
  const float bias = dtb[fch], skip = dskip[fch];
  // Windows of 64 tokens move along the rows, so that a thread's places in them never change; what is past a sequence's end, or no
  // state, reads as 0 and is not written.
  constexpr unsigned E = sizeof(T), NOWHERE = ~0u - 64;
  unsigned ox[4], oz[4], od[4], ob[4], oc[4], oo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned t = 16 * i + row;
    ox[i] = (t * ldx + fch) * E;
    oz[i] = (t * ldz + fch) * E;
    od[i] = (t * C + fch) * 4;
    oo[i] = fc < C ? (t * ldo + fc) * E : NOWHERE;
    ob[i] = lane < N ? (t * ldb + lane) * E : NOWHERE;
    oc[i] = lane < N ? (t * ldc + lane) * E : NOWHERE;
  }
  typename Raw<T>::type fx[4], fz[4], fb[4], fcc[4];
  float fd[4];
  auto fetch = [&](int tb) {
    const unsigned n = min(RT, t1 - tb);
    const auto wx = window(x + (size_t)tb * ldx, n * ldx * E), wz = window(z + (size_t)tb * ldz, n * ldz * E),
               wd = window(dtp + (size_t)tb * C, n * C * 4), wb = window(bm + (size_t)tb * ldb, n * ldb * E),
               wc = window(cm + (size_t)tb * ldc, n * ldc * E);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      fd[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(wd, od[i], 0, 0));
      fx[i] = Raw<T>::load(wx, ox[i]);
      fz[i] = Raw<T>::load(wz, oz[i]);
      fb[i] = Raw<T>::load(wb, ob[i]);
      fcc[i] = Raw<T>::load(wc, oc[i]);
    }
  };
  if (t0 < t1) fetch(t0);
  for (int tb = t0; tb < t1; tb += RT) {
    const int n = min(RT, t1 - tb);
    float gx[4], gz[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * i + row;
      // (past the end tokens that change nothing; a selection would be a branch)
      const float dt = __uint_as_float(__float_as_uint(softplus_fast(fd[i] + bias)) & (t < n ? ~0u : 0u));
      gx[i] = Raw<T>::value(fx[i]);
      gz[i] = Raw<T>::value(fz[i]);
      sdt[lane * DLD + t] = dt;
      sdx[lane * DLD + t] = dt * gx[i];
      sB[lane * RLD + t] = Raw<T>::value(fb[i]);
      sC[lane * RLD + t] = Raw<T>::value(fcc[i]);
    }
    __syncthreads();
    if (tb + RT < t1) fetch(tb + RT);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (16 * u >= n) break;
      float p[16], e[16], in[16], b[16];
      const float *pb = sB + lane * RLD + 16 * u, *pc = sC + lane * RLD + 16 * u;
      float& place = sdt[row * DLD + 16 * u + lane];
      const float dt = place, dx = sdx[row * DLD + 16 * u + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        *reinterpret_cast<f32x4*>(b + 4 * i) = *reinterpret_cast<const f32x4*>(pb + 4 * i);
        *reinterpret_cast<f32x4*>(p + 4 * i) = *reinterpret_cast<const f32x4*>(pc + 4 * i);
      }
      row_tokens(std::make_integer_sequence<int, 16>{}, dt, dx, A, b, e, in);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        st = __builtin_fmaf(e[i], st, in[i]);
        p[i] *= st;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = half_sum<0x128>(p[i], p[i + 8], lane & 8);          // row_ror 8: lane ^ 8
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = half_sum<0x141>(p[i], p[i + 4], lane & 4);          // row_half_mirror: lane ^ 7
#pragma unroll
      for (int i = 0; i < 2; ++i) p[i] = half_sum<0x4E>(p[i], p[i + 2], lane & 2);           // quad_perm [2, 3, 0, 1]
      place = half_sum<0xB1>(p[0], p[1], lane & 1);                                          // quad_perm [1, 0, 3, 2]
    }
    __syncthreads();
    const auto wo = window(out + (size_t)tb * ldo, (unsigned)n * ldo * E);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      Raw<T>::store(wo, oo[i], (sdt[lane * DLD + 16 * i + row] + skip * gx[i]) * silu_fast(gz[i]) * scale);
  }
  if (own) *Sp = st;
}

// The states in front of a sequence's segments, one (channel, state) per thread: they replace the states that the segments left.
__global__ __launch_bounds__(256) void k_selective_walk(const float* __restrict__ a_log, const float* __restrict__ S,
                                                        float* __restrict__ ws, const float* __restrict__ wdt, int C, int N,
                                                        Pieces pc, SeqDesc d) {
  const int s = blockIdx.x;
  const size_t e = (size_t)blockIdx.y * 256 + threadIdx.x, size = (size_t)C * N;
  if ((d.live && !d.live[s]) || e >= size) return;
  int first;
  const int n = own_pieces<0>(d, pc, s, first);
  if (n <= 0) return;
  const float A = -expf(a_log[e]) * 1.4426950408889634f;
  float x = pc.first > 0 || d.pos0[s] > 0 ? S[(size_t)d.slots[s] * size + e] : 0.f;
  float* u = ws + (size_t)first * size + e;
  const float* dt = wdt + (size_t)first * C + e / N;
  constexpr int AHEAD = 16;                         // segments in flight (the last one left nothing)
  float f[AHEAD], g[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (i < n - 1) {
      f[i] = u[i * size];
      g[i] = dt[(size_t)i * C];
    }
  for (int c0 = 0; c0 < n; c0 += AHEAD)
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int c = c0 + i;
      if (c < n) {
        u[c * size] = x;
        if (c < n - 1) x = __builtin_amdgcn_exp2f(g[i] * A) * x + f[i];
        if (c + AHEAD < n - 1) {
          f[i] = u[(c + AHEAD) * size];
          g[i] = dt[(size_t)(c + AHEAD) * C];
        }
      }
    }
}

// ------------------------------------------------------------------------------------------ gated linear attention
// a = sigmoid(z + bias)^(1 / tau) per key channel;  S <- diag(a) S + k v^T;  o = S^T (qscale q).  S [slots, H, dv, dk].
// A lane owns RR rows of CC = 4 columns; R lanes share those columns, a block of 256 threads owns NC = 256 / R * 4 columns
// of one (sequence, head).  The decays are finished in float when a chunk is staged; the next token's vectors are read
// from LDS while the current token is computed.
constexpr int CC = 4;

template <typename T, int RR, int R>
__global__ __launch_bounds__(256) void k_gla_scan(const T* __restrict__ q, int ldq, const T* __restrict__ k, int ldk,
                                                  const T* __restrict__ v, int ldv, const float* __restrict__ z,
                                                  const float* __restrict__ zb, float inv_tau, float qscale,
                                                  float* __restrict__ S, float* __restrict__ out, int H, int dk, int dv,
                                                  SeqDesc d) {
  constexpr int DKP = RR * R, NC = 256 / R * CC, PR = CT * DKP / 256 > 0 ? CT * DKP / 256 : 1, PV = CT * NC / 256;
  __shared__ __attribute__((aligned(16))) float sk[CT * DKP];
  __shared__ __attribute__((aligned(16))) float sq[CT * DKP];
  __shared__ __attribute__((aligned(16))) float sa[CT * DKP];
  __shared__ __attribute__((aligned(16))) float sv[CT * NC];
  __shared__ __attribute__((aligned(16))) float so[CT * NC];       // the tokens' read-outs
  const int s = blockIdx.x / H, hd = blockIdx.x % H, cb = blockIdx.y * NC, tid = threadIdx.x;
  if (d.live && !d.live[s]) return;
  const int lane = tid & 63, grp = (tid >> 6) * (64 / R) + lane_group<R>(lane), row = lane >> 4;
  const int c0 = cb + grp * CC, r0 = lane_part<R>(lane) * RR;
  const int t0 = d.seq_off[s], t1 = d.seq_off[s + 1], p0 = d.pos0[s], slot = d.slots[s];
  float* Sh = S + ((size_t)slot * H + hd) * dv * dk;
  float Sr[CC][RR];
#pragma unroll
  for (int c = 0; c < CC; ++c)
    load_state<RR>(Sh + (size_t)(c0 + c < dv ? c0 + c : 0) * dk, r0, dk, p0 > 0 && c0 + c < dv, Sr[c]);
  static_assert(256 % NC == 0 && 256 % DKP == 0 && CT * DKP >= 256, "a thread keeps its row and its column");
  const int fr = tid % DKP, frt = tid / DKP, frc = hd * dk + min(fr, dk - 1);
  const int fc = cb + tid % NC, fct = tid / NC, fcc = hd * dv + min(fc, dv - 1);
  const float bias = zb[frc];
  T fk[PR], fq[PR], fv[PV];
  float fz[PR];
  auto fetch = [&](int tb) {                             // without branches, as in the selective scan
#pragma unroll
    for (int i = 0; i < PR; ++i) {
      const size_t t = min(tb + frt + 256 / DKP * i, t1 - 1);
      fk[i] = k[t * ldk + frc];
      fq[i] = q[t * ldq + frc];
      fz[i] = z[t * ((size_t)H * dk) + frc];
    }
#pragma unroll
    for (int i = 0; i < PV; ++i) {
      const size_t t = min(tb + fct + 256 / NC * i, t1 - 1);
      fv[i] = v[t * ldv + fcc];
    }
  };
  if (t0 < t1) fetch(t0);
  for (int tb = t0; tb < t1; tb += CT) {
    const int n = min(CT, t1 - tb);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PR; ++i) {
      sk[tid + 256 * i] = fr < dk ? (float)fk[i] : 0.f;       // a padded row never leaves zero
      sq[tid + 256 * i] = fr < dk ? (float)fq[i] * qscale : 0.f;
      const float zt = fz[i] + bias;                           // ln sigmoid(z) = min(z, 0) - ln(1 + e^-|z|)
      sa[tid + 256 * i] = __builtin_amdgcn_exp2f((fminf(zt, 0.f) - log1p_exp_neg(fabsf(zt))) * (inv_tau * 1.4426950408889634f));
    }
#pragma unroll
    for (int i = 0; i < PV; ++i) sv[tid + 256 * i] = (float)fv[i];
    __syncthreads();
    if (tb + CT < t1) fetch(tb + CT);
    struct In {
      f32x4 k[RR / 4], a[RR / 4], q[RR / 4], v;
    };
    auto load = [&](int tt, In& in) {
#pragma unroll
      for (int i4 = 0; i4 < RR / 4; ++i4) {
        in.k[i4] = *reinterpret_cast<const f32x4*>(sk + tt * DKP + r0 + 4 * i4);
        in.a[i4] = *reinterpret_cast<const f32x4*>(sa + tt * DKP + r0 + 4 * i4);
        in.q[i4] = *reinterpret_cast<const f32x4*>(sq + tt * DKP + r0 + 4 * i4);
      }
      in.v = *reinterpret_cast<const f32x4*>(sv + tt * NC + grp * CC);
    };
    auto step = [&](int tt, const In& in) {
      float o[CC] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < RR; ++i)
#pragma unroll
        for (int c = 0; c < CC; ++c) {
          Sr[c][i] = in.a[i >> 2][i & 3] * Sr[c][i] + in.k[i >> 2][i & 3] * in.v[c];
          o[c] += Sr[c][i] * in.q[i >> 2][i & 3];
        }
      const float v = sum_four<R>(o[0], o[1], o[2], o[3]);          // row c of the wave: column c
      if (R == 4 || (lane & (R == 8 ? 1 : 3)) == 0) so[tt * NC + grp * CC + row] = v;
    };
    In a0, a1;
    load(0, a0);
    int tt = 0;
    for (; tt + 1 < n; tt += 2) {
      load(tt + 1, a1);
      step(tt, a0);
      load(min(tt + 2, n - 1), a0);
      step(tt + 1, a1);
    }
    if (tt < n) step(tt, a0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PV; ++i) {
      const int tt = fct + 256 / NC * i;
      if (tt < n && fc < dv) out[((size_t)(tb + tt) * H + hd) * dv + fc] = so[tid + 256 * i];
    }
  }
#pragma unroll
  for (int c = 0; c < CC; ++c)
    if (c0 + c < dv) store_state<RR>(Sh + (size_t)(c0 + c) * dk, r0, dk, Sr[c]);
}

}  // namespace

int seq_selective_max_states() { return 256; }
int seq_gla_max_dk() { return 256; }

// Whether a step runs with a state per lane.  Its longest sequence takes 0.034 us a token, 0.048 where it is the only one and some CUs have
// two of its blocks of 16 channels; the mean length stands for the longest one, half as much again where there are several, most of whose
// blocks then end early.  Beyond 12 waves on a SIMD (49152 channels of sequences) both forms are bound by issue, and eight states per lane
// need fewer instructions; below 32 tokens staging 64 is most of the work.  The form cut over time takes 25 us and 8.5 ps per token and
// channel.  Beside two blocks a CU the two are close: what a state per lane takes more a token, fitted to 94 timed shapes, is 29.6 ns less 4.6
// ps per channel, and what it saves 22 us; the choice is within 1% of the faster one at all of them.
// us, the other form -> a state per lane, 16 states, sequences x tokens x channels: 1 x 256 x 4096 30 -> 12, 1 x 1024 x 1024 37 -> 36 (cut), 1 x
// 1024 x 4096 61 -> 37, 1 x 4096 x 2048 106 -> 134 (cut), 1 x 4096 x 4096 159 -> 134, 1 x 9000 x 4096 325 -> 294, 1 x 9000 x 3072 268 -> 307 (cut),
// 1 x 1024 x 5120 64 -> 52, 1 x 4096 x 5120 181 -> 196 (cut), 1 x 9000 x 4112 353 -> 431 (cut), 1 x 9000 x 6144 475 -> 455, 1 x 9000 x 8192 590 ->
// 446, 2048 + 1337 x 4096 129 -> 84, 4 x 512 x 4096 94 -> 46, 12 x 32 x 4096 14 -> 13, 16 x 16 x 4096 9.5 -> 15 (whole), 24 x 700 x 4096 301 ->
// 332 (whole), 24 x 700 x 2048 219 -> 178.  A sequence that is longer than the guess is the slower for it: 3000 + 3000 x 2560 147 -> 145, but
// 5000 + 1000 161 -> 186.
// Its windows take rows that are no shorter than their columns (where rows repeat or overlap, what stands past a sequence's end is inside the
// window) and 32-bit offsets into 64 of them; other strides take the other form.
bool seq_selective_rows(int T_, int B, int C, int N, int ldx, int ldz, int ldb, int ldc, int ldo) {
  if (std::min({ldx, ldz, ldo}) < C || std::min(ldb, ldc) < N || std::max({ldx, ldz, ldb, ldc, ldo}) >= 1 << 24) return false;
  if (N <= 8 || N > 16 || T_ < 32l * B || (long)B * C > 49152) return false;
  const int blocks = (C + 15) / 16;
  if (B == 1 && blocks > 256 && blocks <= 512) return T_ * (0.0296f - 4.6e-6f * C) < 22.f;
  return 0.034f * (B > 1 ? 1.5f : 1.f) * T_ / B < 8.5e-6f * T_ * C + 25.f;
}

// Tokens of a segment of the scan cut over time, or 0 where sequences run whole.  Whole, a sequence takes `whole` us a token as
// long as the chip is not full, and more after that; cut, a step takes about 25 us and `cut` us per token and channel (every exponential
// twice).  The lengths are not known here: their mean stands for the longest one, so that ragged steps run whole more often than they need.
// us, whole -> cut, tokens x channels: 16 states 4096 x 2048 886 -> 103, 9000 x 4112 1953 -> 353; 8 states 2048 x 4096 444 -> 88, 4 x 1024 x
// 8192 225 -> 227; 32 states 2048 x 8192 394 -> 224,
// 16 x 400 x 1024 85 -> 113 (whole); 64 states 2048 x 4096 379 -> 210, 2048 x 8192 381 -> 398 (whole); 128 states 2048 x 4096 568 -> 396, 4 x
// 1024 x 4096 463 -> 757 (whole); 256 states 2048 x 1024 1098 -> 253, 16 x 400 x 1024 364 -> 730 (whole).
// Segments of 32 tokens where those of 64 would leave the chip idle, else 64: their states pass through memory four times.
static int segment_of(int T_, int B, int C, int N, PiecePlan& plan, size_t most) {
  const struct { int states; float whole, cut; } form[] = {       // (the tilings of seq_selective_scan)
      {16, 0.226f, 8.5e-6f}, {32, 0.192f, 12e-6f}, {64, 0.185f, 23e-6f}, {128, 0.277f, 46e-6f}, {256, 0.54f, 125e-6f}};
  int f = 0;
  while (f < 4 && N > form[f].states) ++f;
  if (B == 0 || form[f].whole * T_ / B < form[f].cut * T_ * C + 25.f) return 0;
  if ((size_t)C * N > (size_t)256 * 65535) return 0;              // (the walk's grid)
  const int seg = (long)T_ * C < (1L << 22) ? 32 : 64;
  plan = plan_pieces(T_, B, seg, (size_t)C * (N + 1), most, form[f].whole);
  return plan.slots == 0 ? 0 : seg;
}
// Floats of its workspace, at most `most` (longer steps run in windows), or 0 where sequences run whole
size_t seq_selective_floats(int T_, int B, int C, int N, size_t most) {
  PiecePlan plan;
  return segment_of(T_, B, C, N, plan, most) == 0 ? 0 : plan.slots * C * (N + 1);
}

void seq_selective_scan(int code, const void* x, int ldx, const float* dtp, const float* dtb, const void* b, int ldb,
                        const void* c, int ldc, const float* a_log, const float* dskip, const void* z, int ldz, float* S,
                        void* out, int ldo, float scale, int C, int N, float* ws, size_t most, SeqDesc d, hipStream_t st) {
  if (d.B == 0) return;
  PiecePlan plan = {0, 0, 1};
  const int seg = ws != nullptr ? segment_of(d.Ttot, d.B, C, N, plan, most) : 1;
  float* wdt = ws != nullptr ? ws + plan.slots * C * N : nullptr;
  Pieces pc = {seg, 0, plan.count};
#define SEL_LAUNCH_(NS_, R_, MODE_, X_)                                                                                     \
  hipLaunchKernelGGL((k_selective_scan<T, NS_, R_, MODE_>), dim3((unsigned)(X_), (C + 256 / R_ * CH - 1) / (256 / R_ * CH)), \
                     dim3(256), 0, st, (const T*)x, ldx, dtp, dtb, (const T*)b, ldb, (const T*)c, ldc, a_log, dskip,        \
                     (const T*)z, ldz, S, (T*)out, ldo, scale, C, N, ws, wdt, pc, d)
#define SEL_LAUNCH(NS_, R_)                                                                                              \
  do {                                                                                                                   \
    if (ws == nullptr) {                                                                                                 \
      SEL_LAUNCH_(NS_, R_, WHOLE, d.B);                                                                                  \
      break;                                                                                                             \
    }                                                                                                                    \
    for (int w = 0; w < plan.windows; ++w, pc.first += plan.count) {                                                     \
      SEL_LAUNCH_(NS_, R_, LEAVES, plan.slots);                                                                          \
      hipLaunchKernelGGL(k_selective_walk, dim3(d.B, (unsigned)(((size_t)C * N + 255) / 256)), dim3(256), 0, st, a_log, S, ws, \
                         wdt, C, N, pc, d);                                                                                   \
      SEL_LAUNCH_(NS_, R_, FROM, plan.slots);                                                                            \
    }                                                                                                                    \
  } while (0)
  SEQ_DISPATCH_T(code, {
    if (seq_selective_rows(d.Ttot, d.B, C, N, ldx, ldz, ldb, ldc, ldo))
      hipLaunchKernelGGL((k_selective_row<T>), dim3((C + 15) / 16, d.B), dim3(256), 0, st, (const T*)x, ldx, dtp, dtb, (const T*)b, ldb,
                         (const T*)c, ldc, a_log, dskip, (const T*)z, ldz, S, (T*)out, ldo, scale, C, N, d);
    else if (N <= 16)
      SEL_LAUNCH(4, 4);
    else if (N <= 32)
      SEL_LAUNCH(4, 8);
    else if (N <= 64)
      SEL_LAUNCH(4, 16);
    else if (N <= 128)
      SEL_LAUNCH(8, 16);
    else
      SEL_LAUNCH(16, 16);
  });
#undef SEL_LAUNCH
#undef SEL_LAUNCH_
  LIPA_CHECK_LAUNCH();
}

void seq_gla_scan(int code, const void* q, int ldq, const void* k, int ldk, const void* v, int ldv, const float* z,
                  const float* zb, float inv_tau, float qscale, float* S, float* out, int H, int dk, int dv, SeqDesc d,
                  hipStream_t st) {
  if (d.B == 0) return;
#define GLA_LAUNCH(RR_, R_)                                                                                              \
  hipLaunchKernelGGL((k_gla_scan<T, RR_, R_>), dim3(d.B * H, (dv + 256 / R_ * CC - 1) / (256 / R_ * CC)), dim3(256), 0, st, \
                     (const T*)q, ldq, (const T*)k, ldk, (const T*)v, ldv, z, zb, inv_tau, qscale, S, out, H, dk, dv, d)
  SEQ_DISPATCH_T(code, {
    if (dk <= 16)
      GLA_LAUNCH(4, 4);
    else if (dk <= 32)
      GLA_LAUNCH(4, 8);
    else if (dk <= 64)
      GLA_LAUNCH(4, 16);
    else if (dk <= 128)
      GLA_LAUNCH(8, 16);
    else
      GLA_LAUNCH(16, 16);
  });
#undef GLA_LAUNCH
  LIPA_CHECK_LAUNCH();
}
