// W4A16 GEMM for decode batches and short prefills (the AWQ / GPTQ / RTN int4 serving
// artifact of Quantization/LoRA-AWQ and Deployment/litellm-proxy/docker-compose-router-lb.yaml:85):
//     y[M, N] = x[M, K] · deq(W)ᵀ (+ residual),   M <= 64,   deq(W)[n, k] = q·s[n, g] + b[n, g]
// with W as 4-bit codes (uint8 [N, K/2], high nibble = even k) and one fp32 (scale, bias = −zero·scale)
// per (row, 128·j-deep group).
//
// At these M the cost is streaming W once (N·K/2 bytes), so the design is about bytes in flight and
// a cheap dequant, with the matrix cores doing the arithmetic:
//  * grid = (N/128 column spans) × (KS K-slices); a 256-thread workgroup owns 128 columns × 128·NKB
//    of K, each wave 32 columns (two 16-column MFMA tiles); every code (16 B per lane per tile and
//    128-deep block) and scale of the wave's whole slice is loaded up front — 4-16 KB per wave in
//    flight, the whole matrix in flight across the chip;
//  * dequant in 7 VALU per 8 weights and no conversion: a nibble q becomes the bf16 bit pattern
//    0x4300|q = 128+q by a byte permute (v_perm with a 0x43 byte plane), so the MFMA accumulates
//    G = Σ x·(128+q) per group; X = Σ x per (row, group) is reduced once while x is staged, and the
//    group folds as y += s·G + (b − 128·s)·X — scale and zero point never touch the weights;
//  * the permute yields the lane's 8 weights in k order (1,3,5,7,0,2,4,6); x is staged once per
//    workgroup into LDS (M × 128·NKB, 16-B padded rows: conflict-free ds_read_b128) in the same
//    order, so every A/B k-slot pair matches (the MFMA sum is order-free);
//  * v_mfma_f32_16x16x32_bf16 with x as A (rows = tokens, 16 per tile, RT tiles) and the codes as B;
//    the lane's B column is its load column, so its output column needs just its own (s, c) pair;
//  * KS > 1: fp32 partials [KS, M, N] + one reduce launch (the residual folds there); KS = 1 writes
//    bf16 directly.  XCD-aware block order: the column spans of one K-slice (same x slice) share an
//    L2.
#include "common.h"

using namespace lipa;

namespace {

constexpr int W4_CT = 2;                      // 16-column MFMA tiles per wave
constexpr int W4_COLS = 4 * 16 * W4_CT;       // columns per workgroup

__device__ __forceinline__ uint32_t vperm(uint32_t hi, uint32_t lo, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}

// one code dword (k = 0..7; byte i = q[2i] << 4 | q[2i+1]) → four bf16 pairs of 128+q in k order
// (1,3) (5,7) (0,2) (4,6)
__device__ __forceinline__ bf16x8 i4_bf16(uint32_t w) {
  constexpr uint32_t C = 0x43434343u;
  const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
  u32x4 o;
  o[0] = vperm(C, lo, 0x04010400u);
  o[1] = vperm(C, lo, 0x04030402u);
  o[2] = vperm(C, hi, 0x04010400u);
  o[3] = vperm(C, hi, 0x04030402u);
  return __builtin_bit_cast(bf16x8, o);
}

// 8 bf16 of x in k order → the same (1,3,5,7,0,2,4,6) order
__device__ __forceinline__ u32x4 x_perm(u32x4 d) {
  u32x4 o;
  o[0] = vperm(d[1], d[0], 0x07060302u);
  o[1] = vperm(d[3], d[2], 0x07060302u);
  o[2] = vperm(d[1], d[0], 0x05040100u);
  o[3] = vperm(d[3], d[2], 0x05040100u);
  return o;
}

template <int RT, int NKB>
__global__ __launch_bounds__(256) void w4mm_k(const bf16* __restrict__ X, int ldx, const uint8_t* __restrict__ codes,
                                              const float2* __restrict__ sc, int gs, const bf16* __restrict__ residual,
                                              bf16* __restrict__ out, float* __restrict__ part, int M, int N, int K,
                                              int ncs) {
  constexpr int KR = 128 * NKB;           // K per workgroup
  constexpr int LDXS = KR + 8;            // LDS row stride (bf16): 16-B pad
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];
  bf16* xs = reinterpret_cast<bf16*>(lds_raw);
  const int KS = gridDim.x / ncs;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int cs = id % ncs, ks = id / ncs;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, li = lane & 15, q = lane >> 4;
  const int k0 = ks * KR;
  const int G = K / gs;

  // 1) the wave's codes and (scale, c) pairs for the whole K slice, all in flight at once
  u32x4 cq[NKB][W4_CT];
  float2 s2[NKB][W4_CT];
  int ncol[W4_CT];
#pragma unroll
  for (int ct = 0; ct < W4_CT; ++ct) ncol[ct] = min(cs * W4_COLS + 32 * w + 16 * ct + li, N - 1);
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
    for (int ct = 0; ct < W4_CT; ++ct) {
      const int kk = k0 + 128 * kb;
      cq[kb][ct] = *reinterpret_cast<const u32x4*>(codes + (size_t)ncol[ct] * (K / 2) + (kk + 32 * q) / 2);
      s2[kb][ct] = sc[(size_t)ncol[ct] * G + kk / gs];
    }

  // 2) x slice → LDS, permuted to the dequant's k order; rows >= M are zero.  The 16 lanes that hold one
  //    128-deep group of a row also reduce its sum Σx (xsum[kb][row], fp32) for the group fold
  constexpr int CH = KR / 8;              // 16-B chunks per row (a multiple of 16)
  constexpr int RWS = RT * 16;
  float* xsum = reinterpret_cast<float*>(lds_raw + (size_t)RWS * LDXS * 2);
  for (int c = tid; c < RWS * CH; c += 256) {
    const int r = c / CH, kc = c - r * CH;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (r < M) v = *reinterpret_cast<const u32x4*>(X + (size_t)r * ldx + k0 + 8 * kc);
    const bf16x8 xb = __builtin_bit_cast(bf16x8, v);
    float t = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) t += (float)xb[e];
    t += __shfl_xor(t, 1, 64);
    t += __shfl_xor(t, 2, 64);
    t += __shfl_xor(t, 4, 64);
    t += __shfl_xor(t, 8, 64);
    if ((kc & 15) == 0) xsum[(kc >> 4) * RWS + r] = t;
    *reinterpret_cast<u32x4*>(xs + r * LDXS + 8 * kc) = x_perm(v);
  }
  __syncthreads();

  f32x4 acc[W4_CT][RT];
#pragma unroll
  for (int ct = 0; ct < W4_CT; ++ct)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[ct][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int kb = 0; kb < NKB; ++kb) {
    bf16x8 bq[W4_CT][4];
#pragma unroll
    for (int ct = 0; ct < W4_CT; ++ct)
#pragma unroll
      for (int j = 0; j < 4; ++j) bq[ct][j] = i4_bf16(cq[kb][ct][j]);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      bf16x8 xa[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xa[j] = *reinterpret_cast<const bf16x8*>(xs + (16 * rt + li) * LDXS + 128 * kb + 32 * q + 8 * j);
      const f32x4 ax = *reinterpret_cast<const f32x4*>(xsum + kb * RWS + 16 * rt + 4 * q);   // Σx of rows 4q..4q+3
#pragma unroll
      for (int ct = 0; ct < W4_CT; ++ct) {
        f32x4 g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[0], bq[ct][0], zero, 0, 0, 0);
#pragma unroll
        for (int j = 1; j < 4; ++j) g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[j], bq[ct][j], g, 0, 0, 0);
        const float s = s2[kb][ct].x, cc = s2[kb][ct].y;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[ct][rt][i] = fmaf(s, g[i], fmaf(cc, ax[i], acc[ct][rt][i]));
      }
    }
  }

  // 3) lane holds y[m = 16·rt + 4q + i][n = its load column]
#pragma unroll
  for (int ct = 0; ct < W4_CT; ++ct) {
    const int n = cs * W4_COLS + 32 * w + 16 * ct + li;
    if (n >= N) continue;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = 16 * rt + 4 * q + i;
        if (m >= M) continue;
        if (KS == 1) {
          float v = acc[ct][rt][i];
          if (residual) v += (float)residual[(size_t)m * N + n];
          out[(size_t)m * N + n] = (bf16)v;
        } else {
          part[((size_t)ks * M + m) * N + n] = acc[ct][rt][i];
        }
      }
  }
}

// out[m, n] = Σ_s part[s, m, n] (+ residual) → bf16; 2 outputs per thread and every slice's load issued
// before the adds (the grid is small at decode sizes — M·N/512 workgroups — so each thread's slice loads
// must overlap, not run as KS dependent round trips)
template <int SU>
__global__ __launch_bounds__(256) void w4mm_reduce_k(const float* __restrict__ part, const bf16* __restrict__ res,
                                                     bf16* __restrict__ out, int S, size_t MN) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 2;
  if (i >= MN) return;
  float2 v = {0.f, 0.f};
  for (int s0 = 0; s0 < S; s0 += SU) {
    float2 t[SU];
#pragma unroll
    for (int u = 0; u < SU; ++u)
      t[u] = s0 + u < S ? *reinterpret_cast<const float2*>(part + (size_t)(s0 + u) * MN + i) : float2{0.f, 0.f};
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      v.x += t[u].x;
      v.y += t[u].y;
    }
  }
  if (res) {
    v.x += (float)res[i];
    v.y += (float)res[i + 1];
  }
  bf16x2 o = {(bf16)v.x, (bf16)v.y};
  *reinterpret_cast<bf16x2*>(out + i) = o;
}

// ============================================================================ w4row: M <= 32, one launch
// w4mm's slices and sums with all of K in one workgroup: it owns 16·CT columns at a time, its waves take the 128·NKB-deep slices, and
// the slices' tiles meet in LDS, added in order — the bits of w4mm and its reduce without the second launch, and with the
// residual or SwiGLU (GLU: CT/2 gate and CT/2 up tiles of W [2N, K], products rounded to bf16 first) in the end.
//  * as many waves as slices (long K: w4long_k).  A wave keeps its slice of x in MFMA order, with its sums, in registers and walks column tiles:
//    x is read once per workgroup, not per 16 columns.
//  * codes and their scales come by LDS-DMA, a unit (16 columns × the slice) a slot of a ring that belongs to one wave: whole pieces of 256
//    B of a row, no register, and no wait but the wave's own.  As operands straight from memory (16 rows × 64 B and 16 times
//    a scale an instruction, half of them scales) a wave stood 3 µs in front of its first products until the loads were taken, and as long
//    again at each tile.  µs, 12 rows, W cold: 24576 × 4096 ended in SwiGLU 20.4 → 16.4 (3.5 TB/s), 6144 × 4096 10.2 → 8.2, 4096 × 4096 8.3 →
//    6.5 (1.7 of them the launch), 2 × 9728 × 2560 in SwiGLU 13.2 → 12.1, 2 × 3072 × 1024 5.8 → 5.4; 24 rows of 24576 × 4096 24.2 → 19.4.
//  * x comes in whole rows of 256 B and turns through LDS, in the place of units that are not on their way yet (as fragments straight from
//    memory, 64 lines a load, the 16 rows of 4096 x 12288 took 20 µs, not 16).  Rows past M repeat row M - 1 and are not stored.
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __amdgpu_buffer_rsrc_t rsrc;

__device__ __forceinline__ rsrc window(const void* base, uint32_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p), hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}
// 64 lanes x 16 (4) bytes from memory into LDS [dst, ..), lane after lane; M0 is put back
__device__ __forceinline__ void to_lds16(const rsrc& rs, uint32_t dst, uint32_t voff, uint32_t soff) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(dst), "v"(voff), "s"(rs), "s"(soff) : "memory");
}
__device__ __forceinline__ void to_lds4(const rsrc& rs, uint32_t dst, uint32_t voff, uint32_t soff) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dword %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(dst), "v"(voff), "s"(rs), "s"(soff) : "memory");
}
// until at most n of a wave's loads are on their way, n rounded down to a multiple of S, or to R · S
template <int S, int R>
__device__ __forceinline__ void wait_loads(int n) {
  if constexpr (R == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    if (n >= R * S)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R * S) : "memory");
    else
      wait_loads<S, R - 1>(n);
  }
}
// Σ of a row over its four lanes (li + 16 q), the rows 4 q .. 4 q + 3 of them in every lane of q
template <int I>
__device__ __forceinline__ float row_sum_of(float v) {
  const int x = __float_as_int(v);
  int r = __builtin_amdgcn_update_dpp(0, x, 0x150 + I, 0x1, 0xF, false);         // row_newbcast, each into its own row of lanes
  r = __builtin_amdgcn_update_dpp(r, x, 0x154 + I, 0x2, 0xF, false);
  r = __builtin_amdgcn_update_dpp(r, x, 0x158 + I, 0x4, 0xF, false);
  return __int_as_float(__builtin_amdgcn_update_dpp(r, x, 0x15C + I, 0x8, 0xF, false));
}
__device__ __forceinline__ f32x4 rows_sums(float v) {
  const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
  const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
  return f32x4{row_sum_of<0>(v), row_sum_of<1>(v), row_sum_of<2>(v), row_sum_of<3>(v)};
}
// codes: chunk c (16 B) of row r of a slice stands in this slot of the row, so that 16 rows of a column of chunks meet every bank once
template <int NKB>
__device__ __forceinline__ int turned(int c, int r) { return NKB == 4 ? c ^ (r & 15) : c ^ ((r >> 1) & 7); }
// a barrier that leaves loads on their way (a fence would wait for them)
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

constexpr int W4_SLICES = 32;                  // of w4long_k, 1 KB of sums each

template <int RT, int NKB, int CT, bool GLU, bool RES>
__global__ __launch_bounds__(NKB == 2 ? 1024 : 512) void w4row_k(const bf16* __restrict__ X, int ldx, const uint8_t* __restrict__ codes,
                                                                        const float2* __restrict__ sc, int gs, const bf16* __restrict__ residual,
                                                                        bf16* __restrict__ out, int M, int N, int K) {
  constexpr int WAVES = NKB == 2 ? 16 : 8, CO = GLU ? CT / 2 : CT, TILE = CT * RT * 256;       // TILE: floats of one slice's sums
  constexpr int UB = NKB * (1024 + 128), LOADS = NKB + NKB / 2;              // a unit: bytes of codes and of scales, the loads that bring it
  constexpr int LDS = 160 * 1024, SUMS = WAVES * TILE * 4;
  constexpr int RING = WAVES * 4 * UB + SUMS <= LDS ? 4 : 3;
  constexpr int TURN = NKB / 2;                                             // 128-deep blocks of x that turn at once
  constexpr int OWN = RING * UB;                                             // a wave's share of LDS
  constexpr int FIRST = (RING * UB - TURN * 4096) / UB;                      // units on their way while x turns
  constexpr bool TWICE = WAVES * OWN + 2 * SUMS <= LDS;               // two places for the sums
  static_assert(FIRST >= 1 && RING * LOADS < 64, "ring");
  __shared__ __attribute__((aligned(1024))) char smem[WAVES * OWN + (TWICE ? 2 : 1) * SUMS];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, q = lane >> 4;
  // (blockDim and gridDim where they are used are loads, which are waited for with all that is on its way)
  const int KS = K / (128 * NKB), G = K / gs, nt = N / (16 * CO), per = gs / 128;
  const int nw = __builtin_amdgcn_readfirstlane(KS), blocks = __builtin_amdgcn_readfirstlane(gridDim.x);
  char* own = smem + w * OWN;
  char* xw = own + FIRST * UB;
  char* sums = smem + WAVES * OWN;
  const uint32_t ring = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)smem) + w * OWN;
  const uint32_t row_bytes = (uint32_t)K / 2, rows_w = (uint32_t)(GLU ? 2 * N : N);
  const rsrc rc = window(codes, rows_w * row_bytes), rs = window(sc, rows_w * (uint32_t)G * 8u);
  constexpr int CH = 4 * NKB;                    // chunks of a row
  uint32_t vc[NKB];
#pragma unroll
  for (int i = 0; i < NKB; ++i) {
    const int r = i * (64 / CH) + lane / CH;
    vc[i] = r * row_bytes + 16 * turned<NKB>(lane % CH, r);
  }
  // scales: (scale, c) of block b of row r at dword (r · NKB + b) · 2
  const int sr = lane / (2 * NKB), sb = lane % (2 * NKB) >> 1;
  auto fill = [&](int slot, int tile, int ct, int slice) {
    const uint32_t dst = ring + slot * UB, n0 = (GLU && ct >= CO ? N : 0) + tile * 16 * CO + 16 * (ct % CO);
#pragma unroll
    for (int i = 0; i < NKB; ++i) to_lds16(rc, dst + i * 1024, vc[i], n0 * row_bytes + slice * 64 * NKB);
#pragma unroll
    for (int i = 0; i < NKB / 2; ++i)
      to_lds4(rs, dst + NKB * 1024 + i * 256,
              ((uint32_t)(sr + i * (32 / NKB)) * G + (uint32_t)(slice * NKB + sb) / (uint32_t)per) * 8u + 4u * (lane & 1), n0 * (uint32_t)G * 8u);
  };
  struct Rows {
    u32x4 x[NKB][RT][4];
  };
  auto load_rows = [&](Rows& s, int slice) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const bf16* xp = X + (size_t)min(16 * rt + 4 * p + q, M - 1) * ldx + slice * 128 * NKB + 8 * li;
#pragma unroll
        for (int b = 0; b < NKB; ++b) s.x[b][rt][p] = *reinterpret_cast<const u32x4*>(xp + 128 * b);
      }
  };
  bf16x8 xa[NKB][RT][4];
  f32x4 ax[NKB][RT];                             // Σx of rows 4q .. 4q+3
  auto turn = [&](const Rows& s) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int b0 = 0; b0 < NKB; b0 += TURN) {
        asm volatile("" ::: "memory");           // (a wave's LDS accesses are in order)
#pragma unroll
        for (int b = 0; b < TURN; ++b)
#pragma unroll
          for (int p = 0; p < 4; ++p)
            *reinterpret_cast<u32x4*>(xw + 4096 * b + (4 * p + q) * 256 + 16 * (li ^ (4 * p + q))) = s.x[b0 + b][rt][p];
        asm volatile("" ::: "memory");
#pragma unroll
        for (int b = 0; b < TURN; ++b) {
          float t[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const u32x4 d = *reinterpret_cast<const u32x4*>(xw + 4096 * b + li * 256 + 16 * ((4 * q + j) ^ li));
            const bf16x8 v = __builtin_bit_cast(bf16x8, d);
            t[j] = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) t[j] += (float)v[e];
            xa[b0 + b][rt][j] = __builtin_bit_cast(bf16x8, x_perm(d));
          }
          ax[b0 + b][rt] = rows_sums((t[0] + t[1]) + (t[2] + t[3]));         // (the pairs of w4mm_k's staging: same bits)
        }
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");               // (units take the place of what has been read)
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // the unit in a slot times the slice of x in registers; next() may fill the slot again
  auto multiply = [&](int slot, f32x4 (&acc)[RT], auto next) {
    const char* p = own + slot * UB;
    u32x4 c[NKB];
    f32x4 s[NKB / 2];
#pragma unroll
    for (int b = 0; b < NKB; ++b) c[b] = *reinterpret_cast<const u32x4*>(p + li * (64 * NKB) + 16 * turned<NKB>(4 * b + q, li));
#pragma unroll
    for (int b = 0; b < NKB / 2; ++b) s[b] = *reinterpret_cast<const f32x4*>(p + NKB * 1024 + (li * NKB + 2 * b) * 8);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    next();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt] = zero;
#pragma unroll
    for (int b = 0; b < NKB; ++b) {
      bf16x8 bq[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) bq[j] = i4_bf16(c[b][j]);
      const float sv = s[b >> 1][2 * (b & 1)], cc = s[b >> 1][2 * (b & 1) + 1];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        f32x4 g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[b][rt][0], bq[0], zero, 0, 0, 0);
#pragma unroll
        for (int j = 1; j < 4; ++j) g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[b][rt][j], bq[j], g, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rt][i] = fmaf(sv, g[i], fmaf(cc, ax[b][rt][i], acc[rt][i]));
      }
    }
  };
  auto row_of = [&](int e) { return 16 * ((e >> 8) % RT) + 4 * ((e >> 6) & 3) + (e & 3); };       // element e: y[m = 16·rt + 4q + i][its column]
  auto col_of = [&](int e, int tile) { return tile * 16 * CO + 16 * ((e >> 8) / RT) + ((e >> 2) & 15); };
  // a thread's first residual, on its way under the products
  const int e0 = min(tid, CO * RT * 256 - 1);
  auto first_residual = [&](int tile) -> unsigned {
    return RES ? __builtin_bit_cast(unsigned short, residual[(size_t)min(row_of(e0), M - 1) * N + col_of(e0, tile)]) : 0u;
  };
  auto finish = [&](const char* from, int tile, unsigned res) {
    const float* rf = reinterpret_cast<const float*>(from);
    for (int e = tid; e < CO * RT * 256; e += 64 * nw) {
      float v = 0.f, up = 0.f;
#pragma unroll 8
      for (int s = 0; s < KS; ++s) {
        v += rf[s * TILE + e];
        if (GLU) up += rf[s * TILE + CO * RT * 256 + e];
      }
      if (row_of(e) >= M) continue;
      const size_t at = (size_t)row_of(e) * N + col_of(e, tile);
      if (GLU) {
        const float gt = (float)(bf16)v, ut = (float)(bf16)up;
        v = gt / (1.f + __expf(-gt)) * ut;
      } else if (RES) {
        v += e == tid ? __uint_as_float(res << 16) : (float)residual[at];
      }
      out[at] = (bf16)v;
    }
  };
  auto leave = [&](char* to, int ct, const f32x4 (&acc)[RT]) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) *reinterpret_cast<f32x4*>(to + ((ct * RT + rt) * 64 + lane) * 16) = acc[rt];
  };
  const int b0 = blockIdx.x, cnt = (nt - b0 + blocks - 1) / blocks * CT;         // units of this wave
  int fu = 0, ft = b0, fs = 0;                                                   // the next one to come, its tile and slot
  auto fill_next = [&] {
    if (fu >= cnt) return;
    fill(fs, ft, CT == 1 ? 0 : fu % CT, w);
    if (CT == 1 || fu % CT == CT - 1) ft += blocks;
    ++fu;
    fs = fs + 1 == RING ? 0 : fs + 1;
  };
  {
    Rows x;
    load_rows(x, w);
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));                        // vmcnt(0): what the compiler counts has come
#pragma unroll
    for (int i = 0; i < FIRST; ++i) fill_next();
    turn(x);
  }
#pragma unroll
  for (int i = FIRST; i < RING; ++i) fill_next();
  int u = 0, slot = 0, buf = 0;
  for (int tile = b0; tile < nt; tile += blocks) {
    const unsigned res = first_residual(tile);
    char* to = sums + buf * SUMS;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct, ++u) {
      f32x4 acc[RT];
      wait_loads<LOADS, RING - 1>((cnt - 1 - u) * LOADS);
      multiply(slot, acc, fill_next);
      slot = slot + 1 == RING ? 0 : slot + 1;
      leave(to + w * TILE * 4, ct, acc);
    }
    lds_barrier();
    finish(to, tile, res);
    if (TWICE)
      buf ^= 1;                                // (the other place is read before the next of these barriers)
    else if (tile + blocks < nt)
      lds_barrier();
  }
}

// The same sums for long K and up to 16 rows: 12 waves take the slices of one tile in turns.  x comes by LDS-DMA too, 128-deep blocks in a
// ring of two (XI: loads of four rows each, as many as M needs); a slice's codes and scales wait in LDS until the wave takes them all into
// registers and the next slice's follow.  4096 x 12288, 12 rows: 16.5 -> 13.1 µs, x through registers, a slice of it on its way, against
// this.  Bound by what a workgroup does with x beside its one tile (24 slices of its sums, 80 of 160 vector instructions a block) and by the
// address unit; 8 waves took 14.8, blocks of codes and scales brought one by one 14.1.
template <int NKB, int XI>
__global__ __launch_bounds__(XI == 4 ? 640 : 768) void w4long_k(const bf16* __restrict__ X, int ldx, const uint8_t* __restrict__ codes,
                                                const float2* __restrict__ sc, int gs, const bf16* __restrict__ residual,
                                                bf16* __restrict__ out, int M, int N, int K) {
  constexpr int WAVES = XI == 4 ? 10 : 12, RING = 2, XB = 1024 * XI, OWN = RING * XB + NKB * (1024 + 128), CH = 4 * NKB;
  __shared__ __attribute__((aligned(1024))) char smem[WAVES * OWN + W4_SLICES * 1024];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, q = lane >> 4, tile = blockIdx.x;
  const int KS = K / (128 * NKB), G = K / gs, per = gs / 128;
  const int m = 4 * ((tid >> 6) & 3) + (tid & 3), n = tile * 16 + ((tid >> 2) & 15);            // y[m][n] is this thread's to finish
  float* sums = reinterpret_cast<float*>(smem + WAVES * OWN);
  float res = 0.f;
  if (residual != nullptr) res = (float)residual[(size_t)min(m, M - 1) * N + n];
  const char* own = smem + w * OWN;
  const uint32_t xs = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr)smem) + w * OWN, cs = xs + RING * XB;
  const uint32_t row_bytes = (uint32_t)K / 2, n0 = (uint32_t)tile * 16;
  const rsrc rx = window(X, ((uint32_t)(M - 1) * (uint32_t)ldx + (uint32_t)K) * 2u), rc = window(codes, (uint32_t)N * row_bytes),
             rs = window(sc, (uint32_t)N * (uint32_t)G * 8u);
  uint32_t vx[XI], vc[NKB];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = 4 * i + q;
    vx[i] = (uint32_t)min(r, M - 1) * (uint32_t)ldx * 2u + 16 * (li ^ r);
  }
#pragma unroll
  for (int i = 0; i < NKB; ++i) {
    const int r = i * (64 / CH) + lane / CH;
    vc[i] = r * row_bytes + 16 * turned<NKB>(lane % CH, r);
  }
  auto fill_x = [&](int place, int block) {
#pragma unroll
    for (int i = 0; i < XI; ++i) to_lds16(rx, xs + place * XB + i * 1024, vx[i], block * 256);
  };
  // a slice's scales, NKB a row: by 16 (8 ..) bytes where its groups are neighbours
  const bool wide = NKB == 4 && per == 1 && G % 2 == 0 && ((uintptr_t)sc & 15) == 0;
  const uint32_t vs = wide ? (uint32_t)((lane >> 1) & 15) * G * 8u + 16 * (lane & 1) : 4u * (lane & 1);
  const int sr = lane / (2 * NKB), sb = lane % (2 * NKB) >> 1;
  constexpr int SCALES = NKB / 2;                // loads of them (wide: the second one is left out, and one counted too many)
  auto fill_codes = [&](int slice) {
#pragma unroll
    for (int i = 0; i < NKB; ++i) to_lds16(rc, cs + i * 1024, vc[i], n0 * row_bytes + slice * 64 * NKB);
    if (wide) {
      const uint32_t dst = __builtin_amdgcn_readfirstlane(cs + NKB * 1024);        // (an address kept in a vector register has no place in M0)
      if (lane < 32) to_lds16(rs, dst, vs, (n0 * G + slice * NKB) * 8u);
    } else {
#pragma unroll
      for (int i = 0; i < SCALES; ++i)
        to_lds4(rs, cs + NKB * 1024 + i * 256, ((uint32_t)(sr + i * (32 / NKB)) * G + (uint32_t)(slice * NKB + sb) / (uint32_t)per) * 8u + vs,
                n0 * (uint32_t)G * 8u);
    }
  };
  constexpr int C = NKB + 1;                     // (the fewest loads that bring a slice's codes)
  if (w < KS) {
    fill_codes(w);
    fill_x(0, w * NKB);
    fill_x(1, w * NKB + 1);
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int slice = w; slice < KS; slice += WAVES) {
    const int next = slice + WAVES;
    const bool more = next < KS;
    if (slice == w || NKB == RING) wait_loads<RING * XI, 1>(RING * XI);         // (later ones are older than x that has been waited for)
    u32x4 c[NKB];
    f32x4 s[NKB / 2];
#pragma unroll
    for (int b = 0; b < NKB; ++b) c[b] = *reinterpret_cast<const u32x4*>(own + RING * XB + li * (64 * NKB) + 16 * turned<NKB>(4 * b + q, li));
#pragma unroll
    for (int b = 0; b < NKB / 2; ++b) s[b] = *reinterpret_cast<const f32x4*>(own + RING * XB + NKB * 1024 + (li * NKB + 2 * b) * 8);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (more) fill_codes(next);
    f32x4 acc = zero;
#pragma unroll
    for (int b = 0; b < NKB; ++b) {
      // younger: the next block of x, and the next slice's codes where they went out behind this one
      if (more) {
        if (b < RING) wait_loads<XI + C, 1>(XI + C); else wait_loads<XI, 1>(XI);
      } else if (b < NKB - 1) {
        wait_loads<XI, 1>(XI);
      } else {
        wait_loads<1, 0>(0);
      }
      const char* p = own + b % RING * XB;
      u32x4 d[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = *reinterpret_cast<const u32x4*>(p + min(li, 4 * XI - 1) * 256 + 16 * ((4 * q + j) ^ min(li, 4 * XI - 1)));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (b + RING < NKB)
        fill_x(b % RING, slice * NKB + b + RING);
      else if (more)
        fill_x(b % RING, next * NKB + b + RING - NKB);
      float t[4];
      f32x4 g = zero;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bf16x8 v = __builtin_bit_cast(bf16x8, d[j]);
        t[j] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) t[j] += (float)v[e];
        g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x_perm(d[j])), i4_bf16(c[b][j]), g, 0, 0, 0);
      }
      const f32x4 ax = rows_sums((t[0] + t[1]) + (t[2] + t[3]));
      const float sv = s[b >> 1][2 * (b & 1)], cc = s[b >> 1][2 * (b & 1) + 1];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(sv, g[i], fmaf(cc, ax[i], acc[i]));
    }
    *reinterpret_cast<f32x4*>(sums + slice * 256 + lane * 4) = acc;
  }
  __syncthreads();
  if (tid >= 256 || m >= M) return;
  float v = 0.f;
#pragma unroll 8
  for (int s = 0; s < KS; ++s) v += sums[s * 256 + tid];
  if (residual != nullptr) v += res;
  out[(size_t)m * N + n] = (bf16)v;
}

// ============================================================================ w4g: 32 < M <= 64
// The same dequant and group fold, tiled for decode batches: a workgroup owns BM = 16·RT rows × BN = 64·CT
// columns (4 waves × 16·CT, each wave every row) over a K slice of nkb 128-deep blocks.  x is streamed per
// block through a double-buffered LDS tile (permuted to the dequant's k order), x, the codes and (scale, c)
// pairs PD blocks ahead in a register ring — so x crosses L2→LDS once per column span (not once per K-slice × span
// as in w4mm), each code dword feeds RT MFMAs, and PD·CT·16 B per lane of codes stay in flight.  Σx per (row,
// block) for the zero-point fold is one more MFMA chain against a ones operand (no cross-lane reduction).
// Split-K (KS > 1) writes fp32 partials for w4mm_reduce_k.  Measured (profiles/r5/w4g_decode.txt): ahead of
// w4mm and gemm4w W4=2 on the Qwen3-8B projections at M = 33..64; at M = 128 / 256 gemm4w W4=2 wins (the
// per-block fold and x restaging scale with the rows), and prefetching 3 blocks instead of 2 loses.
template <int RT, int CT, int PD>
__global__ __launch_bounds__(256, 2) void w4g_k(const bf16* __restrict__ X, int ldx, const uint8_t* __restrict__ codes,
                                                const float2* __restrict__ sc, int gs, const bf16* __restrict__ residual,
                                                bf16* __restrict__ out, float* __restrict__ part, int M, int N, int K,
                                                int ncs, int nrb, int nkb) {
  constexpr int BM = 16 * RT, LDXS = 128 + 8;   // 272-B rows: the 16 rows of a ds_read_b128 group hit distinct banks
  constexpr int NR = PD + 1;                    // code ring depth
  __shared__ __attribute__((aligned(16))) bf16 xs[2][BM * LDXS];
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int cs = id % ncs, rb = (id / ncs) % nrb, ks = id / (ncs * nrb);
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, li = lane & 15, q = lane >> 4;
  const int m0 = rb * BM, kb0 = ks * nkb;
  const int G = K / gs;
  const uint8_t* cp[CT];
  const float2* sp[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int n = cs * (64 * CT) + 16 * CT * w + 16 * ct + li;
    cp[ct] = codes + (size_t)n * (K / 2) + 16 * q;
    sp[ct] = sc + (size_t)n * G;
  }

  u32x4 cq[NR][CT];
  float2 s2[NR][CT];
  auto load_codes = [&](int set, int kb) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      cq[set][ct] = *reinterpret_cast<const u32x4*>(cp[ct] + (size_t)kb * 64);
      s2[set][ct] = sp[ct][kb * 128 / gs];
    }
  };
  // x block: BM rows × 16 chunks of 16 B, RT chunks per thread, in the same ring as the codes
  u32x4 xr[NR][RT];
  auto load_x = [&](int set, int kb) {
#pragma unroll
    for (int p = 0; p < RT; ++p) {
      const int r = 16 * p + (tid >> 4), kc = tid & 15;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (m0 + r < M) v = *reinterpret_cast<const u32x4*>(X + (size_t)(m0 + r) * ldx + kb * 128 + 8 * kc);
      xr[set][p] = v;
    }
  };
  auto store_x = [&](int set, int buf) {
#pragma unroll
    for (int p = 0; p < RT; ++p) {
      const int r = 16 * p + (tid >> 4), kc = tid & 15;
      *reinterpret_cast<u32x4*>(xs[buf] + r * LDXS + 8 * kc) = x_perm(xr[set][p]);
    }
  };

  f32x4 acc[CT][RT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[ct][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (bf16)1.f;

  // blocks 0..PD-1 in flight; block 0's x staged
#pragma unroll
  for (int d = 0; d < PD; ++d)
    if (d < nkb) {
      load_codes(d, kb0 + d);
      load_x(d, kb0 + d);
    }
  store_x(0, 0);
  __syncthreads();
  for (int i0 = 0; i0 < nkb; i0 += NR) {
#pragma unroll
    for (int u = 0; u < NR; ++u) {   // static ring slot u = block i % NR
      const int i = i0 + u;
      if (i >= nkb) break;
      if (i + PD < nkb) {
        load_codes((u + PD) % NR, kb0 + i + PD);
        load_x((u + PD) % NR, kb0 + i + PD);
      }
      const int buf = i & 1;
      bf16x8 bq[CT][4];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j) bq[ct][j] = i4_bf16(cq[u][ct][j]);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        bf16x8 xa[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          xa[j] = *reinterpret_cast<const bf16x8*>(xs[buf] + (16 * rt + li) * LDXS + 32 * q + 8 * j);
        f32x4 ax = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[0], ones, zero, 0, 0, 0);   // Σx, rows 4q..4q+3
#pragma unroll
        for (int j = 1; j < 4; ++j) ax = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[j], ones, ax, 0, 0, 0);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          f32x4 g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[0], bq[ct][0], zero, 0, 0, 0);
#pragma unroll
          for (int j = 1; j < 4; ++j) g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[j], bq[ct][j], g, 0, 0, 0);
          const float sv = s2[u][ct].x, c = s2[u][ct].y;
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[ct][rt][e] = fmaf(sv, g[e], fmaf(c, ax[e], acc[ct][rt][e]));
        }
      }
      if (i + 1 < nkb) store_x((u + 1) % NR, buf ^ 1);   // block i+1 (loaded PD-1 blocks ago) into the buffer block i-1 used
      __syncthreads();
    }
  }
  // lane holds y[m = m0 + 16·rt + 4q + e][n]
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + 16 * rt + 4 * q + e, n = cs * (64 * CT) + 16 * CT * w + 16 * ct + li;
        if (m >= M) continue;
        if (!part) {
          float v = acc[ct][rt][e];
          if (residual) v += (float)residual[(size_t)m * N + n];
          out[(size_t)m * N + n] = (bf16)v;
        } else {
          part[((size_t)ks * M + m) * N + n] = acc[ct][rt][e];
        }
      }
}

}  // namespace

bool w4g_supported(int M, int N, int K, int gs) {
  return M >= 1 && M <= 64 && N % 128 == 0 && K % 128 == 0 && gs % 128 == 0 && K % gs == 0;
}

// K slices: the fewest (halving the 128-deep blocks per workgroup, at least 2 left) that put >= 256 workgroups
// on the 256 CUs (BN = 128: 32 columns per wave; 64 per wave halves the x re-reads of wide N but spills)
int w4g_splits(int M, int N, int K) {
  const int ncs = N / 128, kb = K / 128;
  int ks = 1;
  while (ncs * ks < 256 && kb % (2 * ks) == 0 && kb / (2 * ks) >= 2) ks *= 2;
  return ks;
}

void launch_w4g(const void* X, int ldx, const uint8_t* codes, const float* sc2, int gs, const void* res, void* out,
                float* part, int M, int N, int K, int ks, hipStream_t st) {
  const int ncs = N / 128, nkb = K / 128 / ks, grid = ncs * ks;
  w4g_k<4, 2, 2><<<grid, 256, 0, st>>>((const bf16*)X, ldx, codes, (const float2*)sc2, gs,
                                       ks > 1 ? nullptr : (const bf16*)res, (bf16*)out, ks > 1 ? part : nullptr, M, N,
                                       K, ncs, 1, nkb);
  if (ks > 1 && out != nullptr) {                        // (without out the slices' sums are left where they are)
    const size_t MN = (size_t)M * N;
    w4mm_reduce_k<8><<<(MN / 2 + 255) / 256, 256, 0, st>>>(part, (const bf16*)res, (bf16*)out, ks, MN);
  }
  LIPA_CHECK_LAUNCH();
}

bool w4mm_supported(int M, int N, int K, int gs) {
  return M >= 1 && M <= 64 && N % W4_COLS == 0 && K % 128 == 0 && gs % 128 == 0 && K % gs == 0;
}

// 128-deep blocks per workgroup (measured per shape at M = 1..64 with the unrolled reduce,
// profiles/r4/w4a16_w4mm_reduce.txt): 4, or 2 for M <= 8 when 4 would leave fewer than 512 workgroups
// (q|k|v, o: more, shorter weight streams win there); 2 / 1 when K allows nothing larger
int w4mm_nkb(int M, int N, int K) {
  const int ncs = N / W4_COLS, kb = K / 128;
  if (kb % 4 == 0 && !(M <= 8 && ncs * (kb / 4) < 512)) return 4;
  return kb % 2 == 0 ? 2 : 1;
}

// Does one launch serve (N: columns of the result)?  Against w4mm_k and its reduce, us in a captured graph at 12 / 24 rows:
// 6144 x 4096 8.4 / 11.6 (13.4 / 17.4), 4096 x 4096 6.7 / 9.5 (11.2 / 14.0), 24576 x 4096 16.0 / 19.8 (27.4 / 37.4; ended in SwiGLU
// 16.8 at 12 rows, but 31.5 at 24, where 32 rows of x and two tiles of sums left the registers).  Where w4mm_k is the better one, us of
// one launch against it:
//  * one workgroup holds all of x: a single slice is a single wave, too few for the codes of 3 tiles or more (28672 x 512, 12 rows, 11.6
//    against 6.9).  32 blocks over few tiles, a chain of 16 waves' sums, are ahead by now (1024 x 4096, 3 rows, 5.3 against 7.2; ended in
//    SwiGLU 6.1, 7.0 at 12) and still left to it.
//  * slices in turns: from the second tile on x is read again (27648 x 5120, 12 rows, 44.5 against 36.4, 5120 x 13824 25.3 against 22.5,
//    5120 x 5120 13.1 against 13.7; one tile each, 4096 x 12288 13.1, 16 rows 14.7 against 18.8, 2560 x 9728 10.4 against 14.0); few tiles of
//    a long K leave the chip idle (1024 x 12288, 16 rows, 12.6 against 11.5; 2048 x 12288, 12 rows, 11.8 against 14.3, 1024 x 8192 8.0
//    against 10.1).
bool w4row_serves(int M, int N, int K, int nkb, bool glu) {
  const int KS = K / (128 * nkb), RT = M <= 16 ? 1 : 2, tiles = N / 16, per = (tiles + 255) / 256;
  const bool one = KS * nkb <= 32;               // (8 waves of 4 blocks or 16 of 2 hold x)
  if (M > (glu ? 16 : 32) || (nkb != 2 && nkb != 4) || ((RT == 2 || glu) && !one) || (!one && KS > W4_SLICES)) return false;
  return one ? (KS > 1 || per < 3) && !(KS * nkb == 32 && tiles < 160 && (glu || nkb == 2)) : per == 1 && (tiles >= 128 || K <= 8192);
}

// One launch of w4row_k, or false where it does not serve (w4mm_k then does).
bool launch_w4row(const void* X, int ldx, const uint8_t* codes, const float* sc2, int gs, const void* res, void* out, int M,
                  int N, int K, int nkb, bool glu, hipStream_t st) {
  if (!w4row_serves(M, N, K, nkb, glu)) return false;
  if (K > 128 * nkb * (nkb == 4 ? 8 : 16) && ((uint64_t)(M - 1) * ldx + K) * 2 > 0xFFFFFFFFull) return false;       // (w4long_k's offsets into x)
  const int KS = K / (128 * nkb), RT = M <= 16 ? 1 : 2, tiles = N / 16;
  const bool one = KS * nkb <= 32;
  const int per = (tiles + 255) / 256, grid = one ? (tiles + per - 1) / per : tiles;   // tiles of a workgroup: even shares
#define L(RT_, NKB_, CT_, GLU_)                                                                                      \
  do {                                                                                                             \
    const auto k = res && !GLU_ ? w4row_k<RT_, NKB_, CT_, GLU_, !GLU_> : w4row_k<RT_, NKB_, CT_, GLU_, false>;      \
    k<<<grid, 64 * KS, 0, st>>>((const bf16*)X, ldx, codes, (const float2*)sc2, gs, (const bf16*)res, (bf16*)out, M, N, K); \
  } while (0)
#define LONG(NKB_, XI_)                                                                                             \
  w4long_k<NKB_, XI_><<<grid, XI_ == 4 ? 640 : 768, 0, st>>>((const bf16*)X, ldx, codes, (const float2*)sc2, gs, (const bf16*)res, (bf16*)out, M, N, K)
  if (one && glu) {
    if (nkb == 4) L(1, 4, 2, true);
    else L(1, 2, 2, true);
  } else if (one && RT == 1) {
    if (nkb == 4) L(1, 4, 1, false);
    else L(1, 2, 1, false);
  } else if (one) {
    if (nkb == 4) L(2, 4, 1, false);
    else L(2, 2, 1, false);
  } else if (nkb == 4) {
    if (M <= 8) LONG(4, 2); else if (M <= 12) LONG(4, 3); else LONG(4, 4);
  } else {
    if (M <= 8) LONG(2, 2); else if (M <= 12) LONG(2, 3); else LONG(2, 4);
  }
#undef LONG
#undef L
  LIPA_CHECK_LAUNCH();
  return true;
}

void launch_w4mm(const void* X, int ldx, const uint8_t* codes, const float* sc2, int gs, const void* res, void* out,
                 float* part, int M, int N, int K, int nkb, hipStream_t st) {
  const int ncs = N / W4_COLS, KS = K / (128 * nkb);
  const int RT = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const size_t lds = (size_t)RT * 16 * (128 * nkb + 8) * 2 + (size_t)nkb * RT * 16 * 4;
#define L(RT_, NKB_)                                                                                            \
  w4mm_k<RT_, NKB_><<<ncs * KS, 256, lds, st>>>((const bf16*)X, ldx, codes, (const float2*)sc2, gs,             \
                                                (const bf16*)res, (bf16*)out, part, M, N, K, ncs)
#define LN(RT_)                                                                                                 \
  do {                                                                                                          \
    if (nkb == 8) L(RT_, 8); else if (nkb == 4) L(RT_, 4); else if (nkb == 2) L(RT_, 2); else L(RT_, 1);       \
  } while (0)
  if (RT == 1) LN(1); else if (RT == 2) LN(2); else LN(4);
#undef LN
#undef L
  if (KS > 1 && out != nullptr) {                        // (without out the slices' sums are left where they are)
    const size_t MN = (size_t)M * N;
    w4mm_reduce_k<8><<<(MN / 2 + 255) / 256, 256, 0, st>>>(part, (const bf16*)res, (bf16*)out, KS, MN);
  }
  LIPA_CHECK_LAUNCH();
}
