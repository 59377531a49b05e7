// Cross-entropy forward+backward in one pass over a logits chunk (K7).
//
// One 512-thread workgroup per token row of V logits (V = 151,936 for Qwen3): an online
// (max, sum-exp) reduction over 16-B vector loads, then a second sweep that overwrites the
// bf16 logits IN PLACE with dlogits = (softmax - onehot) * scale (scale = 1/n_valid), so
// the LM-head backward GEMM reads them directly.  Ignored rows (label == ignore_index)
// write zeros.  Returns per-row loss (fp32, already unscaled).
#include "common.h"

using namespace lipa;

namespace {

constexpr int NT = 512, NW = NT / 64;

template <typename T>
__global__ __launch_bounds__(NT) void ce_fwd_bwd_k(T* __restrict__ logits, const int64_t* __restrict__ labels,
                                                   float* __restrict__ row_loss, int V, int ignore_index,
                                                   const float* __restrict__ scale_ptr, float scale_val,
                                                   int rows_per_scale) {
  __shared__ float red[NW];
  const int row = blockIdx.x;
  T* lr = logits + (size_t)row * V;
  const int64_t lab = labels[row];
  // per-group scale (gradient-accumulation micro-batches fused into one pass: 1/(G·n_valid_g))
  const float scale = scale_ptr ? scale_ptr[rows_per_scale > 0 ? row / rows_per_scale : 0] : scale_val;
  if (lab == ignore_index) {
    for (int v = threadIdx.x * 8; v < V; v += NT * 8) {
      if (v + 8 <= V) {
        float z[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        store8(lr + v, z);
      } else {
        for (int i = v; i < V; ++i) lr[i] = (T)0.f;
      }
    }
    if (threadIdx.x == 0) row_loss[row] = 0.f;
    return;
  }
  // pass 1: online max / sum-exp
  float m = -INFINITY, s = 0.f;
  for (int v = threadIdx.x * 8; v < V; v += NT * 8) {
    float x[8];
    int n = 8;
    if (v + 8 <= V) load8(lr + v, x);
    else {
      n = V - v;
      for (int i = 0; i < 8; ++i) x[i] = i < n ? (float)lr[v + i] : -INFINITY;
    }
    float mx = x[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, x[i]);
    const float mn = fmaxf(m, mx);
    float acc = s * __expf(m - mn);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc += __expf(x[i] - mn);
    m = mn;
    s = acc;
  }
  // combine (m, s) across the block
  float gm = block_max<NW>(m, red);
  __syncthreads();
  float gs = block_sum<NW>(s * __expf(m - gm), red);
  const float lse = gm + __logf(gs);
  const float xl = (float)lr[lab];
  __syncthreads();
  // pass 2: dlogits in place
  for (int v = threadIdx.x * 8; v < V; v += NT * 8) {
    if (v + 8 <= V) {
      float x[8];
      load8(lr + v, x);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = (__expf(x[i] - lse) - (v + i == lab ? 1.f : 0.f)) * scale;
      store8(lr + v, x);
    } else {
      for (int i = v; i < V; ++i) lr[i] = (T)((__expf((float)lr[i] - lse) - (i == lab ? 1.f : 0.f)) * scale);
    }
  }
  if (threadIdx.x == 0) row_loss[row] = lse - xl;
}

// What stands round the loss, each one launch where torch takes two to seven (a small model's step is bound by the host, 5 to 8 µs a
// launch; the kernels themselves are a launch's 2 µs): labels moved by one, the row groups' scales, the loss from the rows' losses, and
// the gradient times the loss's own.
__global__ __launch_bounds__(256) void shift_labels_k(const int64_t* __restrict__ in, int64_t* __restrict__ out, size_t n, int S,
                                                      int64_t ignore_index) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = i % S == (size_t)S - 1 ? ignore_index : in[i + 1];
}

// inv[g] = 1 / (groups · labels of group g that count, at least 1)
__global__ __launch_bounds__(256) void ce_scale_k(const int64_t* __restrict__ labels, float* __restrict__ inv, int rows,
                                                  int64_t ignore_index) {
  __shared__ int part[4];
  int n = 0;
  for (int i = threadIdx.x; i < rows; i += 256) n += labels[(size_t)blockIdx.x * rows + i] != ignore_index;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) inv[blockIdx.x] = 1.f / ((float)max(part[0] + part[1] + part[2] + part[3], 1) * (float)gridDim.x);
}

// loss = (add ? loss : 0) + Σ_g inv[g] Σ row_loss of group g, one block, summed in 64 bits
__global__ __launch_bounds__(256) void ce_loss_k(const float* __restrict__ row_loss, const float* __restrict__ inv, float* __restrict__ loss,
                                                 int M, int rows, int add) {
  __shared__ double part[4];
  double t = 0.0;
  for (int i = threadIdx.x; i < M; i += 256) t += (double)row_loss[i] * (double)inv[i / rows];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) *loss = (float)((add ? (double)*loss : 0.0) + ((part[0] + part[1]) + (part[2] + part[3])));
}

// y = x · bf16(*s)
__global__ __launch_bounds__(256) void scale_bf16_k(const bf16* __restrict__ x, const float* __restrict__ s, bf16* __restrict__ y, size_t n) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
  const float f = (float)(bf16)*s;
  if (i + 8 <= n) {
    float v[8];
    load8(x + i, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] *= f;
    store8(y + i, v);
  } else {
    for (size_t j = i; j < n; ++j) y[j] = (bf16)((float)x[j] * f);
  }
}

}  // namespace

void launch_shift_labels(const int64_t* in, int64_t* out, size_t n, int S, int64_t ignore_index, hipStream_t st) {
  if (n == 0) return;
  shift_labels_k<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(in, out, n, S, ignore_index);
  LIPA_CHECK_LAUNCH();
}
void launch_ce_scale(const int64_t* labels, float* inv, int groups, int rows, int64_t ignore_index, hipStream_t st) {
  ce_scale_k<<<groups, 256, 0, st>>>(labels, inv, rows, ignore_index);
  LIPA_CHECK_LAUNCH();
}
void launch_ce_loss(const float* row_loss, const float* inv, float* loss, int M, int rows, bool add, hipStream_t st) {
  ce_loss_k<<<1, 256, 0, st>>>(row_loss, inv, loss, M, rows, add);
  LIPA_CHECK_LAUNCH();
}
void launch_scale_bf16(const void* x, const float* s, void* y, size_t n, hipStream_t st) {
  if (n == 0) return;
  scale_bf16_k<<<(unsigned)((n + 2047) / 2048), 256, 0, st>>>((const bf16*)x, s, (bf16*)y, n);
  LIPA_CHECK_LAUNCH();
}

void launch_ce_fwd_bwd(int dtype, void* logits, const int64_t* labels, float* row_loss, int M, int V,
                       int ignore_index, const float* scale_ptr, float scale_val, int rows_per_scale,
                       hipStream_t st) {
  if (dtype == 1)
    ce_fwd_bwd_k<bf16><<<M, NT, 0, st>>>((bf16*)logits, labels, row_loss, V, ignore_index, scale_ptr, scale_val,
                                         rows_per_scale);
  else
    ce_fwd_bwd_k<float><<<M, NT, 0, st>>>((float*)logits, labels, row_loss, V, ignore_index, scale_ptr, scale_val,
                                          rows_per_scale);
  LIPA_CHECK_LAUNCH();
}
