// MLP surrogate of the MPC runs: FP32 master weights, BF16 operands on the
// MFMA units (v_mfma_f32_16x16x32_bf16, FP32 accumulation), hand-written
// forward and backward passes and Adam, all on the device.  It maps the
// parameters of a run (radii, bond length, interaction energies, reaction
// probability, rate constants) to the time-averaged body-frame density field
// and the propulsion velocity that full MPC runs produce.  No reference
// counterpart: the reference has no learned part.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>
#include <algorithm>
#include <vector>
#include "mpcx_device.h"
#include "mpcx_host.h"
#include "mpcx_stage.h"
#include "../../include/mpcx.h"

namespace mpcx {
namespace ml {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ layouts
// Every product is C[m][n] = sum_k A[m][k] B[n][k] of two BF16 operands whose
// contraction index is contiguous, so a lane's fragment of eight is one 16-byte
// load from L2 and no operand is staged, transposed or bounds-checked on the
// way: the weights are kept as W (n_next x n_prev) and as its transpose, and a
// layer's activations and gradients are written by the product that makes them
// both by row and transposed, with zeros up to the next multiple of 32.
// (Element-wise staging through LDS with a 64 x 64 block tile left 4 to 33
// workgroups a product and 22 us of loads in each: a training step of the
// 8-256-256-256-2049 network, batch 64, took 460 us; 61 us so.)
constexpr int PAD = 32;
static inline int up32(int n) { return (n + PAD - 1) / PAD * PAD; }

__device__ __forceinline__ __bf16 to_bf16(float f) { return (__bf16)f; }   // round to nearest even

// One wave's tile of 16 TM x 16 TN.  Loads run U steps of 32 ahead of the
// matrix instructions (65 steps at the widest contraction, one wave a SIMD:
// latency, not rate, bounds the small products).  Accumulation over k is in
// ascending order whatever the tile.
template <int TM, int TN>
__device__ __forceinline__ void tile_product(const __bf16* __restrict__ A, int lda, const __bf16* __restrict__ B, int ldb,
                                             int K, int m0, int n0, f32x4 (&acc)[TM][TN]) {
  constexpr int U = TM * TN > 1 ? 2 : 4;
  const int lane = threadIdx.x & 63, rr = lane & 15, kq = (lane >> 4) * 8;
  const __bf16* pa = A + (size_t)(m0 + rr) * lda + kq;
  const __bf16* pb = B + (size_t)(n0 + rr) * ldb + kq;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  bf16x8 a[U][TM], b[U][TN];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + u * 32 < K) {
#pragma unroll
        for (int i = 0; i < TM; i++) a[u][i] = *(const bf16x8*)(pa + (size_t)i * 16 * lda + k0 + u * 32);
#pragma unroll
        for (int j = 0; j < TN; j++) b[u][j] = *(const bf16x8*)(pb + (size_t)j * 16 * ldb + k0 + u * 32);
      }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += U * 32) {
    bf16x8 ca[U][TM], cb[U][TN];
#pragma unroll
    for (int u = 0; u < U; u++) {
#pragma unroll
      for (int i = 0; i < TM; i++) ca[u][i] = a[u][i];
#pragma unroll
      for (int j = 0; j < TN; j++) cb[u][j] = b[u][j];
    }
    if (k0 + U * 32 < K) fetch(k0 + U * 32);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + u * 32 < K) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ca[u][i], cb[u][j], acc[i][j], 0, 0, 0);
      }
  }
}
// the wave's tile of a grid of mt x nt tiles, four waves a workgroup along n
// (then along m): first output row and column, or false beyond the last
template <int TM, int TN>
__device__ __forceinline__ bool my_tile(int mt, int nt, int blk, int& m0, int& n0) {
  const int t = blk * 4 + (threadIdx.x >> 6);
  if (t >= mt * nt) return false;
  m0 = (t / nt) * 16 * TM;
  n0 = (t % nt) * 16 * TN;
  return true;
}
// element (i, j, t) of a lane: column lane % 16, rows 4 (lane / 16) + t
#define TILE_ROW(i) (m0 + (i)*16 + ((int)(threadIdx.x & 63) >> 4) * 4)
#define TILE_COL(j) (n0 + (j)*16 + (int)(threadIdx.x & 15))

__device__ __forceinline__ void store4(__bf16* p, const float (&v)[4]) {   // four consecutive, 8-byte aligned
  bf16x4 o;
#pragma unroll
  for (int t = 0; t < 4; t++) o[t] = to_bf16(v[t]);
  *(bf16x4*)p = o;
}

// A layer's activations or gradients: FP32 by row (may be null), BF16 by row
// and transposed (null where nothing reads them)
struct Act {
  float* f;
  __bf16* b;
  __bf16* t;
  int cols, ldb, ldt;
};

// H = act(A W^T + bias), rows < rows; the rows up to the next multiple of 32
// are written as zeros (dW's contraction runs over them).
template <int TM, int TN>
__global__ __launch_bounds__(256) void layer_forward(int rows, int mt, int nt, int K, const __bf16* __restrict__ A, int lda,
                                                     const __bf16* __restrict__ W, int ldw,
                                                     const float* __restrict__ bias, int relu, Act H) {
  int m0, n0;
  if (!my_tile<TM, TN>(mt, nt, blockIdx.x, m0, n0)) return;
  f32x4 acc[TM][TN];
  tile_product<TM, TN>(A, lda, W, ldw, K, m0, n0, acc);
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int gn = TILE_COL(j);
    if (gn >= H.cols) continue;
    const float bv = bias ? bias[gn] : 0.f;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int gm = TILE_ROW(i);
      float v[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        v[t] = acc[i][j][t] + bv;
        if (relu) v[t] = v[t] > 0.f ? v[t] : 0.f;
        if (gm + t >= rows) v[t] = 0.f;
        if (H.f && gm + t < rows) H.f[(size_t)(gm + t) * H.cols + gn] = v[t];
        if (H.b) H.b[(size_t)(gm + t) * H.ldb + gn] = to_bf16(v[t]);
      }
      if (H.t) store4(H.t + (size_t)gn * H.ldt + gm, v);
    }
  }
}

// The output layer of a training step with its loss: Y = A W^T + bias stays in
// registers; the wave's share of sum_c wout[c] (Y - T)^2 goes to part[tile],
// the gradient 2 w (Y - T) / rows to dZ.  Target row r is row idx[r] of T
// (idx null: row r).
__global__ __launch_bounds__(256) void output_loss(int rows, int mt, int nt, int K, const __bf16* __restrict__ A, int lda,
                                                   const __bf16* __restrict__ W, int ldw, const float* __restrict__ bias,
                                                   const float* __restrict__ T, const int* __restrict__ idx,
                                                   const float* __restrict__ wout, Act dZ, double* __restrict__ part) {
  int m0, n0;
  if (!my_tile<1, 1>(mt, nt, blockIdx.x, m0, n0)) return;
  const int gn = TILE_COL(0), gm = TILE_ROW(0);
  const bool col = gn < dZ.cols;
  float tv[4];   // the targets' loads run beside the product
#pragma unroll
  for (int t = 0; t < 4; t++)
    tv[t] = col && gm + t < rows ? T[(size_t)(idx ? idx[gm + t] : gm + t) * dZ.cols + gn] : 0.f;
  const float bv = col ? bias[gn] : 0.f, wv = col ? wout[gn] : 0.f;
  f32x4 acc[1][1];
  tile_product<1, 1>(A, lda, W, ldw, K, m0, n0, acc);
  double loss = 0.0;
  float g[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    g[t] = 0.f;
    if (!col || gm + t >= rows) continue;
    const float d = (acc[0][0][t] + bv) - tv[t];
    loss += (double)wv * (double)d * (double)d;
    g[t] = 2.f * wv * d / (float)rows;
    dZ.f[(size_t)(gm + t) * dZ.cols + gn] = g[t];
  }
  if (col) {
#pragma unroll
    for (int t = 0; t < 4; t++) dZ.b[(size_t)(gm + t) * dZ.ldb + gn] = to_bf16(g[t]);
    store4(dZ.t + (size_t)gn * dZ.ldt + gm, g);
  }
  loss = wave_sum(loss);
  if ((threadIdx.x & 63) == 0) part[blockIdx.x * 4 + (threadIdx.x >> 6)] = loss;
}
// loss of each step of an epoch: its tiles' shares in tile order (one wave a step)
__global__ __launch_bounds__(64) void loss_sums(int tiles, long long stride, const double* __restrict__ part,
                                                double* __restrict__ loss) {
  double s = 0.0;
  for (int j = threadIdx.x; j < tiles; j += 64) s += part[blockIdx.x * stride + j];
  s = wave_sum(s);
  if (threadIdx.x == 0) loss[blockIdx.x] = s;
}

// dZ_l = (dZ_{l+1} W) * (H_l > 0), A = dZ_{l+1} by row, WT the transposed weights
__global__ __launch_bounds__(256) void layer_backward(int rows, int mt, int nt, int K, const __bf16* __restrict__ A, int lda,
                                                      const __bf16* __restrict__ WT, int ldw, const float* __restrict__ H,
                                                      Act dZ) {
  int m0, n0;
  if (!my_tile<1, 1>(mt, nt, blockIdx.x, m0, n0)) return;
  const int gn = TILE_COL(0), gm = TILE_ROW(0);
  const bool col = gn < dZ.cols;
  bool on[4];
#pragma unroll
  for (int t = 0; t < 4; t++) on[t] = col && gm + t < rows && H[(size_t)(gm + t) * dZ.cols + gn] > 0.f;
  f32x4 acc[1][1];
  tile_product<1, 1>(A, lda, WT, ldw, K, m0, n0, acc);
  if (!col) return;
  float g[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    g[t] = on[t] ? acc[0][0][t] : 0.f;
    if (gm + t < rows) dZ.f[(size_t)(gm + t) * dZ.cols + gn] = g[t];
    dZ.b[(size_t)(gm + t) * dZ.ldb + gn] = to_bf16(g[t]);
  }
  store4(dZ.t + (size_t)gn * dZ.ldt + gm, g);
}

// Adam on one FP32 master parameter
struct Adam {
  float lr, b1, b2, eps, c1, c2;
  int on;
};
__device__ __forceinline__ float adam_one(const Adam& a, float p, float gi, float* __restrict__ m, float* __restrict__ v) {
  const float mi = a.b1 * *m + (1.f - a.b1) * gi;
  const float vi = a.b2 * *v + (1.f - a.b2) * gi * gi;
  *m = mi;
  *v = vi;
  return p - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

// Weight and bias gradients of up to MAXL layers in one launch, and the Adam
// step on them where they are made (a.on; else the gradients go to g): dW_l =
// dZ_{l+1}^T H_l over the batch, db_l the column sums of dZ_{l+1} in row order.
// Nothing else of the step reads the weights any more, so the BF16 copies are
// renewed here too.
constexpr int MAXL = 8;
struct GradLayer {
  const __bf16 *dZt, *Ht;   // transposed, contraction over the batch
  const float* dZ;          // FP32 by row, for the bias
  __bf16 *w, *wt;           // BF16 copies of the weights
  long long woff, boff;     // in the flat parameters
  int N, K, ldw, ldwt, nt;  // dims, leading dimensions, tiles along K
  int ldh;                  // leading dimension of Ht
  int blk0, bias0;          // first workgroup of its tiles and of its bias
};
struct GradArgs {
  GradLayer l[MAXL];
  int n;
};
__global__ __launch_bounds__(256) void layer_grads(GradArgs G, int rows, int ldt, Adam a, float* __restrict__ p,
                                                   float* __restrict__ g, float* __restrict__ m, float* __restrict__ v) {
  int q = 0;
  while (q + 1 < G.n && (int)blockIdx.x >= G.l[q + 1].blk0) q++;
  const GradLayer& L = G.l[q];
  if ((int)blockIdx.x >= L.bias0) {
    const int c = ((int)blockIdx.x - L.bias0) * 256 + (int)threadIdx.x;
    if (c >= L.N) return;
    float s = 0.f;
    for (int r0 = 0; r0 < rows; r0 += 16) {   // sixteen loads in flight, added in row order
      float x[16];
#pragma unroll
      for (int r = 0; r < 16; r++) x[r] = r0 + r < rows ? L.dZ[(size_t)(r0 + r) * L.N + c] : 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++)
        if (r0 + r < rows) s += x[r];
    }
    const long long o = L.boff + c;
    if (a.on) p[o] = adam_one(a, p[o], s, m + o, v + o);
    else g[o] = s;
    return;
  }
  int m0, n0;
  if (!my_tile<1, 1>((L.N + 15) / 16, L.nt, (int)blockIdx.x - L.blk0, m0, n0)) return;
  const int gn = TILE_COL(0), gm = TILE_ROW(0);
  f32x4 acc[1][1];
  tile_product<1, 1>(L.dZt, ldt, L.Ht, L.ldh, (rows + PAD - 1) / PAD * PAD, m0, n0, acc);
  if (gn >= L.K) return;
  float w[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    w[t] = 0.f;
    if (gm + t >= L.N) continue;
    const long long o = L.woff + (long long)(gm + t) * L.K + gn;
    if (!a.on) { g[o] = acc[0][0][t]; continue; }
    w[t] = adam_one(a, p[o], acc[0][0][t], m + o, v + o);
    p[o] = w[t];
    L.w[(size_t)(gm + t) * L.ldw + gn] = to_bf16(w[t]);
  }
  if (a.on) store4(L.wt + (size_t)gn * L.ldwt + gm, w);
}

// BF16 copies of one layer's weights, by row and transposed
__global__ void weights_bf16(int N, int K, const float* __restrict__ W, __bf16* __restrict__ w, int ldw,
                             __bf16* __restrict__ wt, int ldwt) {
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < (long long)N * K;
       e += (long long)gridDim.x * blockDim.x) {
    const int n = (int)(e / K), k = (int)(e % K);
    const __bf16 b = to_bf16(W[e]);
    w[(size_t)n * ldw + k] = b;
    wt[(size_t)k * ldwt + n] = b;
  }
}

// The input rows of `steps` batches in a row, BF16 by row and transposed, zeros
// to the batches' padded sizes: row r of batch s is row idx[s*batch + r] of X
// (idx null: row s*batch + r), of the n rows left.
__global__ void input_rows(int n, int batch, int steps, int cols, const float* __restrict__ X, const int* __restrict__ idx,
                           __bf16* __restrict__ hb, int ldb, __bf16* __restrict__ ht, int ldt, int cols_p) {
  const long long per = (long long)ldt * cols;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < per * steps;
       e += (long long)gridDim.x * blockDim.x) {
    const int s = (int)(e / per), r = (int)(e % per / cols), c = (int)(e % cols);
    const long long q = (long long)s * batch + r;
    const __bf16 v = to_bf16(r < batch && q < n ? X[(size_t)(idx ? idx[q] : q) * cols + c] : 0.f);
    hb[((size_t)s * ldt + r) * ldb + c] = v;
    ht[((size_t)s * cols_p + c) * ldt + r] = v;
  }
}
// x (rows x cols, FP32) -> BF16 with leading dimension ld (transposed if tr)
__global__ void to_bf16_padded(int rows, int cols, const float* __restrict__ x, __bf16* __restrict__ y, int ld, int tr) {
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < (long long)rows * cols;
       e += (long long)gridDim.x * blockDim.x) {
    const int r = (int)(e / cols), c = (int)(e % cols);
    y[tr ? (size_t)c * ld + r : (size_t)r * ld + c] = to_bf16(x[e]);
  }
}

}  // namespace ml
}  // namespace mpcx

using namespace mpcx;
using namespace mpcx::ml;

struct mpcx_mlp {
  int n_in, n_hid, n_layers, n_out;   // n_layers hidden layers
  std::vector<int> dims;              // dims[l] -> dims[l+1]
  std::vector<long long> woff, boff;  // offsets of W_l and b_l in the flat parameter vector
  long long nparam = 0;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  std::vector<__bf16*> w, wt;         // BF16 copies of W_l: (up32(n_next) x up32(n_prev)) and transposed
  // forward buffers (fcap rows): activations BF16 by row, the output in FP32
  int fcap = 0;
  std::vector<__bf16*> Fb;
  float *Fx = nullptr, *Fy = nullptr;
  // training buffers (cap rows a batch)
  int cap = 0;
  std::vector<Act> H, dZ;             // H[0]: the input rows of several batches (its ldt: the call's padded batch)
  long long in_rows = 0;              // rows H[0] holds
  double *part = nullptr, *loss = nullptr;
  long long part_n = 0, loss_n = 0;
  int* idx = nullptr;
  long long idx_n = 0;
  float *X = nullptr, *T = nullptr, *W = nullptr;   // dataset on the device
  long long x_n = 0, t_n = 0;
  hipStream_t st = nullptr;
  long long t = 0;                    // Adam step counter
  double gemm_ms = 0;
  long long gemm_flops = 0;
};

#define MLCHK(x)                                                              \
  do {                                                                        \
    hipError_t _r = (x);                                                      \
    if (_r != hipSuccess) return set_error(MPCX_E_HIP, hipGetErrorString(_r)); \
  } while (0)

static inline unsigned blocks_for(long long n) { return (unsigned)std::min<long long>((n + 255) / 256, 4096); }

template <typename T>
static void release(T*& q) {
  if (q) (void)hipFree(q);
  q = nullptr;
}
// a buffer of at least n elements; a new one is all zeros (padding is never written)
template <typename T>
static int grow(hipStream_t st, T*& q, long long& have, long long n) {
  if (n <= have) return 0;
  release(q);
  have = 0;
  MLCHK(mpcx::device_alloc(&q, (size_t)n * sizeof(T)));
  MLCHK(hipMemsetAsync(q, 0, (size_t)n * sizeof(T), st));
  have = n;
  return 0;
}
template <typename T>
static int zeroed(hipStream_t st, T*& q, size_t n) {
  long long have = 0;
  return grow(st, q, have, (long long)n);
}
static void release_act(Act& a) { release(a.f); release(a.b); release(a.t); }
static int make_act(hipStream_t st, Act& a, long long rows, int ldt, int cols) {
  int rc;
  a.cols = cols; a.ldb = up32(cols); a.ldt = ldt;
  if ((rc = zeroed(st, a.f, (size_t)rows * cols)) || (rc = zeroed(st, a.b, (size_t)rows * a.ldb)) ||
      (rc = zeroed(st, a.t, (size_t)a.ldb * rows)))
    return rc;
  return 0;
}

// Training buffers for batches of `batch` rows, `steps` of them an epoch; held:
// the batches whose input rows and loss shares are on the device together.
// These are laid out for the call's own batch, and an epoch of more than
// HELD_BYTES of them is taken in parts: with the largest batch seen as their
// stride, or a whole epoch held, the memory of a small batch's epoch was the
// product of two sizes that need not meet (320 GB for 50,000 rows one at a time
// after a gradient of all of them).
constexpr long long HELD_BYTES = 64ll << 20;
static long long part_stride(const mpcx_mlp* e) {
  return (long long)(e->H[0].ldt / 16) * ((e->n_out + 15) / 16) + 4;
}
static int train_buffers(mpcx_mlp* e, int batch, long long steps, long long& held) {
  const int L = (int)e->dims.size(), R = up32(batch);
  int rc;
  if (batch > e->cap) {
    for (auto& a : e->H) release_act(a);
    for (auto& a : e->dZ) release_act(a);
    e->H.assign(L, Act{}); e->dZ.assign(L, Act{});
    e->cap = 0;
    e->in_rows = 0;
    for (int l = 1; l < L; l++) {
      if (l + 1 < L && (rc = make_act(e->st, e->H[l], R, R, e->dims[l]))) return rc;
      if ((rc = make_act(e->st, e->dZ[l], R, R, e->dims[l]))) return rc;
    }
    e->cap = batch;
  }
  Act& in = e->H[0];
  in.cols = e->n_in; in.ldb = up32(e->n_in); in.ldt = R;
  held = std::max(1ll, std::min(steps, HELD_BYTES / ((long long)R * in.ldb * 4 + part_stride(e) * 8)));
  if (R * held > e->in_rows) {
    release_act(in);
    e->in_rows = 0;
    if ((rc = zeroed(e->st, in.b, (size_t)R * held * in.ldb)) || (rc = zeroed(e->st, in.t, (size_t)R * held * in.ldb)))
      return rc;
    e->in_rows = R * held;
  }
  return grow(e->st, e->part, e->part_n, part_stride(e) * held);
}

// one training step's forward and backward on batch s of the held input
// rows; the loss shares into the step's part, the gradients applied (a.on) or into g
static void train_step(mpcx_mlp* e, int rows, long long s, const float* T, const int* idx, const float* wout, Adam a) {
  const int L = (int)e->dims.size(), ldt = up32(e->cap), Rp = up32(rows), mt = Rp / 16;
  hipStream_t st = e->st;
  const Act& X = e->H[0];
  const __bf16* in = X.b + (size_t)s * X.ldt * X.ldb;
  const __bf16* int_ = X.t + (size_t)s * X.ldt * X.ldb;
  for (int l = 0; l + 1 < L; l++) {
    const int K = up32(e->dims[l]), N = e->dims[l + 1], nt = (N + 15) / 16;
    const unsigned grid = (unsigned)((mt * nt + 3) / 4);
    const __bf16* A = l ? e->H[l].b : in;
    if (l + 2 < L)
      hipLaunchKernelGGL((layer_forward<1, 1>), dim3(grid), dim3(256), 0, st, rows, mt, nt, K, A, K,
                         (const __bf16*)e->w[l], K, (const float*)(e->p + e->boff[l]), 1, e->H[l + 1]);
    else
      hipLaunchKernelGGL(output_loss, dim3(grid), dim3(256), 0, st, rows, mt, nt, K, A, K, (const __bf16*)e->w[l], K,
                         (const float*)(e->p + e->boff[l]), T, idx, wout, e->dZ[l + 1], e->part + s * part_stride(e));
    e->gemm_flops += 2ll * rows * N * e->dims[l];
  }
  for (int l = L - 2; l >= 1; l--) {
    const int K = up32(e->dims[l + 1]), N = e->dims[l], nt = (N + 15) / 16;
    hipLaunchKernelGGL(layer_backward, dim3((unsigned)((mt * nt + 3) / 4)), dim3(256), 0, st, rows, mt, nt, K,
                       (const __bf16*)e->dZ[l + 1].b, K, (const __bf16*)e->wt[l], K, (const float*)e->H[l].f, e->dZ[l]);
    e->gemm_flops += 2ll * rows * N * e->dims[l + 1];
  }
  for (int l0 = 0; l0 + 1 < L; l0 += MAXL) {
    GradArgs G{};
    int blk = 0;
    for (int l = l0; l + 1 < L && l < l0 + MAXL; l++) {
      GradLayer& q = G.l[G.n++];
      const int N = e->dims[l + 1], K = e->dims[l];
      q = GradLayer{e->dZ[l + 1].t, l ? e->H[l].t : int_, e->dZ[l + 1].f, e->w[l], e->wt[l], e->woff[l], e->boff[l],
                    N, K, up32(K), up32(N), (K + 15) / 16, l ? ldt : X.ldt, blk, 0};
      blk += ((N + 15) / 16 * q.nt + 3) / 4;
      q.bias0 = blk;
      blk += (N + 255) / 256;
      e->gemm_flops += 2ll * rows * N * K;
    }
    hipLaunchKernelGGL(layer_grads, dim3((unsigned)blk), dim3(256), 0, st, G, rows, ldt, a, e->p, e->g, e->m, e->v);
  }
}

static void refresh_bf16(mpcx_mlp* e) {
  for (size_t l = 0; l + 1 < e->dims.size(); l++)
    hipLaunchKernelGGL(weights_bf16, dim3(blocks_for((long long)e->dims[l] * e->dims[l + 1])), dim3(256), 0, e->st,
                       e->dims[l + 1], e->dims[l], (const float*)(e->p + e->woff[l]), e->w[l], up32(e->dims[l]), e->wt[l],
                       up32(e->dims[l + 1]));
}

extern "C" int mpcx_mlp_destroy(mpcx_mlp* e) {
  if (!e) return 0;
  mpcx::handle_del(mpcx::H_MLP, e);
  if (e->st) (void)hipStreamSynchronize(e->st);
  release(e->p); release(e->g); release(e->m); release(e->v);
  for (auto& q : e->w) release(q);
  for (auto& q : e->wt) release(q);
  for (auto& q : e->Fb) release(q);
  for (auto& a : e->H) release_act(a);
  for (auto& a : e->dZ) release_act(a);
  release(e->Fx); release(e->Fy); release(e->part); release(e->loss); release(e->idx);
  release(e->X); release(e->T); release(e->W);
  if (e->st) (void)hipStreamDestroy(e->st);
  delete e;
  return 0;
}

extern "C" int mpcx_mlp_create(mpcx_mlp** out, int32_t n_in, int32_t n_hidden, int32_t n_layers, int32_t n_out,
                               uint64_t seed) {
  if (!out || n_in < 1 || n_hidden < 1 || n_layers < 1 || n_out < 1) return set_error(MPCX_E_ARG, "bad sizes");
  mpcx_mlp* e = new mpcx_mlp();
  e->n_in = n_in; e->n_hid = n_hidden; e->n_layers = n_layers; e->n_out = n_out;
  e->dims.push_back(n_in);
  for (int l = 0; l < n_layers; l++) e->dims.push_back(n_hidden);
  e->dims.push_back(n_out);
  long long o = 0;
  for (size_t l = 0; l + 1 < e->dims.size(); l++) {
    e->woff.push_back(o); o += (long long)e->dims[l] * e->dims[l + 1];
    e->boff.push_back(o); o += e->dims[l + 1];
  }
  e->nparam = o;
  // He-uniform initial weights from a 64-bit LCG (Knuth MMIX constants), zero biases
  std::vector<float> p(o, 0.f);
  unsigned long long s = seed * 6364136223846793005ull + 1442695040888963407ull;
  for (size_t l = 0; l + 1 < e->dims.size(); l++) {
    const double lim = sqrt(6.0 / e->dims[l]);
    for (long long i = 0; i < (long long)e->dims[l] * e->dims[l + 1]; i++) {
      s = s * 6364136223846793005ull + 1442695040888963407ull;
      const double u = (double)(s >> 11) * (1.0 / 9007199254740992.0);
      p[e->woff[l] + i] = (float)((2.0 * u - 1.0) * lim);
    }
  }
  if (hipStreamCreateWithFlags(&e->st, hipStreamNonBlocking) != hipSuccess ||
      mpcx::device_alloc(&e->p, o * 4) != hipSuccess || mpcx::device_alloc(&e->g, o * 4) != hipSuccess ||
      mpcx::device_alloc(&e->m, o * 4) != hipSuccess || mpcx::device_alloc(&e->v, o * 4) != hipSuccess) {
    mpcx_mlp_destroy(e);
    return set_error(MPCX_E_HIP, "device allocation failed");
  }
  const size_t nl = e->dims.size() - 1;
  e->w.assign(nl, nullptr);
  e->wt.assign(nl, nullptr);
  for (size_t l = 0; l < nl; l++) {
    const size_t n = (size_t)up32(e->dims[l]) * up32(e->dims[l + 1]);
    if (zeroed(e->st, e->w[l], n) || zeroed(e->st, e->wt[l], n)) {
      mpcx_mlp_destroy(e);
      return MPCX_E_HIP;
    }
  }
  MLCHK(hipMemcpy(e->p, p.data(), o * 4, hipMemcpyHostToDevice));
  MLCHK(hipMemset(e->m, 0, o * 4));
  MLCHK(hipMemset(e->v, 0, o * 4));
  MLCHK(hipMemset(e->g, 0, o * 4));
  refresh_bf16(e);
  MLCHK(hipStreamSynchronize(e->st));
  *out = e;
  mpcx::handle_add(mpcx::H_MLP, e);
  return 0;
}

extern "C" int64_t mpcx_mlp_num_params(mpcx_mlp* e) { return e ? e->nparam : 0; }

extern "C" int mpcx_mlp_get_params(mpcx_mlp* e, float* flat) {
  if (!e || !flat) return set_error(MPCX_E_ARG, "null argument");
  return mpcx::copy_out({{flat, e->p, (size_t)e->nparam * 4}}, e->st);
}

extern "C" int mpcx_mlp_set_params(mpcx_mlp* e, const float* flat) {
  if (!e || !flat) return set_error(MPCX_E_ARG, "null argument");
  MLCHK(hipStreamSynchronize(e->st));
  MLCHK(hipMemcpy(e->p, flat, e->nparam * 4, hipMemcpyHostToDevice));
  refresh_bf16(e);
  MLCHK(hipStreamSynchronize(e->st));
  return 0;
}

// Forward pass.  32 x 32 tiles once a layer has enough of them to fill the
// chip's 1024 SIMDs several times over (they read half as much per product),
// 16 x 16 below that, where the number of waves is what counts.
extern "C" int mpcx_mlp_forward(mpcx_mlp* e, int32_t rows, const float* x, float* y) {
  if (!e || rows < 1 || !x || !y) return set_error(MPCX_E_ARG, "bad arguments");
  const int L = (int)e->dims.size(), Rp = up32(rows);
  int rc;
  if (rows > e->fcap) {
    for (auto& q : e->Fb) release(q);
    release(e->Fx); release(e->Fy);
    e->fcap = 0;
    e->Fb.assign(L - 1, nullptr);
    for (int l = 0; l + 1 < L; l++)
      if ((rc = zeroed(e->st, e->Fb[l], (size_t)Rp * up32(e->dims[l])))) return rc;
    MLCHK(mpcx::device_alloc(&e->Fx, (size_t)rows * e->n_in * 4));
    MLCHK(mpcx::device_alloc(&e->Fy, (size_t)rows * e->n_out * 4));
    e->fcap = rows;
  }
  MLCHK(hipMemcpyAsync(e->Fx, x, (size_t)rows * e->n_in * 4, hipMemcpyHostToDevice, e->st));
  hipLaunchKernelGGL(to_bf16_padded, dim3(blocks_for((long long)rows * e->n_in)), dim3(256), 0, e->st, rows, e->n_in,
                     (const float*)e->Fx, e->Fb[0], up32(e->n_in), 0);
  for (int l = 0; l + 1 < L; l++) {
    const int K = up32(e->dims[l]), N = e->dims[l + 1];
    const bool last = l + 2 == L;
    const Act H{last ? e->Fy : nullptr, last ? nullptr : e->Fb[l + 1], nullptr, N, up32(N), 0};
    const bool big = (long long)(Rp / 16) * ((N + 15) / 16) >= 4096;
    const int mt = Rp / (big ? 32 : 16), nt = big ? up32(N) / 32 : (N + 15) / 16;
    const dim3 grid((unsigned)(((long long)mt * nt + 3) / 4));
    auto launch = [&](auto k) {
      hipLaunchKernelGGL(k, grid, dim3(256), 0, e->st, (int)rows, mt, nt, K, (const __bf16*)e->Fb[l], K,
                         (const __bf16*)e->w[l], K, (const float*)(e->p + e->boff[l]), last ? 0 : 1, H);
    };
    if (big) launch(layer_forward<2, 2>);
    else launch(layer_forward<1, 1>);
    e->gemm_flops += 2ll * rows * N * e->dims[l];
  }
  return mpcx::copy_out({{y, e->Fy, (size_t)rows * e->n_out * 4}}, e->st);
}

// dataset rows, targets and output weights on the device
static int upload_data(mpcx_mlp* e, long long n, const float* x, const float* target, const float* wout) {
  int rc;
  long long w_n = e->W ? e->n_out : 0;
  if ((rc = grow(e->st, e->X, e->x_n, n * e->n_in)) || (rc = grow(e->st, e->T, e->t_n, n * e->n_out)) ||
      (rc = grow(e->st, e->W, w_n, e->n_out)))
    return rc;
  return mpcx::copy_in({mpcx::upload(e->X, x, (size_t)n * e->n_in * 4), mpcx::upload(e->T, target, (size_t)n * e->n_out * 4),
                        mpcx::upload(e->W, wout, (size_t)e->n_out * 4)}, e->st);
}
static void launch_inputs(mpcx_mlp* e, long long n, int batch, long long steps, const int* idx) {
  const Act& a = e->H[0];
  hipLaunchKernelGGL(input_rows, dim3(blocks_for((long long)a.ldt * a.cols * steps)), dim3(256), 0, e->st, (int)n, batch,
                     (int)steps, a.cols, (const float*)e->X, idx, a.b, a.ldb, a.t, a.ldt, a.ldb);
}
// losses of the held steps s0 .. s0 + steps
static void launch_loss(mpcx_mlp* e, int tiles, long long s0, long long steps, double* out) {
  hipLaunchKernelGGL(loss_sums, dim3((unsigned)steps), dim3(64), 0, e->st, tiles, part_stride(e),
                     (const double*)(e->part + s0 * part_stride(e)), out);
}
static int loss_tiles(const mpcx_mlp* e, int rows) { return (up32(rows) / 16) * ((e->n_out + 15) / 16); }

extern "C" int mpcx_mlp_loss_grad(mpcx_mlp* e, int32_t rows, const float* x, const float* target, const float* wout,
                                  double* loss, float* grad) {
  if (!e || rows < 1 || !x || !target || !wout || !loss) return set_error(MPCX_E_ARG, "bad arguments");
  int rc;
  long long held;
  if ((rc = train_buffers(e, rows, 1, held)) || (rc = upload_data(e, rows, x, target, wout)) ||
      (rc = grow(e->st, e->loss, e->loss_n, 1)))
    return rc;
  launch_inputs(e, rows, rows, 1, nullptr);
  train_step(e, rows, 0, e->T, nullptr, e->W, Adam{});
  launch_loss(e, loss_tiles(e, rows), 0, 1, e->loss);
  MLCHK(hipMemcpyAsync(loss, e->loss, 8, hipMemcpyDeviceToHost, e->st));
  if (grad) MLCHK(hipMemcpyAsync(grad, e->g, e->nparam * 4, hipMemcpyDeviceToHost, e->st));
  MLCHK(hipStreamSynchronize(e->st));
  *loss = *loss / rows;
  return 0;
}

// Minibatch Adam over a dataset held on the device.  Each epoch visits the n
// rows in an order shuffled by a 64-bit LCG seeded with `seed` and the epoch.
// The host only makes the orders, a few epochs at a time, and launches: the
// losses stay on the device until the end of the run (waiting for each
// minibatch's, the allocations and 21 launches a step, took 460 us a step).
extern "C" int mpcx_mlp_train(mpcx_mlp* e, int64_t n, const float* x, const float* target, const float* wout,
                              int32_t batch, int32_t epochs, float lr, uint64_t seed, double* epoch_loss) {
  if (!e || n < 1 || !x || !target || !wout || batch < 1 || epochs < 0) return set_error(MPCX_E_ARG, "bad arguments");
  batch = (int32_t)std::min<int64_t>(batch, n);
  const long long steps = (n + batch - 1) / batch;
  const int CHUNK = (int)std::max<int64_t>(1, std::min<int64_t>(64, (1 << 22) / n));   // epochs whose orders are uploaded together
  int rc;
  long long held;
  if ((rc = train_buffers(e, batch, steps, held)) || (rc = upload_data(e, n, x, target, wout)) ||
      (rc = grow(e->st, e->idx, e->idx_n, n * CHUNK)) || (rc = grow(e->st, e->loss, e->loss_n, steps * std::max(epochs, 1))))
    return rc;
  std::vector<int> order((size_t)n * std::min(CHUNK, std::max(epochs, 1)));
  hipEvent_t a0, a1;
  (void)hipEventCreate(&a0);
  (void)hipEventCreate(&a1);
  (void)hipEventRecord(a0, e->st);
  e->gemm_flops = 0;
  const int tail = (int)(n - (steps - 1) * batch);
  for (int e0 = 0; e0 < epochs && !rc; e0 += CHUNK) {
    const int ne = std::min(CHUNK, epochs - e0);
    if (e0) rc = hipStreamSynchronize(e->st) == hipSuccess ? 0 : set_error(MPCX_E_HIP, "hipStreamSynchronize failed");
    for (int q = 0; q < ne; q++) {
      int* o = order.data() + (size_t)q * n;
      for (long long i = 0; i < n; i++) o[i] = (int)i;
      unsigned long long s = (seed + 1) * 6364136223846793005ull + (unsigned long long)(e0 + q) * 1442695040888963407ull;
      for (long long i = n - 1; i > 0; i--) {   // Fisher-Yates
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        const long long j = (long long)((s >> 33) % (unsigned long long)(i + 1));
        std::swap(o[i], o[j]);
      }
    }
    if (!rc && hipMemcpyAsync(e->idx, order.data(), (size_t)ne * n * 4, hipMemcpyHostToDevice, e->st) != hipSuccess)
      rc = set_error(MPCX_E_HIP, "hipMemcpyAsync failed");
    for (int q = 0; q < ne && !rc; q++) {
      const int* idx = e->idx + (size_t)q * n;
      double* lo = e->loss + (size_t)(e0 + q) * steps;
      for (long long s0 = 0; s0 < steps; s0 += held) {
        const long long ns = std::min(held, steps - s0), full = s0 + ns < steps ? ns : ns - 1;
        launch_inputs(e, n - s0 * batch, batch, ns, idx + s0 * batch);
        for (long long s = 0; s < ns; s++) {
          e->t += 1;
          const float c1 = 1.f - powf(0.9f, (float)e->t), c2 = 1.f - powf(0.999f, (float)e->t);
          train_step(e, s < full ? batch : tail, s, e->T, idx + (s0 + s) * batch, e->W,
                     Adam{lr, 0.9f, 0.999f, 1e-8f, c1, c2, 1});
        }
        if (full) launch_loss(e, loss_tiles(e, batch), 0, full, lo + s0);
        if (full < ns) launch_loss(e, loss_tiles(e, tail), full, 1, lo + s0 + full);
      }
    }
  }
  (void)hipEventRecord(a1, e->st);
  std::vector<double> loss((size_t)steps * std::max(epochs, 1));
  if (!rc && epochs > 0 &&
      hipMemcpyAsync(loss.data(), e->loss, (size_t)steps * epochs * 8, hipMemcpyDeviceToHost, e->st) != hipSuccess)
    rc = set_error(MPCX_E_HIP, "hipMemcpyAsync failed");
  const hipError_t sr = hipStreamSynchronize(e->st);   // the orders and the caller's arrays are read until here
  float ms = 0;
  (void)hipEventElapsedTime(&ms, a0, a1);
  e->gemm_ms = ms;
  (void)hipEventDestroy(a0);
  (void)hipEventDestroy(a1);
  if (rc) return rc;
  MLCHK(sr);
  if (epoch_loss)
    for (int ep = 0; ep < epochs; ep++) {
      double tot = 0.0;
      for (long long s = 0; s < steps; s++) {
        const int rows = s + 1 < steps ? batch : tail;
        tot += loss[(size_t)ep * steps + s] / rows * rows;
      }
      epoch_loss[ep] = tot / (double)n;
    }
  return 0;
}

// wall time (ms) and GEMM flops of the last mpcx_mlp_train
extern "C" int mpcx_mlp_train_stats(mpcx_mlp* e, double* ms, double* gemm_flops) {
  if (!e) return set_error(MPCX_E_ARG, "null engine");
  if (ms) *ms = e->gemm_ms;
  if (gemm_flops) *gemm_flops = (double)e->gemm_flops;
  return 0;
}

// C (M x N, FP32) = A (M x K) B (K x N) with A, B rounded to BF16 and FP32
// accumulation on the MFMA units; row-major host arrays.  For tests and timing.
extern "C" int mpcx_gemm_bf16(int32_t M, int32_t N, int32_t K, const float* A, const float* B, float* C, int32_t reps,
                              double* ms) {
  if (M < 1 || N < 1 || K < 1 || !A || !B || !C || reps < 1) return set_error(MPCX_E_ARG, "bad arguments");
  const int Mp = up32(M), Np = up32(N), Kp = up32(K);
  float *Af = nullptr, *Bf = nullptr, *Cd = nullptr;
  __bf16 *Ab = nullptr, *Bb = nullptr;
  MLCHK(mpcx::device_alloc(&Af, (size_t)M * K * 4)); MLCHK(mpcx::device_alloc(&Bf, (size_t)K * N * 4));
  MLCHK(mpcx::device_alloc(&Ab, (size_t)Mp * Kp * 2)); MLCHK(mpcx::device_alloc(&Bb, (size_t)Np * Kp * 2));
  MLCHK(mpcx::device_alloc(&Cd, (size_t)M * N * 4));
  MLCHK(hipMemset(Ab, 0, (size_t)Mp * Kp * 2));
  MLCHK(hipMemset(Bb, 0, (size_t)Np * Kp * 2));
  MLCHK(hipMemcpy(Af, A, (size_t)M * K * 4, hipMemcpyHostToDevice));
  MLCHK(hipMemcpy(Bf, B, (size_t)K * N * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(to_bf16_padded, dim3(1024), dim3(256), 0, 0, M, K, (const float*)Af, Ab, Kp, 0);
  hipLaunchKernelGGL(to_bf16_padded, dim3(1024), dim3(256), 0, 0, K, N, (const float*)Bf, Bb, Kp, 1);
  hipEvent_t a0, a1;
  (void)hipEventCreate(&a0);
  (void)hipEventCreate(&a1);
  const bool big = (long long)(Mp / 16) * ((N + 15) / 16) >= 4096;
  const int mt = Mp / (big ? 32 : 16), nt = big ? Np / 32 : (N + 15) / 16;
  const Act C_{Cd, nullptr, nullptr, N, 0, 0};
  auto product = [&](auto k) {
    hipLaunchKernelGGL(k, dim3((unsigned)(((long long)mt * nt + 3) / 4)), dim3(256), 0, 0, (int)M, mt, nt, Kp,
                       (const __bf16*)Ab, Kp, (const __bf16*)Bb, Kp, (const float*)nullptr, 0, C_);
  };
  auto once = [&] { if (big) product(layer_forward<2, 2>); else product(layer_forward<1, 1>); };
  once();
  (void)hipEventRecord(a0, 0);
  for (int r = 0; r < reps; r++) once();
  (void)hipEventRecord(a1, 0);
  hipError_t rr = hipEventSynchronize(a1);
  float t = 0;
  (void)hipEventElapsedTime(&t, a0, a1);
  if (ms) *ms = t / reps;
  if (rr == hipSuccess) rr = hipMemcpy(C, Cd, (size_t)M * N * 4, hipMemcpyDeviceToHost);
  (void)hipEventDestroy(a0);
  (void)hipEventDestroy(a1);
  (void)hipFree(Af); (void)hipFree(Bf); (void)hipFree(Ab); (void)hipFree(Bb); (void)hipFree(Cd);
  if (rr != hipSuccess) return set_error(MPCX_E_HIP, hipGetErrorString(rr));
  return 0;
}
