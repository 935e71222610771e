// wg_mlp.hip -- the calibration surrogate: a 16-128-128-128-1 GELU perceptron
// trained and evaluated on the GPU with hand-written BF16 MFMA kernels (FP32
// accumulation).  No counterpart in the reference: it stands in for the γ search
// of calibration.cpp:266-636 by proposing γ from basin features.
//
// Precision: FP32 master parameters; BF16 copies of the weights and of every
// GEMM operand (inputs, hidden activations, back-propagated deltas); FP32
// accumulation, biases, pre-activations, GELU, loss and Adam.
//
// All GEMMs are C[M][N] = sum_k A[m][k] * Bt[n][k] with both operands K-contiguous
// BF16, on v_mfma_f32_16x16x32_bf16 (lane l: A row l%16 and B column l%16 with
// k = (l/16)*8 .. +7; C column l%16, rows (l/16)*4 .. +3), accumulated in K order.
//
// A training step is two launches.  mlp_rows takes 16 batch rows per workgroup through
// all layers and back, activations and deltas in LDS and registers; what the weight
// gradients need goes to memory transposed ([unit][row]), so that every operand of
// mlp_update, which forms the gradients and applies Adam, is K-contiguous too.  The
// sums over rows (biases, output weights, loss) keep row order: mlp_update stages
// their terms in LDS and adds them serially, one lane a sum.  (One launch per layer
// and sum, the sums read from memory term by term, took 1,080 us a batch of 1,024.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/watergap2_amd.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
using bf16 = __bf16;

constexpr int kHid = 128;   // hidden units
constexpr int kIn = 16;     // features
constexpr int kInPad = 32;  // features padded to one MFMA K step

// parameter offsets in the flat FP32 vector
constexpr int64_t kOffW1 = 0;
constexpr int64_t kOffB1 = kOffW1 + int64_t(kHid) * kIn;
constexpr int64_t kOffW2 = kOffB1 + kHid;
constexpr int64_t kOffB2 = kOffW2 + int64_t(kHid) * kHid;
constexpr int64_t kOffW3 = kOffB2 + kHid;
constexpr int64_t kOffB3 = kOffW3 + int64_t(kHid) * kHid;
constexpr int64_t kOffW4 = kOffB3 + kHid;
constexpr int64_t kOffB4 = kOffW4 + kHid;
constexpr int64_t kNParams = kOffB4 + 1;

__device__ inline float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float z) {
  return 0.5f * (1.f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// Buffers of one batch of R rows (a multiple of 32), n of them valid, the rest zero
// features and no loss; rows of xs and ts through idx, or in order when idx is NULL.
struct RowBatch {
  const float *xs, *ts;
  const int32_t *idx;
  int n, R;
  bf16 *xt;           // [16][R] features
  bf16 *ht[3];        // [128][R] hidden activations
  bf16 *dt[3];        // [128][R] deltas
  float *et[3];       // [128][R] deltas in FP32
  float *y, *dy, *sq; // [R] output, its loss gradient, squared error
};

// BF16 weights for mlp_rows and mlp_update, and the FP32 master parameters.
struct Weights {
  float *p;
  bf16 *w1, *w2, *w2t, *w3, *w3t, *w4;
};

constexpr int kRowTile = 16;
constexpr int kLdA = kHid + 8;    // LDS rows padded by 16 bytes: the 16 rows that a
constexpr int kLdX = kInPad + 8;  // wavefront reads together fall on different banks

__device__ inline bf16x8 frag(const bf16 *row, int k) { return *reinterpret_cast<const bf16x8 *>(row + k); }

// acc[j] += A (16 rows in LDS) x this wavefront's two column blocks; b: K / 32 x 2
// operand fragments.
template <int kSteps>
__device__ inline void mma(const bf16 *a_row, int kq, const bf16x8 (&b)[kSteps][2], f32x4 (&acc)[2]) {
#pragma unroll
  for (int j = 0; j < 2; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < kSteps; k++) {
    const bf16x8 a = frag(a_row, k * 32 + kq);
#pragma unroll
    for (int j = 0; j < 2; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[k][j], acc[j], 0, 0, 0);
  }
}

template <int kSteps>
__device__ inline void load_frags(const bf16 *w, int n0, int r, int kq, bf16x8 (&b)[kSteps][2]) {
#pragma unroll
  for (int k = 0; k < kSteps; k++)
#pragma unroll
    for (int j = 0; j < 2; j++) b[k][j] = frag(w + (n0 + 16 * j + r) * (kSteps * 32), k * 32 + kq);
}

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

// Forward pass of 16 rows per tile and, for training (kTrain), the backward pass to
// the deltas of the first layer.  Four wavefronts, 32 units each; every weight
// fragment a wavefront needs is loaded once, before the first tile.  Latency bounds a
// batch: eight dependent stages of a few MFMAs between barriers; 16 rows a
// workgroup put a batch of 1,024 on 64 CUs.  Without kTrain only y is written, and
// workgroups take several tiles.
template <bool kTrain>
__global__ __launch_bounds__(256) void mlp_rows(RowBatch q, Weights w) {
  __shared__ bf16 s_x[kRowTile * kLdX];
  __shared__ bf16 s_a[2][kRowTile * kLdA];
  __shared__ float s_w4[kHid];
  __shared__ float s_dy[kRowTile];
  const int tid = threadIdx.x, l = tid & 63;
  const int n0 = (tid >> 6) * 32;  // first unit of this wavefront
  const int r = l & 15, kq = (l >> 4) * 8, row4 = (l >> 4) * 4;
  bf16x8 b1[1][2], b2[4][2], b3[4][2], c3[4][2], c2[4][2];
  load_frags(w.w1, n0, r, kq, b1);
  load_frags(w.w2, n0, r, kq, b2);
  load_frags(w.w3, n0, r, kq, b3);
  if (kTrain) {
    load_frags(w.w3t, n0, r, kq, c3);
    load_frags(w.w2t, n0, r, kq, c2);
  }
  float bias[3][2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int col = n0 + 16 * j + r;
    bias[0][j] = w.p[kOffB1 + col];
    bias[1][j] = w.p[kOffB2 + col];
    bias[2][j] = w.p[kOffB3 + col];
  }
  const float b4 = w.p[kOffB4];
  if (tid < kHid) s_w4[tid] = float(w.w4[tid]);
  for (int t0 = blockIdx.x * kRowTile; t0 < q.R; t0 += gridDim.x * kRowTile) {
    {
      const int row = tid >> 4, k = tid & 15, g = t0 + row;
      const bool ok = g < q.n;
      const int64_t s = ok ? (q.idx ? q.idx[g] : g) : 0;
      const bf16 v = bf16(ok ? q.xs[s * kIn + k] : 0.f);
      s_x[row * kLdX + k] = v;
      s_x[row * kLdX + kIn + k] = bf16(0.f);
      if (kTrain) q.xt[int64_t(k) * q.R + g] = v;
    }
    __syncthreads();
    f32x4 acc[2], z[3][2];
    auto layer = [&](int n, bf16 *out) {  // GELU of layer n + 1 from acc
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int col = n0 + 16 * j + r;
        bf16x4 h;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          z[n][j][e] = acc[j][e] + bias[n][j];
          h[e] = bf16(gelu(z[n][j][e]));
          out[(row4 + e) * kLdA + col] = h[e];
        }
        if (kTrain) *reinterpret_cast<bf16x4 *>(q.ht[n] + int64_t(col) * q.R + t0 + row4) = h;
      }
      __syncthreads();
    };
    mma<1>(s_x + r * kLdX, kq, b1, acc);
    layer(0, s_a[0]);
    mma<4>(s_a[0] + r * kLdA, kq, b2, acc);
    layer(1, s_a[1]);
    mma<4>(s_a[1] + r * kLdA, kq, b3, acc);
    layer(2, s_a[0]);
    // output layer: y = h3 . w4 + b4 (FP32, sequential over units), one lane a row
    if (tid < kRowTile) {
      float s = 0.f;
#pragma unroll 4
      for (int k = 0; k < kHid; k += 8) {
        const bf16x8 h = frag(s_a[0] + tid * kLdA, k);
#pragma unroll
        for (int e = 0; e < 8; e++) s += float(h[e]) * s_w4[k + e];
      }
      const float y = s + b4;
      const int g = t0 + tid;
      if (kTrain) {
        const bool ok = g < q.n;
        const float t = ok ? q.ts[q.idx ? q.idx[g] : g] : 0.f;
        const float d = ok ? 2.f * (y - t) / float(q.n) : 0.f;
        s_dy[tid] = d;
        q.dy[g] = d;
        q.sq[g] = (y - t) * (y - t);
      } else if (g < q.n) {
        q.y[g] = y;
      }
    }
    __syncthreads();
    if (kTrain) {
      auto delta = [&](int n, auto value, bf16 *out) {  // deltas of layer n + 1
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const int col = n0 + 16 * j + r;
          bf16x4 h;
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            v[e] = value(j, e, col);
            h[e] = bf16(v[e]);
            if (out) out[(row4 + e) * kLdA + col] = h[e];
          }
          *reinterpret_cast<f32x4 *>(q.et[n] + int64_t(col) * q.R + t0 + row4) = v;
          *reinterpret_cast<bf16x4 *>(q.dt[n] + int64_t(col) * q.R + t0 + row4) = h;
        }
        __syncthreads();
      };
      delta(2, [&](int j, int e, int col) { return s_dy[row4 + e] * s_w4[col] * gelu_grad(z[2][j][e]); }, s_a[1]);
      mma<4>(s_a[1] + r * kLdA, kq, c3, acc);
      delta(1, [&](int j, int e, int) { return acc[j][e] * gelu_grad(z[1][j][e]); }, s_a[0]);
      mma<4>(s_a[0] + r * kLdA, kq, c2, acc);
      delta(0, [&](int j, int e, int) { return acc[j][e] * gelu_grad(z[0][j][e]); }, nullptr);
    }
  }
}

// Adam's constants of one step.
struct AdamStep {
  float lr, b1, b2, eps, c1, c2;
};

// Gradient g of parameter i: stored, or (kAdam) applied to the FP32 master parameter.
// Returns the parameter's value afterwards.
template <bool kAdam>
__device__ inline float take_grad(float g, int64_t i, float *p, float *grad, float *m1, float *m2,
                                  const AdamStep &st) {
  if (!kAdam) {
    grad[i] = g;
    return 0.f;
  }
  const float a = st.b1 * m1[i] + (1.f - st.b1) * g;
  const float b = st.b2 * m2[i] + (1.f - st.b2) * g * g;
  m1[i] = a;
  m2[i] = b;
  const float v = p[i] - st.lr * (a / st.c1) / (sqrtf(b / st.c2) + st.eps);
  p[i] = v;
  return v;
}

// Work of mlp_update's workgroups, in order: 16 x 16 tiles of dW3, dW2 (64 each) and
// dW1 (8), a wavefront a tile; then sums over rows, kSumCols columns a workgroup: the
// biases (3 x 128), the output weights (128), and the output bias with the loss.
constexpr int kTileBlocks = (64 + 64 + 8) / 4;
constexpr int kSumCols = 32, kSumChunk = 1024, kSumLd = kSumChunk + 4;
constexpr int kSumBlocks = 4 * (kHid / kSumCols) + 1;
constexpr int kSumLdsBytes = kSumCols * kSumLd * int(sizeof(float));

// Weight gradients dW[m][n] = sum_rows delta[row][m] act[row][n], bias and output
// gradients, and the loss; with kAdam the parameters and their BF16 copies are
// updated in place, by the owner of each gradient, and loss accumulates the mean
// squared error of the batch.  The tiles take R / 32 dependent MFMAs, eight pairs of
// loads in flight; a sum takes R dependent additions of terms read from LDS.
template <bool kAdam>
__global__ __launch_bounds__(256) void mlp_update(RowBatch q, Weights w, float *grad, float *m1, float *m2,
                                                  AdamStep st, float *loss) {
  extern __shared__ float s_t[];
  const int tid = threadIdx.x, l = tid & 63, R = q.R;
  if (blockIdx.x < kTileBlocks) {
    int tile = blockIdx.x * 4 + (tid >> 6);
    const bf16 *A, *B;
    int64_t off;
    int tn, ld;
    bf16 *wb, *wt;  // BF16 copy, and its transpose where the backward pass reads one
    if (tile < 64) {
      A = q.dt[2], B = q.ht[1], off = kOffW3, tn = tile & 7, tile >>= 3, ld = kHid, wb = w.w3, wt = w.w3t;
    } else if (tile < 128) {
      tile -= 64;
      A = q.dt[1], B = q.ht[0], off = kOffW2, tn = tile & 7, tile >>= 3, ld = kHid, wb = w.w2, wt = w.w2t;
    } else {
      tile -= 128;
      A = q.dt[0], B = q.xt, off = kOffW1, tn = 0, ld = kIn, wb = w.w1, wt = nullptr;
    }
    const int r = l & 15, kq = (l >> 4) * 8;
    const bf16 *pa = A + int64_t(tile * 16 + r) * R + kq, *pb = B + int64_t(tn * 16 + r) * R + kq;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int k0 = 0;
    for (; k0 + 256 <= R; k0 += 256) {
      bf16x8 a[8], b[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        a[u] = frag(pa, k0 + 32 * u);
        b[u] = frag(pb, k0 + 32 * u);
      }
#pragma unroll
      for (int u = 0; u < 8; u++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b[u], acc, 0, 0, 0);
    }
    for (; k0 < R; k0 += 32)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(pa, k0), frag(pb, k0), acc, 0, 0, 0);
    const int n = tn * 16 + r;
    const int ldb = ld == kIn ? kInPad : ld;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int m = tile * 16 + (l >> 4) * 4 + e;
      const float v = take_grad<kAdam>(acc[e], off + int64_t(m) * ld + n, w.p, grad, m1, m2, st);
      if (kAdam) {
        const bf16 h = bf16(v);
        wb[m * ldb + n] = h;
        if (wt) wt[n * kHid + m] = h;
      }
    }
    return;
  }
  const int sb = blockIdx.x - kTileBlocks, kind = sb / (kHid / kSumCols);
  const int c0 = (sb % (kHid / kSumCols)) * kSumCols;
  const int cols = kind == 4 ? 2 : kSumCols;
  float s = 0.f;
  for (int r0 = 0; r0 < R; r0 += kSumChunk) {
    const int m = R - r0 < kSumChunk ? R - r0 : kSumChunk;
    // the chunk's terms, columns row-contiguous
    for (int i = tid * 4; i < cols * m; i += 256 * 4) {
      const int c = i / m, k = i - c * m;  // m is a multiple of 32
      f32x4 v;
      if (kind < 3) {
        v = *reinterpret_cast<const f32x4 *>(q.et[kind] + int64_t(c0 + c) * R + r0 + k);
      } else if (kind == 3) {
        const f32x4 d = *reinterpret_cast<const f32x4 *>(q.dy + r0 + k);
        const bf16x4 h = *reinterpret_cast<const bf16x4 *>(q.ht[2] + int64_t(c0 + c) * R + r0 + k);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = d[e] * float(h[e]);
      } else {
        v = *reinterpret_cast<const f32x4 *>((c == 0 ? q.dy : q.sq) + r0 + k);
      }
      *reinterpret_cast<f32x4 *>(s_t + c * kSumLd + k) = v;
    }
    __syncthreads();
    if (tid < cols) {
      const float *t = s_t + tid * kSumLd;
      // the loss counts the valid rows only
      const int end = kind == 4 && tid == 1 ? (q.n - r0 < m ? (q.n > r0 ? q.n - r0 : 0) : m) : m;
      int k = 0;
      for (; k + 16 <= end; k += 16) {
        f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = *reinterpret_cast<const f32x4 *>(t + k + 4 * u);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
          for (int e = 0; e < 4; e++) s += v[u][e];
      }
      for (; k < end; k++) s += t[k];
    }
    __syncthreads();
  }
  if (tid >= cols) return;
  if (kind == 4 && tid == 1) {
    loss[0] += s / float(q.n);
    return;
  }
  constexpr int64_t kOff[5] = {kOffB1, kOffB2, kOffB3, kOffW4, kOffB4};
  int64_t off = kOff[4];
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (kind == k) off = kOff[k];
  const float v = take_grad<kAdam>(s, off + c0 + tid, w.p, grad, m1, m2, st);
  if (kAdam && kind == 3) w.w4[c0 + tid] = bf16(v);
}

// BF16 weight copies for the GEMMs: W1 padded [128][32], W2, W3 and their transposes, w4.
__global__ void mlp_pack(const float *__restrict__ p, bf16 *__restrict__ w1, bf16 *__restrict__ w2,
                         bf16 *__restrict__ w2t, bf16 *__restrict__ w3, bf16 *__restrict__ w3t,
                         bf16 *__restrict__ w4) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kHid * kInPad) {
    const int n = i / kInPad, k = i % kInPad;
    w1[i] = bf16(k < kIn ? p[kOffW1 + n * kIn + k] : 0.f);
  }
  if (i < kHid * kHid) {
    const int n = i / kHid, k = i % kHid;
    const bf16 a = bf16(p[kOffW2 + i]), b = bf16(p[kOffW3 + i]);
    w2[i] = a;
    w2t[k * kHid + n] = a;
    w3[i] = b;
    w3t[k * kHid + n] = b;
  }
  if (i < kHid) w4[i] = bf16(p[kOffW4 + i]);
}

}  // namespace

struct wg_mlp {
  std::string err;
  hipStream_t stream = nullptr;
  int device = 0;
  Weights w{};
  float *g = nullptr, *m1 = nullptr, *m2 = nullptr, *loss = nullptr;
  int64_t adam_t = 0;
  // batch buffers of R rows, and the samples of a call with their host staging
  // (pinned): kept and grown up to kKeepBatch and kKeepRows rows, larger ones live for
  // one call
  RowBatch q{};
  void *batch = nullptr;
  int R = 0;
  float *dx = nullptr, *dt = nullptr, *stage = nullptr;
  int32_t *didx = nullptr;
  int rows = 0;
};

namespace {

int mlp_fail(wg_mlp *h, int code, const std::string &msg) {
  if (h) h->err = msg;
  return code;
}

#define MLP_CHECK(h, x)                                                              \
  do {                                                                               \
    hipError_t e_ = (x);                                                             \
    if (e_ != hipSuccess) return mlp_fail(h, WG_E_HIP, std::string(#x ": ") + hipGetErrorString(e_)); \
  } while (0)

template <class T>
int mlp_alloc(wg_mlp *h, T **p, size_t n) {
  hipError_t e = hipMalloc(reinterpret_cast<void **>(p), std::max<size_t>(n, 1) * sizeof(T));
  if (e != hipSuccess) return mlp_fail(h, WG_E_NOMEM, "hipMalloc failed");
  e = hipMemsetAsync(*p, 0, std::max<size_t>(n, 1) * sizeof(T), h->stream);
  if (e != hipSuccess) return mlp_fail(h, WG_E_HIP, "hipMemsetAsync failed");
  return WG_OK;
}

// Batch buffers for R rows (a multiple of 32) in one allocation.
int ensure_batch(wg_mlp *h, int R) {
  if (R > h->R) {
    MLP_CHECK(h, hipStreamSynchronize(h->stream));
    if (h->batch) (void)hipFree(h->batch);
    h->batch = nullptr;
    h->R = 0;
    const size_t per_row = kIn * sizeof(bf16) + 6 * kHid * sizeof(bf16) + (3 * kHid + 2) * sizeof(float);
    if (hipMalloc(&h->batch, per_row * R) != hipSuccess) return mlp_fail(h, WG_E_NOMEM, "hipMalloc failed");
    h->R = R;
  }
  char *at = static_cast<char *>(h->batch);
  auto take = [&](auto *&ptr, size_t n) {
    ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(at);
    at += n * sizeof(*ptr) * size_t(h->R);
  };
  for (int k = 0; k < 3; k++) take(h->q.et[k], kHid);
  take(h->q.dy, 1);
  take(h->q.sq, 1);
  for (int k = 0; k < 3; k++) take(h->q.ht[k], kHid);
  for (int k = 0; k < 3; k++) take(h->q.dt[k], kHid);
  take(h->q.xt, kIn);
  return WG_OK;
}

int pack(wg_mlp *h) {
  const Weights &w = h->w;
  hipLaunchKernelGGL(mlp_pack, dim3((kHid * kHid + 255) / 256), dim3(256), 0, h->stream, w.p, w.w1, w.w2, w.w2t, w.w3,
                     w.w3t, w.w4);
  MLP_CHECK(h, hipGetLastError());
  return WG_OK;
}

// Forward pass of `rows` device rows x into y on a stream; workgroups beyond 512 (two
// per CU) would only load the weights again.
int launch_forward(wg_mlp *h, hipStream_t stream, const float *x, int rows, float *y) {
  RowBatch q{};
  q.xs = x;
  q.n = rows;
  q.R = (rows + kRowTile - 1) / kRowTile * kRowTile;
  q.y = y;
  hipLaunchKernelGGL(mlp_rows<false>, dim3(std::min(q.R / kRowTile, 512)), dim3(256), 0, stream, q, h->w);
  MLP_CHECK(h, hipGetLastError());
  return WG_OK;
}

// Forward and backward pass and the gradients of one batch (or Adam's step on them).
int launch_batch(wg_mlp *h, const float *xs, const float *ts, const int32_t *idx, int n, int R, const AdamStep *st) {
  RowBatch q = h->q;
  q.xs = xs;
  q.ts = ts;
  q.idx = idx;
  q.n = n;
  q.R = R;
  hipLaunchKernelGGL(mlp_rows<true>, dim3(R / kRowTile), dim3(256), 0, h->stream, q, h->w);
  auto *update = st ? mlp_update<true> : mlp_update<false>;
  hipLaunchKernelGGL(update, dim3(kTileBlocks + kSumBlocks), dim3(256), kSumLdsBytes, h->stream, q, h->w, h->g, h->m1,
                     h->m2, st ? *st : AdamStep{}, h->loss);
  MLP_CHECK(h, hipGetLastError());
  return WG_OK;
}

int round32(int r) { return (r + 31) / 32 * 32; }

constexpr int kKeepRows = 1 << 18, kKeepBatch = kKeepRows / 8;

void free_samples(wg_mlp *h) {
  void *bufs[] = {h->dx, h->dt, h->didx};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  if (h->stage) (void)hipHostFree(h->stage);
  h->dx = h->dt = h->stage = nullptr;
  h->didx = nullptr;
  h->rows = 0;
}

// Device copies of n samples: h->dx and, with targets, h->dt; up to kKeepRows through
// the pinned staging buffer (free again: a call ends with the stream idle).
int upload_samples(wg_mlp *h, const float *x, const float *t, int n) {
  if (n > h->rows) {
    MLP_CHECK(h, hipStreamSynchronize(h->stream));
    free_samples(h);
    // dt also holds the outputs of a forward pass
    if (hipMalloc(&h->dx, size_t(n) * kIn * sizeof(float)) != hipSuccess ||
        hipMalloc(&h->dt, size_t(n) * sizeof(float)) != hipSuccess ||
        hipMalloc(&h->didx, size_t(n) * sizeof(int32_t)) != hipSuccess ||
        (n <= kKeepRows &&
         hipHostMalloc(&h->stage, size_t(n) * (kIn + 1) * sizeof(float), hipHostMallocDefault) != hipSuccess)) {
      free_samples(h);
      (void)hipGetLastError();
      return mlp_fail(h, WG_E_NOMEM, "sample buffers: out of memory");
    }
    h->rows = n;
  }
  const size_t xb = size_t(n) * kIn * sizeof(float), tb = size_t(n) * sizeof(float);
  if (h->stage) {
    std::memcpy(h->stage, x, xb);
    x = h->stage;
    if (t) t = static_cast<const float *>(std::memcpy(h->stage + size_t(n) * kIn, t, tb));
  }
  MLP_CHECK(h, hipMemcpyAsync(h->dx, x, xb, hipMemcpyHostToDevice, h->stream));
  if (t) MLP_CHECK(h, hipMemcpyAsync(h->dt, t, tb, hipMemcpyHostToDevice, h->stream));
  return WG_OK;
}

// Ends a call: the stream is idle and buffers beyond what a handle keeps are given back.
int end_call(wg_mlp *h, int rc) {
  const hipError_t e = hipStreamSynchronize(h->stream);
  if (h->rows > kKeepRows) free_samples(h);
  if (h->R > kKeepBatch) {
    (void)hipFree(h->batch);
    h->batch = nullptr;
    h->R = 0;
  }
  if (!rc && e != hipSuccess) return mlp_fail(h, WG_E_HIP, std::string("stream: ") + hipGetErrorString(e));
  return rc;
}

}  // namespace

extern "C" int wg_mlp_create(uint64_t seed, wg_mlp **out) {
  if (!out) return WG_E_ARG;
  *out = nullptr;
  wg_mlp *h = new (std::nothrow) wg_mlp();
  if (!h) return WG_E_NOMEM;
  *out = h;
  MLP_CHECK(h, hipGetDevice(&h->device));
  MLP_CHECK(h, hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  int rc = mlp_alloc(h, &h->w.p, kNParams);
  if (!rc) rc = mlp_alloc(h, &h->g, kNParams);
  if (!rc) rc = mlp_alloc(h, &h->m1, kNParams);
  if (!rc) rc = mlp_alloc(h, &h->m2, kNParams);
  if (!rc) rc = mlp_alloc(h, &h->w.w1, size_t(kHid) * kInPad);
  if (!rc) rc = mlp_alloc(h, &h->w.w2, size_t(kHid) * kHid);
  if (!rc) rc = mlp_alloc(h, &h->w.w2t, size_t(kHid) * kHid);
  if (!rc) rc = mlp_alloc(h, &h->w.w3, size_t(kHid) * kHid);
  if (!rc) rc = mlp_alloc(h, &h->w.w3t, size_t(kHid) * kHid);
  if (!rc) rc = mlp_alloc(h, &h->w.w4, kHid);
  if (!rc) rc = mlp_alloc(h, &h->loss, 1);
  if (rc) return rc;
  // He-uniform initial weights from a 64-bit LCG (host), zero biases
  std::vector<float> p(kNParams, 0.f);
  uint64_t s = seed * 6364136223846793005ULL + 1442695040888963407ULL;
  auto uni = [&]() {
    s = s * 6364136223846793005ULL + 1442695040888963407ULL;
    return float((s >> 40) * (1.0 / 16777216.0)) * 2.f - 1.f;
  };
  auto fill = [&](int64_t off, int n_out, int n_in) {
    const float a = std::sqrt(6.f / float(n_in));
    for (int64_t i = 0; i < int64_t(n_out) * n_in; i++) p[off + i] = a * uni();
  };
  fill(kOffW1, kHid, kIn);
  fill(kOffW2, kHid, kHid);
  fill(kOffW3, kHid, kHid);
  fill(kOffW4, 1, kHid);
  MLP_CHECK(h, hipMemcpyAsync(h->w.p, p.data(), kNParams * sizeof(float), hipMemcpyHostToDevice, h->stream));
  rc = pack(h);
  if (rc) return rc;
  MLP_CHECK(h, hipStreamSynchronize(h->stream));
  return WG_OK;
}

extern "C" int wg_mlp_destroy(wg_mlp *h) {
  if (!h) return WG_E_ARG;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  free_samples(h);
  const Weights &w = h->w;
  void *bufs[] = {w.p, w.w1, w.w2, w.w2t, w.w3, w.w3t, w.w4, h->g, h->m1, h->m2, h->loss, h->batch};
  for (void *q : bufs)
    if (q) (void)hipFree(q);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return WG_OK;
}

extern "C" const char *wg_mlp_last_error(const wg_mlp *h) { return h ? h->err.c_str() : "null handle"; }

extern "C" int64_t wg_mlp_n_params(void) { return kNParams; }

extern "C" int wg_mlp_get_params(wg_mlp *h, float *out) {
  if (!h || !out) return WG_E_ARG;
  MLP_CHECK(h, hipMemcpyAsync(out, h->w.p, kNParams * sizeof(float), hipMemcpyDeviceToHost, h->stream));
  MLP_CHECK(h, hipStreamSynchronize(h->stream));
  return WG_OK;
}

extern "C" int wg_mlp_set_params(wg_mlp *h, const float *in) {
  if (!h || !in) return WG_E_ARG;
  MLP_CHECK(h, hipMemcpyAsync(h->w.p, in, kNParams * sizeof(float), hipMemcpyHostToDevice, h->stream));
  int rc = pack(h);
  if (rc) return rc;
  MLP_CHECK(h, hipStreamSynchronize(h->stream));
  return WG_OK;
}

extern "C" int wg_mlp_forward(wg_mlp *h, int32_t rows, const float *x, float *y) {
  if (!h || rows <= 0 || !x || !y) return WG_E_ARG;
  int rc = upload_samples(h, x, nullptr, rows);
  if (!rc) rc = launch_forward(h, h->stream, h->dx, rows, h->dt);
  // the outputs come back through the staging buffer's second part
  float *st = rc || !h->stage ? y : h->stage + size_t(rows) * kIn;
  if (!rc && hipMemcpyAsync(st, h->dt, size_t(rows) * sizeof(float), hipMemcpyDeviceToHost, h->stream) != hipSuccess)
    rc = mlp_fail(h, WG_E_HIP, "forward copy");
  if (!rc) {
    const hipError_t e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) rc = mlp_fail(h, WG_E_HIP, std::string("forward: ") + hipGetErrorString(e));
  }
  if (!rc && st != y) std::memcpy(y, st, size_t(rows) * sizeof(float));
  return end_call(h, rc);
}

extern "C" int wg_mlp_forward_noalloc(wg_mlp *h, int32_t rows, const float *x, float *y, void *stream) {
  if (!h || !x || !y) return WG_E_ARG;
  if (rows <= 0 || rows > WG_MLP_NOALLOC_MAX_ROWS)
    return mlp_fail(h, WG_E_ARG, "wg_mlp_forward_noalloc: rows must be 1.." + std::to_string(WG_MLP_NOALLOC_MAX_ROWS) +
                                     ", got " + std::to_string(rows));
  return launch_forward(h, stream ? static_cast<hipStream_t>(stream) : h->stream, x, rows, y);
}

extern "C" int wg_mlp_gradient(wg_mlp *h, int32_t rows, const float *x, const float *t, float *loss, float *grad) {
  if (!h || rows <= 0 || !x || !t || !grad) return WG_E_ARG;
  const int R = round32(rows);
  int rc = upload_samples(h, x, t, rows);
  if (!rc) rc = ensure_batch(h, R);
  if (!rc && hipMemsetAsync(h->loss, 0, sizeof(float), h->stream) != hipSuccess) rc = mlp_fail(h, WG_E_HIP, "loss");
  if (!rc) rc = launch_batch(h, h->dx, h->dt, nullptr, rows, R, nullptr);
  if (!rc) {
    hipError_t e = hipMemcpyAsync(grad, h->g, kNParams * sizeof(float), hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess && loss) e = hipMemcpyAsync(loss, h->loss, sizeof(float), hipMemcpyDeviceToHost, h->stream);
    if (e != hipSuccess) rc = mlp_fail(h, WG_E_HIP, "gradient copy");
  }
  return end_call(h, rc);
}

extern "C" int wg_mlp_train(wg_mlp *h, int32_t n_samples, const float *x, const float *t, int32_t epochs,
                            int32_t batch, float lr, uint64_t seed, float *epoch_loss) {
  if (!h || n_samples <= 0 || !x || !t || epochs <= 0 || batch < 32 || batch % 32) return WG_E_ARG;
  int rc = upload_samples(h, x, t, n_samples);
  if (!rc) rc = ensure_batch(h, std::min(batch, round32(n_samples)));
  std::vector<int32_t> perm(n_samples);
  for (int i = 0; i < n_samples; i++) perm[i] = i;
  uint64_t s = seed ^ 0x9E3779B97F4A7C15ULL;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int ep = 0; !rc && ep < epochs; ep++) {
    // Fisher-Yates shuffle of the sample order (host)
    for (int i = n_samples - 1; i > 0; i--) {
      s = s * 6364136223846793005ULL + 1442695040888963407ULL;
      const int j = int((s >> 33) % uint64_t(i + 1));
      std::swap(perm[i], perm[j]);
    }
    hipError_t e = hipMemcpyAsync(h->didx, perm.data(), n_samples * sizeof(int32_t), hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess) e = hipMemsetAsync(h->loss, 0, sizeof(float), h->stream);
    if (e != hipSuccess) { rc = mlp_fail(h, WG_E_HIP, "epoch setup"); break; }
    int n_batches = 0;
    for (int r0 = 0; r0 < n_samples; r0 += batch) {
      const int n = std::min(batch, n_samples - r0);
      h->adam_t++;
      const float c1 = 1.f - std::pow(b1, float(h->adam_t)), c2 = 1.f - std::pow(b2, float(h->adam_t));
      const AdamStep st{lr, b1, b2, eps, c1, c2};
      rc = launch_batch(h, h->dx, h->dt, h->didx + r0, n, round32(n), &st);
      if (rc) break;
      n_batches++;
    }
    if (rc) break;
    float l = 0.f;
    e = hipMemcpyAsync(&l, h->loss, sizeof(float), hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) { rc = mlp_fail(h, WG_E_HIP, "loss copy"); break; }
    if (epoch_loss) epoch_loss[ep] = l / float(std::max(n_batches, 1));
  }
  return end_call(h, rc);
}
