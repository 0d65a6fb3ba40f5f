// rk_mlp.hip -- the rebuild-interval proposal network: an MLP
// 16 -> 64 (tanh) -> 64 (tanh) -> 1 in FP32, with its forward, backward and
// Adam kernels.  It has no counterpart in the reference: it only chooses how
// many iterations the host enqueues before it reads the device displacement
// guard (rk_engine.cpp run_guarded), so it never changes a result.
//
// Parameters, one float array of kMlpParams:
//   W1[64][16] b1[64] W2[64][64] b2[64] W3[64] b3[1]
// Training: k_mlp_pass computes a tile of 16 samples' activations and
// back-propagated deltas per workgroup; k_mlp_grad then sums each parameter's
// gradient over chunks of 256 samples, in sample order within a chunk and
// the chunks' sums in order (k_mlp_reduce), so gradients are deterministic.
// A batch of one chunk takes its Adam step in k_mlp_grad itself, a larger one
// in k_mlp_adam.  Loss = mean of (y - t)^2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/rockable_amd.h"

namespace {

constexpr int kIn = 16, kH = 64;
constexpr int oW1 = 0, oB1 = oW1 + kH * kIn, oW2 = oB1 + kH, oB2 = oW2 + kH * kH, oW3 = oB2 + kH, oB3 = oW3 + kH;
constexpr int kMlpParams = oB3 + 1;  // 5313
constexpr int kBlock = 256;

static_assert(oW2 % 4 == 0 && oW1 % 4 == 0, "the weights are read as float4");
constexpr int kTile = 16;    // samples per workgroup of k_mlp_pass
constexpr int kChunk = 256;  // samples per gradient chunk
constexpr int kPad = kH + 1; // LDS row of a transposed weight matrix

enum { MLP_FORWARD, MLP_LOSS, MLP_GRAD };

// The network on a tile of 16 samples (rows idx[s] of X, or s without idx):
// its output (MLP_FORWARD), its squared errors (MLP_LOSS), or with those the
// activations h1, h2, the deltas d1, d2 (dL/d pre-activation) and
// e = dL/dy = 2 (y - t) / n that the gradient sums over (MLP_GRAD).
// Thread (j, g) computes unit j of samples 4 g .. 4 g + 3: the weights lie
// transposed in LDS (rows of 65, so that both the forward's reads along j
// and the backward's along i fall on different banks), the four samples'
// inputs come as one broadcast 16-byte read, and each weight read serves
// four multiply-adds.  Every sum keeps the order of the plain loops (bias
// first, then the inputs in turn).  Bound by LDS reads and the latency of its
// five dependent stages.  One thread per sample, its activations in scratch
// memory and only n / 256 workgroups, took 87 us for a minibatch of 256 and
// 101 us for 20 000 samples; this takes 9.3 us and 29 us.
template <int MODE>
__global__ void __launch_bounds__(kBlock) k_mlp_pass(const float* __restrict__ P, const float* __restrict__ X,
                                                     const float* __restrict__ T, const int32_t* __restrict__ idx,
                                                     int n, float* __restrict__ Y, float* __restrict__ H1,
                                                     float* __restrict__ H2, float* __restrict__ D1,
                                                     float* __restrict__ D2, float* __restrict__ E,
                                                     float* __restrict__ SQ) {
  __shared__ float w1[kIn * kPad], w2[kH * kPad], rest[3 * kH + 1];  // rest: b1 b2 W3 b3
  __shared__ __align__(16) float sx[kIn * kTile], sh1[kH * kTile], sh2[kH * kTile], sd2[kH * kTile];
  __shared__ float se[kTile];
  const int t = threadIdx.x, j = t & (kH - 1), s4 = 4 * (t >> 6);
  const int s0 = blockIdx.x * kTile;
  // every global load first (the sample's index, then its row, last), so that
  // one latency covers the weights
  const int s = t / kIn, i = t % kIn;  // 16 samples of 16 inputs: one each
  const bool live = s0 + s < n;
  const int row = live ? (idx ? idx[s0 + s] : s0 + s) : 0;
  const float4 v1 = *reinterpret_cast<const float4*>(P + oW1 + 4 * t);
  float4 v2[4];
#pragma unroll
  for (int k = 0; k < 4; k++) v2[k] = *reinterpret_cast<const float4*>(P + oW2 + 4 * (t + kBlock * k));
  if (t < kH) {
    rest[t] = P[oB1 + t];
    rest[kH + t] = P[oB2 + t];
    rest[2 * kH + t] = P[oW3 + t];
    if (t == 0) rest[3 * kH] = P[oB3];
  }
  const float xv = live ? X[(size_t)row * kIn + i] : 0.0f;
  {
    const int r = t / 4, c = 4 * (t % 4);  // row r of W1, columns c ...
    w1[c * kPad + r] = v1.x;
    w1[(c + 1) * kPad + r] = v1.y;
    w1[(c + 2) * kPad + r] = v1.z;
    w1[(c + 3) * kPad + r] = v1.w;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int r = t / 16 + 16 * k, c = 4 * (t % 16);
    w2[c * kPad + r] = v2[k].x;
    w2[(c + 1) * kPad + r] = v2[k].y;
    w2[(c + 2) * kPad + r] = v2[k].z;
    w2[(c + 3) * kPad + r] = v2[k].w;
  }
  sx[i * kTile + s] = xv;
  __syncthreads();
  float a[4], h1[4], h2[4];
#pragma unroll
  for (int k = 0; k < 4; k++) a[k] = rest[j];
#pragma unroll
  for (int i = 0; i < kIn; i++) {
    const float w = w1[i * kPad + j];
    const float4 x = *reinterpret_cast<const float4*>(sx + i * kTile + s4);
    a[0] += w * x.x;
    a[1] += w * x.y;
    a[2] += w * x.z;
    a[3] += w * x.w;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) h1[k] = tanhf(a[k]);
  *reinterpret_cast<float4*>(sh1 + j * kTile + s4) = make_float4(h1[0], h1[1], h1[2], h1[3]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; k++) a[k] = rest[kH + j];
#pragma unroll 16
  for (int i = 0; i < kH; i++) {
    const float w = w2[i * kPad + j];
    const float4 x = *reinterpret_cast<const float4*>(sh1 + i * kTile + s4);
    a[0] += w * x.x;
    a[1] += w * x.y;
    a[2] += w * x.z;
    a[3] += w * x.w;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) h2[k] = tanhf(a[k]);
  *reinterpret_cast<float4*>(sh2 + j * kTile + s4) = make_float4(h2[0], h2[1], h2[2], h2[3]);
  __syncthreads();
  if (t < kTile) {
    float y = rest[3 * kH];
#pragma unroll 16
    for (int i = 0; i < kH; i++) y += rest[2 * kH + i] * sh2[i * kTile + t];
    if (s0 + t < n) {
      if (MODE == MLP_FORWARD) {
        Y[s0 + t] = y;
      } else {
        const float r = y - T[idx ? idx[s0 + t] : s0 + t];
        const float e = 2.0f * r / (float)n;
        SQ[s0 + t] = r * r;
        if (MODE == MLP_GRAD) {
          E[s0 + t] = e;
          se[t] = e;
        }
      }
    }
  }
  if (MODE != MLP_GRAD) return;
  __syncthreads();
  float d2[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const bool in = s0 + s4 + k < n;
    d2[k] = in ? se[s4 + k] * rest[2 * kH + j] * (1.0f - h2[k] * h2[k]) : 0.0f;
    if (in) {
      const size_t o = (size_t)(s0 + s4 + k) * kH + j;
      H1[o] = h1[k];
      H2[o] = h2[k];
      D2[o] = d2[k];
    }
  }
  *reinterpret_cast<float4*>(sd2 + j * kTile + s4) = make_float4(d2[0], d2[1], d2[2], d2[3]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; k++) a[k] = 0.0f;
#pragma unroll 16
  for (int q = 0; q < kH; q++) {  // unit j's delta: over the second layer's units q
    const float w = w2[j * kPad + q];
    const float4 x = *reinterpret_cast<const float4*>(sd2 + q * kTile + s4);
    a[0] += w * x.x;
    a[1] += w * x.y;
    a[2] += w * x.z;
    a[3] += w * x.w;
  }
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (s0 + s4 + k < n) D1[(size_t)(s0 + s4 + k) * kH + j] = a[k] * (1.0f - h1[k] * h1[k]);
}

struct AdamArgs {
  float *P, *M, *V;
  float lr, b1t, b2t;
};
__device__ __forceinline__ void adam_update(const AdamArgs& A, int q, float g) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float m = b1 * A.M[q] + (1.0f - b1) * g;
  const float v = b2 * A.V[q] + (1.0f - b2) * g * g;
  A.M[q] = m;
  A.V[q] = v;
  A.P[q] -= A.lr * (m / (1.0f - A.b1t)) / (sqrtf(v / (1.0f - A.b2t)) + eps);
}

// The gradient of the samples [256 c, 256 c + 256) of a chunk c, each
// parameter summed in sample order by one thread from operands staged
// in LDS: workgroups 0-15 take the 16 x 16 blocks of W2, 16-19 those of W1,
// 20-22 b1, b2 and W3 with b3 and the loss (the last column).  Chunk c's sums
// go to out[c kOut ...], or with ADAM (one chunk) straight into the
// parameters.  Bound by latency: the staging loads, then 256 dependent
// additions; blocks of 16 x 16 give 23 workgroups per chunk, so that a
// minibatch spreads over 23 CUs and 20 000 samples fill the chip.  One
// thread per parameter over all samples, its operands from memory at every
// sample, took 85 us for a minibatch of 256 and 5.1 ms for 20 000 samples;
// this takes 7.7 us (the Adam step in it) and 23 us.
constexpr int kOut = kMlpParams + 1;  // a chunk's sums: the parameters, then the loss
constexpr int kGradTiles = 23;
template <bool ADAM>
__global__ void __launch_bounds__(kBlock) k_mlp_grad(const float* __restrict__ X, const int32_t* __restrict__ idx, int n,
                                                     const float* __restrict__ H1, const float* __restrict__ H2,
                                                     const float* __restrict__ D1, const float* __restrict__ D2,
                                                     const float* __restrict__ E, const float* __restrict__ SQ,
                                                     float* __restrict__ out, AdamArgs A) {
  __shared__ float sa[kChunk * 16], sb[kChunk * 16], sc[kChunk];
  const int t = threadIdx.x, b = blockIdx.x % kGradTiles, chunk = blockIdx.x / kGradTiles;
  const int s0 = chunk * kChunk, m = min(kChunk, n - s0);
  float* o = out + (size_t)chunk * kOut;
  if (b < 20) {
    const bool second = b < 16;
    const int j0 = second ? (b >> 2) * 16 : (b - 16) * 16, i0 = second ? (b & 3) * 16 : 0;
    const float* D = second ? D2 : D1;
    const int r = t >> 4, c = t & 15;
    // (rows past the last sample repeat it, so that all loads go out at
    // once without a branch; the sum stops at m)
    float xa[16], xb[16];
#pragma unroll
    for (int k = 0; k < 16; k++) xa[k] = D[(size_t)(s0 + min(16 * k + r, m - 1)) * kH + j0 + c];
    if (second) {
#pragma unroll
      for (int k = 0; k < 16; k++) xb[k] = H1[(size_t)(s0 + min(16 * k + r, m - 1)) * kH + i0 + c];
    } else {
      int row[16];
#pragma unroll
      for (int k = 0; k < 16; k++) {
        row[k] = s0 + min(16 * k + r, m - 1);
        if (idx) row[k] = idx[row[k]];
      }
#pragma unroll
      for (int k = 0; k < 16; k++) xb[k] = X[(size_t)row[k] * kIn + c];
    }
#pragma unroll
    for (int k = 0; k < 16; k++) {
      sa[(16 * k + r) * 16 + c] = xa[k];
      sb[(16 * k + r) * 16 + c] = xb[k];
    }
    __syncthreads();
    float g = 0.0f;
#pragma unroll 16
    for (int s = 0; s < m; s++) g += sa[s * 16 + r] * sb[s * 16 + c];
    const int q = second ? oW2 + (j0 + r) * kH + i0 + c : oW1 + (j0 + r) * kIn + c;
    if (ADAM)
      adam_update(A, q, g);
    else
      o[q] = g;
    return;
  }
  // a column sum per thread of 64: D1, D2, or E H2; in two pieces of 128 samples
  const float* src = b == 20 ? D1 : b == 21 ? D2 : H2;
  float e = 0.0f, sq = 0.0f;
  if (b == 22) {
    e = E[s0 + min(t, m - 1)];
    if (!ADAM) sq = SQ[s0 + min(t, m - 1)];
    sc[t] = e;
  }
  float g = 0.0f;
  for (int p = 0; p < m; p += 128) {
    const int len = min(128, m - p);
    float x[32];
#pragma unroll
    for (int k = 0; k < 32; k++) x[k] = src[(size_t)(s0 + min(p + 4 * k + (t >> 6), m - 1)) * kH + (t & 63)];
    __syncthreads();  // the last piece's sums are done
#pragma unroll
    for (int k = 0; k < 32; k++) {
      const int s = 4 * k + (t >> 6);
      (s < 64 ? sa : sb)[(s & 63) * kH + (t & 63)] = x[k];
    }
    __syncthreads();
    if (t < kH) {
      for (int h = 0; h < len; h += 64) {
        const float* tile = h ? sb : sa;
        const int end = min(64, len - h);
        if (b == 22) {
#pragma unroll 16
          for (int s = 0; s < end; s++) g += sc[p + h + s] * tile[s * kH + t];
        } else {
#pragma unroll 16
          for (int s = 0; s < end; s++) g += tile[s * kH + t];
        }
      }
    }
  }
  if (t < kH) {
    const int q = (b == 20 ? oB1 : b == 21 ? oB2 : oW3) + t;
    if (ADAM)
      adam_update(A, q, g);
    else
      o[q] = g;
  }
  if (b != 22) return;
  // b3: the sum of E; then the loss: the sum of the squared errors
  __syncthreads();
  sb[t] = sq;
  __syncthreads();
  if (t == 0) {
    g = 0.0f;
#pragma unroll 16
    for (int s = 0; s < m; s++) g += sc[s];
    if (ADAM)
      adam_update(A, oB3, g);
    else
      o[oB3] = g;
  } else if (!ADAM && t == 64) {
    g = 0.0f;
#pragma unroll 16
    for (int s = 0; s < m; s++) g += sb[s];
    o[kMlpParams] = g;
  }
}

// The chunks' sums added in order; the loss (the last column) over n.
__global__ void __launch_bounds__(64) k_mlp_reduce(const float* __restrict__ part, int chunks, int n,
                                                   float* __restrict__ G, float* __restrict__ loss) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q > kMlpParams) return;
  float g = part[q];
#pragma unroll 16
  for (int c = 1; c < chunks; c++) g += part[(size_t)c * kOut + q];
  if (q == kMlpParams)
    *loss = g / (float)n;
  else
    G[q] = g;
}

// The loss alone: the sums of 256 squared errors, then as k_mlp_reduce.
__global__ void __launch_bounds__(kBlock) k_mlp_loss(const float* __restrict__ SQ, int n, float* __restrict__ loss) {
  __shared__ float s[kBlock];
  const int chunks = (n + kChunk - 1) / kChunk;
  float total = 0.0f;
  for (int c0 = 0; c0 < chunks; c0 += kBlock) {
    const int c = c0 + (int)threadIdx.x;
    float g = 0.0f;
    if (c < chunks) {
      const int end = min(n, (c + 1) * kChunk);
#pragma unroll 16
      for (int k = c * kChunk; k < end; k++) g += SQ[k];
    }
    s[threadIdx.x] = g;
    __syncthreads();
    if (threadIdx.x == 0)
      for (int k = 0; k < min(kBlock, chunks - c0); k++) total += s[k];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = total / (float)n;
}

__global__ void __launch_bounds__(kBlock) k_mlp_adam(const float* __restrict__ G, AdamArgs A) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < kMlpParams) adam_update(A, q, G[q]);
}

inline int nblk(long n) { return (int)((n + kBlock - 1) / kBlock); }

}  // namespace

struct rk_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  float* P = nullptr;  // parameters
  float *M = nullptr, *V = nullptr, *G = nullptr, *loss = nullptr;
  int64_t adam_t = 0;
  // sample buffers
  size_t cap = 0;
  float *X = nullptr, *T = nullptr, *Y = nullptr, *H1 = nullptr, *H2 = nullptr, *D1 = nullptr, *D2 = nullptr,
        *E = nullptr, *SQ = nullptr;
  // the gradient chunks' sums, and the training's sample order: one epoch's
  // on the device in each of two slots, from pinned host memory
  size_t part_cap = 0, order_cap = 0;
  float* part = nullptr;
  int32_t *order = nullptr, *order_host = nullptr;
  hipEvent_t order_ev[2] = {};
};

namespace {

int mfail(rk_mlp* m, const std::string& s) {
  if (m) m->err = s;
  return -1;
}
#define MCHK(x)                                                                          \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) return mfail(mlp, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

int reserve(rk_mlp* mlp, size_t n) {
  if (n <= mlp->cap) return 0;
  float** bufs[] = {&mlp->X, &mlp->T, &mlp->Y, &mlp->H1, &mlp->H2, &mlp->D1, &mlp->D2, &mlp->E, &mlp->SQ};
  for (float** b : bufs)
    if (*b) (void)hipFree(*b);
  const size_t c = n + n / 2 + 64;
  const size_t sz[] = {kIn, 1, 1, kH, kH, kH, kH, 1, 1};
  for (int k = 0; k < 9; k++) MCHK(hipMalloc(bufs[k], c * sz[k] * sizeof(float)));
  mlp->cap = c;
  return 0;
}

// the gradient chunks' sums of n samples
int reserve_part(rk_mlp* mlp, size_t n) {
  const size_t need = (n + kChunk - 1) / kChunk;
  if (need <= mlp->part_cap) return 0;
  if (mlp->part) (void)hipFree(mlp->part);
  mlp->part = nullptr;
  mlp->part_cap = 0;
  MCHK(hipMalloc(&mlp->part, need * kOut * sizeof(float)));
  mlp->part_cap = need;
  return 0;
}

// two epochs' sample orders
int reserve_order(rk_mlp* mlp, size_t n) {
  for (hipEvent_t& e : mlp->order_ev)
    if (!e) MCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (n <= mlp->order_cap) return 0;
  if (mlp->order) (void)hipFree(mlp->order);
  if (mlp->order_host) (void)hipHostFree(mlp->order_host);
  mlp->order = mlp->order_host = nullptr;
  mlp->order_cap = 0;
  MCHK(hipMalloc(&mlp->order, 2 * n * sizeof(int32_t)));
  MCHK(hipHostMalloc((void**)&mlp->order_host, 2 * n * sizeof(int32_t), hipHostMallocDefault));
  mlp->order_cap = n;
  return 0;
}

int npass(int n) { return (n + kTile - 1) / kTile; }
int nchunks(int n) { return (n + kChunk - 1) / kChunk; }

// loss and gradient (into loss, G) of n samples: rows idx[s] (or s) of X, T
void launch_gradient(rk_mlp* mlp, const int32_t* idx, int n) {
  hipLaunchKernelGGL(k_mlp_pass<MLP_GRAD>, dim3(npass(n)), dim3(kBlock), 0, mlp->stream, mlp->P, mlp->X, mlp->T, idx, n,
                     mlp->Y, mlp->H1, mlp->H2, mlp->D1, mlp->D2, mlp->E, mlp->SQ);
  hipLaunchKernelGGL(k_mlp_grad<false>, dim3(kGradTiles * nchunks(n)), dim3(kBlock), 0, mlp->stream, mlp->X, idx, n,
                     mlp->H1, mlp->H2, mlp->D1, mlp->D2, mlp->E, mlp->SQ, mlp->part, AdamArgs{});
  hipLaunchKernelGGL(k_mlp_reduce, dim3((kOut + 63) / 64), dim3(64), 0, mlp->stream, mlp->part, nchunks(n), n, mlp->G,
                     mlp->loss);
}

// one Adam step on the n samples idx[0..n) of X, T.  Up to one chunk the
// gradient kernel takes the step itself: two launches instead of four.
int adam_step(rk_mlp* mlp, const int32_t* idx, int n, float lr) {
  mlp->adam_t++;
  AdamArgs A;
  A.P = mlp->P;
  A.M = mlp->M;
  A.V = mlp->V;
  A.lr = lr;
  A.b1t = (float)std::pow(0.9, (double)mlp->adam_t);
  A.b2t = (float)std::pow(0.999, (double)mlp->adam_t);
  if (n <= kChunk) {
    hipLaunchKernelGGL(k_mlp_pass<MLP_GRAD>, dim3(npass(n)), dim3(kBlock), 0, mlp->stream, mlp->P, mlp->X, mlp->T, idx,
                       n, mlp->Y, mlp->H1, mlp->H2, mlp->D1, mlp->D2, mlp->E, mlp->SQ);
    hipLaunchKernelGGL(k_mlp_grad<true>, dim3(kGradTiles), dim3(kBlock), 0, mlp->stream, mlp->X, idx, n, mlp->H1,
                       mlp->H2, mlp->D1, mlp->D2, mlp->E, mlp->SQ, mlp->part, A);
  } else {
    launch_gradient(mlp, idx, n);
    hipLaunchKernelGGL(k_mlp_adam, dim3(nblk(kMlpParams)), dim3(kBlock), 0, mlp->stream, mlp->G, A);
  }
  MCHK(hipGetLastError());
  return 0;
}

}  // namespace

// device entry used by the engine: y[0] = MLP(x) for one feature vector
// already on the device, on the given stream
int rk_mlp_forward_device(rk_mlp* mlp, const float* x_dev, float* y_dev, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_pass<MLP_FORWARD>, dim3(1), dim3(kBlock), 0, s, mlp->P, x_dev, nullptr, nullptr, 1, y_dev,
                     nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" {

int rk_mlp_create(rk_mlp** out, int device, uint64_t seed) {
  if (!out) return -1;
  *out = nullptr;
  int nd = 0;
  if (hipGetDeviceCount(&nd) != hipSuccess || device < 0 || device >= nd) return -2;
  if (hipSetDevice(device) != hipSuccess) return -2;
  rk_mlp* mlp = new rk_mlp();
  mlp->device = device;
  if (hipStreamCreate(&mlp->stream) != hipSuccess) {
    delete mlp;
    return -2;
  }
  // Glorot-uniform weights, zero biases
  std::vector<float> p(kMlpParams, 0.0f);
  std::mt19937_64 rng(seed);
  auto fill = [&](int off, int fan_out, int fan_in) {
    const float a = std::sqrt(6.0f / (float)(fan_in + fan_out));
    std::uniform_real_distribution<float> u(-a, a);
    for (int k = 0; k < fan_out * fan_in; k++) p[off + k] = u(rng);
  };
  fill(oW1, kH, kIn);
  fill(oW2, kH, kH);
  fill(oW3, 1, kH);
  std::vector<float> zero(kMlpParams, 0.0f);
  if (hipMalloc(&mlp->P, kMlpParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&mlp->M, kMlpParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&mlp->V, kMlpParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&mlp->G, kMlpParams * sizeof(float)) != hipSuccess ||
      hipMalloc(&mlp->loss, sizeof(float)) != hipSuccess ||
      hipMemcpy(mlp->P, p.data(), kMlpParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(mlp->M, zero.data(), kMlpParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(mlp->V, zero.data(), kMlpParams * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
    rk_mlp_destroy(mlp);
    return -2;
  }
  *out = mlp;
  return 0;
}

void rk_mlp_destroy(rk_mlp* mlp) {
  if (!mlp) return;
  float* bufs[] = {mlp->P, mlp->M, mlp->V, mlp->G, mlp->loss, mlp->X, mlp->T, mlp->Y,
                   mlp->H1, mlp->H2, mlp->D1, mlp->D2, mlp->E, mlp->SQ, mlp->part};
  for (float* b : bufs)
    if (b) (void)hipFree(b);
  if (mlp->order) (void)hipFree(mlp->order);
  if (mlp->order_host) (void)hipHostFree(mlp->order_host);
  for (hipEvent_t e : mlp->order_ev)
    if (e) (void)hipEventDestroy(e);
  if (mlp->stream) (void)hipStreamDestroy(mlp->stream);
  delete mlp;
}

const char* rk_mlp_last_error(const rk_mlp* mlp) { return mlp ? mlp->err.c_str() : "null model"; }

int rk_mlp_nparams(void) { return kMlpParams; }

int rk_mlp_get_params(rk_mlp* mlp, float* out, size_t n) {
  if (!mlp || !out || n < (size_t)kMlpParams) return mfail(mlp, "rk_mlp_get_params: buffer too small");
  MCHK(hipStreamSynchronize(mlp->stream));
  MCHK(hipMemcpy(out, mlp->P, kMlpParams * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int rk_mlp_set_params(rk_mlp* mlp, const float* in, size_t n) {
  if (!mlp || !in || n < (size_t)kMlpParams) return mfail(mlp, "rk_mlp_set_params: buffer too small");
  MCHK(hipStreamSynchronize(mlp->stream));
  MCHK(hipMemcpy(mlp->P, in, kMlpParams * sizeof(float), hipMemcpyHostToDevice));
  std::vector<float> zero(kMlpParams, 0.0f);
  MCHK(hipMemcpy(mlp->M, zero.data(), kMlpParams * sizeof(float), hipMemcpyHostToDevice));
  MCHK(hipMemcpy(mlp->V, zero.data(), kMlpParams * sizeof(float), hipMemcpyHostToDevice));
  mlp->adam_t = 0;
  return 0;
}

int rk_mlp_forward(rk_mlp* mlp, const float* X, size_t n, float* y) {
  if (!mlp || (!X && n) || (!y && n)) return -1;
  if (n == 0) return 0;
  (void)hipSetDevice(mlp->device);
  if (reserve(mlp, n)) return -1;
  MCHK(hipMemcpyAsync(mlp->X, X, n * kIn * sizeof(float), hipMemcpyHostToDevice, mlp->stream));
  hipLaunchKernelGGL(k_mlp_pass<MLP_FORWARD>, dim3(npass((int)n)), dim3(kBlock), 0, mlp->stream, mlp->P, mlp->X, nullptr,
                     nullptr, (int)n, mlp->Y, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
  MCHK(hipGetLastError());
  MCHK(hipMemcpyAsync(y, mlp->Y, n * sizeof(float), hipMemcpyDeviceToHost, mlp->stream));
  MCHK(hipStreamSynchronize(mlp->stream));
  return 0;
}

int rk_mlp_loss_grad(rk_mlp* mlp, const float* X, const float* t, size_t n, float* loss, float* grad) {
  if (!mlp || !X || !t || n == 0) return mfail(mlp, "rk_mlp_loss_grad: empty input");
  (void)hipSetDevice(mlp->device);
  if (reserve(mlp, n) || reserve_part(mlp, n)) return -1;
  MCHK(hipMemcpyAsync(mlp->X, X, n * kIn * sizeof(float), hipMemcpyHostToDevice, mlp->stream));
  MCHK(hipMemcpyAsync(mlp->T, t, n * sizeof(float), hipMemcpyHostToDevice, mlp->stream));
  launch_gradient(mlp, nullptr, (int)n);
  MCHK(hipGetLastError());
  if (grad) MCHK(hipMemcpyAsync(grad, mlp->G, kMlpParams * sizeof(float), hipMemcpyDeviceToHost, mlp->stream));
  if (loss) MCHK(hipMemcpyAsync(loss, mlp->loss, sizeof(float), hipMemcpyDeviceToHost, mlp->stream));
  MCHK(hipStreamSynchronize(mlp->stream));
  return 0;
}

int rk_mlp_train(rk_mlp* mlp, const float* X, const float* t, size_t n, int epochs, int batch, float lr,
                 uint64_t seed, float* final_loss) {
  if (!mlp || !X || !t || n == 0 || epochs < 1 || batch < 1) return mfail(mlp, "rk_mlp_train: bad arguments");
  (void)hipSetDevice(mlp->device);
  const size_t b = std::min<size_t>((size_t)batch, n);
  if (reserve(mlp, n) || reserve_part(mlp, b) || reserve_order(mlp, n)) return -1;
  // the samples go to the device once; each epoch sends its shuffled order
  // and the minibatches read their rows through it, so that nothing waits
  // between two Adam steps (copying each minibatch and waiting for it took
  // 30 us a step)
  MCHK(hipMemcpyAsync(mlp->X, X, n * kIn * sizeof(float), hipMemcpyHostToDevice, mlp->stream));
  MCHK(hipMemcpyAsync(mlp->T, t, n * sizeof(float), hipMemcpyHostToDevice, mlp->stream));
  std::vector<size_t> order(n);
  for (size_t k = 0; k < n; k++) order[k] = k;
  std::mt19937_64 rng(seed);
  for (int ep = 0; ep < epochs; ep++) {
    std::shuffle(order.begin(), order.end(), rng);
    int32_t* host = mlp->order_host + (size_t)(ep & 1) * n;
    int32_t* dev = mlp->order + (size_t)(ep & 1) * n;
    if (ep >= 2) MCHK(hipEventSynchronize(mlp->order_ev[ep & 1]));  // the slot's last epoch is done
    for (size_t k = 0; k < n; k++) host[k] = (int32_t)order[k];
    MCHK(hipMemcpyAsync(dev, host, n * sizeof(int32_t), hipMemcpyHostToDevice, mlp->stream));
    for (size_t s0 = 0; s0 + b <= n; s0 += b)
      if (adam_step(mlp, dev + s0, (int)b, lr)) return -1;
    MCHK(hipEventRecord(mlp->order_ev[ep & 1], mlp->stream));
  }
  float l = 0.0f;
  if (final_loss) {
    hipLaunchKernelGGL(k_mlp_pass<MLP_LOSS>, dim3(npass((int)n)), dim3(kBlock), 0, mlp->stream, mlp->P, mlp->X, mlp->T,
                       nullptr, (int)n, mlp->Y, nullptr, nullptr, nullptr, nullptr, nullptr, mlp->SQ);
    hipLaunchKernelGGL(k_mlp_loss, dim3(1), dim3(kBlock), 0, mlp->stream, mlp->SQ, (int)n, mlp->loss);
    MCHK(hipGetLastError());
    MCHK(hipMemcpyAsync(&l, mlp->loss, sizeof l, hipMemcpyDeviceToHost, mlp->stream));
  }
  MCHK(hipStreamSynchronize(mlp->stream));
  if (final_loss) *final_loss = l;
  return 0;
}

}  // extern "C"
