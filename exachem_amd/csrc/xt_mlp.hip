// Task cost model: a 7 -> 64 -> 64 -> 1 FP32 multilayer perceptron (ReLU
// hidden layers, linear output) with its inference, back-propagation and
// Adam kernels.  Every reduction over samples runs in a fixed order (one
// thread per parameter looping over samples), so a training run gives the
// same parameters bit for bit on every call.
//
// Parameter layout (kMlpParams floats):
//   W1[7][64] | b1[64] | W2[64][64] | b2[64] | w3[64] | b3
// Loss: mean squared error over the batch.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "xt_device.h"

namespace xt {
namespace {

constexpr int IN = kMlpIn, H = kMlpHidden;
constexpr int OW1 = 0, OB1 = OW1 + IN * H, OW2 = OB1 + H, OB2 = OW2 + H * H, OW3 = OB2 + H,
              OB3 = OW3 + H;
static_assert(OB3 + 1 == kMlpParams, "parameter layout");

// One forward pass of SB samples per workgroup, thread (sample tid / 64, unit
// tid % 64); with BACK also the error signals of both hidden layers:
//   DY = 2 (y - t) / n, D2 = DY w3 [a2 > 0], D1 = (W2 D2) [a1 > 0],
//   SQ = (y - t)^2 for the loss.
// Every sum runs over its index in order in one thread, so the values do not
// depend on the split.  What bounds it is latency (a batch is a few hundred
// samples): with one thread per sample a batch of 512 filled two workgroups,
// and forward and backward took 40 + 39 us; with one thread per unit and one
// kernel 9 us.  The parameters are staged in LDS (W2 with a padded row: the
// backward product reads it along its rows).  inc: the Adam step count is
// advanced here, once per step, for the update kernel that follows.
constexpr int SB = 4;
constexpr int LW = H + 1;

template<bool BACK>
__global__ void __launch_bounds__(SB * H) k_mlp_pass(const float* __restrict__ P,
                                                     const float* __restrict__ X,
                                                     const float* __restrict__ T, long n,
                                                     float* __restrict__ Y, float* __restrict__ A1,
                                                     float* __restrict__ A2, float* __restrict__ DY,
                                                     float* __restrict__ D1, float* __restrict__ D2,
                                                     float* __restrict__ SQ, int* step) {
  __shared__ float w1[IN * H + H], w2[H * LW], wo[2 * H + 1];
  __shared__ float u[SB][H], v[SB][H], yo[SB];
  const int tid = threadIdx.x, k = tid >> 6, h = tid & 63;
  if(BACK && step && blockIdx.x == 0 && tid == 0) step[0] += 1;
  for(int i = tid; i < OW2; i += SB * H) w1[i] = P[i];
  for(int i = tid; i < H * H; i += SB * H) w2[(i >> 6) * LW + (i & 63)] = P[OW2 + i];
  for(int i = tid; i < 2 * H + 1; i += SB * H) wo[i] = P[OB2 + i];  // b2, w3, b3
  __syncthreads();
  // the same trip count for every thread of the workgroup
  for(long s0 = (long) blockIdx.x * SB; s0 < n; s0 += (long) gridDim.x * SB) {
    const long s  = s0 + k;
    const bool on = s < n;
    float      a1 = 0.f, a2 = 0.f;
    if(on) {
      float z = w1[OB1 + h];
#pragma unroll
      for(int i = 0; i < IN; i++) z = fmaf(X[s * IN + i], w1[i * H + h], z);
      a1 = fmaxf(z, 0.f);
      if(A1) A1[s * H + h] = a1;
    }
    u[k][h] = a1;
    __syncthreads();
    {
      float z = wo[h];
#pragma unroll 16
      for(int a = 0; a < H; a++) z = fmaf(u[k][a], w2[a * LW + h], z);
      a2      = fmaxf(z, 0.f);
      v[k][h] = a2;
      if(on && A2) A2[s * H + h] = a2;
    }
    __syncthreads();
    if(h == 0 && on) {
      float y = wo[2 * H];
#pragma unroll 16
      for(int b = 0; b < H; b++) y = fmaf(v[k][b], wo[H + b], y);
      Y[s]  = y;
      yo[k] = y;
    }
    __syncthreads();
    if(BACK) {
      float d2 = 0.f;
      if(on) {
        const float r  = yo[k] - T[s];
        const float dy = 2.f * r / (float) n;
        if(h == 0) {
          SQ[s] = r * r;
          DY[s] = dy;
        }
        d2            = a2 > 0.f ? dy * wo[H + h] : 0.f;
        D2[s * H + h] = d2;
      }
      v[k][h] = d2;
      __syncthreads();
      float g = 0.f;
#pragma unroll 16
      for(int b = 0; b < H; b++) g = fmaf(w2[h * LW + b], v[k][b], g);
      if(on) D1[s * H + h] = a1 > 0.f ? g : 0.f;
      __syncthreads();
    }
  }
}

// The forward pass of large batches, one thread per sample: every lane reads the
// same weight from LDS at a time, four per read, where k_mlp_pass reads a weight
// per lane and product and runs the last layer on one lane.  The same order of
// every sum, so the same bits.  Bound: LDS reads and FP32 products.
__global__ void __launch_bounds__(256) k_mlp_forward(const float* __restrict__ P,
                                                     const float* __restrict__ X, long n,
                                                     float* __restrict__ Y) {
  __shared__ float w[kMlpParams];
  for(int i = threadIdx.x; i < kMlpParams; i += blockDim.x) w[i] = P[i];
  __syncthreads();
  const long s = (long) blockIdx.x * blockDim.x + threadIdx.x;
  if(s >= n) return;
  float x[IN];
#pragma unroll
  for(int i = 0; i < IN; i++) x[i] = X[s * IN + i];
  float a1[H];
#pragma unroll
  for(int h = 0; h < H; h++) {
    float z = w[OB1 + h];
#pragma unroll
    for(int i = 0; i < IN; i++) z = fmaf(x[i], w[OW1 + i * H + h], z);
    a1[h] = fmaxf(z, 0.f);
  }
  float y = w[OB3];
  for(int b = 0; b < H; b++) {
    float z = w[OB2 + b];
#pragma unroll
    for(int a = 0; a < H; a++) z = fmaf(a1[a], w[OW2 + a * H + b], z);
    y = fmaf(fmaxf(z, 0.f), w[OW3 + b], y);
  }
  Y[s] = y;
}

// Parameter gradients, and with TRAIN the Adam update of the same parameters:
// one thread per parameter, samples summed in order, chunks of CS samples of
// the factors staged through LDS with samples contiguous.  Bound: latency.  With
// one thread per parameter reading both factors from L2 sample by sample the
// gradient kernel took 120 us for 512 samples; here it takes 16 us with the
// update (chunks of 128: 20 us).
//   workgroups 0..15: a 16 x 16 tile of W2 (A1 x D2)
//   workgroups 16, 17: W1 and b1 (X with a constant 1 x D1), inputs 4 (w - 16) ..
//   workgroups 18, 19: b2 (sum of D2), b3 (sum of DY) and the loss; w3 (DY x A2)
constexpr int CS = 64, GT = 256, LS = CS + 4;
constexpr int kGradGroups = 20;

template<bool TRAIN>
__device__ __forceinline__ void update(float* P, float* G, float* M1, float* M2, int p, float g,
                                       float lr, float c1, float c2) {
  G[p] = g;
  if(!TRAIN) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float m = b1 * M1[p] + (1.f - b1) * g;
  const float v = b2 * M2[p] + (1.f - b2) * g * g;
  M1[p]         = m;
  M2[p]         = v;
  const float mh = m / c1;
  const float vh = v / c2;
  P[p] -= lr * mh / (sqrtf(vh) + eps);
}

__device__ __forceinline__ float fma4(const float4& u, const float4& v, float g) {
  g = fmaf(u.x, v.x, g);
  g = fmaf(u.y, v.y, g);
  g = fmaf(u.z, v.z, g);
  return fmaf(u.w, v.w, g);
}

template<bool TRAIN>
__global__ void __launch_bounds__(GT) k_mlp_grad(MlpWork W, long n, float lr, float* loss_hist) {
  __shared__ __align__(16) float fa[16][LS];
  __shared__ __align__(16) float fd[H][LS];
  const int tid = threadIdx.x, w = blockIdx.x, sl = tid >> 2, q = tid & 3;
  float     c1 = 1.f, c2 = 1.f, g = 0.f;
  int       t = 0;
  if(TRAIN) {
    t  = W.step[0];  // already counts this step
    c1 = 1.f - powf(0.9f, (float) t);
    c2 = 1.f - powf(0.999f, (float) t);
  }
  if(w < 18) {
    const bool   hid = w < 16;
    const int    a0 = hid ? 16 * (w >> 2) : 4 * (w - 16), b0 = hid ? 16 * (w & 3) : 0;
    const int    row = hid ? tid >> 4 : tid >> 6, col = hid ? tid & 15 : tid & 63;
    const float* D = hid ? W.D2 : W.D1;
    float        ra[4], rd[16];
    auto         load = [&](long s0) {
      const long s  = s0 + sl;
      const bool on = s < n;
      if(hid) {
#pragma unroll
        for(int j = 0; j < 4; j++) ra[j] = on ? W.A1[s * H + a0 + 4 * q + j] : 0.f;
#pragma unroll
        for(int j = 0; j < 4; j++) rd[j] = on ? D[s * H + b0 + 4 * q + j] : 0.f;
      }
      else {
        const int i = a0 + q;
        ra[0]       = !on ? 0.f : i < IN ? W.X[s * IN + i] : 1.f;
#pragma unroll
        for(int j = 0; j < 16; j++) rd[j] = on ? D[s * H + 16 * q + j] : 0.f;
      }
    };
    load(0);
    for(long s0 = 0; s0 < n; s0 += CS) {
      __syncthreads();
      if(hid) {
#pragma unroll
        for(int j = 0; j < 4; j++) {
          fa[4 * q + j][sl] = ra[j];
          fd[4 * q + j][sl] = rd[j];
        }
      }
      else {
        fa[q][sl] = ra[0];
#pragma unroll
        for(int j = 0; j < 16; j++) fd[16 * q + j][sl] = rd[j];
      }
      __syncthreads();
      if(s0 + CS < n) load(s0 + CS);
      if(s0 + CS <= n)
#pragma unroll
        for(int s = 0; s < CS; s += 4)
          g = fma4(*reinterpret_cast<const float4*>(&fa[row][s]),
                   *reinterpret_cast<const float4*>(&fd[col][s]), g);
      else
        for(int s = 0; s < (int) (n - s0); s++) g = fmaf(fa[row][s], fd[col][s], g);
    }
    const int p = hid ? OW2 + (a0 + row) * H + b0 + col : a0 + row < IN ? OW1 + (a0 + row) * H + col : OB1 + col;
    update<TRAIN>(W.P, W.G, W.M1, W.M2, p, g, lr, c1, c2);
    return;
  }
  const bool   out = w == 19;
  const float* F   = out ? W.A2 : W.D2;
  float        rd[16], ry = 0.f, rq = 0.f;
  double       l    = 0.0;
  auto         load = [&](long s0) {
    const long s  = s0 + sl;
    const bool on = s < n;
#pragma unroll
    for(int j = 0; j < 16; j++) rd[j] = on ? F[s * H + 16 * q + j] : 0.f;
    if(q == 0) {
      ry = on ? W.DY[s] : 0.f;
      rq = on ? W.SQ[s] : 0.f;
    }
  };
  load(0);
  for(long s0 = 0; s0 < n; s0 += CS) {
    __syncthreads();
#pragma unroll
    for(int j = 0; j < 16; j++) fd[16 * q + j][sl] = rd[j];
    if(q == 0) {
      fa[0][sl] = ry;
      fa[1][sl] = rq;
    }
    __syncthreads();
    if(s0 + CS < n) load(s0 + CS);
    const float* x = tid < 64 ? fd[tid] : fa[tid == 65];
    if(tid > 65 || (out && tid > 63)) continue;
    if(s0 + CS <= n) {
#pragma unroll
      for(int s = 0; s < CS; s += 4) {
        const float4 v = *reinterpret_cast<const float4*>(&x[s]);
        if(out) g = fma4(*reinterpret_cast<const float4*>(&fa[0][s]), v, g);
        else if(tid == 65) {
          l += v.x;
          l += v.y;
          l += v.z;
          l += v.w;
        }
        else {
          g += v.x;
          g += v.y;
          g += v.z;
          g += v.w;
        }
      }
    }
    else
      for(int s = 0; s < (int) (n - s0); s++) {
        if(out) g = fmaf(fa[0][s], x[s], g);
        else if(tid == 65) l += x[s];
        else g += x[s];
      }
  }
  if(tid < 64) update<TRAIN>(W.P, W.G, W.M1, W.M2, (out ? OW3 : OB2) + tid, g, lr, c1, c2);
  else if(!out && tid == 64) update<TRAIN>(W.P, W.G, W.M1, W.M2, OB3, g, lr, c1, c2);
  else if(!out && tid == 65) {
    const float m = (float) (l / (double) n);
    W.loss[0]     = m;
    // step[1]: value of step[0] when the training call began
    if(TRAIN && loss_hist) loss_hist[t - 1 - W.step[1]] = m;
  }
}

inline unsigned blocks(long n, int t) { return (unsigned) ((n + t - 1) / t); }

}  // namespace

// From here on one thread per sample is faster (xt_mlp_predict, us, with a thread
// per hidden unit and with one per sample: 16,384 samples 69 and 82, 32,768 97 and
// 98, 65,536 162 and 141, 1,000,000 1,815 and 1,350).
constexpr long kManySamples = 32768;

int mlp_forward(const float* P, const float* X, long n, float* Y, float* A1, float* A2,
                void* stream) {
  if(n <= 0) return 0;
  if(n >= kManySamples && !A1 && !A2) {
    hipLaunchKernelGGL(k_mlp_forward, dim3(blocks(n, 256)), dim3(256), 0, (hipStream_t) stream, P, X, n, Y);
    return (int) hipGetLastError();
  }
  // workgroups loop over samples: staging the parameters costs more than one group of samples
  hipLaunchKernelGGL(k_mlp_pass<false>, dim3(std::min(blocks(n, SB), 1024u)), dim3(SB * H), 0,
                     (hipStream_t) stream, P, X, (const float*) nullptr, n, Y, A1, A2, (float*) nullptr,
                     (float*) nullptr, (float*) nullptr, (float*) nullptr, (int*) nullptr);
  return (int) hipGetLastError();
}

static int pass(const MlpWork& W, long n, int* step, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_pass<true>, dim3(std::min(blocks(n, SB), 1024u)), dim3(SB * H), 0, st, W.P, W.X, W.T,
                     n, W.Y, W.A1, W.A2, W.DY, W.D1, W.D2, W.SQ, step);
  return (int) hipGetLastError();
}

int mlp_loss_grad(const MlpWork& W, long n, void* stream) {
  hipStream_t st  = (hipStream_t) stream;
  const int   err = pass(W, n, nullptr, st);
  if(err) return err;
  hipLaunchKernelGGL(k_mlp_grad<false>, dim3(kGradGroups), dim3(GT), 0, st, W, n, 0.f, (float*) nullptr);
  return (int) hipGetLastError();
}

int mlp_train_step(const MlpWork& W, long n, float lr, float* loss_hist, void* stream) {
  hipStream_t st  = (hipStream_t) stream;
  const int   err = pass(W, n, W.step, st);
  if(err) return err;
  hipLaunchKernelGGL(k_mlp_grad<true>, dim3(kGradGroups), dim3(GT), 0, st, W, n, lr, loss_hist);
  return (int) hipGetLastError();
}

}  // namespace xt
