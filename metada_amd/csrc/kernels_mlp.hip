// Learned inflation network (no counterpart in the reference): a per-column
// MLP 8 -> 64 -> 64 -> 1 with tanh hidden layers and rho = 1 + softplus(out),
// in FP32, with its forward pass, the gradient of the mean squared error
// against target inflations, and an Adam update.
//
// Parameter layout (4801 floats): W1[64][8], b1[64], W2[64][64], b2[64],
// W3[64], b3.
//
// All products run on FP32 matrix cores (v_mfma_f32_16x16x4f32: FP32 products
// and accumulation; A[l%16][l/16], B[l/16][l%16], D[4(l/16)+r][l%16]), 16
// samples per wavefront and step.  Activations sit as [unit][sample]: register
// (t, r) of lane (i16, kk) holds unit 16t + 4kk + r of sample i16, which is the
// right operand of the product step over the units {16t + 4kk + r : kk}, so a
// layer's output feeds the next one from its registers.
//   forward      weights as operand fragments in registers;
//   loss/grad    (a) forward, then g2 = dL/d(pre-activation 2) and g1 likewise
//                    through W2^T; the deltas and activations pass through LDS
//                    once, where the contraction over samples needs them the
//                    other way round; a wavefront accumulates every weight's
//                    gradient over its samples in registers, a block's four
//                    meet in LDS, one partial per block;
//                (b) fixed-order sum of the partials, so the gradient is
//                    deterministic;
//   Adam         elementwise with bias correction.
#include <algorithm>

#include "mda_device.hpp"
#include "mda_internal.hpp"

namespace mda {

constexpr int MLP_IN = 8, MLP_H = 64;
constexpr int MLP_NP = MLP_H * MLP_IN + MLP_H + MLP_H * MLP_H + MLP_H + MLP_H + 1;  // 4801
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + MLP_H * MLP_IN, OFF_W2 = OFF_B1 + MLP_H,
              OFF_B2 = OFF_W2 + MLP_H * MLP_H, OFF_W3 = OFF_B2 + MLP_H, OFF_B3 = OFF_W3 + MLP_H;
static_assert(OFF_B3 + 1 == MLP_NP, "parameter layout");

__device__ inline float softplus_f(float v) { return v > 30.f ? v : log1pf(expf(v)); }
__device__ inline float sigmoid_f(float v) { return 1.f / (1.f + expf(-v)); }

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ inline f4 mfma_f32(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Forward operands of one wavefront: w1[s][tj] = W1[16 tj + i16][4s + kk],
// w2[t][r][tj] = W2[16 tj + i16][16 t + 4 kk + r]; biases and W3 at unit
// 16 t + 4 kk + r.
struct mlp_operands {
  float w1[2][4], w2[4][4][4], b1[4][4], b2[4][4], w3[4][4], b3;
  __device__ void load(const float* __restrict__ P) {
    const int lane = threadIdx.x & 63, i16 = lane & 15, kk = lane >> 4;
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) {
#pragma unroll
      for (int s = 0; s < 2; ++s) w1[s][tj] = P[OFF_W1 + (16 * tj + i16) * MLP_IN + 4 * s + kk];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          w2[t][r][tj] = P[OFF_W2 + (16 * tj + i16) * MLP_H + 16 * t + 4 * kk + r];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int u = 16 * t + 4 * kk + r;
        b1[t][r] = P[OFF_B1 + u];
        b2[t][r] = P[OFF_B2 + u];
        w3[t][r] = P[OFF_W3 + u];
      }
    b3 = P[OFF_B3];
  }
  // x[s] = feature 4s + kk of sample i16; returns the output's pre-activation
  // of sample i16 (in every lane of it)
  __device__ float forward(const float (&x)[2], float (&h1)[4][4], float (&h2)[4][4]) const {
    f4 a[4];
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) {
      a[tj] = f4{b1[tj][0], b1[tj][1], b1[tj][2], b1[tj][3]};
#pragma unroll
      for (int s = 0; s < 2; ++s) a[tj] = mfma_f32(w1[s][tj], x[s], a[tj]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) h1[t][r] = tanhf(a[t][r]);
#pragma unroll
    for (int tj = 0; tj < 4; ++tj) a[tj] = f4{b2[tj][0], b2[tj][1], b2[tj][2], b2[tj][3]};
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) a[tj] = mfma_f32(w2[t][r][tj], h1[t][r], a[tj]);
    float out = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        h2[t][r] = tanhf(a[t][r]);
        out = fmaf(w3[t][r], h2[t][r], out);
      }
    out += __shfl_xor(out, 16);
    out += __shfl_xor(out, 32);
    return out + b3;
  }
};

// Bound by the tanh evaluations.  m = 131,072: 35 us (49 us with one thread
// per sample and the parameters read from LDS, one broadcast per FMA).
__global__ __launch_bounds__(256) void k_mlp_forward(const float* __restrict__ params,
                                                     const float* __restrict__ feat, int64_t m,
                                                     float* __restrict__ rho) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, kk = lane >> 4;
  mlp_operands W;
  W.load(params);
  for (int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); 16 * g < m;
       g += (int64_t)gridDim.x * 4) {
    const int64_t s = 16 * g + i16;
    float x[2], h1[4][4], h2[4][4];
#pragma unroll
    for (int q = 0; q < 2; ++q) x[q] = s < m ? feat[s * MLP_IN + 4 * q + kk] : 0.f;
    const float out = W.forward(x, h1, h2);
    if (kk == 0 && s < m) rho[s] = 1.f + softplus_f(out);
  }
}

// (a) forward, backward and the gradient's partial of one block.
// m = 32,768: 44 us; forward and deltas by one thread per sample took 80 us,
// the outer products by one thread per parameter 665 us.
constexpr int MLP_TS = 17;  // LDS row stride of [unit][16 samples]

__global__ __launch_bounds__(256) void k_mlp_grad(const float* __restrict__ params,
                                                  const float* __restrict__ feat,
                                                  const float* __restrict__ target, int64_t m,
                                                  float* __restrict__ part,
                                                  double* __restrict__ part_loss) {
  // per wavefront g1, g2, h1 [64][MLP_TS] and x [8][MLP_TS]; the block's sums
  // [4801] afterwards
  extern __shared__ float sh[];
  __shared__ double lsum[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i16 = lane & 15, kk = lane >> 4;
  float* tg1 = sh + wv * (3 * MLP_H + MLP_IN) * MLP_TS;
  float* tg2 = tg1 + MLP_H * MLP_TS;
  float* th1 = tg2 + MLP_H * MLP_TS;
  float* tx = th1 + MLP_H * MLP_TS;
  mlp_operands W;
  W.load(params);
  float w2t[4][4][4];  // W2^T: [16 tj + i16] of row 16 t + 4 kk + r
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int tj = 0; tj < 4; ++tj)
        w2t[t][r][tj] = params[OFF_W2 + (16 * t + 4 * kk + r) * MLP_H + 16 * tj + i16];
  f4 dw2[4][4], dw1[4];
  float db1[4][4], db2[4][4], dw3[4][4], db3 = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    dw1[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      dw2[t][r] = f4{0.f, 0.f, 0.f, 0.f};
      db1[t][r] = db2[t][r] = dw3[t][r] = 0.f;
    }
  }
  double loss = 0.0;
  for (int64_t g = (int64_t)blockIdx.x * 4 + wv; 16 * g < m; g += (int64_t)gridDim.x * 4) {
    const int64_t s = 16 * g + i16;
    const bool in = s < m;
    float x[2], h1[4][4], h2[4][4];
#pragma unroll
    for (int q = 0; q < 2; ++q) x[q] = in ? feat[s * MLP_IN + 4 * q + kk] : 0.f;
    const float a = W.forward(x, h1, h2);
    const float res = in ? 1.f + softplus_f(a) - target[s] : 0.f;
    const float ga = 2.f * res * sigmoid_f(a) / (float)m;  // 0 past m
    if (kk == 0) {
      loss += (double)(res * res);
      db3 += ga;
    }
    f4 c[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) c[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int u = 16 * t + 4 * kk + r;
        const float g2 = ga * W.w3[t][r] * (1.f - h2[t][r] * h2[t][r]);
        dw3[t][r] = fmaf(ga, h2[t][r], dw3[t][r]);
        db2[t][r] += g2;
        tg2[u * MLP_TS + i16] = g2;
        th1[u * MLP_TS + i16] = h1[t][r];
#pragma unroll
        for (int tj = 0; tj < 4; ++tj) c[tj] = mfma_f32(w2t[t][r][tj], g2, c[tj]);
      }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float g1 = c[t][r] * (1.f - h1[t][r] * h1[t][r]);
        db1[t][r] += g1;
        tg1[(16 * t + 4 * kk + r) * MLP_TS + i16] = g1;
      }
#pragma unroll
    for (int q = 0; q < 2; ++q) tx[(4 * q + kk) * MLP_TS + i16] = x[q];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // contraction over the 16 samples: A[unit i16][sample kk], B[sample kk][i16]
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int sc = 4 * q + kk;
      float av[4], bv[4], a1[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        av[t] = tg2[(16 * t + i16) * MLP_TS + sc];
        bv[t] = th1[(16 * t + i16) * MLP_TS + sc];
        a1[t] = tg1[(16 * t + i16) * MLP_TS + sc];
      }
      const float xv = i16 < MLP_IN ? tx[(i16 & 7) * MLP_TS + sc] : 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int u = 0; u < 4; ++u) dw2[t][u] = mfma_f32(av[t], bv[u], dw2[t][u]);
        dw1[t] = mfma_f32(a1[t], xv, dw1[t]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // bias and W3 sums over the samples (i16)
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      for (int off = 1; off < 16; off <<= 1) {
        db1[t][r] += __shfl_xor(db1[t][r], off);
        db2[t][r] += __shfl_xor(db2[t][r], off);
        dw3[t][r] += __shfl_xor(dw3[t][r], off);
      }
  for (int off = 1; off < 16; off <<= 1) {
    db3 += __shfl_xor(db3, off);
    loss += __shfl_xor(loss, off);
  }
  if (lane == 0) lsum[wv] = loss;
  // the block's sums, one wavefront after the other
  float* sum = sh;
  for (int w = 0; w < 4; ++w) {
    __syncthreads();
    if (wv != w) continue;
    auto add = [&](int p, float v) { sum[p] = (w == 0 ? 0.f : sum[p]) + v; };
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int u = 16 * t + 4 * kk + r;  // D row
#pragma unroll
        for (int c = 0; c < 4; ++c) add(OFF_W2 + u * MLP_H + 16 * c + i16, dw2[t][c][r]);
        if (i16 < MLP_IN) add(OFF_W1 + u * MLP_IN + i16, dw1[t][r]);
        if (i16 == 0) {
          add(OFF_B1 + u, db1[t][r]);
          add(OFF_B2 + u, db2[t][r]);
          add(OFF_W3 + u, dw3[t][r]);
        }
      }
    if (lane == 0) add(OFF_B3, db3);
  }
  __syncthreads();
  float* out = part + (size_t)blockIdx.x * MLP_NP;
  for (int p = threadIdx.x; p < MLP_NP; p += 256) out[p] = sum[p];
  if (threadIdx.x == 0) part_loss[blockIdx.x] = (lsum[0] + lsum[1]) + (lsum[2] + lsum[3]);
}

// (b) sum over the blocks, eight threads per parameter, each a contiguous
// eighth of them, added in order; the last block sums the loss
__global__ __launch_bounds__(512) void k_mlp_grad_final(const float* __restrict__ part,
                                                        const double* __restrict__ part_loss,
                                                        int nblocks, int64_t m,
                                                        float* __restrict__ grad,
                                                        double* __restrict__ loss) {
  __shared__ float red[8][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int p = blockIdx.x * 64 + lane;
  const int per = (nblocks + 7) / 8, b0 = q * per, b1 = b0 + per < nblocks ? b0 + per : nblocks;
  float s = 0.f;
  if (p < MLP_NP) {
#pragma unroll 8
    for (int b = b0; b < b1; ++b) s += part[(size_t)b * MLP_NP + p];
  }
  red[q][lane] = s;
  __syncthreads();
  if (q == 0 && p < MLP_NP) {
    float t = red[0][lane];
    for (int i = 1; i < 8; ++i) t += red[i][lane];
    grad[p] = t;
  }
  if (blockIdx.x == gridDim.x - 1 && q == 1) {
    double l = 0.0;
    for (int b = lane; b < nblocks; b += 64) l += part_loss[b];
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
    if (lane == 0) *loss = l / (double)m;
  }
}

__global__ void k_mlp_adam(float* __restrict__ params, float* __restrict__ m1,
                           float* __restrict__ m2, const float* __restrict__ grad, float lr,
                           float b1, float b2, float eps, float c1, float c2) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= MLP_NP) return;
  const float g = grad[p];
  const float a = b1 * m1[p] + (1.f - b1) * g;
  const float v = b2 * m2[p] + (1.f - b2) * g * g;
  m1[p] = a;
  m2[p] = v;
  params[p] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
}

// blocks of four wavefronts, each at least one step of 16 samples
static unsigned mlp_blocks(int64_t m, int64_t cap) {
  return (unsigned)std::min<int64_t>((m + 63) / 64, cap);
}

void launch_mlp_forward(hipStream_t s, const float* params, const float* feat, int64_t m,
                        float* rho) {
  if (m <= 0) return;
  hipLaunchKernelGGL(k_mlp_forward, dim3(mlp_blocks(m, 1024)), dim3(256), 0, s, params, feat, m,
                     rho);
  MDA_LAUNCH_CHECK();
}

void launch_mlp_loss_grad(mda_ctx* c, hipStream_t s, const float* params, const float* feat,
                          const float* target, int64_t m, float* grad, double* loss) {
  MDA_REQUIRE(m > 0 && m < (int64_t)1 << 31, "bad number of samples");
  const unsigned nb = mlp_blocks(m, 256);
  float* part = c->get<float>("mlp_part", (size_t)nb * MLP_NP);
  double* pl = c->get<double>("mlp_part_loss", nb);
  const size_t shm = sizeof(float) * 4 * (3 * MLP_H + MLP_IN) * MLP_TS;
  static_assert(4 * (3 * MLP_H + MLP_IN) * MLP_TS >= MLP_NP, "the block's sums reuse the tiles");
  hipLaunchKernelGGL(k_mlp_grad, dim3(nb), dim3(256), shm, s, params, feat, target, m, part, pl);
  MDA_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_mlp_grad_final, dim3((MLP_NP + 63) / 64), dim3(512), 0, s, part, pl,
                     (int)nb, m, grad, loss);
  MDA_LAUNCH_CHECK();
}

void launch_mlp_adam(hipStream_t s, float* params, float* m1, float* m2, const float* grad,
                     int64_t step, float lr, float b1, float b2, float eps) {
  MDA_REQUIRE(step >= 1, "Adam step counts from 1");
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_NP + 255) / 256), dim3(256), 0, s, params, m1, m2,
                     grad, lr, b1, b2, eps, c1, c2);
  MDA_LAUNCH_CHECK();
}

}  // namespace mda
