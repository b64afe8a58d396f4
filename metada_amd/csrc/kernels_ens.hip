// Streaming ensemble kernels and the global (all-observation) EnKF / ETKF
// pieces: ensemble mean and perturbations, H x with observation-space
// statistics, Y'^T R^-1 [Y' | d] reductions, the k x k solves, the global
// transform and Metrics.
#include <algorithm>

#include "mda_device.hpp"
#include "mda_internal.hpp"

namespace mda {

__global__ void k_zero_words(uint32_t* p, int64_t nwords) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nwords;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

void launch_zero(hipStream_t s, void* ptr, size_t bytes) {
  int64_t nw = (int64_t)(bytes / 4);
  hipLaunchKernelGGL(k_zero_words, dim3(grid_for(nw, 256, 4096)), dim3(256), 0, s,
                     (uint32_t*)ptr, nw);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Ensemble::RecomputeMean / RecomputePerturbations (Ensemble.hpp:105-151):
// sequential sum over members, times the reciprocal 1/k, then (x - mean)*scale.
// Member-major [k][n]; each thread owns state indices, loads are coalesced.
// ---------------------------------------------------------------------------
__global__ void k_mean_pert(const double* __restrict__ X, int k, int64_t n, double scale,
                            double* __restrict__ mean, double* __restrict__ pert) {
  const double rk = 1.0 / (double)k;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int j = 0; j < k; ++j) s += X[(size_t)j * n + i];
    double m = s * rk;
    if (mean) mean[i] = m;
    if (pert)
      for (int j = 0; j < k; ++j) pert[(size_t)j * n + i] = (X[(size_t)j * n + i] - m) * scale;
  }
}

void launch_mean_pert(hipStream_t s, const double* X, int k, int64_t n, double scale,
                      double* mean, double* pert) {
  hipLaunchKernelGGL(k_mean_pert, dim3(grid_for(n, 256, 65536)), dim3(256), 0, s, X, k, n,
                     scale, mean, pert);
  MDA_LAUNCH_CHECK();
}

// sum of squares, one partial per block (launch_reduce_partials adds them in order)
__global__ void k_sumsq(const double* __restrict__ X, int64_t count, double* partial) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count;
       i += (int64_t)gridDim.x * blockDim.x)
    acc += X[i] * X[i];
  acc = block_sum(acc, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

void launch_sumsq(hipStream_t s, const double* X, int64_t count, double* partial,
                  int nblocks) {
  hipLaunchKernelGGL(k_sumsq, dim3(nblocks), dim3(256), 0, s, X, count, partial);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Observation space (EnKF.hpp:168-184, LETKF.hpp:197-211): hx_j = H x_j for
// every member (CSR stencil gather, or a caller-supplied member-major H(x)),
// ybar = mean over members, Y' = hx - ybar, d = y_o - ybar.  A block owns 64
// observations; the [64][k] tile is assembled in LDS so that the obs-major Y'
// rows go out as contiguous, coalesced stores.  With `order`, the block's
// observations are order[t] for its 64 positions t (for the LETKF, sorted by
// the grid position of their first stencil tap, groups of four levels
// together, so that neighbouring observations' state gathers share cache
// lines); without `opos` observation
// order[t] is written at position t, with `opos` at position opos[order[t]].
// Blocks map XCD-contiguously (block i -> slice i mod 8), so consecutive
// tiles share an L2.
// ---------------------------------------------------------------------------
constexpr int OBS_TILE = 64;
constexpr int OBS_TAPS = 8;  // stencils held in registers (trilinear: 8)

__global__ __launch_bounds__(256) void k_obs_stats(
    const double* __restrict__ X, int k, int64_t n, int64_t p,
    const int64_t* __restrict__ row_ptr, const int64_t* __restrict__ col,
    const double* __restrict__ w, const double* __restrict__ hx_mm,
    const double* __restrict__ yo, const uint32_t* __restrict__ order,
    const uint32_t* __restrict__ opos, double* __restrict__ ybar,
    double* __restrict__ yp_om, double* __restrict__ d, double* __restrict__ yp_mm,
    float* __restrict__ y32, int* __restrict__ status) {
  extern __shared__ double tile[];  // [OBS_TILE][k + 1] (padded rows)
  const int kp = k + 1;
  __shared__ double mean_s[OBS_TILE];
  __shared__ int64_t pos_s[OBS_TILE];
  const int tid = threadIdx.x, nt = blockDim.x;
  const int64_t nb = gridDim.x;  // a multiple of 8
  const int64_t vb = (int64_t)(blockIdx.x % 8) * (nb / 8) + blockIdx.x / 8;
  const int64_t o0 = vb * OBS_TILE;
  if (o0 >= p) return;
  const int nob = (int)((p - o0) < OBS_TILE ? (p - o0) : OBS_TILE);
  if (hx_mm) {
    // H x_j: entry (ob, j) with ob fastest so hx_mm reads are coalesced
    for (int e = tid; e < nob * k; e += nt) {
      int ob = e % nob, j = e / nob;
      const int64_t o = order ? (int64_t)order[o0 + ob] : o0 + ob;
      tile[ob * kp + j] = hx_mm[(size_t)j * p + o];
    }
  } else {
    // Stencil: lane ob of every wave owns observation ob, wave g members
    // g, g + 4, ...  A stencil of up to OBS_TAPS taps is read once into
    // registers and its gathers for one member go out together; the sum
    // runs over the taps in stencil order.
    const int ob = tid & 63, jg = tid >> 6;
    if (ob < nob) {
      const int64_t o = order ? (int64_t)order[o0 + ob] : o0 + ob;
      const int64_t t0 = row_ptr[o], t1 = row_ptr[o + 1];
      if (t1 - t0 <= OBS_TAPS) {
        const int nt_o = (int)(t1 - t0);
        int64_t cc[OBS_TAPS];
        double ww[OBS_TAPS];
#pragma unroll
        for (int q = 0; q < OBS_TAPS; ++q) {
          cc[q] = q < nt_o ? col[t0 + q] : 0;  // absent taps read entry 0, unused
          ww[q] = q < nt_o ? w[t0 + q] : 0.0;
        }
#pragma unroll 2
        for (int j = jg; j < k; j += nt / 64) {
          const double* xj = X + (size_t)j * n;
          double xv[OBS_TAPS];
#pragma unroll
          for (int q = 0; q < OBS_TAPS; ++q) xv[q] = xj[cc[q]];
          double v = 0.0;
#pragma unroll
          for (int q = 0; q < OBS_TAPS; ++q)
            if (q < nt_o) v += ww[q] * xv[q];
          tile[ob * kp + j] = v;
        }
      } else {
        for (int j = jg; j < k; j += nt / 64) {
          const double* xj = X + (size_t)j * n;
          double v = 0.0;
          for (int64_t t = t0; t < t1; ++t) v += w[t] * xj[col[t]];
          tile[ob * kp + j] = v;
        }
      }
    }
  }
  __syncthreads();
  for (int ob = tid; ob < nob; ob += nt) {
    double s = 0.0;
    for (int j = 0; j < k; ++j) s += tile[ob * kp + j];
    double m = s / (double)k;
    mean_s[ob] = m;
    const int64_t o = order ? (int64_t)order[o0 + ob] : o0 + ob;
    const int64_t q = opos ? (int64_t)opos[o] : o0 + ob;  // output position
    pos_s[ob] = q;
    const double dv = yo[o] - m;
    if (ybar) ybar[q] = m;
    if (d) d[q] = dv;
    // a non-finite H(x) (hence mean, Y' row and innovation) or observation
    if (status && !isfinite(dv)) atomicOr(status, MDA_ST_NONFINITE_OBS);
  }
  __syncthreads();
  for (int e = tid; e < nob * k; e += nt) {
    int ob = e / k, j = e % k;
    double v = tile[ob * kp + j] - mean_s[ob];
    const size_t at = (size_t)pos_s[ob] * k + j;
    if (yp_om) yp_om[at] = v;
    if (y32) y32[at] = (float)v;
    tile[ob * kp + j] = v;
  }
  if (yp_mm) {
    __syncthreads();
    for (int e = tid; e < nob * k; e += nt) {
      int ob = e % nob, j = e / nob;
      yp_mm[(size_t)j * p + pos_s[ob]] = tile[ob * kp + j];
    }
  }
}

void launch_obs_stats(hipStream_t s, const double* X, int k, int64_t n, int64_t p,
                      const int64_t* row_ptr, const int64_t* col, const double* w,
                      const double* hx_mm, const double* yo, double* ybar, double* yp_om,
                      double* d, double* yp_mm, const uint32_t* order, float* y32,
                      const uint32_t* opos, int* status) {
  if (p <= 0) return;
  const int64_t tiles = (p + OBS_TILE - 1) / OBS_TILE;
  MDA_REQUIRE(tiles < ((int64_t)1 << 31) - 8, "too many observations");
  const unsigned nb = (unsigned)((tiles + 7) / 8 * 8);
  size_t shm = sizeof(double) * OBS_TILE * (k + 1);
  hipLaunchKernelGGL(k_obs_stats, dim3(nb), dim3(256), shm, s, X, k, n, p, row_ptr, col, w,
                     hx_mm, yo, order, opos, ybar, yp_om, d, yp_mm, y32, status);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Global Gram over all observations (ETKF.hpp:150-155; EnKF via Woodbury):
//   mode 0: G[a][c] = sum_o Y'[o][a] Y'[o][c] / var_o (c < k), and
//           G[a][k] = sum_o Y'[o][a] d_o / var_o
//   mode 1: G[a][j] = sum_o Y'[o][a] D[o][j] / var_o with the perturbed
//           innovation D[o][j] = d_o + sqrt(var_o) Z[o][j] - Y'[o][j]
//           (EnKF.hpp:212-224; Z is [p][k]).
// On FP64 MFMA, four observations a step (lane (i16, kk): member 16t + i16 of
// observation 4 step + kk, 128-byte row segments): mode 0 on the lower 16 x 16
// tiles, mode 1 on all.  KT = ceil(k / 16) tile rows; up to 4 the block's four
// wavefronts take different steps, beyond that two take each step, with the
// even and the odd tile rows.  The wavefronts' sums meet in LDS, one partial
// per block, then a fixed-order reduction (none for a single block).
// p = 100,000, k = 64: 48 us (451 us with one product per thread and
// observation out of LDS, and 64 us for a serial sum of the partials).
// ---------------------------------------------------------------------------
template <int KT, int MODE>
__global__ __launch_bounds__(256) void k_global_gram(const double* __restrict__ yp_om,
                                                     const double* __restrict__ d,
                                                     const double* __restrict__ var,
                                                     const double* __restrict__ Z, int k,
                                                     int64_t p, double* __restrict__ partial) {
  constexpr int NG = KT > 4 ? 2 : 1, WS = 4 / NG;  // row groups, wavefronts over steps
  constexpr int NR = (KT + NG - 1) / NG;           // tile rows of a group
  constexpr int NA = NR * KT;
  extern __shared__ double out[];  // [k][kq]
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, i16 = lane & 15, kk = lane >> 4;
  const int grp = wv % NG, ws = wv / NG;
  const int kq = MODE == 0 ? k + 1 : k;
  const int64_t nstep = (p + 3) / 4;
  d4 acc[NA];
#pragma unroll
  for (int t = 0; t < NA; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
  double bp[NR];
#pragma unroll
  for (int t = 0; t < NR; ++t) bp[t] = 0.0;
  for (int64_t st = (int64_t)blockIdx.x * WS + ws; st < nstep; st += (int64_t)gridDim.x * WS) {
    const int64_t o = 4 * st + kk;
    const bool in = o < p;
    const double vr = in ? var[o] : INFINITY, dv = in ? d[o] : 0.0;
    const double rinv = 1.0 / vr;  // 0 for an invalid observation (var = +inf)
    double y[KT], z[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const int m = 16 * t + i16;
      const bool mv = in && m < k;
      y[t] = mv ? yp_om[(size_t)o * k + m] : 0.0;
      if (MODE == 1) z[t] = mv && !isinf(vr) ? Z[(size_t)o * k + m] : 0.0;
    }
    if (MODE == 1) {
      const double sr = isinf(vr) ? 0.0 : sqrt(vr);
#pragma unroll
      for (int t = 0; t < KT; ++t) z[t] = isinf(vr) ? 0.0 : dv + sr * z[t] - y[t];
    }
#pragma unroll
    for (int t = 0; t < NR; ++t) {
      // tile row t NG + grp, by selects on the uniform grp (static indices)
      double ya = y[t * NG];
      if (NG == 2) ya = grp ? (t * NG + 1 < KT ? y[t * NG + 1 < KT ? t * NG + 1 : 0] : 0.0) : ya;
      const double aw = rinv * ya;
      if (MODE == 0) bp[t] = fma(aw, dv, bp[t]);
#pragma unroll
      for (int tb = 0; tb < KT; ++tb)
        if (MODE == 1 || tb <= t * NG + NG - 1)
          acc[t * KT + tb] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              aw, MODE == 0 ? y[tb] : z[tb], acc[t * KT + tb], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < NR; ++t) {
    bp[t] += __shfl_xor(bp[t], 16);
    bp[t] += __shfl_xor(bp[t], 32);
  }
  for (int w = 0; w < WS; ++w) {
    if (ws == w) {
#pragma unroll
      for (int t = 0; t < NR; ++t) {
        const int ta = t * NG + grp;
#pragma unroll
        for (int tb = 0; tb < KT; ++tb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = 16 * ta + kk + 4 * r, col = 16 * tb + i16;
            const bool use = row < k && col < k && (MODE == 1 || col <= row);
            if (use && (MODE == 1 || tb <= t * NG + NG - 1)) {
              const double v = acc[t * KT + tb][r] + (w == 0 ? 0.0 : out[row * kq + col]);
              out[row * kq + col] = v;
              if (MODE == 0 && row != col) out[col * kq + row] = v;
            }
          }
        if (MODE == 0 && kk == 0 && 16 * ta + i16 < k) {
          const int row = 16 * ta + i16;
          out[row * kq + k] = bp[t] + (w == 0 ? 0.0 : out[row * kq + k]);
        }
      }
    }
    __syncthreads();
  }
  double* pb = partial + (size_t)blockIdx.x * k * kq;
  for (int e = tid; e < k * kq; e += 256) pb[e] = out[e];
}

// out[e] = sum over blocks of partial[b][e]: eight threads per entry, each a
// contiguous eighth of the blocks, added in order
__global__ __launch_bounds__(512) void k_reduce_partials(const double* __restrict__ partial,
                                                         int nblocks, int ne,
                                                         double* __restrict__ out) {
  __shared__ double red[8][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int e = blockIdx.x * 64 + lane;
  const int per = (nblocks + 7) / 8, b0 = q * per,
            b1 = b0 + per < nblocks ? b0 + per : nblocks;
  double s = 0.0;
  if (e < ne) {
#pragma unroll 8
    for (int b = b0; b < b1; ++b) s += partial[(size_t)b * ne + e];
  }
  red[q][lane] = s;
  __syncthreads();
  if (q == 0 && e < ne) {
    double t = red[0][lane];
    for (int i = 1; i < 8; ++i) t += red[i][lane];
    out[e] = t;
  }
}

void launch_reduce_partials(hipStream_t s, const double* partial, int nblocks, int ne,
                            double* out) {
  hipLaunchKernelGGL(k_reduce_partials, dim3((ne + 63) / 64), dim3(512), 0, s, partial, nblocks,
                     ne, out);
  MDA_LAUNCH_CHECK();
}

void launch_global_gram(hipStream_t s, const double* yp_om, const double* d,
                        const double* var, const double* Z, int k, int64_t p, int mode,
                        double* partial, int nblocks, double* out) {
  MDA_REQUIRE(k >= 1 && k <= 128, "global Gram supports k <= 128");
  const int kq = mode == 0 ? k + 1 : k, kt = (k + 15) / 16;
  // at least eight steps of four observations per wavefront
  const int ws = kt > 4 ? 2 : 4;
  const int64_t want = ((p + 3) / 4 + 8 * ws - 1) / (8 * ws);
  const int nb = (int)std::min<int64_t>(nblocks, std::max<int64_t>(1, want));
  double* part = nb > 1 ? partial : out;
  const size_t shm = sizeof(double) * k * kq;
#define MDA_GG(KT)                                                                               \
  case KT:                                                                                       \
    if (mode == 0)                                                                               \
      hipLaunchKernelGGL((k_global_gram<KT, 0>), dim3(nb), dim3(256), shm, s, yp_om, d, var, Z,  \
                         k, p, part);                                                            \
    else                                                                                         \
      hipLaunchKernelGGL((k_global_gram<KT, 1>), dim3(nb), dim3(256), shm, s, yp_om, d, var, Z,  \
                         k, p, part);                                                            \
    break;
  switch (kt) { MDA_GG(1) MDA_GG(2) MDA_GG(3) MDA_GG(4) MDA_GG(5) MDA_GG(6) MDA_GG(7) MDA_GG(8) }
#undef MDA_GG
  MDA_LAUNCH_CHECK();
  if (nb == 1) return;
  launch_reduce_partials(s, partial, nb, k * kq, out);
}

// ---------------------------------------------------------------------------
// k x k solves of the global filters, one workgroup, k <= 128: M = E + (k-1) I
// = L L^T (EB is [k][k+1] = [E | b]) with the identity's rows carried through
// the factorisation, so that W = L^-T (upper triangular) comes with it.  Both
// triangles packed in LDS (132 KB at k = 128).  The matrix in global memory,
// a barrier per column and a serial inverse took 545 us (ETKF, k = 64) and
// 960 us (EnKF, k = 80); this takes 62 and 182 us.
// ---------------------------------------------------------------------------
constexpr int KS_THREADS = 512;
__host__ __device__ inline size_t ks_tri(int k) { return (size_t)k * (k + 1) / 2; }

struct ks_lds {
  double* M;  // lower triangle, row i at i (i + 1) / 2
  double* W;  // upper triangle, row i holds the columns i .. k-1
  int k;
  __device__ double* lrow(int i) const { return M + (size_t)i * (i + 1) / 2; }
  // W[i][j] = wrow(i)[j], j >= i
  __device__ double* wrow(int i) const {
    return W + ((ptrdiff_t)i * k - (ptrdiff_t)i * (i - 1) / 2 - i);
  }
};

// M (rows and columns in reversed order with rev) and W = L^-T; false when M
// is not positive definite
__device__ inline bool ks_factor(const ks_lds& f, const double* __restrict__ EB, bool rev) {
  const int k = f.k, tid = threadIdx.x;
  for (int idx = tid; idx < k * k; idx += KS_THREADS) {
    const int i = idx / k, j = idx % k;
    if (j > i) continue;
    const int si = rev ? k - 1 - i : i, sj = rev ? k - 1 - j : j;
    f.lrow(i)[j] = EB[si * (k + 1) + sj] + (i == j ? (double)(k - 1) : 0.0);
    f.wrow(j)[i] = i == j ? 1.0 : 0.0;
  }
  __syncthreads();
  return block_row_cholesky(
      k, 2 * k, [&](int i) { return i < k ? f.lrow(i) : f.wrow(i - k); },
      [&](int i) { return i - k; });
}

// ETKF (ETKF.hpp:150-159): Pa = M^-1, wa = Pa b, Wa = sqrt(k-1) chol_L(Pa),
// T = wa 1^T + Wa so that X_a = xbar + X' T.  With the order of the members
// reversed (J M J = L L^T), chol_L(Pa) = J L^-T J: entry (i, j), j <= i, is
// W[k-1-i][k-1-j].
__global__ __launch_bounds__(KS_THREADS) void k_etkf_solve(int k, const double* __restrict__ EB,
                                                           double* __restrict__ T, int* status) {
  extern __shared__ double sh[];
  __shared__ double y[128], wa[128];
  const int tid = threadIdx.x;
  const ks_lds f{sh, sh + ks_tri(k), k};
  const bool ok = ks_factor(f, EB, true);
  if (!ok) {  // the same in every thread; T is not used then
    if (tid == 0) atomicOr(status, MDA_ST_NOT_SPD);
    return;
  }
  auto lp = [&](int i, int j) { return f.wrow(k - 1 - i)[k - 1 - j]; };
  if (tid < k) {
    double s = 0.0;
    for (int i = tid; i < k; ++i) s = fma(lp(i, tid), EB[i * (k + 1) + k], s);
    y[tid] = s;
  }
  __syncthreads();
  if (tid < k) {
    double s = 0.0;
    for (int j = 0; j <= tid; ++j) s = fma(lp(tid, j), y[j], s);
    wa[tid] = s;
  }
  __syncthreads();
  const double sq = sqrt((double)(k - 1));
  for (int idx = tid; idx < k * k; idx += KS_THREADS) {
    const int i = idx / k, j = idx % k;
    T[idx] = wa[i] + (j <= i ? sq * lp(i, j) : 0.0);
  }
}

void launch_etkf_solve_ws(hipStream_t s, int k, const double* EB, double* T, int* status) {
  MDA_REQUIRE(k <= 128, "ETKF supports k <= 128");
  hipLaunchKernelGGL(k_etkf_solve, dim3(1), dim3(KS_THREADS), sizeof(double) * 2 * ks_tri(k), s, k,
                     EB, T, status);
  MDA_LAUNCH_CHECK();
}

// EnKF: with M = (k-1) I + Y'^T R^-1 Y' the Woodbury identity gives
// Y'^T S^-1 / (k-1) = M^-1 Y'^T R^-1 for S = Y'Y'^T/(k-1) + R
// (EnKF.hpp:193-199), so K D = X' M^-1 F with F = Y'^T R^-1 D and the update
// x_a = xbar + X'_j + K D_j (EnKF.hpp:216-226) is X_a = xbar + X'(I + M^-1 F).
// Outputs T = I + M^-1 F and M^-1 = W W^T.
__global__ __launch_bounds__(KS_THREADS) void k_enkf_solve(int k, const double* __restrict__ EB,
                                                           const double* __restrict__ F,
                                                           double* __restrict__ T,
                                                           double* __restrict__ Minv,
                                                           int* status) {
  extern __shared__ double sh[];
  const int tid = threadIdx.x;
  const ks_lds f{sh, sh + ks_tri(k), k};
  const bool ok = ks_factor(f, EB, false);
  if (!ok) {
    if (tid == 0) atomicOr(status, MDA_ST_NOT_SPD);
    return;
  }
  // M^-1 into the place of L (W has all it needs)
  for (int idx = tid; idx < k * k; idx += KS_THREADS) {
    const int i = idx / k, j = idx % k;
    if (j > i) continue;
    const double *wi = f.wrow(i), *wj = f.wrow(j);
    double s = 0.0;
#pragma unroll 4
    for (int c = i; c < k; ++c) s = fma(wi[c], wj[c], s);
    f.lrow(i)[j] = s;
    Minv[i * k + j] = s;
    Minv[j * k + i] = s;
  }
  __syncthreads();
  for (int idx = tid; idx < (k + 3) / 4 * k; idx += KS_THREADS) {
    const int i0 = idx / k * 4, j = idx % k;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int c = 0; c < k; ++c) {
      const double fv = F[(size_t)c * k + j];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + r < k ? i0 + r : k - 1;
        s[r] = fma(i >= c ? f.lrow(i)[c] : f.lrow(c)[i], fv, s[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (i0 + r < k) T[(size_t)(i0 + r) * k + j] = (i0 + r == j ? 1.0 : 0.0) + s[r];
  }
}

void launch_enkf_solve_ws(hipStream_t s, int k, const double* EB, const double* F, double* T,
                          double* Minv, int* status) {
  MDA_REQUIRE(k <= 128, "EnKF supports k <= 128");
  hipLaunchKernelGGL(k_enkf_solve, dim3(1), dim3(KS_THREADS), sizeof(double) * 2 * ks_tri(k), s, k,
                     EB, F, T, Minv, status);
  MDA_LAUNCH_CHECK();
}

// [max, min, sum, sum] of nb partial quadruples, one block, in a fixed order
__global__ __launch_bounds__(256) void k_fold_extremes(const double* __restrict__ partial,
                                                       int64_t nb, double* __restrict__ out) {
  __shared__ double r0[256], r1[256], r2[256], r3[256];
  const int tid = threadIdx.x;
  double mx = -INFINITY, mn = INFINITY, s2 = 0.0, s3 = 0.0;
#pragma unroll 4
  for (int64_t b = tid; b < nb; b += 256) {
    mx = fmax(mx, partial[4 * b]);
    mn = fmin(mn, partial[4 * b + 1]);
    s2 += partial[4 * b + 2];
    s3 += partial[4 * b + 3];
  }
  r0[tid] = mx; r1[tid] = mn; r2[tid] = s2; r3[tid] = s3;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (tid < st) {
      r0[tid] = fmax(r0[tid], r0[tid + st]);
      r1[tid] = fmin(r1[tid], r1[tid + st]);
      r2[tid] += r2[tid + st];
      r3[tid] += r3[tid + st];
    }
    __syncthreads();
  }
  if (tid == 0) { out[0] = r0[0]; out[1] = r1[0]; out[2] = r2[0]; out[3] = r3[0]; }
}

void launch_fold_extremes(hipStream_t s, const double* partial, int64_t nb, double* out4) {
  hipLaunchKernelGGL(k_fold_extremes, dim3(1), dim3(256), 0, s, partial, nb, out4);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Global transform: X_a[j][i] = xbar_i + sum_m (scale (x_m,i - xbar_i)) T[m][j]
// (ETKF.hpp:163-169, EnKF.hpp:216-227) on FP64 MFMA, in place.  T sits in LDS
// in fragment order (one 512-byte read per two products: A = T^T, rows =
// analysis members), a wavefront takes 32 points with all their members in
// registers (B, columns = points), so X is read and written once in 128-byte
// segments.  Bound by HBM: n = 2,097,152, k = 64 moves 2.15 GB in 0.55 ms
// (3.9 TB/s; one LDS broadcast per FMA took 2.50 ms).
// Nothing is written when an earlier stage of the analysis failed (status bits
// MDA_ST_SKIP_UPDATE); a non-finite background value sets
// MDA_ST_NONFINITE_STATE (the analysis at that index is then non-finite, as
// the reference's arithmetic makes it).  With `partial`, each block leaves
// [-1e308, 1e308, 0, sum of (x_a - mean_a)^2] for the analysis spread
// (EnKF.hpp:246-253): sums of the deviations from member 0's increment, which
// are of the spread's own size.
// ---------------------------------------------------------------------------
constexpr int TG_THREADS = 512, TG_POINTS = TG_THREADS / 64 * 32;

template <int NS>
__global__ __launch_bounds__(TG_THREADS) void k_transform_global(
    double* __restrict__ X, int k, int64_t n, double scale, const double* __restrict__ T,
    int* __restrict__ status, double* __restrict__ partial) {
  constexpr int NT = NS / 4;
  extern __shared__ double Tf[];  // [NS][NT][64]
  __shared__ double red[TG_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, i16 = lane & 15, kk = lane >> 4;
  double ss = 0.0;
  if (!(status && (*status & MDA_ST_SKIP_UPDATE))) {
    for (int e = tid; e < NS * NT * 64; e += TG_THREADS) {
      const int l = e & 63, tj = (e >> 6) % NT, st = (e >> 6) / NT;
      const int m = 4 * st + (l >> 4), j = 16 * tj + (l & 15);
      Tf[e] = m < k && j < k ? T[m * k + j] : 0.0;
    }
    __syncthreads();
    for (int64_t b0 = (int64_t)blockIdx.x * TG_POINTS; b0 < n;
         b0 += (int64_t)gridDim.x * TG_POINTS) {
      const int64_t i0 = b0 + 32 * wv;
      if (i0 >= n) continue;
      double v[2][NS], mean[2], sh[2] = {0.0, 0.0}, s1[2] = {0.0, 0.0}, s2[2] = {0.0, 0.0};
      load_pert<NS, 2>(X, k, n, scale, i0, v, mean);
      if (status && (!isfinite(mean[0]) || !isfinite(mean[1])))
        atomicOr(status, MDA_ST_NONFINITE_STATE);
#pragma unroll 1
      for (int tj = 0; tj < NT; ++tj) {
        d4 acc[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
        const double* tf = Tf + tj * 64 + lane;
#pragma unroll
        for (int st = 0; st < NS; ++st) {
          const double a = tf[st * NT * 64];
          acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, v[0][st], acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, v[1][st], acc[1], 0, 0, 0);
        }
        // D[kk + 4r][i16]: member 16 tj + kk + 4r, point i16
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int64_t i = i0 + 16 * t + i16;
          if (tj == 0) sh[t] = __shfl(acc[t][0], i16);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = 16 * tj + kk + 4 * r;
            if (j < k && i < n) {
              X[(size_t)j * n + i] = mean[t] + acc[t][r];
              const double dv = acc[t][r] - sh[t];
              s1[t] += dv;
              s2[t] = fma(dv, dv, s2[t]);
            }
          }
        }
      }
      if (partial) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          for (int off = 16; off < 64; off <<= 1) {
            s1[t] += __shfl_xor(s1[t], off);
            s2[t] += __shfl_xor(s2[t], off);
          }
          if (kk == 0) ss += s2[t] - s1[t] * s1[t] / (double)k;
        }
      }
    }
  }
  if (!partial) return;
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  if (lane == 0) red[wv] = ss;
  __syncthreads();
  if (tid == 0) {
    double t = 0.0;
    for (int w = 0; w < TG_THREADS / 64; ++w) t += red[w];
    double* out = partial + 4 * (size_t)blockIdx.x;
    out[0] = -1.0e308;
    out[1] = 1.0e308;
    out[2] = 0.0;
    out[3] = t;
  }
}

unsigned transform_global_blocks(int64_t n) {
  return grid_for(n, TG_POINTS, 4096);
}

void launch_transform_global(hipStream_t s, double* X, int k, int64_t n, double scale,
                             const double* T, int* status, double* partial, double* out4) {
  MDA_REQUIRE(k <= 128, "global transform supports k <= 128");
  const unsigned g = transform_global_blocks(n);
#define MDA_TG(NS)                                                                           \
  hipLaunchKernelGGL(k_transform_global<NS>, dim3(g), dim3(TG_THREADS),                      \
                     sizeof(double) * NS * (NS / 4) * 64, s, X, k, n, scale, T, status, partial)
  MDA_MEMBER_STEPS(k, MDA_TG)
#undef MDA_TG
  MDA_LAUNCH_CHECK();
  if (partial) launch_fold_extremes(s, partial, g, out4);
}

// ---------------------------------------------------------------------------
// EnKF diagnostics: max / min of K = X' G with G = M^-1 Y'^T R^-1 (k x p),
// EnKF.hpp:202-203, and the background's sum of squares (:334).  G is formed
// first in fragment order, Gf[tile of 16 observations][step][lane] =
// G[4 step + kk][16 tile + i16], 512 contiguous bytes per MFMA step.  Then K
// is formed tile by tile on the matrix cores and folded into the extremes at
// once; it never reaches memory.  Bound by the FP64 matrix rate (2 n p k
// FLOP): one 16x16x4 product takes 64 cycles of its SIMD, so a fragment load
// per two products (two tiles of points per wavefront) leaves the caches
// idle.  The observation tiles are split over gridDim.y when the points alone
// leave SIMDs empty.  n = 262,144, p = 1,500, k = 80: 73.7 ms with one thread
// per point (its perturbations in scratch memory), 1.11 ms here (57 TFLOP/s; a
// large FP64 matrix product reaches 72 on this card).
// ---------------------------------------------------------------------------
__global__ void k_enkf_G(const double* __restrict__ Minv, const double* __restrict__ yp_om,
                         const double* __restrict__ var, int k, int64_t p, int ns,
                         int64_t ntile, double* __restrict__ Gf) {
  const int64_t total = ntile * ns * 64;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(e & 63);
    const int64_t ts = e >> 6;
    const int64_t o = ts / ns * 16 + (lane & 15);
    const int a = 4 * (int)(ts % ns) + (lane >> 4);
    double g = 0.0;
    if (o < p && a < k) {
      const double* mr = Minv + (size_t)a * k;
      const double* yr = yp_om + (size_t)o * k;
      double s0 = 0.0, s1 = 0.0;
      int b = 0;
#pragma unroll 4
      for (; b + 1 < k; b += 2) {
        s0 = fma(mr[b], yr[b], s0);
        s1 = fma(mr[b + 1], yr[b + 1], s1);
      }
      if (b < k) s0 = fma(mr[b], yr[b], s0);
      g = (s0 + s1) / var[o];
    }
    Gf[e] = g;
  }
}

template <int NS>
__global__ __launch_bounds__(256) void k_enkf_gain_minmax(const double* __restrict__ X, int k,
                                                          int64_t n, double scale,
                                                          const double* __restrict__ Gf,
                                                          int64_t p, int64_t ntile, int64_t per,
                                                          double* __restrict__ partial) {
  __shared__ double red[3][4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i16 = lane & 15, kk = lane >> 4;
  const int64_t i0 = ((int64_t)blockIdx.x * 4 + wv) * 32;
  double a[2][NS], mean[2];
  load_pert<NS, 2>(X, k, n, scale, i0, a, mean);
  double mx = -1.0e308, mn = 1.0e308, ss = 0.0;
  if (blockIdx.y == 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < NS; ++s) ss = fma(a[t][s], a[t][s], ss);
  }
  const int64_t t0 = blockIdx.y * per, t1 = t0 + per < ntile ? t0 + per : ntile;
  if (i0 < n) {
    for (int64_t ot = t0; ot < t1; ++ot) {
      const double* gf = Gf + (size_t)ot * NS * 64 + lane;
      d4 acc[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const double b = gf[64 * s];
        acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[0][s], b, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[1][s], b, acc[1], 0, 0, 0);
      }
      // D[kk + 4r][i16]: point kk + 4r of the tile, observation i16
      const bool ov = 16 * ot + i16 < p;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double v = acc[t][r];
          const bool in = ov && i0 + 16 * t + kk + 4 * r < n;
          mx = in && v > mx ? v : mx;
          mn = in && v < mn ? v : mn;
        }
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    mx = fmax(mx, __shfl_xor(mx, off));
    mn = fmin(mn, __shfl_xor(mn, off));
    ss += __shfl_xor(ss, off);
  }
  if (lane == 0) { red[0][wv] = mx; red[1][wv] = mn; red[2][wv] = ss; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double* out = partial + 4 * ((size_t)blockIdx.y * gridDim.x + blockIdx.x);
    out[0] = fmax(fmax(red[0][0], red[0][1]), fmax(red[0][2], red[0][3]));
    out[1] = fmin(fmin(red[1][0], red[1][1]), fmin(red[1][2], red[1][3]));
    out[2] = (red[2][0] + red[2][1]) + (red[2][2] + red[2][3]);
    out[3] = 0.0;
  }
}

// Launch shape: one block per 128 points; with fewer than 1024 blocks (one
// wavefront per SIMD of the chip) the observation tiles are split further.
enkf_gain_shape enkf_gain_plan(int k, int64_t n, int64_t p) {
  enkf_gain_shape g;
  g.ns = (k + 15) / 16 * 4;
  g.ntile = (p + 15) / 16;
  g.nbx = (n + 127) / 128;
  const int64_t want = std::max<int64_t>(1, 1024 / g.nbx);
  g.per = (g.ntile + want - 1) / want;
  g.nby = (g.ntile + g.per - 1) / g.per;
  return g;
}

void launch_enkf_gain_minmax(hipStream_t s, const double* X, int k, int64_t n, double scale,
                             const double* Minv, const double* yp_om, const double* var,
                             int64_t p, const enkf_gain_shape& g, double* Gf, double* partial,
                             double* out4) {
  MDA_REQUIRE(k <= 128, "gain diagnostics support k <= 128");
  MDA_REQUIRE(g.nbx < (int64_t)1 << 31 && g.nby < 65536, "gain grid too large");
  hipLaunchKernelGGL(k_enkf_G, dim3(grid_for(g.ntile * g.ns * 64, 256, 4096)), dim3(256), 0, s,
                     Minv, yp_om, var, k, p, g.ns, g.ntile, Gf);
  MDA_LAUNCH_CHECK();
#define MDA_GAIN(NS)                                                                              \
  hipLaunchKernelGGL(k_enkf_gain_minmax<NS>, dim3((unsigned)g.nbx, (unsigned)g.nby), dim3(256),  \
                     0, s, X, k, n, scale, Gf, p, g.ntile, g.per, partial)
  MDA_MEMBER_STEPS(k, MDA_GAIN)
#undef MDA_GAIN
  MDA_LAUNCH_CHECK();
  launch_fold_extremes(s, partial, g.nbx * g.nby, out4);
}

// ---------------------------------------------------------------------------
// Metrics::CalculateAll (Metrics.hpp:74-94): per-block partial sums of
// [rmse^2, bias, sum mean, sum truth, sum mean*truth, sum mean^2,
//  sum truth^2, spread, crps].
// One point per thread.  Up to 128 members sit in registers (KM of them), and
// the CRPS's k^2 differences take each member once more from the cache against
// all the registers, against itself in place of the entries past k: two FP64
// operations a pair and X read from HBM once.  n = 1,048,576, k = 40: 184 us
// (3.56 ms with both members of every pair loaded).  Beyond 128 members
// (KM = 0) that form remains.
// ---------------------------------------------------------------------------
template <int KM, bool WHOLE>  // WHOLE: k = KM
__global__ __launch_bounds__(256) void k_metrics(const double* __restrict__ X, int k, int64_t n,
                                                 const double* __restrict__ truth,
                                                 double* __restrict__ partial) {
  __shared__ double red[256];
  double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double t = truth[i];
    double m = 0.0, sp = 0.0, sd = 0.0, st = 0.0;
    if constexpr (KM > 0) {
      double x[KM];
#pragma unroll
      for (int j = 0; j < KM; ++j) x[j] = WHOLE || j < k ? X[(size_t)j * n + i] : 0.0;
#pragma unroll
      for (int j = 0; j < KM; ++j) m += x[j];
      m /= (double)k;  // Metrics.hpp:111-113 divides
#pragma unroll
      for (int j = 0; j < KM; ++j) {
        const double df = x[j] - m;
        if (WHOLE || j < k) {
          sp += df * df;
          st += fabs(x[j] - t);
        }
      }
      // entries that every k of this kernel fills
      constexpr int FULL = WHOLE ? KM : KM - (KM > 64 ? 16 : 8) + 1;
      double d0 = 0.0, d1 = 0.0;
      double xn = x[0];
      for (int a = 0; a < k; ++a) {
        const double xa = xn;
        if (a + 1 < k) xn = X[(size_t)(a + 1) * n + i];  // in flight during the pairs
#pragma unroll
        for (int b = 0; b < KM; b += 2) {
          d0 += fabs(xa - (b < FULL || b < k ? x[b] : xa));
          d1 += fabs(xa - (b + 1 < FULL || b + 1 < k ? x[b + 1] : xa));
        }
      }
      sd = d0 + d1;
    } else {
      for (int j = 0; j < k; ++j) m += X[(size_t)j * n + i];
      m /= (double)k;
      for (int j = 0; j < k; ++j) {
        double df = X[(size_t)j * n + i] - m;
        sp += df * df;
      }
      for (int a = 0; a < k; ++a) {
        double xa = X[(size_t)a * n + i];
        for (int b = 0; b < k; ++b) sd += fabs(xa - X[(size_t)b * n + i]);
        st += fabs(xa - t);
      }
    }
    sp = sqrt(sp / (double)(k - 1));
    const double df = m - t;
    acc[0] += df * df; acc[1] += df; acc[2] += m; acc[3] += t; acc[4] += m * t;
    acc[5] += m * m; acc[6] += t * t; acc[7] += sp;
    acc[8] += st / k - sd / (2.0 * k * k);
  }
  for (int q = 0; q < 9; ++q) {
    double v = block_sum(acc[q], red);
    if (threadIdx.x == 0) partial[(size_t)blockIdx.x * 9 + q] = v;
  }
}

void launch_metrics(hipStream_t s, const double* X, int k, int64_t n, const double* truth,
                    double* partial, double* out9) {
  const unsigned nb = grid_for(n, 256, METRICS_BLOCKS);
#define MDA_MTL(KM, WHOLE)                                                                 \
  hipLaunchKernelGGL((k_metrics<KM, WHOLE>), dim3(nb), dim3(256), 0, s, X, k, n, truth, partial)
#define MDA_MT(KM)                \
  {                               \
    if (k == KM)                  \
      MDA_MTL(KM, true);          \
    else                          \
      MDA_MTL(KM, false);         \
  }
  if (k <= 8) MDA_MT(8)
  else if (k <= 16) MDA_MT(16)
  else if (k <= 24) MDA_MT(24)
  else if (k <= 32) MDA_MT(32)
  else if (k <= 40) MDA_MT(40)
  else if (k <= 48) MDA_MT(48)
  else if (k <= 56) MDA_MT(56)
  else if (k <= 64) MDA_MT(64)
  else if (k <= 80) MDA_MT(80)
  else if (k <= 96) MDA_MT(96)
  else if (k <= 112) MDA_MT(112)
  else if (k <= 128) MDA_MT(128)
  else MDA_MTL(0, false);
#undef MDA_MT
#undef MDA_MTL
  MDA_LAUNCH_CHECK();
  launch_reduce_partials(s, partial, (int)nb, 9, out9);
}

}  // namespace mda
