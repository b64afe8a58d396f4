// Dense p x p linear algebra of the global filters, kept in device memory:
//   - the EnKF's S = Y'Y'^T/(k-1) + R and its condition number
//     (EnKF.hpp:188-209: JacobiSVD singular values), from the k x k side
//     when p > 128,
//   - Householder tridiagonalisation of a symmetric matrix, whose extreme
//     eigenvalues (and the one nearest zero) are then found by multisection on
//     Sturm counts of the tridiagonal,
//   - Gauss-Jordan elimination with partial pivoting, A^-1 B for p x m B (the
//     S^-1 products of EnKF.hpp:199 and LWEnKF.hpp:273-276).
// Each elimination step is a short sequence of launches over the trailing
// matrix: O(p^3) work, as the reference's own dense algebra.  Sizes are
// bounded by MDA_DENSE_MAX.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "mda_device.hpp"
#include "mda_internal.hpp"

namespace mda {

// S[a][b] = (sum_j Y'[a][j] Y'[b][j]) / (k-1) + (a == b ? var[a] : 0), Y'
// obs-major [p][k]; the member sum runs in member order (as EnKF.hpp:193).
__global__ void k_form_enkf_S(const double* __restrict__ yp, const double* __restrict__ var,
                              int k, int64_t p, double* __restrict__ S) {
  const int64_t total = p * p;
  const double rk1 = 1.0 / (double)(k - 1);
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t a = e / p, b = e % p;
    const double* ya = yp + (size_t)a * k;
    const double* yb = yp + (size_t)b * k;
    double s = 0.0;
    for (int j = 0; j < k; ++j) s += ya[j] * yb[j];
    S[e] = s * rk1 + (a == b ? var[a] : 0.0);
  }
}

void launch_form_enkf_S(hipStream_t s, const double* yp, const double* var, int k, int64_t p,
                        double* S) {
  hipLaunchKernelGGL(k_form_enkf_S, dim3(grid_for(p * p, 256, 8192)), dim3(256), 0, s, yp, var,
                     k, p, S);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Householder tridiagonalisation, step j (m = p - j - 1 trailing rows):
//   x = A[j+1:, j], alpha = -sign(x_0) ||x||, u = x - alpha e_1,
//   tau = 2 / u^T u, pv = tau A' u, w = pv - (tau/2)(pv^T u) u,
//   A' <- A' - u w^T - w u^T;  d_j = A[j][j], e_j = alpha.
// ---------------------------------------------------------------------------
__device__ inline double block_reduce_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if (lane == 0) red[wv] = v;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}

__global__ __launch_bounds__(1024) void k_hh_vec(int64_t p, int64_t j, const double* __restrict__ A,
                                                 double* __restrict__ u, double* __restrict__ sc,
                                                 double* __restrict__ d, double* __restrict__ e) {
  __shared__ double red[16];
  double s = 0.0;
  for (int64_t r = j + 1 + threadIdx.x; r < p; r += blockDim.x) {
    const double x = A[(size_t)r * p + j];
    s += x * x;
  }
  const double nrm2 = block_reduce_sum(s, red);
  const double x0 = A[(size_t)(j + 1) * p + j];
  const bool nz = nrm2 > 0.0;
  const double alpha = nz ? (x0 > 0.0 ? -1.0 : 1.0) * sqrt(nrm2) : 0.0;
  const double tau = nz ? 2.0 / (nrm2 - 2.0 * alpha * x0 + alpha * alpha) : 0.0;
  for (int64_t r = threadIdx.x; r < p; r += blockDim.x) {
    double v = 0.0;
    if (r > j && nz) v = A[(size_t)r * p + j] - (r == j + 1 ? alpha : 0.0);
    u[r] = v;
  }
  if (threadIdx.x == 0) {
    sc[0] = tau;
    d[j] = A[(size_t)j * p + j];
    e[j] = alpha;
  }
}

// pv[r] = tau sum_{c > j} A[r][c] u[c] for r > j: one wavefront per row
__global__ __launch_bounds__(256) void k_hh_symv(int64_t p, int64_t j, const double* __restrict__ A,
                                                 const double* __restrict__ u,
                                                 const double* __restrict__ sc,
                                                 double* __restrict__ pv) {
  const int lane = threadIdx.x & 63;
  const int64_t nw = (int64_t)gridDim.x * (blockDim.x >> 6);
  const double tau = sc[0];
  for (int64_t r = j + 1 + blockIdx.x * (int64_t)(blockDim.x >> 6) + (threadIdx.x >> 6); r < p;
       r += nw) {
    const double* row = A + (size_t)r * p;
    double s = 0.0;
    for (int64_t c = j + 1 + lane; c < p; c += 64) s += row[c] * u[c];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) pv[r] = tau * s;
  }
}

// w = pv - (tau/2)(pv^T u) u (one block)
__global__ __launch_bounds__(1024) void k_hh_w(int64_t p, int64_t j, const double* __restrict__ u,
                                               const double* __restrict__ pv,
                                               const double* __restrict__ sc,
                                               double* __restrict__ w) {
  __shared__ double red[16];
  double s = 0.0;
  for (int64_t r = j + 1 + threadIdx.x; r < p; r += blockDim.x) s += pv[r] * u[r];
  const double K = 0.5 * sc[0] * block_reduce_sum(s, red);
  for (int64_t r = j + 1 + threadIdx.x; r < p; r += blockDim.x) w[r] = pv[r] - K * u[r];
}

// A' <- A' - u w^T - w u^T on the trailing block (two FMAs per entry)
__global__ __launch_bounds__(256) void k_hh_syr2(int64_t p, int64_t j, double* __restrict__ A,
                                                 const double* __restrict__ u,
                                                 const double* __restrict__ w) {
  const int64_t m = p - j - 1;
  const int64_t total = m * m;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = j + 1 + t / m, c = j + 1 + t % m;
    double& a = A[(size_t)r * p + c];
    a = fma(-u[r], w[c], fma(-w[r], u[c], a));
  }
}

// last 2 x 2 block of the tridiagonal
__global__ void k_hh_tail(int64_t p, const double* __restrict__ A, double* __restrict__ d,
                          double* __restrict__ e) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  if (p >= 2) {
    d[p - 2] = A[(size_t)(p - 2) * p + (p - 2)];
    e[p - 2] = A[(size_t)(p - 1) * p + (p - 2)];
  }
  d[p - 1] = A[(size_t)(p - 1) * p + (p - 1)];
  e[p - 1] = 0.0;
}

void dense_tridiagonalise(hipStream_t s, int64_t p, double* A, double* d, double* e, double* u,
                          double* pv, double* w, double* sc) {
  MDA_REQUIRE(p >= 1 && p <= MDA_DENSE_MAX, "dense matrix size out of range");
  for (int64_t j = 0; j + 2 < p; ++j) {
    const int64_t m = p - j - 1;
    hipLaunchKernelGGL(k_hh_vec, dim3(1), dim3(1024), 0, s, p, j, A, u, sc, d, e);
    MDA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_hh_symv, dim3(grid_for(m, 4, 2048)), dim3(256), 0, s, p, j, A, u, sc, pv);
    MDA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_hh_w, dim3(1), dim3(1024), 0, s, p, j, u, pv, sc, w);
    MDA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_hh_syr2, dim3(grid_for(m * m, 256, 8192)), dim3(256), 0, s, p, j, A, u, w);
    MDA_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_hh_tail, dim3(1), dim3(64), 0, s, p, A, d, e);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// The same reduction for n <= SYM_LDS_N in one launch: a workgroup of 512
// threads holds the matrix in LDS (row stride = 4 mod 32 doubles: the four
// threads of a row and eight rows of a half wavefront fall on 32 different
// bank pairs).  Norms and dot products of a step are formed by every
// wavefront for itself, so a step costs three barriers.  Bound by those and
// by LDS latency: n = 20 61 us with the extremes below, against 167 us for a
// one-workgroup Jacobi of the matrix in global memory.
// ---------------------------------------------------------------------------
constexpr int SYM_LDS_N = 128;

__device__ inline double wave_sum_xor(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

__global__ __launch_bounds__(512) void k_sym_tridiag_lds(const double* __restrict__ A,
                                                         int64_t lda, int n, int ld,
                                                         double* __restrict__ d,
                                                         double* __restrict__ e) {
  extern __shared__ double sh[];
  double* a = sh;                     // [n][ld]
  double* u = a + (size_t)n * ld;     // [SYM_LDS_N]
  double* pv = u + SYM_LDS_N;         // [SYM_LDS_N]
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = tid >> 2, h = tid & 3;
  for (int idx = tid; idx < n * n; idx += 512)
    a[(idx / n) * ld + idx % n] = A[(size_t)(idx / n) * lda + idx % n];
  if (tid < SYM_LDS_N) { u[tid] = 0.0; pv[tid] = 0.0; }
  __syncthreads();
  for (int j = 0; j + 2 < n; ++j) {
    // x = A[j][j+1..] (row j equals column j): entries lane and lane + 64
    const double x0 = lane > j && lane < n ? a[j * ld + lane] : 0.0;
    const double x1 = lane + 64 > j && lane + 64 < n ? a[j * ld + lane + 64] : 0.0;
    const double nrm2 = wave_sum_xor(fma(x0, x0, x1 * x1));
    const double xh = a[j * ld + j + 1];
    const bool nz = nrm2 > 0.0;
    const double alpha = nz ? (xh > 0.0 ? -1.0 : 1.0) * sqrt(nrm2) : 0.0;
    const double tau = nz ? 2.0 / (nrm2 - 2.0 * alpha * xh + alpha * alpha) : 0.0;
    const double u0 = nz ? x0 - (lane == j + 1 ? alpha : 0.0) : 0.0;
    const double u1 = nz ? x1 - (lane + 64 == j + 1 ? alpha : 0.0) : 0.0;
    if (tid < 64) {
      u[lane] = u0;
      u[lane + 64] = u1;
      if (lane == 0) { d[j] = a[j * ld + j]; e[j] = alpha; }
    }
    __syncthreads();
    const bool live = r > j && r < n;
    double pr = 0.0;
    if (live)
      for (int c = h; c < n; c += 4) pr = fma(a[r * ld + c], u[c], pr);  // u = 0 up to j
    pr += __shfl_xor(pr, 1);
    pr += __shfl_xor(pr, 2);
    pr *= tau;
    if (h == 0 && live) pv[r] = pr;
    __syncthreads();
    const double p0 = lane > j && lane < n ? pv[lane] : 0.0;
    const double p1 = lane + 64 > j && lane + 64 < n ? pv[lane + 64] : 0.0;
    const double K = 0.5 * tau * wave_sum_xor(fma(p0, u0, p1 * u1));
    if (live) {
      const double ur = u[r], wr = pr - K * ur;
      for (int c = h; c < n; c += 4)
        if (c > j) {
          const double wc = pv[c] - K * u[c];
          a[r * ld + c] = fma(-ur, wc, fma(-wr, u[c], a[r * ld + c]));
        }
    }
    __syncthreads();
  }
  if (tid == 0) {
    if (n >= 2) {
      d[n - 2] = a[(n - 2) * ld + n - 2];
      e[n - 2] = a[(n - 2) * ld + n - 1];
    }
    d[n - 1] = a[(n - 1) * ld + n - 1];
    e[n - 1] = 0.0;
  }
}

// ---------------------------------------------------------------------------
// Extreme eigenvalues of a symmetric tridiagonal (d, e), one workgroup:
// multisection on Sturm counts, 128 threads (points) for each of the smallest,
// the largest, the largest negative and the smallest non-negative eigenvalue,
// 7 bits a round.  count(x) = number of eigenvalues < x from the pivots of
// the LDL^T factorisation of T - x I.  out = [lmin, lmax, |l|min, |l|max].
// ---------------------------------------------------------------------------
__device__ inline int sturm_count(const double* d, const double* e2, int n, double x,
                                  double pivmin) {
  int cnt = 0;
  double q = 1.0;
  for (int i = 0; i < n; ++i) {
    q = (d[i] - x) - (i > 0 ? e2[i - 1] / q : 0.0);
    if (fabs(q) < pivmin) q = -pivmin;
    cnt += q < 0.0;
  }
  return cnt;
}

__global__ __launch_bounds__(512) void k_tridiag_extremes(const double* __restrict__ dg,
                                                          const double* __restrict__ eg, int n,
                                                          double* __restrict__ out) {
  extern __shared__ double sh[];  // d [n], e^2 [n]
  __shared__ double red[3][8], slo[4], shi[4];
  __shared__ uint64_t bal[8];
  double* d = sh;
  double* e2 = sh + n;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double lo = INFINITY, hi = -INFINITY, em = 0.0;
  for (int i = tid; i < n; i += 512) {
    const double di = dg[i], ei = i + 1 < n ? fabs(eg[i]) : 0.0;
    const double r = (i > 0 ? fabs(eg[i - 1]) : 0.0) + ei;
    d[i] = di;
    e2[i] = ei * ei;
    lo = fmin(lo, di - r);
    hi = fmax(hi, di + r);
    em = fmax(em, ei);
  }
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off));
    hi = fmax(hi, __shfl_xor(hi, off));
    em = fmax(em, __shfl_xor(em, off));
  }
  if (lane == 0) { red[0][wv] = lo; red[1][wv] = hi; red[2][wv] = em; }
  __syncthreads();
  for (int w = 0; w < 8; ++w) {
    lo = fmin(lo, red[0][w]);
    hi = fmax(hi, red[1][w]);
    em = fmax(em, red[2][w]);
  }
  const double span = fmax(fabs(lo), fabs(hi));
  lo -= 1e-14 * span + 1e-300;
  hi += 1e-14 * span + 1e-300;
  const double pivmin = fmax(1e-300, 1e-300 * em * em);
  const int neg = sturm_count(d, e2, n, 0.0, pivmin);
  const int tg = tid >> 7, t = tid & 127;
  const int idx = tg == 0 ? 0 : tg == 1 ? n - 1 : tg == 2 ? neg - 1 : neg;
  if (t == 0) {
    slo[tg] = tg == 3 ? 0.0 : lo;
    shi[tg] = tg == 2 ? 0.0 : hi;
  }
  __syncthreads();
  for (int round = 0; round < 10; ++round) {
    const double a = slo[tg], b = shi[tg], w = b - a;
    const double x = a + w * ((double)(t + 1) / 129.0);
    const bool above = idx >= 0 && idx < n && sturm_count(d, e2, n, x, pivmin) > idx;
    const uint64_t m = __ballot(above);
    if (lane == 0) bal[wv] = m;
    __syncthreads();
    if (t == 0) {
      const uint64_t b0 = bal[2 * tg], b1 = bal[2 * tg + 1];
      const int f = b0 ? __builtin_ctzll(b0) : b1 ? 64 + __builtin_ctzll(b1) : 128;
      if (f > 0) slo[tg] = a + w * ((double)f / 129.0);
      if (f < 128) shi[tg] = a + w * ((double)(f + 1) / 129.0);
    }
    __syncthreads();
  }
  if (tid == 0) {
    const double l0 = 0.5 * (slo[0] + shi[0]), l1 = 0.5 * (slo[1] + shi[1]);
    double am = INFINITY;
    if (neg > 0) am = fmin(am, fabs(0.5 * (slo[2] + shi[2])));
    if (neg < n) am = fmin(am, fabs(0.5 * (slo[3] + shi[3])));
    out[0] = l0;
    out[1] = l1;
    out[2] = am;
    out[3] = fmax(fabs(l0), fabs(l1));
  }
}

void dense_sym_extremes(mda_ctx* c, double* A, int64_t p, int64_t lda, double* out) {
  hipStream_t s = c->stream;
  if (lda == 0) lda = p;
  double* d = c->get<double>("dense_d", p);
  double* e = c->get<double>("dense_e", p);
  if (p <= SYM_LDS_N) {
    const int n = (int)p, ld = (n + 27) / 32 * 32 + 4;  // the next row stride = 4 mod 32
    const size_t shm = sizeof(double) * ((size_t)n * ld + 2 * SYM_LDS_N);
    hipLaunchKernelGGL(k_sym_tridiag_lds, dim3(1), dim3(512), shm, s, A, lda, n, ld, d, e);
    MDA_LAUNCH_CHECK();
  } else {
    MDA_REQUIRE(lda == p, "the large reduction takes contiguous rows");
    double* u = c->get<double>("dense_u", p);
    double* pv = c->get<double>("dense_pv", p);
    double* w = c->get<double>("dense_w", p);
    double* sc = c->get<double>("dense_sc", 4);
    dense_tridiagonalise(s, p, A, d, e, u, pv, w, sc);
  }
  hipLaunchKernelGGL(k_tridiag_extremes, dim3(1), dim3(512), sizeof(double) * 2 * p, s, d, e,
                     (int)p, out);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Extreme eigenvalues of S = R + Y Y^T / (k-1), R = diag(r), Y [p][k], without
// forming S.  By the inertia of the block matrix [[R - x, Y], [Y^T, -(k-1) I]]
// (its two Schur complements):
//   x > lambda_max  <=>  (k-1) I - Y^T (x - R)^-1 Y is positive definite
//                        (x > max r);
//   x < lambda_min  <=>  W W^T - D is positive definite, with the rows split
//                        by r: A = (k-1) I + sum_{r_o > x} y_o y_o^T / (r_o - x)
//                        = L L^T, W = Y_- L^-T and D = diag(x - r_o) over the q
//                        rows with r_o <= x (never, when q > k).
// Both are decided by Cholesky factorisations of definite matrices.  A round
// tests 128 points inside each of the two brackets, one workgroup per point
// (256 workgroups, one per CU): the weighted Gram on FP64 MFMA, the rows of
// Y_- carried through the factorisation of A, all in LDS.  Eight rounds narrow
// each bracket by 129^8 = 8e16.  At p = 1,500, k = 80 the dense reduction of S
// took 33 ms (four launches per column), this 1.8 ms.
// ---------------------------------------------------------------------------
constexpr int CE_PTS = 128, CE_ROUNDS = 8;

// sorted rows: Yf[step][tile][lane] = y of row 4 step + kk, member 16 tile + i16
// (zeros past p and k), rs = r (+inf past p), ss = |y|^2 per row
__global__ void k_ce_rows(const double* __restrict__ yp, const double* __restrict__ var,
                          const uint32_t* __restrict__ order, int k, int kt, int64_t p,
                          int64_t nstep, double* __restrict__ Yf, double* __restrict__ rs,
                          double* __restrict__ ss) {
  const int64_t total = nstep * kt * 64;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(e & 63);
    const int64_t st = (e >> 6) / kt, t = 4 * st + (lane >> 4);
    const int m = 16 * (int)((e >> 6) % kt) + (lane & 15);
    Yf[e] = t < p && m < k ? yp[(size_t)order[t] * k + m] : 0.0;
  }
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < 4 * nstep;
       t += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    if (t < p)
      for (int m = 0; m < k; ++m) {
        const double v = yp[(size_t)order[t] * k + m];
        s = fma(v, v, s);
      }
    rs[t] = t < p ? var[order[t]] : INFINITY;
    ss[t] = s;
  }
}

// The bracket of kind 0 (lambda_max) or 1 (lambda_min) after `rounds` rounds,
// the same in every workgroup; 256 threads, red: 8 doubles of LDS.
__device__ inline void ce_bracket(int kind, int rounds, int k, int64_t p,
                                  const double* __restrict__ rs, const double* __restrict__ ss,
                                  const int* __restrict__ flags, double* red, double& lo,
                                  double& hi) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const double rk1 = 1.0 / (double)(k - 1);
  double tr = 0.0, mn = INFINITY;
  for (int64_t t = tid; t < p; t += 256) {
    tr += ss[t];
    mn = fmin(mn, fma(ss[t], rk1, rs[t]));
  }
  tr = wave_sum_xor(tr);
  for (int off = 32; off > 0; off >>= 1) mn = fmin(mn, __shfl_xor(mn, off));
  __syncthreads();
  if (lane == 0) { red[wv] = tr; red[4 + wv] = mn; }
  __syncthreads();
  tr = (red[0] + red[1]) + (red[2] + red[3]);
  mn = fmin(fmin(red[4], red[5]), fmin(red[6], red[7]));
  if (kind == 0) {
    lo = rs[p - 1];
    hi = (lo + tr * rk1) * (1.0 + 1e-14);
  } else {
    lo = rs[0];
    hi = mn * (1.0 + 1e-14);
  }
  for (int r = 0; r < rounds; ++r) {
    const int* f = flags + (2 * r + kind) * CE_PTS;
    const uint64_t b0 = __ballot(f[lane] != 0), b1 = __ballot(f[lane + 64] != 0);
    const int i = b0 ? __builtin_ctzll(b0) : b1 ? 64 + __builtin_ctzll(b1) : CE_PTS;
    const double a = lo, w = hi - lo;
    if (i > 0) lo = a + w * ((double)i / (CE_PTS + 1));
    if (i < CE_PTS) hi = a + w * ((double)(i + 1) / (CE_PTS + 1));
  }
}

template <int KT>
__global__ __launch_bounds__(256) void k_ce_round(const double* __restrict__ Yf,
                                                  const double* __restrict__ rs,
                                                  const double* __restrict__ ss, int k,
                                                  int64_t p, int64_t nstep, int round, int qcap,
                                                  double* __restrict__ wglobal,
                                                  int* __restrict__ flags) {
  constexpr int NT = KT * (KT + 1) / 2;
  extern __shared__ double sh[];
  __shared__ double red[8];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, i16 = lane & 15, kk = lane >> 4;
  const int kind = blockIdx.x / CE_PTS, pt = blockIdx.x % CE_PTS;
  double lo, hi;
  ce_bracket(kind, round, k, p, rs, ss, flags, red, lo, hi);
  const double x = lo + (hi - lo) * ((double)(pt + 1) / (CE_PTS + 1));
  int* flag = flags + (2 * round + kind) * CE_PTS + pt;
  // rows with r <= x
  int64_t q = 0;
  if (kind == 1) {
    int64_t a = 0, b = p;
    while (a < b) {
      const int64_t m = (a + b) >> 1;
      if (rs[m] <= x) a = m + 1; else b = m;
    }
    q = a;
    if (q > k) {
      if (tid == 0) *flag = 1;
      return;  // block-uniform
    }
  }
  double* M = sh;                                   // lower triangle, packed rows
  const int wld = k | 1;                            // odd stride of the rows of W
  double* W = q <= qcap ? sh + (size_t)k * (k + 1) / 2
                        : wglobal + (size_t)blockIdx.x * k * wld;
  {
    d4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
    for (int64_t st = wv; st < nstep; st += 4) {
      const double r = rs[4 * st + kk];
      // past p: r = +inf, weight 0
      const double w = kind == 0 ? (r < INFINITY ? 1.0 / (x - r) : 0.0)
                                 : (r > x ? 1.0 / (r - x) : 0.0);
      double y[KT];
#pragma unroll
      for (int t = 0; t < KT; ++t) y[t] = Yf[(size_t)(st * KT + t) * 64 + lane];
      int tile = 0;
#pragma unroll
      for (int ta = 0; ta < KT; ++ta) {
        const double aw = w * y[ta];
#pragma unroll
        for (int tb = 0; tb <= ta; ++tb, ++tile)
          acc[tile] = __builtin_amdgcn_mfma_f64_16x16x4f64(aw, y[tb], acc[tile], 0, 0, 0);
      }
    }
    // the four wavefronts' sums, one after the other
    for (int w = 0; w < 4; ++w) {
      if (wv == w) {
        int tile = 0;
#pragma unroll
        for (int ta = 0; ta < KT; ++ta)
#pragma unroll
          for (int tb = 0; tb <= ta; ++tb, ++tile)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int row = 16 * ta + kk + 4 * r, col = 16 * tb + i16;
              if (row < k && col <= row) {
                double* m = M + (size_t)row * (row + 1) / 2 + col;
                const double v = kind == 0 ? -acc[tile][r] : acc[tile][r];
                *m = (w == 0 ? (row == col ? (double)(k - 1) : 0.0) : *m) + v;
              }
            }
      }
      __syncthreads();
    }
  }
  if (kind == 0) {
    const bool spd = block_row_cholesky(k, k, [&](int i) { return M + (size_t)i * (i + 1) / 2; },
                                        [](int) { return 0; });
    if (tid == 0) *flag = spd ? 1 : 0;
    return;
  }
  // rows of Y_-: row t of the sorted order, out of the fragments
  const int nq = (int)q;
  for (int e = tid; e < nq * k; e += 256) {
    const int t = e / k, m = e % k;
    W[t * wld + m] = Yf[((size_t)(t / 4) * KT + m / 16) * 64 + (t % 4) * 16 + m % 16];
  }
  __syncthreads();
  bool below = block_row_cholesky(
      k, k + nq,
      [&](int i) { return i < k ? M + (size_t)i * (i + 1) / 2 : W + (size_t)(i - k) * wld; },
      [](int) { return 0; });
  if (below) {
    // N = W W^T - D in the triangle's place
    for (int e = tid; e < nq * nq; e += 256) {
      const int a = e / nq, b = e % nq;
      if (b > a) continue;
      const double *wa = W + (size_t)a * wld, *wb = W + (size_t)b * wld;
      double s0 = 0.0, s1 = 0.0;
      int m = 0;
      for (; m + 1 < k; m += 2) {
        s0 = fma(wa[m], wb[m], s0);
        s1 = fma(wa[m + 1], wb[m + 1], s1);
      }
      if (m < k) s0 = fma(wa[m], wb[m], s0);
      M[(size_t)a * (a + 1) / 2 + b] = s0 + s1 - (a == b ? x - rs[a] : 0.0);
    }
    __syncthreads();
    below = block_row_cholesky(nq, nq, [&](int i) { return M + (size_t)i * (i + 1) / 2; },
                               [](int) { return 0; });
  }
  if (tid == 0) *flag = below ? 0 : 1;
}

__global__ __launch_bounds__(256) void k_ce_final(const double* __restrict__ rs,
                                                  const double* __restrict__ ss, int k,
                                                  int64_t p, const int* __restrict__ flags,
                                                  double* __restrict__ out) {
  __shared__ double red[8];
  double lo, hi;
  for (int kind = 0; kind < 2; ++kind) {
    ce_bracket(kind, CE_ROUNDS, k, p, rs, ss, flags, red, lo, hi);
    if (threadIdx.x == 0) out[kind] = 0.5 * (lo + hi);
  }
}

void lowrank_spd_extremes(mda_ctx* c, const double* yp, const double* var, const double* hvar,
                          int k, int64_t p, double* out) {
  MDA_REQUIRE(k >= 2 && k <= 128 && p >= 1, "condition number: size out of range");
  hipStream_t s = c->stream;
  std::vector<uint32_t> order(p);
  std::iota(order.begin(), order.end(), 0u);
  std::stable_sort(order.begin(), order.end(),
                   [&](uint32_t a, uint32_t b) { return hvar[a] < hvar[b]; });
  uint32_t* dord = c->get<uint32_t>("ce_order", p);
  h2d(c, dord, order.data(), sizeof(uint32_t) * p);
  const int kt = (k + 15) / 16;
  const int64_t nstep = (p + 3) / 4;
  double* Yf = c->get<double>("ce_rows", (size_t)nstep * kt * 64);
  double* rs = c->get<double>("ce_r", 4 * nstep);
  double* ss = c->get<double>("ce_s", 4 * nstep);
  int* flags = c->get<int>("ce_flags", 2 * CE_PTS * CE_ROUNDS);
  // W in LDS up to qcap rows (144 KB with the triangle; all k rows for
  // k <= 110), else in a global scratch
  const size_t tri = (size_t)k * (k + 1) / 2, wld = k | 1, cap = 18432;
  const int qcap = (int)std::min<size_t>(k, (cap - tri) / wld);
  double* wg = qcap < k ? c->get<double>("ce_w", (size_t)2 * CE_PTS * k * wld) : nullptr;
  const size_t shm = sizeof(double) * (tri + qcap * wld);
  hipLaunchKernelGGL(k_ce_rows, dim3(grid_for(nstep * kt * 64, 256, 4096)), dim3(256), 0, s, yp,
                     var, dord, k, kt, p, nstep, Yf, rs, ss);
  MDA_LAUNCH_CHECK();
  for (int r = 0; r < CE_ROUNDS; ++r) {
#define MDA_CE(KT)                                                                             \
  case KT:                                                                                     \
    hipLaunchKernelGGL(k_ce_round<KT>, dim3(2 * CE_PTS), dim3(256), shm, s, Yf, rs, ss, k, p,  \
                       nstep, r, qcap, wg, flags);                                             \
    break;
    switch (kt) { MDA_CE(1) MDA_CE(2) MDA_CE(3) MDA_CE(4) MDA_CE(5) MDA_CE(6) MDA_CE(7) MDA_CE(8) }
#undef MDA_CE
    MDA_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_ce_final, dim3(1), dim3(256), 0, s, rs, ss, k, p, flags, out);
  MDA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Gauss-Jordan elimination with partial pivoting on [A | B] (A p x p, B p x m,
// both row-major, destroyed): B <- A^-1 B.  Step j: the pivot row is the
// first row r >= j with the largest |A[r][j]| (the choice of partial-pivot
// LU); rows j and r swap; row j is divided by the pivot; every other row r
// takes -A[r][j] times row j (columns > j of A, all of B).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void k_gj_pivot(int64_t p, int64_t j, const double* __restrict__ A,
                                                   int64_t* __restrict__ piv,
                                                   double* __restrict__ pval,
                                                   int* __restrict__ status) {
  __shared__ double bv[1024];
  __shared__ int64_t bi[1024];
  double best = -1.0;
  int64_t bidx = j;
  for (int64_t r = j + threadIdx.x; r < p; r += blockDim.x) {
    const double v = fabs(A[(size_t)r * p + j]);
    if (v > best) { best = v; bidx = r; }
  }
  bv[threadIdx.x] = best;
  bi[threadIdx.x] = bidx;
  __syncthreads();
  for (int s2 = blockDim.x / 2; s2 > 0; s2 >>= 1) {
    if ((int)threadIdx.x < s2) {
      const double v2 = bv[threadIdx.x + s2];
      const int64_t i2 = bi[threadIdx.x + s2];
      if (v2 > bv[threadIdx.x] || (v2 == bv[threadIdx.x] && i2 < bi[threadIdx.x])) {
        bv[threadIdx.x] = v2;
        bi[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    piv[0] = bi[0];
    const double pv = A[(size_t)bi[0] * p + j];
    pval[0] = pv;
    if (!(pv != 0.0) || !isfinite(pv)) atomicOr(status, MDA_ST_NOT_SPD);
  }
}

// swap rows j and piv of [A | B] and divide row j by the pivot (columns >= j
// of A, all of B); one thread per column
__global__ void k_gj_swap_scale(int64_t p, int64_t m, int64_t j, double* __restrict__ A,
                                double* __restrict__ B, const int64_t* __restrict__ piv,
                                const double* __restrict__ pval) {
  const int64_t r = piv[0];
  const double inv = 1.0 / pval[0];
  const int64_t ncols = (p - j) + m;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < ncols;
       t += (int64_t)gridDim.x * blockDim.x) {
    double* M;
    int64_t ld, cidx;
    if (t < p - j) { M = A; ld = p; cidx = j + t; } else { M = B; ld = m; cidx = t - (p - j); }
    double* rowj = M + (size_t)j * ld + cidx;
    double* rowr = M + (size_t)r * ld + cidx;
    const double vj = *rowj, vr = *rowr;
    *rowr = vj;
    *rowj = vr * inv;
  }
}

// row r != j:  X[r][c] -= A[r][j] X[j][c]  for c > j in A and every c of B
// (column j of A itself is left as it is: later steps never read it)
__global__ void k_gj_eliminate(int64_t p, int64_t m, int64_t j, double* __restrict__ A,
                               double* __restrict__ B) {
  const int64_t nca = p - j - 1, ncols = nca + m;
  const int64_t total = p * ncols;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = t / ncols, cc = t % ncols;
    if (r == j) continue;
    const double f = A[(size_t)r * p + j];
    if (cc < nca) {
      const int64_t c = j + 1 + cc;
      A[(size_t)r * p + c] = fma(-f, A[(size_t)j * p + c], A[(size_t)r * p + c]);
    } else {
      const int64_t c = cc - nca;
      B[(size_t)r * m + c] = fma(-f, B[(size_t)j * m + c], B[(size_t)r * m + c]);
    }
  }
}

void dense_gauss_jordan(hipStream_t s, int64_t p, int64_t m, double* A, double* B,
                        int64_t* piv, double* pval, int* status) {
  MDA_REQUIRE(p >= 1 && p <= MDA_DENSE_MAX && m >= 1, "dense solve size out of range");
  for (int64_t j = 0; j < p; ++j) {
    hipLaunchKernelGGL(k_gj_pivot, dim3(1), dim3(1024), 0, s, p, j, A, piv, pval, status);
    MDA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_gj_swap_scale, dim3(grid_for(p - j + m, 256, 1024)), dim3(256), 0, s, p,
                       m, j, A, B, piv, pval);
    MDA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_gj_eliminate, dim3(grid_for(p * (p - j - 1 + m), 256, 8192)), dim3(256),
                       0, s, p, m, j, A, B);
    MDA_LAUNCH_CHECK();
  }
}

}  // namespace mda
