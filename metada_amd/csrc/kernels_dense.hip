// Dense p x p linear algebra of the global filters, kept in device memory:
//   - the EnKF's S = Y'Y'^T/(k-1) + R and its condition number
//     (EnKF.hpp:188-209: JacobiSVD singular values), from the k x k side
//     when p > 128,
//   - Householder tridiagonalisation of a symmetric matrix, whose extreme
//     eigenvalues (and the one nearest zero) are then found by multisection on
//     Sturm counts of the tridiagonal,
//   - Gauss-Jordan elimination with partial pivoting, A^-1 B for p x m B (the
//     S^-1 products of EnKF.hpp:199 and LWEnKF.hpp:273-276).
// Each step is one or two launches over the trailing matrix: O(p^3) work, as
// the reference's own dense algebra.  Sizes are bounded by MDA_DENSE_MAX.
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

// Lane shifts in the vector unit (DPP), a few cycles each where a shuffle
// through LDS takes over a hundred; lanes without a source, and rows outside
// ROWS, take `none`.
template <int CTRL, int ROWS = 0xf>
__device__ inline double dpp(double v, double none) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(none), __double2loint(v), CTRL, ROWS,
                                             0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(none), __double2hiint(v), CTRL, ROWS,
                                             0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ inline double read_lane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// row_shr 1, 2, 4, 8: lane 15 of a row of 16 holds the row's result; row_bcast
// 15 and 31 carry it on, lane 63 holds the wavefront's
__device__ inline double wave_sum(double v) {
  v += dpp<0x111>(v, 0.0);
  v += dpp<0x112>(v, 0.0);
  v += dpp<0x114>(v, 0.0);
  v += dpp<0x118>(v, 0.0);
  v += dpp<0x142, 0xa>(v, 0.0);
  v += dpp<0x143, 0xc>(v, 0.0);
  return read_lane(v, 63);
}

__device__ inline double row_max(double v) {  // in lane 15 of each row
  v = fmax(v, dpp<0x111>(v, v));
  v = fmax(v, dpp<0x112>(v, v));
  v = fmax(v, dpp<0x114>(v, v));
  return fmax(v, dpp<0x118>(v, v));
}

__device__ inline double wave_max(double v) {
  v = row_max(v);
  v = fmax(v, dpp<0x142>(v, v));
  v = fmax(v, dpp<0x143>(v, v));
  return read_lane(v, 63);
}

// sum over the block's wavefronts (at most 16), in every thread
__device__ inline double block_wave_sum(double v, double* red) {
  v = wave_sum(v);
  const int nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}

// ---------------------------------------------------------------------------
// Householder tridiagonalisation, step j (m = p - j - 1 trailing rows):
//   x = A[j+1:, j], alpha = -sign(x_0) ||x||, u = x - alpha e_1,
//   tau = 2 / u^T u, pv = tau A' u, w = pv - (tau/2)(pv^T u) u,
//   A' <- A' - u w^T - w u^T;  d_j = A[j][j], e_j = alpha.
// One launch per step.  A step's rank-2 update is applied by the next step's
// launch: every block forms w of the step before and the new column j (row j,
// which no block writes) for itself, O(p) work, and then takes its rows, each
// updated, stored and multiplied by the new u in the same pass.  The vectors
// of successive steps alternate between two buffers.  Bound by the latency of a
// launch and its dependent reads up to p of about 1,000 (p = 512: 2.7 ms, 5.3 us
// a step; 7.1 ms with four launches a step) and by the one read and write of the
// trailing matrix beyond.
// ---------------------------------------------------------------------------
struct hh_vectors {  // of one step: u [p], pv [p], tau
  double *u, *pv, *tau;
};

constexpr int HH_PF = 8;

__global__ __launch_bounds__(256) void k_hh_step(int p, int j, double* __restrict__ A,
                                                 hh_vectors prev, hh_vectors next,
                                                 double* __restrict__ d, double* __restrict__ e) {
  extern __shared__ double sh[];  // u and w of the step before, u of this one
  __shared__ double red[4];
  double *up = sh, *wp = sh + p, *un = sh + 2 * p;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  // the first HH_PF entries a lane takes of its wavefront's first row, on
  // their way while the vectors are formed
  const int r0 = j + 1 + blockIdx.x * 4 + wv;
  double pf[HH_PF];
#pragma unroll
  for (int q = 0; q < HH_PF; ++q) {
    const int c = j + 1 + lane + 64 * q;
    pf[q] = r0 < p && c < p ? A[(size_t)r0 * p + c] : 0.0;
  }
  double part = 0.0;
  for (int c = j + tid; c < p; c += 256) {
    const double a = j > 0 ? prev.u[c] : 0.0, b = j > 0 ? prev.pv[c] : 0.0;
    up[c] = a;
    wp[c] = b;
    un[c] = A[(size_t)j * p + c];
    part = fma(a, b, part);
  }
  const double K = j > 0 ? 0.5 * *prev.tau * block_wave_sum(part, red) : 0.0;
  for (int c = j + tid; c < p; c += 256) wp[c] -= K * up[c];
  __syncthreads();
  const double upj = up[j], wpj = wp[j];
  double s2 = 0.0;
  for (int c = j + tid; c < p; c += 256) {
    const double x = fma(-upj, wp[c], fma(-wpj, up[c], un[c]));
    un[c] = x;
    if (c > j) s2 = fma(x, x, s2);
  }
  const double nrm2 = block_wave_sum(s2, red);  // its barriers order un
  const double x0 = un[j + 1], dj = un[j];
  const bool nz = nrm2 > 0.0;
  const double alpha = nz ? (x0 > 0.0 ? -1.0 : 1.0) * sqrt(nrm2) : 0.0;
  const double tau = nz ? 2.0 / (nrm2 - 2.0 * alpha * x0 + alpha * alpha) : 0.0;
  __syncthreads();  // every thread has read x0
  for (int c = j + tid; c < p; c += 256) {
    const double v = c == j || !nz ? 0.0 : un[c] - (c == j + 1 ? alpha : 0.0);
    un[c] = v;
    if (blockIdx.x == 0) next.u[c] = v;
  }
  if (blockIdx.x == 0 && tid == 0) {
    d[j] = dj;
    e[j] = alpha;
    *next.tau = tau;
  }
  __syncthreads();
  for (int r = r0; r < p; r += gridDim.x * 4) {
    const double ur = up[r], wr = wp[r];
    double* row = A + (size_t)r * p;
    double acc = 0.0;
    int c = j + 1 + lane;
    if (r == r0) {
#pragma unroll
      for (int q = 0; q < HH_PF; ++q, c += 64)
        if (c < p) {
          const double a = fma(-ur, wp[c], fma(-wr, up[c], pf[q]));
          row[c] = a;
          acc = fma(a, un[c], acc);
        }
    }
#pragma unroll 4
    for (; c < p; c += 64) {
      const double a = fma(-ur, wp[c], fma(-wr, up[c], row[c]));
      row[c] = a;
      acc = fma(a, un[c], acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) next.pv[r] = tau * acc;
  }
}

// last 2 x 2 block, with the last step's update still to apply
__global__ void k_hh_tail(int p, const double* __restrict__ A, hh_vectors prev,
                          double* __restrict__ d, double* __restrict__ e) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const int a = p - 2, b = p - 1;
  const double ua = prev.u[a], ub = prev.u[b];
  const double K = 0.5 * *prev.tau * fma(prev.pv[a], ua, prev.pv[b] * ub);
  const double wa = prev.pv[a] - K * ua, wb = prev.pv[b] - K * ub;
  d[a] = fma(-ua, wa, fma(-wa, ua, A[(size_t)a * p + a]));
  e[a] = fma(-ub, wa, fma(-wb, ua, A[(size_t)b * p + a]));
  d[b] = fma(-ub, wb, fma(-wb, ub, A[(size_t)b * p + b]));
  e[b] = 0.0;
}

// p >= 3; work: 4 p + 2 doubles
static void dense_tridiagonalise(hipStream_t s, int p, double* A, double* d, double* e,
                                 double* work) {
  MDA_REQUIRE(p >= 3 && p <= MDA_DENSE_MAX, "dense matrix size out of range");
  hh_vectors v[2];
  for (int i = 0; i < 2; ++i)
    v[i] = {work + (size_t)i * 2 * p, work + (size_t)i * 2 * p + p, work + (size_t)4 * p + i};
  for (int j = 0; j + 2 < p; ++j) {
    hipLaunchKernelGGL(k_hh_step, dim3(grid_for(p - j - 1, 4, 1024)), dim3(256),
                       sizeof(double) * 3 * p, s, p, j, A, v[(j + 1) & 1], v[j & 1], d, e);
    MDA_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_hh_tail, dim3(1), dim3(64), 0, s, p, A, v[(p - 3) & 1], d, e);
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
    const double nrm2 = wave_sum(fma(x0, x0, x1 * x1));
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
    const double K = 0.5 * tau * wave_sum(fma(p0, u0, p1 * u1));
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
// multisection on Sturm counts, 128 points a round for each of the smallest,
// the largest, the largest negative and the smallest non-negative eigenvalue.
// out = [lmin, lmax, |l|min, |l|max].  Bound by the chain of the counts, n = 512:
// 0.16 ms (0.5 ms with the counts by quotients).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void k_tridiag_extremes(const double* __restrict__ dg,
                                                          const double* __restrict__ eg, int n,
                                                          double* __restrict__ out) {
  extern __shared__ d2 de[];
  __shared__ double red[2][8], slo[4], shi[4];
  __shared__ uint64_t bal[8];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double lo = INFINITY, hi = -INFINITY;
  for (int i = tid; i < n; i += 512) {
    const double di = dg[i], ei = i + 1 < n ? fabs(eg[i]) : 0.0;
    const double r = (i > 0 ? fabs(eg[i - 1]) : 0.0) + ei;
    lo = fmin(lo, di - r);
    hi = fmax(hi, di + r);
  }
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off));
    hi = fmax(hi, __shfl_xor(hi, off));
  }
  if (lane == 0) { red[0][wv] = lo; red[1][wv] = hi; }
  __syncthreads();
  for (int w = 0; w < 8; ++w) {
    lo = fmin(lo, red[0][w]);
    hi = fmax(hi, red[1][w]);
  }
  const double span = fmax(fabs(lo), fabs(hi));
  const int sc = span > 0.0 && isfinite(span) ? -ilogb(span) - 1 : 0;
  for (int i = tid; i < (n + 7) / 8 * 8; i += 512) {
    const double ei = i > 0 && i < n ? ldexp(eg[i - 1], sc) : 0.0;
    de[i] = i < n ? sturm_row(ldexp(dg[i], sc), ei) : d2{2.0, 0.0};
  }
  __syncthreads();
  lo = ldexp(lo, sc) - 1e-14;
  hi = ldexp(hi, sc) + 1e-14;
  const int n8 = (n + 7) / 8 * 8;
  const double zero[1] = {0.0};
  int neg1[1];
  sturm_counts(de, n8, zero, neg1);
  const int neg = neg1[0];
  const int tg = tid >> 7, t = tid & 127;
  const int idx = tg == 0 ? 0 : tg == 1 ? n - 1 : tg == 2 ? neg - 1 : neg;
  if (t == 0) {
    slo[tg] = tg == 3 ? 0.0 : lo;
    shi[tg] = tg == 2 ? 0.0 : hi;
  }
  __syncthreads();
  for (int round = 0; round < 10; ++round) {
    const double a = slo[tg], b = shi[tg], w = b - a;
    const double x[1] = {a + w * ((double)(t + 1) / 129.0)};
    int cnt[1];
    sturm_counts(de, n8, x, cnt);
    const uint64_t above = __ballot(idx >= 0 && idx < n && cnt[0] > idx);
    if (lane == 0) bal[wv] = above;
    __syncthreads();
    if (t == 0) {  // f: first point above the eigenvalue
      const uint64_t b0 = bal[2 * tg], b1 = bal[2 * tg + 1];
      const int f = b0 ? __ffsll((long long)b0) - 1 : b1 ? 64 + __ffsll((long long)b1) - 1 : 128;
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
    out[0] = ldexp(l0, -sc);
    out[1] = ldexp(l1, -sc);
    out[2] = ldexp(am, -sc);
    out[3] = ldexp(fmax(fabs(l0), fabs(l1)), -sc);
  }
}

void dense_sym_extremes(mda_ctx* c, hipStream_t s, double* A, int64_t p, int64_t lda,
                        double* out) {
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
    dense_tridiagonalise(s, (int)p, A, d, e, c->get<double>("dense_hh", 4 * p + 2));
  }
  hipLaunchKernelGGL(k_tridiag_extremes, dim3(1), dim3(512), sizeof(double) * 2 * (p + 7), s, d, e,
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
// took 33 ms with four launches per column, this 1.8 ms, on the second stream
// beside the gain.
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
  tr = wave_sum(tr);
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
    // one step's rows ahead of the products, where the registers hold them
    constexpr bool AHEAD = KT < 8;
    double nr = INFINITY, ny[KT];
    auto load = [&](int64_t st) {
      if (st >= nstep) return;
      nr = rs[4 * st + kk];
#pragma unroll
      for (int t = 0; t < KT; ++t) ny[t] = Yf[(size_t)(st * KT + t) * 64 + lane];
    };
    if (AHEAD) load(wv);
    for (int64_t st = wv; st < nstep; st += 4) {
      if (!AHEAD) load(st);
      const double r = nr;
      double y[KT];
#pragma unroll
      for (int t = 0; t < KT; ++t) y[t] = ny[t];
      if (AHEAD) load(st + 4);
      // past p: r = +inf, weight 0
      const double w = kind == 0 ? (r < INFINITY ? 1.0 / (x - r) : 0.0)
                                 : (r > x ? 1.0 / (r - x) : 0.0);
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

void lowrank_spd_extremes(mda_ctx* c, side_branch& br, const double* yp, const double* var,
                          const double* hvar, int k, int64_t p, double* out) {
  MDA_REQUIRE(k >= 2 && k <= 128 && p >= 1, "condition number: size out of range");
  std::vector<uint32_t> order(p);
  std::iota(order.begin(), order.end(), 0u);
  std::stable_sort(order.begin(), order.end(),
                   [&](uint32_t a, uint32_t b) { return hvar[a] < hvar[b]; });
  uint32_t* dord = c->get<uint32_t>("ce_order", p);
  h2d(c, dord, order.data(), sizeof(uint32_t) * p);
  hipStream_t s = br.fork();
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
// both row-major, destroyed): B <- A^-1 B, in blocks of GJ_NB columns, two
// launches each.
//   panel   one workgroup, rows in registers (a thread owns positions tid,
//           tid + NT, ...): LU with partial pivoting of the block's columns over
//           the rows >= j0, the pivot of a column being the first row with the
//           largest entry (entries within 2^-40 of each other count as equal: no
//           multiplier exceeds 1 by more); an entry that is no finite number makes
//           S singular.  With A11 = L11 U11 the pivot rows and l_r the
//           multipliers of any other row, W[r] = -l_r L11^-1, and W[j0 + t] =
//           row t of A11^-1.
//   strips  a workgroup per 32 columns right of the block or of B: the row
//           exchanges, then every row r <- (r not a pivot row ? row r : 0) +
//           W[r] (old pivot rows) on FP64 MFMA.
// Bound by the panel's chain of pivots (p = 512, m = 64: 33 us a panel, 11 us a
// strip launch, 1.4 ms in all; 5.1 ms column by column, three launches each).
// ---------------------------------------------------------------------------
constexpr int GJ_NB = 16, GJ_W = 32;

struct gj_moves {      // of one block, applied to the columns outside it
  int pivot[GJ_NB];    // row that becomes row j0 + t
  int ndisp;           // rows displaced by them: to[i] receives row from[i]
  int to[GJ_NB], from[GJ_NB];
};

template <int NT, int R, int NB>
__global__ __launch_bounds__(NT) void k_gj_panel(int p, int j0, int nb, const double* __restrict__ A,
                                                 double* __restrict__ W,
                                                 gj_moves* __restrict__ moves,
                                                 int* __restrict__ status) {
  constexpr int NW = NT / 64;
  // of a step, by its parity: each wavefront's candidate (value and row index
  // in one key, its row, its row without the multipliers) and the row that the
  // pivot row changes places with
  __shared__ double key[2][NW], cand[2][NW][2][NB], xrow[2][NB], LU[NB][NB + 1];
  __shared__ int piv[NB];
  __shared__ gj_moves mv;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double a[R][NB];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int r = tid + NT * i;
#pragma unroll
    for (int c = 0; c < NB; ++c) a[i][c] = r < p && c < nb ? A[(size_t)r * p + j0 + c] : 0.0;
  }
  // Every step ends by rotating the rows one column to the left, so that the
  // step's column is a[.][0], the loop stays rolled and the columns are in order
  // again after NB steps.
#pragma unroll 1
  for (int t = 0; t < NB; ++t) {
    if (t < nb) {
      // key: |value| with its last 12 bits replaced by 4095 - row, so that the
      // first of the largest wins
      const int par = t & 1;
      double kv = -1.0;
      bool bad = false;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int r = tid + NT * i;
        const double v = fabs(a[i][0]);
        if (r >= j0 + t && r < p) {
          if (v < INFINITY)
            kv = fmax(kv, __hiloint2double(__double2hiint(v),
                                           (__double2loint(v) & ~4095) | (4095 - r)));
          else
            bad = true;
        }
      }
      if (bad) atomicOr(status, MDA_ST_NOT_SPD);
      kv = wave_max(kv);
      const int rw = kv >= 0.0 ? 4095 - (__double2loint(kv) & 4095) : -1;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int r = tid + NT * i;
        if (r == rw) {
#pragma unroll
          for (int c = 0; c < NB; ++c) {
            cand[par][wv][0][c] = a[i][c];
            cand[par][wv][1][c] = c + t < NB ? a[i][c] : 0.0;
          }
        }
        if (r == j0 + t) {
#pragma unroll
          for (int c = 0; c < NB; ++c) xrow[par][c] = a[i][c];
        }
      }
      if (lane == 0) key[par][wv] = kv;
      __syncthreads();
      const double best = read_lane(row_max(key[par][lane % NW]), 15);
      // no finite entry: no exchange, and no finite pivot
      const int bi = best >= 0.0 ? 4095 - (__double2loint(best) & 4095) : j0 + t;
      const int bw = (bi % NT) >> 6;
      const double(&prow)[NB] = cand[par][bw][0];
      const double(&urow)[NB] = cand[par][bw][1];
      const double pvt = best >= 0.0 ? prow[0] : __builtin_nan("");
      if (tid == 0) {
        piv[t] = bi;
        if (!(pvt != 0.0) || !isfinite(pvt)) atomicOr(status, MDA_ST_NOT_SPD);
      }
      const double inv = 1.0 / pvt;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int r = tid + NT * i;
        if (r == j0 + t) {
#pragma unroll
          for (int c = 0; c < NB; ++c) a[i][c] = prow[c];
        } else {
          if (r == bi) {
#pragma unroll
            for (int c = 0; c < NB; ++c) a[i][c] = xrow[par][c];
          }
          if (r < j0 || r > j0 + t) {  // not a pivot row
            const double l = a[i][0] * inv;
            a[i][0] = l;
#pragma unroll
            for (int c = 1; c < NB; ++c) a[i][c] = fma(-l, urow[c], a[i][c]);
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const double a0 = a[i][0];
#pragma unroll
      for (int c = 1; c < NB; ++c) a[i][c - 1] = a[i][c];
      a[i][NB - 1] = a0;
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int r = tid + NT * i;
    if (r >= j0 && r < j0 + nb) {
#pragma unroll
      for (int c = 0; c < NB; ++c) LU[r - j0][c] = a[i][c];
    }
  }
  __syncthreads();  // piv
  if (tid == NT - 1) {
    // the exchanges j0 + t <-> piv[t], one after the other, as moves of rows:
    // row content of the block's positions, and of the positions below it
    int n = 0;
    for (int t = 0; t < nb; ++t) mv.pivot[t] = j0 + t;
    for (int t = 0; t < nb; ++t) {
      const int q = piv[t];
      if (q == j0 + t) continue;
      const int mine = mv.pivot[t];
      if (q < j0 + nb) {
        mv.pivot[t] = mv.pivot[q - j0];
        mv.pivot[q - j0] = mine;
        continue;
      }
      int at = 0;
      while (at < n && mv.to[at] != q) ++at;
      mv.pivot[t] = at < n ? mv.from[at] : q;
      mv.to[at] = q;
      mv.from[at] = mine;
      if (at == n) ++n;
    }
    mv.ndisp = n;
  }
  __syncthreads();
  if (tid < nb) moves->pivot[tid] = mv.pivot[tid];
  if (tid < mv.ndisp) {
    moves->to[tid] = mv.to[tid];
    moves->from[tid] = mv.from[tid];
  }
  if (tid == 0) moves->ndisp = mv.ndisp;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int r = tid + NT * i;
    if (r >= p) continue;
    const bool pr = r >= j0 && r < j0 + nb;
    if (pr) {  // y U = e_t
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        double y = r - j0 == c ? 1.0 : 0.0;
        if (c < nb) {
#pragma unroll
          for (int q = 0; q < c; ++q) y = fma(-a[i][q], LU[q][c], y);
          y /= LU[c][c];
        }
        a[i][c] = c < nb ? y : 0.0;
      }
    }
    // x L = l_r (or y), unit lower L
#pragma unroll
    for (int c = NB - 1; c >= 0; --c) {
      if (c < nb) {
        double x = a[i][c];
#pragma unroll
        for (int q = c + 1; q < NB; ++q)
          if (q < nb) x = fma(-a[i][q], LU[q][c], x);
        a[i][c] = x;
      }
    }
#pragma unroll
    for (int c = 0; c < GJ_NB; ++c) {
      const double x = c < NB && c < nb ? a[i][c < NB ? c : 0] : 0.0;
      W[(size_t)r * GJ_NB + c] = pr ? x : -x;
    }
  }
}

__global__ __launch_bounds__(512) void k_gj_strip(int p, int m, int j0, int nb,
                                                  double* __restrict__ A, double* __restrict__ B,
                                                  const double* __restrict__ W,
                                                  const gj_moves* __restrict__ moves, int na) {
  __shared__ double rows[GJ_NB][GJ_W + 2], disp[GJ_NB][GJ_W + 2];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, i16 = lane & 15, kk = lane >> 4;
  // strip of A's columns right of the block, or of B
  const bool in_a = (int)blockIdx.x < na;
  double* M = in_a ? A : B;
  const int ld = in_a ? p : m;
  const int c0 = in_a ? j0 + nb + GJ_W * blockIdx.x : GJ_W * ((int)blockIdx.x - na);
  const int nc = ld - c0 < GJ_W ? ld - c0 : GJ_W;
  const int nd = moves->ndisp;
  {
    const int t = tid / GJ_W, c = tid % GJ_W;  // 16 rows of 32 columns
    rows[t][c] = t < nb && c < nc ? M[(size_t)moves->pivot[t] * ld + c0 + c] : 0.0;
    disp[t][c] = t < nd && c < nc ? M[(size_t)moves->from[t] * ld + c0 + c] : 0.0;
    __syncthreads();
    if (t < nd && c < nc) M[(size_t)moves->to[t] * ld + c0 + c] = disp[t][c];
    __syncthreads();
  }
  for (int r0 = 16 * wv; r0 < p; r0 += 16 * 8) {
    double w[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      w[s] = r0 + i16 < p ? W[(size_t)(r0 + i16) * GJ_NB + 4 * s + kk] : 0.0;
#pragma unroll
    for (int u = 0; u < GJ_W / 16; ++u) {
      const int c = 16 * u + i16;
      d4 acc;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = r0 + kk + 4 * q;
        acc[q] = r < p && c < nc && (r < j0 || r >= j0 + nb) ? M[(size_t)r * ld + c0 + c] : 0.0;
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(w[s], rows[4 * s + kk][c], acc, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = r0 + kk + 4 * q;
        if (r < p && c < nc) M[(size_t)r * ld + c0 + c] = acc[q];
      }
    }
  }
}

size_t dense_gauss_jordan_work(int64_t p) {
  return (size_t)p * GJ_NB + (sizeof(gj_moves) + 7) / 8;
}

void dense_gauss_jordan(hipStream_t s, int64_t p, int64_t m, double* A, double* B, double* work,
                        int* status) {
  MDA_REQUIRE(p >= 1 && p <= MDA_DENSE_MAX && m >= 1, "dense solve size out of range");
  const int n = (int)p;
  double* W = work;
  gj_moves* mv = reinterpret_cast<gj_moves*>(work + (size_t)p * GJ_NB);
  // blocks of 16 columns while a thread holds one row, of 8 beyond (more
  // exceeds the registers of 1024 threads)
  const int nbmax = p <= 1024 ? 16 : 8;
  for (int j0 = 0; j0 < n; j0 += nbmax) {
    const int nb = n - j0 < nbmax ? n - j0 : nbmax;
#define MDA_GJ(NT, R, NB) \
  hipLaunchKernelGGL((k_gj_panel<NT, R, NB>), dim3(1), dim3(NT), 0, s, n, j0, nb, A, W, mv, status)
    if (p <= 256) MDA_GJ(256, 1, 16);
    else if (p <= 512) MDA_GJ(512, 1, 16);
    else if (p <= 1024) MDA_GJ(1024, 1, 16);
    else if (p <= 2048) MDA_GJ(1024, 2, 8);
    else MDA_GJ(1024, 4, 8);
#undef MDA_GJ
    MDA_LAUNCH_CHECK();
    const int na = (n - j0 - nb + GJ_W - 1) / GJ_W, nbs = ((int)m + GJ_W - 1) / GJ_W;
    hipLaunchKernelGGL(k_gj_strip, dim3(na + nbs), dim3(512), 0, s, n, (int)m, j0, nb, A, B, W, mv,
                       na);
    MDA_LAUNCH_CHECK();
  }
}

}  // namespace mda
