// Device-side helpers: distances, Gaspari-Cohn, and workgroup-cooperative
// dense kernels (Cholesky, SPD inverse, parallel-order Jacobi) that operate on
// matrices in LDS or in global memory through flat pointers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mda {

constexpr double kPi = 3.14159265358979323846;
constexpr double kEarthRadiusKm = 6371.0;

// Location::haversine (Location.hpp:349-357), same formula, constants and
// operation order, with no FMA contraction (the reference's x86-64 build
// rounds every product and sum separately).
__device__ inline double haversine_km(double lat1, double lon1, double lat2, double lon2) {
#pragma clang fp contract(off)
  const double dlat = (lat2 - lat1) * kPi / 180.0;
  const double dlon = (lon2 - lon1) * kPi / 180.0;
  const double s1 = sin(dlat / 2), s2 = sin(dlon / 2);
  const double a = s1 * s1 + cos(lat1 * kPi / 180.0) * cos(lat2 * kPi / 180.0) * s2 * s2;
  const double c = 2 * atan2(sqrt(a), sqrt(1 - a));
  return kEarthRadiusKm * c;
}

// Squared GRID / CARTESIAN distance of Location::distance_to
// (Location.hpp:205-224) in its operation order, (dx dx + dy dy) + dz dz with
// every product rounded (no FMA), so that a distance equal to the radius in
// the reference's arithmetic is equal here too.  dz = 0 for GRID.
__device__ inline double dist2_exact(double dx, double dy, double dz) {
#pragma clang fp contract(off)
  return dx * dx + dy * dy + dz * dz;
}

// Relative half-width of the shell around the GEOGRAPHIC membership
// threshold chord2_r = 4 sin^2(r / 2R) inside which the chord test on unit
// vectors (equal to the haversine test in exact arithmetic) is not trusted:
// |c2 - chord2_r| <= shell_width(chord2_r).  The rounding of c2 (about
// 1.5e-15 |u - v| absolute) is covered 700 times over.
__host__ __device__ inline double shell_width(double chord2_r) {
  return 1e-9 * chord2_r + 1e-12 * sqrt(chord2_r);
}

// Gaspari & Cohn (1999) eq. (4.10) in z = d / c; zero for z >= 2.
__device__ inline double gaspari_cohn(double z) {
  z = fabs(z);
  if (z >= 2.0) return 0.0;
  if (z <= 1.0) return (((-0.25 * z + 0.5) * z + 0.625) * z - 5.0 / 3.0) * z * z + 1.0;
  return ((((z / 12.0 - 0.5) * z + 0.625) * z + 5.0 / 3.0) * z - 5.0) * z + 4.0 -
         2.0 / (3.0 * z);
}

// FP32 form of gaspari_cohn, for weights that feed FP32 / BF16 contractions.
__device__ inline float gaspari_cohn_f32(float z) {
  z = fabsf(z);
  if (z >= 2.f) return 0.f;
  if (z <= 1.f) return (((-0.25f * z + 0.5f) * z + 0.625f) * z - 5.f / 3.f) * z * z + 1.f;
  return ((((z / 12.f - 0.5f) * z + 0.625f) * z + 5.f / 3.f) * z - 5.f) * z + 4.f -
         2.f / (3.f * z);
}

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// FP64 MFMA over state points (v_mfma_f64_16x16x4f64, one wavefront per
// 16 MT points): lane (i16, kk) holds members 4s + kk of point i16 of each
// tile, the layout of either operand (A[l%16][l/16], B[l/16][l%16]).  Member
// loads are 128-byte segments.  An ensemble of k members takes NS = k / 4
// steps, rounded up to a compiled size; the values past k are zero.
// ---------------------------------------------------------------------------
// v[t][s] = (x - mean) scale of the tile's points (0 past n and k); mean[t]
// the mean over the members of point i0 + 16 t + i16
template <int NS, int MT>
__device__ __forceinline__ void load_pert(const double* __restrict__ X, int k, int64_t n,
                                          double scale, int64_t i0, double (&v)[MT][NS],
                                          double (&mean)[MT]) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, kk = lane >> 4;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int64_t i = i0 + 16 * t + i16;
    double sum = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int m = 4 * s + kk;
      v[t][s] = m < k && i < n ? X[(size_t)m * n + i] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) sum += v[t][s];
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    mean[t] = sum * (1.0 / (double)k);
#pragma unroll
    for (int s = 0; s < NS; ++s)
      v[t][s] = 4 * s + kk < k && i < n ? (v[t][s] - mean[t]) * scale : 0.0;
  }
}

// the compiled step counts: k <= 16, 32, ..., 128
#define MDA_MEMBER_STEPS(k, CALL)        \
  switch (((k) + 15) / 16) {             \
    case 1: { CALL(4); } break;          \
    case 2: { CALL(8); } break;          \
    case 3: { CALL(12); } break;         \
    case 4: { CALL(16); } break;         \
    case 5: { CALL(20); } break;         \
    case 6: { CALL(24); } break;         \
    case 7: { CALL(28); } break;         \
    default: { CALL(32); } break;        \
  }

// ---------------------------------------------------------------------------
// workgroup reductions
// ---------------------------------------------------------------------------
__device__ inline double block_sum(double v, double* red) {
  const int tid = threadIdx.x, nt = blockDim.x;
  red[tid] = v;
  __syncthreads();
  for (int s = nt / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  double r = red[0];
  __syncthreads();
  return r;
}

// ---------------------------------------------------------------------------
// Cholesky M = L L^T in place (lower triangle; strict upper set to 0).
// Returns false when a pivot is not positive.  All threads participate.
// ---------------------------------------------------------------------------
__device__ inline bool block_cholesky(double* A, int lda, int n, int* flag) {
  const int tid = threadIdx.x, nt = blockDim.x;
  if (tid == 0) *flag = 0;
  __syncthreads();
  for (int j = 0; j < n; ++j) {
    if (tid == 0) {
      double a = A[j * lda + j];
      if (!(a > 0.0)) *flag = 1;
      A[j * lda + j] = sqrt(a > 0.0 ? a : 1.0);
    }
    __syncthreads();
    double ljj = A[j * lda + j];
    for (int i = j + 1 + tid; i < n; i += nt) A[i * lda + j] /= ljj;
    __syncthreads();
    int m = n - j - 1;
    for (int idx = tid; idx < m * m; idx += nt) {
      int i = j + 1 + idx / m, l = j + 1 + idx % m;
      if (l <= i) A[i * lda + l] -= A[i * lda + j] * A[l * lda + j];
    }
    __syncthreads();
  }
  for (int idx = tid; idx < n * n; idx += nt) {
    int i = idx / n, l = idx % n;
    if (l > i) A[i * lda + l] = 0.0;
  }
  __syncthreads();
  return *flag == 0;
}

// Given L (lower) in A, writes M^-1 = L^-T L^-1 into A, using W as scratch
// for L^-1 (both n x n with their leading dimensions).
__device__ inline void block_spd_inverse_from_chol(double* A, int lda, double* W, int ldw,
                                                   int n) {
  const int tid = threadIdx.x, nt = blockDim.x;
  // column c of L^-1 by forward substitution (one thread per column)
  for (int c = tid; c < n; c += nt) {
    for (int i = 0; i < c; ++i) W[i * ldw + c] = 0.0;
    for (int i = c; i < n; ++i) {
      double s = (i == c) ? 1.0 : 0.0;
      for (int t = c; t < i; ++t) s -= A[i * lda + t] * W[t * ldw + c];
      W[i * ldw + c] = s / A[i * lda + i];
    }
  }
  __syncthreads();
  for (int idx = tid; idx < n * n; idx += nt) {
    int i = idx / n, j = idx % n;
    int t0 = i > j ? i : j;
    double s = 0.0;
    for (int t = t0; t < n; ++t) s += W[t * ldw + i] * W[t * ldw + j];
    A[i * lda + j] = s;
  }
  __syncthreads();
}

// 1 / sqrt(t) for t in the normal range: the hardware estimate (about 2^-24
// relative) refined by one third-order step y (1 + e/2 + 3e^2/8),
// e = 1 - t y^2 (the Taylor series of (1 - e)^(-1/2)), about 1 ulp
__device__ inline double refined_rsqrt(double t) {
  const double y = __builtin_amdgcn_rsq(t);
  const double e = fma(-t * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// ---------------------------------------------------------------------------
// Cholesky of the leading n columns of `rows` >= n rows, one row per thread
// (rows <= blockDim.x), matrix in LDS: row(i)[j] = a_ij becomes
// l_ij = (a_ij - sum_c l_ic l_jc) / l_jj.  Rows i < n hold the columns j <= i;
// rows i >= n hold the columns j >= first(i) (zero before it): b^T becomes
// b^T L^-T.  Four columns at a time: each thread's dot products with the four
// panel rows (one own and four broadcast LDS reads per four FMAs), then every
// thread factors the 4 x 4 block for itself, bound by that chain: its roots and
// quotients are refined reciprocal roots (a chain of some 350 cycles where the
// library's take 1,500; ETKF solve k = 64 74 -> 60 us).  Three barriers per panel;
// false (in every thread) when a pivot is not positive.
// ---------------------------------------------------------------------------
template <class Row, class First>
__device__ inline bool block_row_cholesky(int n, int rows, Row row, First first) {
  const int i = threadIdx.x;
  double* li = row(i < rows ? i : rows - 1);
  const int c0 = i < rows && i >= n ? first(i) : 0;
  for (int j0 = 0; j0 < n; j0 += 4) {
    const int nb = n - j0 < 4 ? n - j0 : 4;
    const double* r0 = row(j0);
    const double* r1 = row(j0 + (nb > 1 ? 1 : 0));
    const double* r2 = row(j0 + (nb > 2 ? 2 : 0));
    const double* r3 = row(j0 + (nb > 3 ? 3 : 0));
    const bool own = i < rows && i >= j0;
    // last panel column this row holds
    const int last = i < n ? (i - j0 < nb - 1 ? i - j0 : nb - 1) : nb - 1;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (own) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (m <= last && j0 + m >= c0) s[m] = li[j0 + m];
#pragma unroll 4
      for (int c = c0; c < j0; ++c) {
        const double v = li[c];
        s[0] = fma(-v, r0[c], s[0]);
        s[1] = fma(-v, r1[c], s[1]);
        s[2] = fma(-v, r2[c], s[2]);
        s[3] = fma(-v, r3[c], s[3]);
      }
    }
    const bool panel = own && i < j0 + nb && i < n;
    __syncthreads();  // the panel rows' entries below j0 + nb have been read
    if (panel) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (m <= last) li[j0 + m] = s[m];
    }
    __syncthreads();
    // L of the 4 x 4 block (rows past nb are not used), d: reciprocals of its
    // diagonal
    const double g00 = r0[j0];
    if (!(g00 > 0.0)) return false;
    const double d0 = refined_rsqrt(g00), l00 = g00 * d0;
    double l10 = 0.0, l11 = 1.0, l20 = 0.0, l21 = 0.0, l22 = 1.0, l30 = 0.0, l31 = 0.0, l32 = 0.0,
           l33 = 1.0, d1 = 1.0, d2 = 1.0, d3 = 1.0;
    if (nb > 1) {
      l10 = r1[j0] * d0;
      const double g = fma(-l10, l10, r1[j0 + 1]);
      if (!(g > 0.0)) return false;
      d1 = refined_rsqrt(g);
      l11 = g * d1;
    }
    if (nb > 2) {
      l20 = r2[j0] * d0;
      l21 = fma(-l20, l10, r2[j0 + 1]) * d1;
      const double g = fma(-l21, l21, fma(-l20, l20, r2[j0 + 2]));
      if (!(g > 0.0)) return false;
      d2 = refined_rsqrt(g);
      l22 = g * d2;
    }
    if (nb > 3) {
      l30 = r3[j0] * d0;
      l31 = fma(-l30, l10, r3[j0 + 1]) * d1;
      l32 = fma(-l31, l21, fma(-l30, l20, r3[j0 + 2])) * d2;
      const double g = fma(-l32, l32, fma(-l31, l31, fma(-l30, l30, r3[j0 + 3])));
      if (!(g > 0.0)) return false;
      d3 = refined_rsqrt(g);
      l33 = g * d3;
    }
    __syncthreads();  // the block has been read
    if (own) {
      double x[4];
      x[0] = s[0] * d0;
      x[1] = fma(-x[0], l10, s[1]) * d1;
      x[2] = fma(-x[1], l21, fma(-x[0], l20, s[2])) * d2;
      x[3] = fma(-x[2], l32, fma(-x[1], l31, fma(-x[0], l30, s[3]))) * d3;
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (m <= last && j0 + m >= c0) li[j0 + m] = x[m];
      if (panel)  // the diagonal entry
        li[i] = i == j0 ? l00 : i == j0 + 1 ? l11 : i == j0 + 2 ? l22 : l33;
    }
    __syncthreads();
  }
  return true;
}

// ---------------------------------------------------------------------------
// Parallel-order cyclic Jacobi (round-robin "circle" ordering: n-1 rounds of
// n/2 disjoint rotations per sweep).  A (n x n symmetric, n even) is
// diagonalised in place; V (may be null) accumulates the rotations so that
// A_in = V diag(A) V^T.  Rotation: symmetric Schur decomposition (Golub & Van
// Loan, sec. 8.5).  Scratch: rc, rs [n/2] doubles, rp, rq [n/2] ints, red
// [blockDim] doubles.  Returns the number of sweeps.
// ---------------------------------------------------------------------------
__device__ inline int rr_player(int pos, int r, int n) {
  return pos == 0 ? 0 : 1 + (pos - 1 + r) % (n - 1);
}

__device__ inline int block_jacobi(double* A, int lda, double* V, int ldv, int n, double* rc,
                                   double* rs, int* rp, int* rq, double* red, int max_sweeps,
                                   double tol) {
  const int tid = threadIdx.x, nt = blockDim.x, h = n / 2;
  if (V)
    for (int idx = tid; idx < n * n; idx += nt) {
      int i = idx / n, j = idx % n;
      V[i * ldv + j] = (i == j) ? 1.0 : 0.0;
    }
  __syncthreads();
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int idx = tid; idx < n * n; idx += nt) {
      int i = idx / n, j = idx % n;
      double v = A[i * lda + j];
      tot += v * v;
      if (i != j) off += v * v;
    }
    off = block_sum(off, red);
    tot = block_sum(tot, red);
    if (off <= tol * tol * tot) break;
    for (int r = 0; r < n - 1; ++r) {
      for (int m = tid; m < h; m += nt) {
        int p = rr_player(m, r, n), q = rr_player(n - 1 - m, r, n);
        if (p > q) { int t = p; p = q; q = t; }
        double apq = A[p * lda + q], c = 1.0, s = 0.0;
        if (apq != 0.0) {
          double app = A[p * lda + p], aqq = A[q * lda + q];
          double theta = (aqq - app) / (2.0 * apq);
          double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(1.0 + theta * theta));
          c = 1.0 / sqrt(1.0 + t * t);
          s = t * c;
        }
        rc[m] = c; rs[m] = s; rp[m] = p; rq[m] = q;
      }
      __syncthreads();
      for (int blk = tid; blk < h * h; blk += nt) {
        int m1 = blk / h, m2 = blk % h;
        int p1 = rp[m1], q1 = rq[m1], p2 = rp[m2], q2 = rq[m2];
        double c1 = rc[m1], s1 = rs[m1], c2 = rc[m2], s2 = rs[m2];
        double a = A[p1 * lda + p2], b = A[p1 * lda + q2];
        double cc = A[q1 * lda + p2], d = A[q1 * lda + q2];
        double a2 = c2 * a - s2 * b, b2 = s2 * a + c2 * b;    // B J2
        double c3 = c2 * cc - s2 * d, d2 = s2 * cc + c2 * d;
        double na = c1 * a2 - s1 * c3, nc = s1 * a2 + c1 * c3;  // J1^T (B J2)
        double nb = c1 * b2 - s1 * d2, nd = s1 * b2 + c1 * d2;
        if (m1 == m2) { nb = 0.0; nc = 0.0; }
        A[p1 * lda + p2] = na; A[p1 * lda + q2] = nb;
        A[q1 * lda + p2] = nc; A[q1 * lda + q2] = nd;
      }
      if (V)
        for (int idx = tid; idx < n * h; idx += nt) {
          int m = idx / n, row = idx % n;
          int p = rp[m], q = rq[m];
          double c = rc[m], s = rs[m];
          double vp = V[row * ldv + p], vq = V[row * ldv + q];
          V[row * ldv + p] = c * vp - s * vq;
          V[row * ldv + q] = s * vp + c * vq;
        }
      __syncthreads();
    }
  }
  return sweep;
}

// Sturm counts: cnt[m] = number of eigenvalues below x[m] of the symmetric
// tridiagonal with rows de[i] = (d_i, e_{i-1}^2), as the sign changes of the leading
// minors of T - x I by their three-term recurrence: one multiply-add deep and five
// instructions per row, where the pivots' quotients (a reciprocal and its
// refinement) are ten deep.  Requires T scaled to largest entry of about 1 (sturm_row);
// n a multiple of 8, filled up with rows (2, 0), which change no sign.  The pair of
// minors is brought to unit size every 4 rows; e^2 is at least 1e-70, so a zero
// minor is followed by a nonzero one of the sign opposite to the one before it, and
// the two steps count one change whatever sign the zero has.
__device__ inline d2 sturm_row(double d, double e) { return d2{d, fmax(e * e, 1e-70)}; }

template <int M>
__device__ inline void sturm_counts(const d2* de, int n, const double (&x)[M], int (&cnt)[M]) {
  double m0[M], m1[M];  // the last two minors
#pragma unroll
  for (int t = 0; t < M; ++t) {
    m0[t] = 0.0;  // what row 0's e^2 multiplies
    m1[t] = 1.0;
    cnt[t] = 0;
  }
  for (int i0 = 0; i0 < n; i0 += 8) {
    unsigned bits[M];
    d2 r[8];
#pragma unroll
    for (int t = 0; t < M; ++t) bits[t] = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) r[q] = de[i0 + q];
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int t = 0; t < M; ++t) {
        const double m = fma(r[q][0] - x[t], m1[t], -r[q][1] * m0[t]);
        bits[t] = __builtin_amdgcn_alignbit(
            bits[t], (unsigned)(__double2hiint(m) ^ __double2hiint(m1[t])), 31);
        m0[t] = m1[t];
        m1[t] = m;
        if (q == 3 || q == 7) {
          const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(m0[t]), fabs(m1[t])));
          m0[t] = __builtin_amdgcn_ldexp(m0[t], ex);
          m1[t] = __builtin_amdgcn_ldexp(m1[t], ex);
        }
      }
#pragma unroll
    for (int t = 0; t < M; ++t) cnt[t] += __popc(bits[t]);
  }
}

}  // namespace mda
