// Local weighted EnKF (LWEnKF.hpp:207-334, 413-668): member weights, a
// weighted observation-space covariance tapered by the index-distance
// localisation, the gain K = X'_rho Y'^T S^-1 / (k-1) tapered again
// element-wise, and the perturbed-observation update of every member.
//
//   S(a, b)  = L_o(a, b) * sum_i (w_i y'_ai) y'_bi + [a == b] r_a
//              L_o(a, b) = f(|a - b| / p / radius)                (:554-575)
//   K(s, b)  = L_g(s, b) * (sum_i X'_rho(s, i) G(b, i)) / (k - 1),
//              G = S^-T Y' (p x k), L_g(s, b) = f(|s - b| / max(n, p) / radius)
//   x_i^a    = xbar + (X'_rho(:, i) + K D(:, i)),
//              D(b, i) = (yo_b + sqrt(r_b) Z_bi) - Yb_bi              (:286-301)
//
// f is the reference's localisation function (:600-636): gaussian
// exp(-nd^2 / 2), exponential exp(-nd), cutoff [nd <= 1], or its
// "gaspari_cohn" polynomial -- which is not Gaspari & Cohn's function (4 at
// 0, -0.125 just below 1, a jump to 0.125, 1.0 just below 2) -- or, on
// request, Gaspari & Cohn (1999) eq. (4.10).  The taper and the weighted
// covariance are evaluated without FMA contraction in the reference's
// operation order, so S matches the reference's to the last bit up to exp().
#include <algorithm>

#include "mda_device.hpp"
#include "mda_internal.hpp"

namespace mda {

__device__ inline double lw_taper(double dist, double radius, int fn, int gc_form) {
#pragma clang fp contract(off)
  const double nd = dist / radius;
  switch (fn) {
    case MDA_LW_LOC_EXPONENTIAL:
      return exp(-nd);
    case MDA_LW_LOC_CUTOFF:
      return nd <= 1.0 ? 1.0 : 0.0;
    case MDA_LW_LOC_GASPARI_COHN:
      if (gc_form == MDA_LW_GC_STANDARD) return gaspari_cohn(nd);
      if (nd >= 2.0) return 0.0;
      if (nd >= 1.0) {
        const double z = nd - 1.0;
        return ((-0.25 * z + 0.5) * z + 0.625) * z + 0.125;
      } else {
        const double z = nd;
        return (((-0.25 * z + 0.5) * z + 0.625) * z - 5.0) * z + 4.0;
      }
    default:  // gaussian
      return exp(-0.5 * nd * nd);
  }
}

// partial[blk][j] = sum over the block's state points of (x_j - mean)^2, the
// mean formed in the same pass over X (32 points a wavefront, their members in
// registers); bound by reading X once.
template <int NS>
__global__ __launch_bounds__(256) void k_lw_member_sumsq(const double* __restrict__ X, int k,
                                                         int64_t n, double* __restrict__ partial) {
  __shared__ double red[4][NS * 4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i16 = lane & 15, kk = lane >> 4;
  double ss[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) ss[s] = 0.0;
  for (int64_t i0 = ((int64_t)blockIdx.x * 4 + wv) * 32; i0 < n; i0 += (int64_t)gridDim.x * 128) {
    double v[2][NS], mean[2];
    load_pert<NS, 2>(X, k, n, 1.0, i0, v, mean);
#pragma unroll
    for (int s = 0; s < NS; ++s) ss[s] = fma(v[0][s], v[0][s], fma(v[1][s], v[1][s], ss[s]));
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    for (int off = 1; off < 16; off <<= 1) ss[s] += __shfl_xor(ss[s], off);
    if (i16 == 0) red[wv][4 * s + kk] = ss[s];
  }
  __syncthreads();
  for (int j = threadIdx.x; j < k; j += 256)
    partial[(size_t)blockIdx.x * k + j] = (red[0][j] + red[1][j]) + (red[2][j] + red[3][j]);
}

// chi2_j = sum_b (yo_b - Yb_bj) / r_b * (yo_b - Yb_bj), Yb = ybar + Y'  (:475-500)
__global__ __launch_bounds__(256) void k_lw_chi2(const double* __restrict__ yo,
                                                 const double* __restrict__ ybar,
                                                 const double* __restrict__ yp_om,
                                                 const double* __restrict__ var, int k,
                                                 int64_t p, double* __restrict__ chi2) {
  __shared__ double red[256];
  const int j = blockIdx.x;
  double acc = 0.0;
  for (int64_t b = threadIdx.x; b < p; b += blockDim.x) {
    const double inn = yo[b] - (ybar[b] + yp_om[(size_t)b * k + j]);
    acc += inn * (1.0 / var[b]) * inn;
  }
  acc = block_sum(acc, red);
  if (threadIdx.x == 0) chi2[j] = acc;
}

// S and its transpose, 16 x 16 tiles with the Y' rows of both sides in LDS
constexpr int LW_ST = 16;

__global__ __launch_bounds__(256) void k_lw_form_S(const double* __restrict__ yp_om,
                                                   const double* __restrict__ w,
                                                   const double* __restrict__ var, int k,
                                                   int64_t p, double radius, int fn, int gc_form,
                                                   double* __restrict__ S,
                                                   double* __restrict__ St) {
#pragma clang fp contract(off)
  extern __shared__ double sm[];
  double* ya = sm;                  // [LW_ST][k]
  double* yb = sm + LW_ST * k;      // [LW_ST][k]
  double* ws = sm + 2 * LW_ST * k;  // [k]
  const int64_t a0 = (int64_t)blockIdx.y * LW_ST, b0 = (int64_t)blockIdx.x * LW_ST;
  const int tid = threadIdx.x;
  for (int e = tid; e < LW_ST * k; e += 256) {
    const int r = e / k, i = e % k;
    ya[e] = a0 + r < p ? yp_om[(size_t)(a0 + r) * k + i] : 0.0;
    yb[e] = b0 + r < p ? yp_om[(size_t)(b0 + r) * k + i] : 0.0;
  }
  for (int i = tid; i < k; i += 256) ws[i] = w[i];
  __syncthreads();
  const int ra = tid / LW_ST, rb = tid % LW_ST;
  const int64_t a = a0 + ra, b = b0 + rb;
  if (a >= p || b >= p) return;
  double acc = 0.0;
  for (int i = 0; i < k; ++i) acc += (ws[i] * ya[ra * k + i]) * yb[rb * k + i];
  const double dist = (double)(a > b ? a - b : b - a) / (double)p;
  double v = acc * lw_taper(dist, radius, fn, gc_form);
  if (a == b) v = v + var[a];
  S[(size_t)a * p + b] = v;
  St[(size_t)b * p + a] = v;
}

// D(b, i) = (yo_b + sqrt(r_b) Z_bi) - (ybar_b + y'_bi), obs-major [p][k]
__global__ void k_lw_innovations(const double* __restrict__ yo, const double* __restrict__ ybar,
                                 const double* __restrict__ yp_om,
                                 const double* __restrict__ var, const double* __restrict__ Z,
                                 int k, int64_t p, double* __restrict__ D) {
#pragma clang fp contract(off)
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < p * k;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = e / k;
    D[e] = (yo[b] + sqrt(var[b]) * Z[e]) - (ybar[b] + yp_om[e]);
  }
}

// ---------------------------------------------------------------------------
// The gain and update, fused, on FP64 MFMA.  A wavefront owns 32 state points
// with all their members in registers and takes 16 observations at a time:
//   K^T tile  = G^T X'_rho   (rows = observations, columns = points; G
//               fragments already divided by k - 1), times the taper,
//   acc      += D^T K^T      (rows = members, columns = points).
// Row kk + 4r of a product's result sits in register r of lane (i16, kk),
// which is the right operand of the step over observations 4r .. 4r + 3, so
// the tapered tile feeds the second product from its registers: K never
// reaches LDS, and X is read and written once.  The result's members match
// the fragments of X'_rho lane by lane as well.
// The taper depends on |s - b| alone: a table of every index distance (one
// evaluation each, instead of one per state point and observation), up to the
// ends of the last block and the last tile, is read in windows of p + 32
// entries.  Fragments go through two LDS buffers shared
// by the block's four wavefronts, and they and the tapers are fetched one tile
// ahead (read where they are used, they left one wavefront per SIMD waiting on
// L2 and HBM: 20.9 ms).
// Bound by the FP64 matrix rate (4 n p k FLOP); 30.8 ms at n = 4,194,304,
// p = 512, k = 64 with 4 x 4 register tiles out of LDS on the vector ALUs,
// 10.8 ms here (51 TFLOP/s).
// ---------------------------------------------------------------------------
// Gf[tile][step][lane] = G[16 tile + i16][4 step + kk] / (k - 1),
// Df[tile][r][tj][lane] = D[16 tile + 4r + kk][16 tj + i16] (ns = 4 nt steps),
// tap[m] = taper at index distance m
__global__ void k_lw_fragments(const double* __restrict__ Gt, const double* __restrict__ D, int k,
                               int64_t p, int ns, int64_t ntile, int64_t n, int64_t ntap,
                               double radius, int fn, int gc_form, double* __restrict__ Gf,
                               double* __restrict__ Df, double* __restrict__ tap) {
  const int64_t total = ntile * ns * 64;
  const int64_t t0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x,
                dt = (int64_t)gridDim.x * blockDim.x;
  const double kden = (double)(k - 1);
  for (int64_t e = t0; e < total; e += dt) {
    const int lane = (int)(e & 63), i16 = lane & 15, kk = lane >> 4;
    const int64_t ot = (e >> 6) / ns;
    const int st = (int)((e >> 6) % ns), nt = ns / 4;
    const int64_t og = 16 * ot + i16, od = 16 * ot + 4 * (st / nt) + kk;
    const int a = 4 * st + kk, m = 16 * (st % nt) + i16;
    Gf[e] = og < p && a < k ? Gt[(size_t)og * k + a] / kden : 0.0;
    Df[e] = od < p && m < k ? D[(size_t)od * k + m] : 0.0;
  }
  const double gdim = (double)(n > p ? n : p);
  for (int64_t e = t0; e < ntap; e += dt) tap[e] = lw_taper((double)e / gdim, radius, fn, gc_form);
}

template <int NS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NS <= 16 ? 2 : 1)))
void k_lw_update(double* __restrict__ X, int k, int64_t n, double scale,
                 const double* __restrict__ Gf, const double* __restrict__ Df,
                 const double* __restrict__ tap, int64_t p, int64_t ntile,
                 double* __restrict__ partial, const int* __restrict__ status) {
  constexpr int NT = NS / 4;
  extern __shared__ double sh[];     // two tiles of [Gf | Df]
  __shared__ double red[4][4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i16 = lane & 15, kk = lane >> 4;
  const int64_t i0 = ((int64_t)blockIdx.x * 4 + wv) * 32;
  double mx = -INFINITY, mn = INFINITY, sb = 0.0, sa = 0.0;
  double v[2][NS], mean[2];
  load_pert<NS, 2>(X, k, n, scale, i0, v, mean);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < NS; ++s) sb = fma(v[t][s], v[t][s], sb);
  d4 acc[NT][2];
#pragma unroll
  for (int tj = 0; tj < NT; ++tj) acc[tj][0] = acc[tj][1] = d4{0.0, 0.0, 0.0, 0.0};
  // the next tile's fragments (this thread's share) and tapers, on their way
  // while a tile is computed
  double gn[NT], dn[NT];
  double tn[2][4];
  auto fetch = [&](int64_t ot) {
    const double* g = Gf + (size_t)ot * NS * 64 + threadIdx.x;
    const double* d = Df + (size_t)ot * NS * 64 + threadIdx.x;
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      gn[q] = g[256 * q];
      dn[q] = d[256 * q];
    }
    const int64_t d0 = i0 + i16 - 16 * ot - kk;  // s - b of register 0, tile 0
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = d0 + 16 * t - 4 * r;
        tn[t][r] = tap[m < 0 ? -m : m];
      }
  };
  auto stage = [&](int b) {
    double* g = sh + (size_t)b * 2 * NS * 64 + threadIdx.x;
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      g[256 * q] = gn[q];
      g[NS * 64 + 256 * q] = dn[q];
    }
  };
  fetch(0);
  stage(0);
  for (int64_t ot = 0; ot < ntile; ++ot) {
    const int b = (int)(ot & 1);
    double tp[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) tp[t][r] = tn[t][r];
    __syncthreads();  // tile ot is in LDS, tile ot - 1 has been read
    if (ot + 1 < ntile) fetch(ot + 1);
    const double* gf = sh + (size_t)b * 2 * NS * 64 + lane;
    const double* df = gf + NS * 64;
    d4 kt[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const double a = gf[64 * s];
      kt[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, v[0][s], kt[0], 0, 0, 0);
      kt[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, v[1][s], kt[1], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double kv = kt[t][r] * tp[t][r];
        kt[t][r] = kv;
        if (16 * ot + kk + 4 * r < p && i0 + 16 * t + i16 < n) {
          mx = fmax(mx, kv);
          mn = fmin(mn, kv);
        }
      }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int tj = 0; tj < NT; ++tj) {
        const double a = df[64 * (r * NT + tj)];
        acc[tj][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, kt[0][r], acc[tj][0], 0, 0, 0);
        acc[tj][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, kt[1][r], acc[tj][1], 0, 0, 0);
      }
    if (ot + 1 < ntile) stage(b ^ 1);
  }
  {
    const bool update = (*status & MDA_ST_SKIP_UPDATE) == 0;
    // x_a = mean + (x'_rho + K D); the spread from the deviations' distance to
    // member 0's
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int64_t i = i0 + 16 * t + i16;
      const double sh = __shfl(v[t][0] + acc[0][t][0], i16);
      double s1 = 0.0, s2 = 0.0;
#pragma unroll
      for (int tj = 0; tj < NT; ++tj)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * tj + kk + 4 * r;
          const double dv = v[t][4 * tj + r] + acc[tj][t][r];
          if (j < k && i < n) {
            if (update) X[(size_t)j * n + i] = mean[t] + dv;
            s1 += dv - sh;
            s2 = fma(dv - sh, dv - sh, s2);
          }
        }
      for (int off = 16; off < 64; off <<= 1) {
        s1 += __shfl_xor(s1, off);
        s2 += __shfl_xor(s2, off);
      }
      if (kk == 0) sa += s2 - s1 * s1 / (double)k;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    mx = fmax(mx, __shfl_xor(mx, off));
    mn = fmin(mn, __shfl_xor(mn, off));
    sb += __shfl_xor(sb, off);
    sa += __shfl_xor(sa, off);
  }
  if (lane == 0) { red[0][wv] = mx; red[1][wv] = mn; red[2][wv] = sb; red[3][wv] = sa; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double* out = partial + 4 * (size_t)blockIdx.x;
    out[0] = fmax(fmax(red[0][0], red[0][1]), fmax(red[0][2], red[0][3]));
    out[1] = fmin(fmin(red[1][0], red[1][1]), fmin(red[1][2], red[1][3]));
    out[2] = (red[2][0] + red[2][1]) + (red[2][2] + red[2][3]);
    out[3] = (red[3][0] + red[3][1]) + (red[3][2] + red[3][3]);
  }
}

// any +inf variance (an invalid observation) -> *flag = 1
__global__ void k_lw_flag_inf(const double* __restrict__ var, int64_t p, int* __restrict__ flag) {
  bool bad = false;
  for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < p;
       o += (int64_t)gridDim.x * blockDim.x)
    bad = bad || isinf(var[o]);
  if (__ballot(bad) != 0ull && (threadIdx.x & 63) == 0) atomicOr(flag, 1);
}

// ---------------------------------------------------------------------------
void launch_lw_member_sumsq(hipStream_t s, const double* X, int k, int64_t n, double* part,
                            double* sumsq) {
  const unsigned nb = grid_for(n, 128, LW_SUMSQ_BLOCKS);
#define MDA_SS(NS) \
  hipLaunchKernelGGL(k_lw_member_sumsq<NS>, dim3(nb), dim3(256), 0, s, X, k, n, part)
  MDA_MEMBER_STEPS(k, MDA_SS)
#undef MDA_SS
  MDA_LAUNCH_CHECK();
  launch_reduce_partials(s, part, (int)nb, k, sumsq);
}

void launch_lw_chi2(hipStream_t s, const double* yo, const double* ybar, const double* yp_om,
                    const double* var, int k, int64_t p, double* chi2) {
  hipLaunchKernelGGL(k_lw_chi2, dim3(k), dim3(256), 0, s, yo, ybar, yp_om, var, k, p, chi2);
  MDA_LAUNCH_CHECK();
}

void launch_lw_form_S(hipStream_t s, const double* yp_om, const double* w, const double* var,
                      int k, int64_t p, double radius, int fn, int gc_form, double* S,
                      double* St) {
  const unsigned nt = (unsigned)((p + LW_ST - 1) / LW_ST);
  const size_t shm = sizeof(double) * (2 * LW_ST * k + k);
  hipLaunchKernelGGL(k_lw_form_S, dim3(nt, nt), dim3(256), shm, s, yp_om, w, var, k, p, radius,
                     fn, gc_form, S, St);
  MDA_LAUNCH_CHECK();
}

void launch_lw_innovations(hipStream_t s, const double* yo, const double* ybar,
                           const double* yp_om, const double* var, const double* Z, int k,
                           int64_t p, double* D) {
  hipLaunchKernelGGL(k_lw_innovations, dim3(grid_for(p * k, 256, 4096)), dim3(256), 0, s, yo,
                     ybar, yp_om, var, Z, k, p, D);
  MDA_LAUNCH_CHECK();
}

lw_update_shape lw_update_plan(int k, int64_t n, int64_t p) {
  lw_update_shape g;
  g.ns = (k + 15) / 16 * 4;
  g.ntile = (p + 15) / 16;
  g.nblk = (n + 127) / 128;
  // whole blocks of points and whole tiles of observations look their distances
  // up: |s - b| < 128 nblk for s >= b, and < 16 ntile otherwise
  g.ntap = std::max(128 * g.nblk, 16 * g.ntile);
  return g;
}

void launch_lw_update(hipStream_t s, double* X, double scale, const double* Gt, const double* D,
                      int k, int64_t n, int64_t p, double radius, int fn, int gc_form,
                      const lw_update_shape& g, double* Gf, double* Df, double* tap,
                      double* partial, double* out4, const int* status) {
  MDA_REQUIRE(k >= 2 && k <= 128, "LWEnKF supports 2 <= k <= 128");
  MDA_REQUIRE(g.nblk < (int64_t)1 << 31, "LWEnKF state too large");
  MDA_REQUIRE(g.ntap >= 128 * g.nblk && g.ntap >= 16 * g.ntile, "LWEnKF taper table too short");
  hipLaunchKernelGGL(k_lw_fragments, dim3(grid_for(std::max(g.frag_doubles(), g.ntap), 256, 4096)),
                     dim3(256), 0, s, Gt, D, k, p, g.ns, g.ntile, n, g.ntap, radius, fn, gc_form,
                     Gf, Df, tap);
  MDA_LAUNCH_CHECK();
#define MDA_LU(NS)                                                                            \
  hipLaunchKernelGGL(k_lw_update<NS>, dim3((unsigned)g.nblk), dim3(256),                     \
                     sizeof(double) * 4 * NS * 64, s, X, k, n, scale, Gf, Df, tap, p, g.ntile, \
                     partial, status)
  MDA_MEMBER_STEPS(k, MDA_LU)
#undef MDA_LU
  MDA_LAUNCH_CHECK();
  launch_fold_extremes(s, partial, g.nblk, out4);
}

void launch_lw_flag_inf(hipStream_t s, const double* var, int64_t p, int* flag) {
  if (p <= 0) return;
  hipLaunchKernelGGL(k_lw_flag_inf, dim3(grid_for(p, 256, 1024)), dim3(256), 0, s, var, p, flag);
  MDA_LAUNCH_CHECK();
}

}  // namespace mda
