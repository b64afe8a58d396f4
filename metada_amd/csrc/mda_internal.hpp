// Internal declarations shared by the HIP sources of libmetada_amd.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <functional>
#include <map>
#include <stdexcept>
#include <string>
#include <vector>

#include "metada_amd.h"

// ---------------------------------------------------------------------------
// errors: every entry point converts these into MDA_E_* codes
// ---------------------------------------------------------------------------
struct mda_error : std::runtime_error {
  int code;
  mda_error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define MDA_HIP(call)                                                              \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess)                                                          \
      throw mda_error(e_ == hipErrorOutOfMemory ? MDA_E_NOMEM : MDA_E_DEVICE,      \
                      std::string(#call) + ": " + hipGetErrorString(e_));          \
  } while (0)

#define MDA_REQUIRE(cond, msg)                                                     \
  do {                                                                             \
    if (!(cond)) throw mda_error(MDA_E_ARG, msg);                                  \
  } while (0)

#define MDA_LAUNCH_CHECK() MDA_HIP(hipGetLastError())

// Bits of an analysis's device status word (zeroed at the start of each
// analysis; kernels OR into it):
//   MDA_ST_NOT_SPD          a Cholesky factor did not exist (non-SPD matrix)
//   MDA_ST_NONFINITE_OBS    a non-finite H(x), observation-space mean or
//                           innovation
//   MDA_ST_NONFINITE_STATE  a non-finite background value reached the update
// The update kernels write nothing when a MDA_ST_SKIP_UPDATE bit is set, so
// an analysis that fails before its update leaves the ensemble unchanged.
//   MDA_ST_BOUNDARY_OVERFLOW more observations at the localisation radius
//                           than the boundary list holds
enum : int {
  MDA_ST_NOT_SPD = 1,
  MDA_ST_NONFINITE_OBS = 2,
  MDA_ST_NONFINITE_STATE = 4,
  MDA_ST_BOUNDARY_OVERFLOW = 8,
  MDA_ST_SKIP_UPDATE = MDA_ST_NOT_SPD | MDA_ST_NONFINITE_OBS | MDA_ST_BOUNDARY_OVERFLOW,
};

// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------
struct mda_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  struct buf {
    void* ptr = nullptr;
    size_t bytes = 0;
  };
  std::map<std::string, buf> ws;  // named device workspace, grown on demand
  hipEvent_t ev[12] = {};
  // batched analyses: extra streams (default priority) for concurrent
  // analyses, fork/join events, instantiated graphs by signature, and the
  // autotuned Gram launch (blocks, work queue) by workload key
  std::vector<hipStream_t> side;
  std::vector<hipEvent_t> fj;
  // timing events of column-chunked analyses (grown on demand)
  std::vector<hipEvent_t> evpool;
  std::map<std::string, hipGraphExec_t> graphs;
  std::map<std::string, std::pair<int, int>> tune;
  // state of the last LETKF call (for mda_letkf_last_transforms)
  int last_k = 0;
  int64_t last_ncol = 0;
  int last_ks = 0;           // block size of last_T
  double* last_T = nullptr;  // device, [ncol][last_ks][last_ks]
  int* last_nloc = nullptr;  // device, [ncol]
  int* last_flag = nullptr;  // device, [ncol] (tridiagonal path only)

  // Staging of small host arrays (create_staging): a pinned buffer with a
  // device buffer of the same layout.  An array goes to its place (stage_place)
  // in the pinned one, its device address lies at the same place in the other;
  // one asynchronous copy (send_staged) carries everything staged since the last,
  // before the first kernel that reads it.  Offsets start again with the first
  // array that an entry point stages, once the stream has drained; one that
  // stages nothing does not wait.  `result` is the pinned end of small copies
  // back.
  static constexpr size_t STAGE_BYTES = 4u << 20, STAGE_MAX = 512u << 10, RESULT_BYTES = 1u << 20;
  char *stage_host = nullptr, *stage_dev = nullptr, *result = nullptr;
  size_t stage_off = 0, stage_sent = 0;
  bool stage_begun = false;  // by the entry point that runs
  int depth = 0;  // nested entry points

  void create_staging() {
    MDA_HIP(hipHostMalloc((void**)&stage_host, STAGE_BYTES));
    MDA_HIP(hipHostMalloc((void**)&result, RESULT_BYTES));
    MDA_HIP(hipMalloc((void**)&stage_dev, STAGE_BYTES));
  }
  void destroy_staging() {
    if (stage_host) (void)hipHostFree(stage_host);
    if (result) (void)hipHostFree(result);
    if (stage_dev) (void)hipFree(stage_dev);
  }
  // place for `bytes` in both buffers (offset), or SIZE_MAX when the array is
  // too large or the buffers are full
  size_t stage_place(size_t bytes) {
    if (bytes > STAGE_MAX) return SIZE_MAX;
    if (!stage_begun) {
      // no copy or kernel of the calls before is left
      if (stage_off) MDA_HIP(hipStreamSynchronize(stream));
      stage_off = stage_sent = 0;
      stage_begun = true;
    }
    if (stage_off + bytes > STAGE_BYTES) return SIZE_MAX;
    const size_t at = stage_off;
    stage_off = (stage_off + bytes + 255) & ~(size_t)255;
    return at;
  }
  void send_staged() {
    if (stage_sent == stage_off) return;
    MDA_HIP(hipMemcpyAsync(stage_dev + stage_sent, stage_host + stage_sent,
                           stage_off - stage_sent, hipMemcpyHostToDevice, stream));
    stage_sent = stage_off;
  }
  void begin_call() {
    stage_begun = false;
    stage_sent = stage_off;  // what a call that failed left unsent
  }

  // returns a device buffer of at least `bytes`; contents are unspecified.
  // Each name has one meaning; a call fetches a name once, since growing a
  // buffer frees the previous allocation.
  void* get(const std::string& name, size_t bytes) {
    if (bytes == 0) bytes = 256;
    buf& b = ws[name];
    if (b.bytes < bytes) {
      // a cached graph may hold the old address: drop them all (their keys
      // hold every address they use, so none would match again anyway)
      drop_graphs();
      forget_results(b.ptr);
      if (b.ptr) MDA_HIP(hipFree(b.ptr));
      b.ptr = nullptr;
      b.bytes = 0;
      size_t want = bytes + bytes / 8;  // headroom: fewer re-allocations
      MDA_HIP(hipMalloc(&b.ptr, want));
      b.bytes = want;
    }
    return b.ptr;
  }
  template <class T>
  T* get(const std::string& name, size_t count) {
    return static_cast<T*>(get(name, count * sizeof(T)));
  }
  // frees the buffers whose names end in `suffix`
  void release(const std::string& suffix) {
    drop_graphs();
    for (auto& kv : ws) {
      const std::string& n = kv.first;
      if (n.size() < suffix.size() || n.compare(n.size() - suffix.size(), suffix.size(), suffix) != 0)
        continue;
      forget_results(kv.second.ptr);
      if (kv.second.ptr) MDA_HIP(hipFree(kv.second.ptr));
      kv.second = buf{};
    }
  }
  // results of the last LETKF call that lie in a buffer about to be freed
  void forget_results(const void* ptr) {
    if (last_T == ptr) last_T = nullptr;
    if (last_nloc == ptr) last_nloc = nullptr;
    if (last_flag == ptr) last_flag = nullptr;
  }
  void drop_graphs() {
    for (auto& kv : graphs)
      if (kv.second) (void)hipGraphExecDestroy(kv.second);
    graphs.clear();
  }
};

// Scoped "make this context's device current".
struct device_guard {
  int prev = 0;
  explicit device_guard(int dev) {
    MDA_HIP(hipGetDevice(&prev));
    if (prev != dev) MDA_HIP(hipSetDevice(dev));
  }
  ~device_guard() { (void)hipSetDevice(prev); }
};

// Host <-> device transfers.  Small arrays go through the context's pinned
// buffers: h2d enqueues its copy (the source may change when it returns), d2h
// enqueues one, waits for the stream and copies out, so a call with a handful
// of small inputs waits once instead of twice per array.  Large host buffers
// are ordinary pageable memory, copied synchronously: the context's stream is
// drained first (it is non-blocking, so the copy would not otherwise wait for
// it).
inline void h2d(mda_ctx* c, void* dst, const void* src, size_t bytes) {
  if (bytes == 0) return;
  const size_t at = c->stage_place(bytes);
  if (at == SIZE_MAX) {
    MDA_HIP(hipStreamSynchronize(c->stream));
    MDA_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return;
  }
  std::memcpy(c->stage_host + at, src, bytes);
  // what was staged before it goes out first; its own bytes go to dst only
  if (c->stage_sent < at)
    MDA_HIP(hipMemcpyAsync(c->stage_dev + c->stage_sent, c->stage_host + c->stage_sent,
                           at - c->stage_sent, hipMemcpyHostToDevice, c->stream));
  MDA_HIP(hipMemcpyAsync(dst, c->stage_host + at, bytes, hipMemcpyHostToDevice, c->stream));
  c->stage_sent = c->stage_off;
}
inline void d2h(mda_ctx* c, void* dst, const void* src, size_t bytes) {
  // kernels enqueued before this may have read staged inputs
  if (c->stage_sent != c->stage_off)
    throw mda_error(MDA_E_DEVICE, "internal: staged inputs were not sent to the device");
  if (bytes == 0) return;
  if (bytes <= mda_ctx::RESULT_BYTES) {
    MDA_HIP(hipMemcpyAsync(c->result, src, bytes, hipMemcpyDeviceToHost, c->stream));
    MDA_HIP(hipStreamSynchronize(c->stream));
    std::memcpy(dst, c->result, bytes);
    return;
  }
  MDA_HIP(hipStreamSynchronize(c->stream));
  MDA_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
}

// Host data staged to the device (no-op when already on the device).  A small
// array is on its way only after send_staged().
template <class T>
const T* to_device(mda_ctx* c, const std::string& name, const T* src, size_t count,
                   bool on_device) {
  if (src == nullptr) return nullptr;
  if (on_device) return src;
  const size_t bytes = count * sizeof(T), at = c->stage_place(bytes);
  if (at != SIZE_MAX) {
    std::memcpy(c->stage_host + at, src, bytes);
    return reinterpret_cast<const T*>(c->stage_dev + at);
  }
  T* d = c->get<T>(name, count);
  h2d(c, d, src, bytes);
  return d;
}

// Work beside the context's stream: what fork() returns runs after everything
// enqueued so far, and what is enqueued after join(), or after the branch has
// gone out of scope, runs after the branch's work.
struct side_branch {
  mda_ctx* c;
  bool open = false;
  explicit side_branch(mda_ctx* ctx) : c(ctx) {
    if (c->side.empty()) {
      hipStream_t st = nullptr;
      MDA_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
      c->side.push_back(st);
    }
    while (c->fj.size() < 2) {
      hipEvent_t e = nullptr;
      MDA_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      c->fj.push_back(e);
    }
  }
  side_branch(const side_branch&) = delete;
  side_branch& operator=(const side_branch&) = delete;
  hipStream_t fork() {
    MDA_HIP(hipEventRecord(c->fj[0], c->stream));
    MDA_HIP(hipStreamWaitEvent(c->side[0], c->fj[0], 0));
    open = true;
    return c->side[0];
  }
  void join() {
    if (!open) return;
    open = false;
    MDA_HIP(hipEventRecord(c->fj[1], c->side[0]));
    MDA_HIP(hipStreamWaitEvent(c->stream, c->fj[1], 0));
  }
  ~side_branch() {  // an error is on its way out
    if (open) (void)hipStreamSynchronize(c->side[0]);
  }
};

inline unsigned grid_for(int64_t n, int block, int64_t cap = 1 << 20) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

// ---------------------------------------------------------------------------
// kernels launched by the API layer (defined in the kernel sources)
// ---------------------------------------------------------------------------
namespace mda {

// clears `bytes` (multiple of 4) with a kernel, so the clear is graph-safe
void launch_zero(hipStream_t s, void* ptr, size_t bytes);
// streaming ensemble statistics
void launch_mean_pert(hipStream_t s, const double* X, int k, int64_t n, double scale,
                      double* mean, double* pert);
void launch_sumsq(hipStream_t s, const double* X, int64_t count, double* partial,
                  int nblocks);
// observation space: Y' obs-major [p][k], ybar, d; optional member-major Y'.
// With `order`, observations are processed in the order order[0], order[1],
// ...; observation order[t] is written at position t, or at opos[order[t]]
// when `opos` is given.  y32 (if not null) receives an FP32 copy of Y'.
void launch_obs_stats(hipStream_t s, const double* X, int k, int64_t n, int64_t p,
                      const int64_t* row_ptr, const int64_t* col, const double* w,
                      const double* hx_mm, const double* yo, double* ybar, double* yp_om,
                      double* d, double* yp_mm, const uint32_t* order = nullptr,
                      float* y32 = nullptr, const uint32_t* opos = nullptr,
                      int* status = nullptr);
// global (all-observation) Gram: G[a][c] = sum_o r_o Y'[o][a] Q[o][c] with Q =
// [Y' | d] (mode 0) or D = d + sigma Z - Y' (mode 1, EnKF); partials reduced.
void launch_global_gram(hipStream_t s, const double* yp_om, const double* d,
                        const double* var, const double* Z, int k, int64_t p, int mode,
                        double* partial, int nblocks, double* out);
// out[e] = sum over blocks of partial[block][e], e < ne
void launch_reduce_partials(hipStream_t s, const double* partial, int nblocks, int ne,
                            double* out);
// [max, min, sum, sum] over nb quadruples
void launch_fold_extremes(hipStream_t s, const double* partial, int64_t nb, double* out4);
// small dense solves on one workgroup (matrices in LDS)
void launch_etkf_solve_ws(hipStream_t s, int k, const double* EB, double* T, int* status);
void launch_enkf_solve_ws(hipStream_t s, int k, const double* EB, const double* F, double* T,
                          double* Minv, int* status);
// X_a = xbar + scale * X' T for all state points (global T); skipped when
// the status word holds a MDA_ST_SKIP_UPDATE bit.  With partial (4 doubles per
// block, transform_global_blocks(n) of them), out4[3] = sum over state and
// members of (x_a - mean_a)^2
unsigned transform_global_blocks(int64_t n);
void launch_transform_global(hipStream_t s, double* X, int k, int64_t n, double scale,
                             const double* T, int* status, double* partial = nullptr,
                             double* out4 = nullptr);
// EnKF diagnostics
struct enkf_gain_shape {
  int ns;              // MFMA steps over the members
  int64_t ntile, per;  // tiles of 16 observations, tiles per block
  int64_t nbx, nby;    // blocks over state points and over observation tiles
  int64_t gf_doubles() const { return ntile * ns * 64; }
  int64_t partial_doubles() const { return 4 * nbx * nby; }
};
enkf_gain_shape enkf_gain_plan(int k, int64_t n, int64_t p);
// out4 = [max K, min K, sum over state and members of ((x - mean) scale)^2, 0]
void launch_enkf_gain_minmax(hipStream_t s, const double* X, int k, int64_t n, double scale,
                             const double* Minv, const double* yp_om, const double* var,
                             int64_t p, const enkf_gain_shape& g, double* Gf, double* partial,
                             double* out4);
// the nine sums of Metrics::CalculateAll; partial: 9 METRICS_BLOCKS doubles
constexpr int METRICS_BLOCKS = 2048;
void launch_metrics(hipStream_t s, const double* X, int k, int64_t n, const double* truth,
                    double* partial, double* out9);

// LETKF
struct bucket_grid {
  int coord;
  int nrow, ncolb;       // bucket rows (lat / y) and bucket columns (lon / x)
  double a0, b0;         // origin of the bucket grid
  double da, db;         // bucket sizes
  int wrap;              // longitude wrap-around
};
// clears status, stats [9], and per column sweeps, flag and (when set) nloc,
// and per pass the fallback and boundary-list counts
struct letkf_begin_args {
  int64_t ncol, npass;
  int *status, *sweeps, *flag, *nloc;
  int64_t* stats;
  unsigned* wcount;
  uint32_t* shell_count;
};
void launch_letkf_begin(hipStream_t s, const letkf_begin_args& a);
// validity, bucket keys and (tkeys set) keys of the first stencil tap, nxy
// points per level; rcoord: latitude (GEOGRAPHIC) or y, ccoord: longitude or x
struct obs_prepare_args {
  int64_t p, nxy;
  const double *yo, *var, *rcoord, *ccoord;
  bucket_grid grid;
  uint32_t *keys, *vals;
  const int64_t *row_ptr, *col;
  uint32_t *tkeys, *tvals;
  int* status;
};
void launch_obs_prepare(hipStream_t s, const obs_prepare_args& a);
// stable sort of up to two sets of p <= SORT_SMALL (key, value) pairs, in place
constexpr int SORT_SMALL = 4096;
struct sort_job {
  uint32_t *keys, *vals;
  int bits;  // of the keys
};
void launch_sort_small(hipStream_t s, const sort_job* jobs, int njobs, int64_t p);
void radix_sort_pairs(hipStream_t s, uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp,
                      uint32_t* vals_tmp, int64_t p, int key_bits, uint32_t* hist,
                      int64_t hist_cap);
void launch_bucket_ranges(hipStream_t s, const uint32_t* sorted_keys, int64_t p,
                          int nbuckets, int* start);
// per-observation data in bucket order (1/var, coordinates; unit vectors of
// GEOGRAPHIC locations when ux is not null; ipos[order[t]] = t when set)
void launch_gather_obs(hipStream_t s, const uint32_t* order, int64_t p, const double* var,
                       const double* oa, const double* ob, const double* oc, int rweight,
                       double* s_rinv, double* s_a, double* s_b, double* s_c, double* ux,
                       double* uy, double* uz, uint32_t* ipos);
// Y' rows and d in bucket order, plus the FP32 copy of Y' when y32 is not null
void launch_gather_rows(hipStream_t s, const uint32_t* order, int64_t p, int k,
                        const double* yp_om, const double* d, double* s_yp, double* s_d,
                        float* y32);
struct letkf_gram_args {
  int k;
  // size of the per-column blocks C [ks][ks] and b [ks]: k, or the padded
  // size of the eigensolver's kernels (letkf_eig_size), zeros past k
  int ks;
  int64_t ncol, nx;
  int coord;
  const double* col_a;
  const double* col_b;
  const double* col_c;
  bucket_grid grid;
  const int* bstart;
  const double* yp;    // sorted obs-major Y'
  const double* d;     // sorted innovations
  const double* rinv;  // sorted 1/var (or 1)
  const double* oa;
  const double* ob;
  const double* oc;
  double radius;
  int localization;
  int precision;
  const float* y32;    // sorted obs-major Y' in FP32 (FP32 / BF16x3 contractions)
  const double* ux;    // sorted unit vectors of GEOGRAPHIC observation locations (any precision)
  const double* uy;
  const double* uz;
  double* C;    // out [ncol][ks][ks]
  // C holds FP32 entries (the FP32 / BF16x3 contractions, whose products are
  // accumulated in FP32): half the buffer is used, E1 widens them to FP64
  int c32;
  double* b;    // out [ncol][ks]
  int* nloc;    // out [ncol]
  // per-column setup records [ncol][96] of the Gram (window rows, row table,
  // reference point), from launch_column_setup
  int* crec;
  // work-queue mode: persistent waves take columns order[0], order[1], ...
  // through the counter `queue` (zeroed before the launch)
  const uint32_t* order;
  uint32_t* queue;
  int nblocks;  // launch size (0: one wave per column)
  // GEOGRAPHIC boundary list of the pass: (column, observation, chord
  // decision) of candidates within shell_width of the threshold, decided
  // exactly by launch_letkf_shell_fixup; its counter is zeroed before the Gram
  int4* shell;
  uint32_t* shell_count;
  int64_t shell_cap;
  // Global index of column 0.  The per-column arrays (col_a/b/c, C, b, nloc)
  // start at that column; col0 only enters where the global index itself
  // matters (grid coordinates of a GRID geometry without coordinates).
  int64_t col0;
};
// setup records of columns [0, a.ncol) for the Gram kernels (a.crec),
// LETKF_CREC_INTS ints per column
constexpr int LETKF_CREC_INTS = 96;
void launch_column_setup(hipStream_t s, const letkf_gram_args& a);
void launch_letkf_gram(hipStream_t s, const letkf_gram_args& a);
// exact decisions of the pass's GEOGRAPHIC boundary list (no-op otherwise)
void launch_letkf_shell_fixup(hipStream_t s, const letkf_gram_args& a, int* status);
// per-column cost estimate (observations in the candidate buckets) as
// descending-order sort keys, and column ids
void launch_column_cost(hipStream_t s, const letkf_gram_args& a, uint32_t* keys,
                        uint32_t* cols);
// learned-inflation inputs: per-observation background variance of the
// sorted Y', then the 8 local statistics of every column
void launch_obs_spread(hipStream_t s, const double* s_yp, int64_t p, int k, double* sp);
void launch_letkf_features(hipStream_t s, const letkf_gram_args& a, double* sp,
                           const double* X, int64_t nlev, const double* rho_prev, float* feat);
// Lorenz-96 forecast of nstates states of size N in place (scheme 0 RK4, 1 Euler)
void launch_l96(hipStream_t s, double* X, int64_t nstates, int64_t N, double F, double dt,
                int nsteps, int scheme);
// learned inflation network
void launch_mlp_forward(hipStream_t s, const float* params, const float* feat, int64_t m,
                        float* rho);
void launch_mlp_loss_grad(mda_ctx* c, hipStream_t s, const float* params, const float* feat,
                          const float* target, int64_t m, float* grad, double* loss);
void launch_mlp_adam(hipStream_t s, float* params, float* m1, float* m2, const float* grad,
                     int64_t step, float lr, float b1, float b2, float eps);
struct letkf_solve_args {
  int k;
  int ks;  // size of the per-column blocks C, T, U, b, lam (letkf_gram_args::ks)
  int64_t ncol;
  int64_t all_cols;  // of the whole analysis, where this is one chunk of it
  const double* C;
  int c32;  // C holds FP32 entries (letkf_gram_args::c32)
  const double* b;
  const int* nloc;
  double rho;
  const double* rho_col;
  int inflation_form, sqrt_form, combine;
  double* T;
  int* sweeps;
  int* status;
  // tridiagonal eigensolver workspace (symmetric square root)
  double* de;    // [ncol][2 ks]
  double* lam;   // [ncol][ks]
  double* U;     // [ncol][ks][ks] Householder reflectors
  int* flag;     // [ncol] columns re-solved by the Jacobi fallback
  // Jacobi whose two matrices exceed the LDS (letkf_solve_v_global): one in a
  // global scratch of letkf_solve_matrix_bytes(k) for each of jblocks blocks
  double* jscratch;
  int jblocks;
  // fallback work list [ncol] and its length (set: only the flagged and empty
  // columns are visited after the tridiagonal eigensolver)
  int* wlist;
  unsigned* wcount;
  int method;    // 0: tridiagonal + Jacobi fallback, 1: Jacobi only
  // set: the columns the tridiagonal kernels work on [ncol], nloc where
  // nloc >= k and 0 elsewhere; the others with observations go to the
  // fallback (k < ks with a reduced-precision Gram, see launch_letkf_solve)
  int* eig_nloc;
  // set: T from the inverse square root corrected against C (k < ks, FP64)
  int refine;
  hipEvent_t ev_stage[3];  // recorded after E1, E2, E3 when set (timing)
  // Reduced-precision Gram: eigenvalues within null_rel * ||A|| of (k-1)/rho
  // are treated as the null space of Y'^T R^-1 Y' (0 for FP64)
  double null_rel;
  // Fused eigenvectors + transform (tridiagonal path, ks in {16, 32, 48, 64},
  // matrix combination, FP64 transform): E3 applies X_a = X T' to the pass's
  // columns [x_col0, x_col0 + ncol) of X (x_ncol columns of x_nlev levels)
  // and writes T only for the columns it leaves to the fallback (flag != 0)
  // and for the empty ones.
  int fuse;
  double* X;
  int64_t x_ncol, x_nlev, x_col0;
};
// true when the tridiagonal eigensolver of block size ks can apply the
// transform itself
bool letkf_eig_fusable(int ks);
size_t letkf_solve_matrix_bytes(int k);
bool letkf_solve_v_global(int k);
void launch_letkf_solve(hipStream_t s, const letkf_solve_args& a);
// block size of the tridiagonal eigensolver for k members: the smallest
// compiled size >= k
int letkf_eig_size(int k);
void launch_letkf_eig(hipStream_t s, const letkf_solve_args& a, double* de, double* lam,
                      int* flag);
// X_a = xbar + X' T for the columns [col0, col0 + nc) of X (ncol columns in
// all; nc < 0: every column); T holds the nc columns' transforms, blocks of
// ks x ks (ks = k, or letkf_eig_size(k)).  Skipped
// when the status word holds a MDA_ST_SKIP_UPDATE bit.  MDA_PREC_BF16X3
// runs X' T as split-precision bf16 products with FP32 accumulation (k a
// multiple of 16, at most 64); otherwise FP64.  `only` ([nc], FP64 MFMA path
// only) restricts the update to the columns with only[g] != 0.
void launch_letkf_transform(hipStream_t s, double* X, int k, int ks, int64_t ncol,
                            int64_t nlev, const double* T, int* status, int64_t col0 = 0, int64_t nc = -1,
                            int precision = MDA_PREC_FP64, const int* only = nullptr);
// [sum, max, #zeros] of each array (v2 may be null), added into out9
void launch_reduce_int(hipStream_t s, const int* v0, const int* v1, const int* v2, int64_t n,
                       int64_t* out9);

// runs f with the context's device current and converts its exceptions into
// MDA_E_* codes (message in ctx->err)
int guarded_call(mda_ctx* ctx, const std::function<void()>& f);

// ETKF (ETKF.hpp:100-178) on device buffers: Y' [p][k], d [p], Gram
// partials [ETKF_GG_BLOCKS][k][k+1], [E | b] [k][k+1], T [k][k] and the status
// word.  etkf_run takes them from the
// context workspace when `bufs` is null.
constexpr int ETKF_GG_BLOCKS = 256;
struct etkf_bufs {
  double *yp, *dd, *part, *EB, *T;
  int* status;
};
void etkf_run(mda_ctx* c, double inflation, mda_ensemble* ens, const mda_obs* obs,
              const mda_hop* hop, const etkf_bufs* bufs);

// IDW4 observation operator on the device (kernels_hop.hip): 4 taps per
// row at row_ptr[o] (rows of invalid observations are empty and skipped)
void launch_idw4_stencil(hipStream_t s, int64_t p, int coord, const double* oa, const double* ob,
                         const double* oc, const double* var, int64_t nx, int64_t ny,
                         int64_t nlev, const double* clat, const double* clon,
                         const double* vcoord, const int64_t* row_ptr, int64_t* col,
                         double* weight);

// dense p x p algebra of the global filters (p <= MDA_DENSE_MAX)
constexpr int64_t MDA_DENSE_MAX = 4096;
void launch_form_enkf_S(hipStream_t s, const double* yp, const double* var, int k, int64_t p,
                        double* S);
// enqueues the extreme eigenvalues of the symmetric device matrix A (destroyed
// beyond 128 rows) into out [4] = lmin, lmax, |l|min, |l|max (device); lda: row
// stride, 0 = p (rows beyond 128 are contiguous)
void dense_sym_extremes(mda_ctx* c, hipStream_t s, double* A, int64_t p, int64_t lda, double* out);
// enqueues lambda_max and lambda_min of S = Y'Y'^T/(k-1) + diag(var), through
// k x k factorisations, into out [2] (device); hvar: the variances on the host,
// finite and > 0
void lowrank_spd_extremes(mda_ctx* c, side_branch& br, const double* yp, const double* var,
                          const double* hvar, int k, int64_t p, double* out);
// B <- A^-1 B by Gauss-Jordan with partial pivoting (A destroyed); a zero
// pivot sets MDA_ST_NOT_SPD in *status; work: dense_gauss_jordan_work(p) doubles
size_t dense_gauss_jordan_work(int64_t p);
void dense_gauss_jordan(hipStream_t s, int64_t p, int64_t m, double* A, double* B, double* work,
                        int* status);

// LWEnKF (kernels_lw.hip)
// sumsq[j] = sum over the state of (x_j - mean)^2; part: LW_SUMSQ_BLOCKS * k
constexpr int LW_SUMSQ_BLOCKS = 1024;
void launch_lw_member_sumsq(hipStream_t s, const double* X, int k, int64_t n, double* part,
                            double* sumsq);
void launch_lw_chi2(hipStream_t s, const double* yo, const double* ybar, const double* yp_om,
                    const double* var, int k, int64_t p, double* chi2);
void launch_lw_form_S(hipStream_t s, const double* yp_om, const double* w, const double* var,
                      int k, int64_t p, double radius, int fn, int gc_form, double* S,
                      double* St);
void launch_lw_innovations(hipStream_t s, const double* yo, const double* ybar,
                           const double* yp_om, const double* var, const double* Z, int k,
                           int64_t p, double* D);
// workspace of the fused gain and update: fragments of G and D, the taper of
// every index distance, per-block partials
struct lw_update_shape {
  int ns;                 // MFMA steps over the members
  int64_t ntile, nblk;    // tiles of 16 observations, blocks of 128 state points
  int64_t ntap;           // taper table entries
  int64_t frag_doubles() const { return ntile * ns * 64; }
};
lw_update_shape lw_update_plan(int k, int64_t n, int64_t p);
// out4 = [max K, min K, sum of squares of X'_rho, sum of (x_a - mean_a)^2]; X is
// left alone when the status word holds a MDA_ST_SKIP_UPDATE bit
void launch_lw_update(hipStream_t s, double* X, double scale, const double* Gt, const double* D,
                      int k, int64_t n, int64_t p, double radius, int fn, int gc_form,
                      const lw_update_shape& g, double* Gf, double* Df, double* tap,
                      double* partial, double* out4, const int* status);
void launch_lw_flag_inf(hipStream_t s, const double* var, int64_t p, int* flag);

}  // namespace mda
