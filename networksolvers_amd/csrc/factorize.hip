// Truncated factorisation theta = U C (ITensors factorize, inserter.jl:23) and the
// QR gauge walk (extracter.jl:6).  FP64 throughout.
//
// "svd" route: an SVD of M itself (svd.hip): one-launch Householder
// bidiagonalisation, the singular values by bisection on the Golub-Kahan matrix,
// the kept singular vectors by inverse iteration, orthonormalised (block CGS2 +
// CholQR2) and back-transformed through the Householder reflectors (compact-WY).
// P = s^2 in decreasing order, with an SVD's accuracy (the Gram matrix would resolve
// P only to eps * P_max).  "eigen" route: rho = M M^T (isometry on the rows; M^T M
// on the columns) by MFMA GEMM, then batched Jacobi for small rho, else the
// one-launch tridiagonal reduction, bisection for every eigenvalue, inverse
// iteration for the kept ones only and the same orthonormalisation and
// back-transformation; the spectrum sorted by decreasing |lambda|.  Sizes beyond
// the one-launch kernels (n > 1024 on the eigen route, s > 2048 on the svd route)
// take rocSOLVER dsyevd on the Gram matrix.  NDTensors truncate! is restated on
// the host; the kept vectors get the gauge fix and C = U^T M by MFMA GEMM.
// rocSOLVER is column-major: a row-major m x n buffer is its n x m transpose.
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <memory>
#include <numeric>

#include "internal.h"

using namespace nsmi;

namespace nsmi {
namespace {

// auxiliary streams for the sector solves of one QN bond
constexpr size_t kAuxStreams = 4;

// restatement of NDTensors truncate! (relative cutoff); returns kept count
int64_t truncate_spectrum(std::vector<double>& P, int64_t mindim, int64_t maxdim, double cutoff, double* truncerr,
                          double* total) {
  const int64_t origm = int64_t(P.size());
  *truncerr = 0.0;
  *total = 0.0;
  if (origm == 0) return 0;
  if (origm == 1) {
    *total = P[0];
    return 1;
  }
  if (P[0] < 0)
    for (auto& v : P) v = -v;
  for (int64_t n = origm - 1; n >= 0; --n) {
    if (P[n] >= 0) break;
    P[n] = 0.0;
  }
  int64_t n = origm;
  double err = 0.0;
  while (n > maxdim) {
    err += P[n - 1];
    --n;
  }
  double scale = 0.0;
  for (double v : P) scale += v;
  *total = scale;
  if (scale == 0.0) scale = 1.0;
  while (n > mindim && (err + P[n - 1] <= cutoff * scale)) {
    err += P[n - 1];
    --n;
  }
  err /= scale;
  if (n < 1) n = 1;
  *truncerr = err;
  return n;
}

// For each of k vectors (row r of a row-major matrix with row stride ld when
// rows == 1, else column c with column stride 1 and row stride ld), find the
// first index of the largest magnitude and write its sign (+1/-1) to sgn.
__global__ void k_gauge_sign(const double* __restrict__ X, int64_t len, int64_t ld, int rows,
                             const int* __restrict__ idx, double* __restrict__ sgn) {
  const int j = blockIdx.x;
  const int64_t base = rows ? int64_t(idx ? idx[j] : j) * ld : int64_t(idx ? idx[j] : j);
  const int64_t step = rows ? 1 : ld;
  double best = -1.0;
  int64_t bi = 0;
  for (int64_t i = threadIdx.x; i < len; i += blockDim.x) {
    const double a = fabs(X[base + i * step]);
    if (a > best) {  // strict: first index wins within a thread's stride
      best = a;
      bi = i;
    }
  }
  __shared__ double sb[256];
  __shared__ int64_t si[256];
  sb[threadIdx.x] = best;
  si[threadIdx.x] = bi;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      const double b2 = sb[threadIdx.x + o];
      const int64_t i2 = si[threadIdx.x + o];
      if (b2 > sb[threadIdx.x] || (b2 == sb[threadIdx.x] && i2 < si[threadIdx.x])) {
        sb[threadIdx.x] = b2;
        si[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) sgn[j] = (X[base + si[0] * step] < 0.0) ? -1.0 : 1.0;
}

// out[j, i] = scale[j] * sgn[j] * X[idx[j], i]   (gather rows; out row-major k x len)
__global__ void k_gather_rows(const double* __restrict__ X, int64_t ld, const int* __restrict__ idx, int k,
                              int64_t len, const double* __restrict__ sgn, const double* __restrict__ scale,
                              double* __restrict__ out) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(k) * len) return;
  const int j = int(t / len);
  const int64_t i = t % len;
  const int src = idx ? idx[j] : j;
  double f = sgn ? sgn[j] : 1.0;
  if (scale) f *= scale[j];
  out[t] = f * X[int64_t(src) * ld + i];
}

// out[i, j] = scale[j] * sgn[j] * X[i, idx[j]]   (gather columns into row-major len x k)
__global__ void k_gather_cols(const double* __restrict__ X, int64_t ld, const int* __restrict__ idx, int k,
                              int64_t len, const double* __restrict__ sgn, const double* __restrict__ scale,
                              double* __restrict__ out) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(k) * len) return;
  const int64_t i = t / k;
  const int j = int(t % k);
  const int src = idx ? idx[j] : j;
  double f = sgn[j];
  if (scale) f *= scale[j];
  out[t] = f * X[i * ld + src];
}

// out (len x k, row-major) = transpose of in (k x len, row-major)
__global__ void k_transpose(const double* __restrict__ in, int k, int64_t len, double* __restrict__ out) {
  __shared__ double tile[32][33];
  const int64_t i0 = int64_t(blockIdx.x) * 32, j0 = int64_t(blockIdx.y) * 32;
  for (int r = threadIdx.y; r < 32; r += blockDim.y) {
    const int64_t j = j0 + r, i = i0 + threadIdx.x;
    if (j < k && i < len) tile[r][threadIdx.x] = in[j * len + i];
  }
  __syncthreads();
  for (int r = threadIdx.y; r < 32; r += blockDim.y) {
    const int64_t i = i0 + r, j = j0 + threadIdx.x;
    if (i < len && j < k) out[i * k + j] = tile[threadIdx.x][r];
  }
}

// out (k x L, row-major) = Y^T padded with zeros: out[j][i] = Y[i][j] for i < len (Y: len x k)
__global__ void k_transpose_pad(const double* __restrict__ Y, int64_t len, int k, int64_t L, double* __restrict__ out) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(k) * L) return;
  const int64_t j = t / L, i = t % L;
  out[t] = i < len ? Y[i * k + j] : 0.0;
}

// R (r x n row-major) from a gelqf/geqrf output read row-major, zeroing the
// triangle below (upper == 1 keeps j >= i) and applying row signs.
__global__ void k_extract_tri(const double* __restrict__ X, int64_t ldx, int64_t r, int64_t n,
                              const double* __restrict__ sgn, double* __restrict__ out, int transpose_out) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= r * n) return;
  const int64_t i = t / n, j = t % n;
  const double v = (j >= i) ? sgn[i] * X[i * ldx + j] : 0.0;
  if (transpose_out)
    out[j * r + i] = v;
  else
    out[t] = v;
}

// R^T (m x r row-major) from a geqrf output read row-major (m x ldx): element
// (j, i) = sgn[i] * X[j*ldx + i] for i <= j, else 0.
__global__ void k_extract_tri_t(const double* __restrict__ X, int64_t ldx, int64_t r, int64_t m,
                                const double* __restrict__ sgn, double* __restrict__ out) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= r * m) return;
  const int64_t j = t / r, i = t % r;
  out[t] = (i <= j) ? sgn[i] * X[j * ldx + i] : 0.0;
}

// Q columns (or rows) times the diagonal signs of R
__global__ void k_scale_cols(double* __restrict__ X, int64_t rows, int64_t cols, const double* __restrict__ sgn) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= rows * cols) return;
  X[t] *= sgn[t % cols];
}
__global__ void k_scale_rows(double* __restrict__ X, int64_t rows, int64_t cols, const double* __restrict__ sgn) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= rows * cols) return;
  X[t] *= sgn[t / cols];
}
// sign of the diagonal entries of a row-major matrix (row stride ld)
__global__ void k_diag_sign(const double* __restrict__ X, int64_t ld, int64_t r, double* __restrict__ sgn) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < r) sgn[i] = X[i * ld + i] < 0.0 ? -1.0 : 1.0;
}

inline unsigned blocks(int64_t n, int t = 256) { return unsigned((n + t - 1) / t); }

GemmDesc gdesc(int64_t M, int64_t N, int64_t K, bool ta, bool tb) {
  GemmDesc g{};
  g.M = M;
  g.N = N;
  g.K = K;
  g.transA = ta;
  g.transB = tb;
  g.lda = ta ? M : K;
  g.ldb = tb ? K : N;
  g.ldc = N;
  g.batch = 1;
  return g;
}

void check_rocsolver(rocblas_status st, const char* what) {
  if (st != rocblas_status_success)
    fail(NSMI_ERR_SOLVER, std::string(what) + " failed with rocblas_status " + std::to_string(int(st)));
}

}  // namespace
}  // namespace nsmi

namespace nsmi {
namespace {

// One real matrix M (m x nc) split into the isometry side (rows of M, or columns
// when rows_trailing) and the rest: phase 1 computes the decomposition and the
// spectrum P sorted as NDTensors sorts it; phase 2 writes U and C for k vectors.
struct FactCore {
  const double* M;
  int64_t m, nc;
  bool rows_trailing;
  int route;
  int64_t iso = 0, oth = 0, full = 0;
  bool tri = false;     // rho holds sytrd reflectors; d (w) and e the tridiagonal, lam its eigenvalues
  bool bid = false;     // svd route: X holds the bidiagonalisation, lam the singular values
  bool jacobi = false;  // rho awaits the batched Jacobi solve (eigenvalues into wdev)
  bool want_v = false;  // bid: the isometry is X's right singular vectors (X = the isometry side transposed)
  bool svd_declined = false;  // the svd route could not launch here: the Gram matrix took its place
  int64_t xr = 0, xs = 0;  // bid: X is xr x xs (xr >= xs)
  std::vector<double> P;
  std::vector<int> order;
  std::unique_ptr<Scratch> rho, z, tau, wdev, w, e, lam, X, tauR, gk;
  SytrdRun sr;             // the one-launch reduction's buffers and host flags
  double* wh = nullptr;    // host copy of the eigenvalues (pinned stage memory, filled asynchronously)
  int* info_h = nullptr;   // host copy of the solver status (pinned stage memory)
  unsigned* orth_h = nullptr;  // host copy of the orthonormalisation's failure flag (fact_emit)
  FactCore(const double* M_, int64_t m_, int64_t nc_, bool rt, int r) : M(M_), m(m_), nc(nc_), rows_trailing(rt),
                                                                         route(r) {
    iso = rt ? nc : m;
    oth = rt ? m : nc;
    full = std::min(m, nc);
  }
};

// Spectrum P in NDTensors' order from the host copy of the eigenvalues.
void fact_spectrum(FactCore& f, std::vector<double>& wh) {
  const int64_t iso = f.iso;
  for (double v : wh)
    if (!std::isfinite(v)) fail(NSMI_ERR_NOT_FINITE, "factorize: non-finite eigenvalue");
  f.order.resize(iso);
  std::iota(f.order.begin(), f.order.end(), 0);
  if (f.route == NSMI_ROUTE_EIGEN) {
    // NDTensors eigen: sort by decreasing |lambda|; truncate! zeroes a negative tail
    std::stable_sort(f.order.begin(), f.order.end(), [&](int a, int b) { return std::fabs(wh[a]) > std::fabs(wh[b]); });
  } else {
    // svd semantics: P = s^2 >= 0 in decreasing order
    for (auto& v : wh) v = std::max(v, 0.0);
    std::stable_sort(f.order.begin(), f.order.end(), [&](int a, int b) { return wh[a] > wh[b]; });
  }
  f.P.resize(iso);
  for (int64_t i = 0; i < iso; ++i) f.P[i] = wh[f.order[i]];
}

// Phases of one factorisation, so that several independent ones (the sectors of a
// QN bond) can run on several streams: the Gram product, then for a small rho the
// batched Jacobi solve; otherwise the one-launch reduction and, once its flags are
// read, rocSOLVER's divide and conquer on T (the back-transformation is deferred
// to fact_emit, where only the kept vectors are transformed), or the library's
// dsyevd when the reduction cannot run.  Every phase only enqueues; fact_finish
// reads the copied status and eigenvalues after the caller's synchronisation.
void fact_gram_gemm(nsmi_ctx* ctx, FactCore& f) {
  // Beyond its one-launch kernels the "svd" route diagonalises the Gram matrix as
  // well: rocSOLVER's dgesvd is ~80x slower than dsyevd at n = 2048 on gfx950 (3.9 s
  // vs 47 ms) and 8x slower than the batched Jacobi solver at n = 32 (4.2 vs 0.55 ms
  // per factorisation).
  const int64_t iso = f.iso, oth = f.oth, m = f.m, nc = f.nc;
  f.rho.reset(new Scratch(ctx, sizeof(double) * size_t(iso) * iso));
  {
    ProfScope ps(ctx, NSMI_K_FACT_GEMM, 2.0 * double(iso) * iso * oth, 8.0 * (double(m) * nc + double(iso) * iso));
    if (!f.rows_trailing)
      gemm_f64(ctx, gdesc(m, m, nc, false, true), 1.0, f.M, f.M, 0.0, f.rho->as<double>(), kRoleFact);
    else
      gemm_f64(ctx, gdesc(nc, nc, m, true, false), 1.0, f.M, f.M, 0.0, f.rho->as<double>(), kRoleFact);
  }
  if (iso <= kJacobiMax) {
    f.jacobi = true;
    f.wdev.reset(new Scratch(ctx, sizeof(double) * size_t(iso)));
    return;
  }
  f.w.reset(new Scratch(ctx, sizeof(double) * size_t(iso)));
  f.e.reset(new Scratch(ctx, sizeof(double) * size_t(iso)));
  f.tau.reset(new Scratch(ctx, sizeof(double) * size_t(std::max<int64_t>(iso, 2))));
}

// the reduction; false when it cannot run here (the caller takes fact_syevd)
bool fact_tri_launch(nsmi_ctx* ctx, FactCore& f) {
  f.tri = sytrd_launch(ctx, f.rho->as<double>(), int(f.iso), f.w->as<double>(), f.e->as<double>(),
                       f.tau->as<double>(), f.sr);
  return f.tri;
}

void fact_readback(nsmi_ctx* ctx, FactCore& f) {
  f.wh = static_cast<double*>(stage_take(ctx, sizeof(double) * size_t(f.iso)));
  f.info_h = static_cast<int*>(stage_take(ctx, sizeof(int)));
  *f.info_h = 0;
  NSMI_HIP(hipMemcpyAsync(f.info_h, ctx->d_info, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  NSMI_HIP(hipMemcpyAsync(f.wh, f.w->p, sizeof(double) * f.iso, hipMemcpyDeviceToHost, ctx->stream));
}

void fact_syevd(nsmi_ctx* ctx, FactCore& f);

// after the reduction's flags are on the host (a group that never started is launched again
// first, spread): every eigenvalue of T by bisection (descending), copied to the host; the
// eigenvectors wait for the truncation
void fact_tri_solve(nsmi_ctx* ctx, FactCore& f) {
  const int64_t iso = f.iso;
  for (int i = 0; i < kRelaunches && reduction_unplaced(f.sr); ++i) {
    f.tri = sytrd_launch(ctx, f.rho->as<double>(), int(iso), f.w->as<double>(), f.e->as<double>(),
                         f.tau->as<double>(), f.sr, true);
    if (!f.tri) return fact_syevd(ctx, f);
    NSMI_HIP(hipStreamSynchronize(ctx->stream));
  }
  sytrd_check(f.sr);
  f.sr.xch.reset();
  f.lam.reset(new Scratch(ctx, sizeof(double) * size_t(iso)));
  tri_bisect(ctx, f.w->as<double>(), f.e->as<double>(), int(iso), 0, int(iso), f.lam->as<double>());
  f.wh = static_cast<double*>(stage_take(ctx, sizeof(double) * size_t(iso)));
  f.info_h = static_cast<int*>(stage_take(ctx, sizeof(int)));
  *f.info_h = 0;
  NSMI_HIP(hipMemcpyAsync(f.wh, f.lam->p, sizeof(double) * iso, hipMemcpyDeviceToHost, ctx->stream));
}

// svd route: the isometry side as a tall matrix X (its left singular vectors, or its
// right ones when the isometry side is the shorter one), bidiagonalised in one launch,
// then the singular values by bisection on the Golub-Kahan matrix (descending),
// copied to the host.  False, with nothing launched, beyond the kernel's range.  spread: as
// for the reduction's launch.
bool fact_svd_launch(nsmi_ctx* ctx, FactCore& f, bool spread = false) {
  f.bid = false;
  const int64_t m = f.m, nc = f.nc;
  f.want_v = f.iso < f.oth;
  const bool x_is_m = f.rows_trailing ? (nc < m) : (m >= nc);
  f.xr = x_is_m ? m : nc;
  f.xs = x_is_m ? nc : m;
  const int r = int(f.xr), s = int(f.xs);
  if (bidiag_groups(r, s) == 0) return false;
  f.X.reset(new Scratch(ctx, sizeof(double) * size_t(r) * s));
  if (x_is_m)
    NSMI_HIP(hipMemcpyAsync(f.X->p, f.M, sizeof(double) * size_t(r) * s, hipMemcpyDeviceToDevice, ctx->stream));
  else {
    hipLaunchKernelGGL(k_transpose, dim3(blocks(nc, 32), blocks(m, 32)), dim3(32, 8), 0, ctx->stream, f.M, int(m),
                       nc, f.X->as<double>());
    NSMI_LAUNCH_CHECK();
  }
  f.w.reset(new Scratch(ctx, sizeof(double) * size_t(s)));
  f.e.reset(new Scratch(ctx, sizeof(double) * size_t(std::max(s - 1, 1))));
  f.tau.reset(new Scratch(ctx, sizeof(double) * size_t(s)));
  f.tauR.reset(new Scratch(ctx, sizeof(double) * size_t(std::max(s - 1, 1))));
  if (!bidiag_launch(ctx, f.X->as<double>(), r, s, f.w->as<double>(), f.e->as<double>(), f.tau->as<double>(),
                     f.tauR->as<double>(), f.sr, spread)) {
    f.X.reset();
    return false;
  }
  f.gk.reset(new Scratch(ctx, sizeof(double) * size_t(std::max(2 * s - 1, 1))));
  gk_offdiag(ctx, f.w->as<double>(), f.e->as<double>(), s, f.gk->as<double>());
  f.lam.reset(new Scratch(ctx, sizeof(double) * size_t(s)));
  tri_bisect(ctx, nullptr, f.gk->as<double>(), 2 * s, 0, s, f.lam->as<double>());
  f.wh = static_cast<double*>(stage_take(ctx, sizeof(double) * size_t(s)));
  f.info_h = static_cast<int*>(stage_take(ctx, sizeof(int)));
  *f.info_h = 0;
  NSMI_HIP(hipMemcpyAsync(f.wh, f.lam->p, sizeof(double) * s, hipMemcpyDeviceToHost, ctx->stream));
  f.bid = true;
  return true;
}

// synchronises (the finiteness check reads a device flag)
void fact_syevd(nsmi_ctx* ctx, FactCore& f) {
  const int64_t iso = f.iso;
  f.tau.reset();
  require_finite(ctx, f.rho->as<double>(), iso * iso, "factorize");
  {
    ProfScope ps(ctx, NSMI_K_FACT_SOLVE, 9.0 * double(iso) * iso * iso, 0.0);
    check_rocsolver(rocsolver_dsyevd(ctx->blas, rocblas_evect_original, rocblas_fill_upper, rocblas_int(iso),
                                     f.rho->as<double>(), rocblas_int(iso), f.w->as<double>(), f.e->as<double>(),
                                     ctx->d_info),
                    "rocsolver_dsyevd");
  }
  fact_readback(ctx, f);
}

// after the stream has passed fact_readback's copies
void fact_finish(FactCore& f) {
  if (f.bid) {
    sytrd_check(f.sr);
    // P = s^2 of the singular values (descending); the host keeps s in wh
    std::vector<double> w(size_t(f.xs));
    for (int64_t i = 0; i < f.xs; ++i) {
      if (!std::isfinite(f.wh[i])) fail(NSMI_ERR_NOT_FINITE, "factorize: non-finite singular value");
      const double sv = std::max(f.wh[i], 0.0);
      w[size_t(i)] = sv * sv;
    }
    f.order.resize(size_t(f.xs));
    std::iota(f.order.begin(), f.order.end(), 0);
    std::stable_sort(f.order.begin(), f.order.end(), [&](int a, int b) { return w[a] > w[b]; });
    f.P.resize(size_t(f.xs));
    for (int64_t i = 0; i < f.xs; ++i) f.P[size_t(i)] = w[size_t(f.order[size_t(i)])];
    return;
  }
  if (*f.info_h != 0) fail(NSMI_ERR_SOLVER, "rocsolver_dsyevd returned info = " + std::to_string(*f.info_h));
  std::vector<double> w(f.wh, f.wh + f.iso);
  fact_spectrum(f, w);
}

// one factorisation on the main stream
void fact_gram(nsmi_ctx* ctx, FactCore& f) {
  fact_gram_gemm(ctx, f);
  if (f.jacobi) return;
  if (fact_tri_launch(ctx, f)) {
    NSMI_HIP(hipStreamSynchronize(ctx->stream));
    fact_tri_solve(ctx, f);
  } else {
    fact_syevd(ctx, f);
  }
  NSMI_HIP(hipStreamSynchronize(ctx->stream));
  fact_finish(f);
}


// The deferred small Gram matrices of several cores in one batched launch:
// enqueue (eigenvalues and the convergence flag copied to the host), then finish
// after the caller's synchronisation.
void fact_jacobi_launch(nsmi_ctx* ctx, const std::vector<FactCore*>& fs, unsigned* unconverged) {
  std::vector<JacobiJob> jobs;
  for (FactCore* f : fs)
    if (f->jacobi) jobs.push_back(JacobiJob{f->rho->as<double>(), f->wdev->as<double>(), int(f->iso)});
  *unconverged = 0u;
  if (jobs.empty()) return;
  jacobi_eig_batched(ctx, jobs, unconverged);
  for (FactCore* f : fs)
    if (f->jacobi) {
      f->wh = static_cast<double*>(stage_take(ctx, sizeof(double) * size_t(f->iso)));
      NSMI_HIP(hipMemcpyAsync(f->wh, f->wdev->p, sizeof(double) * f->iso, hipMemcpyDeviceToHost, ctx->stream));
    }
}

void fact_jacobi_finish(const std::vector<FactCore*>& fs, unsigned unconverged) {
  if (unconverged) fail(NSMI_ERR_SOLVER, "jacobi: a Gram matrix did not converge within the sweep limit");
  for (FactCore* f : fs)
    if (f->jacobi) {
      std::vector<double> w(f->wh, f->wh + f->iso);
      fact_spectrum(*f, w);
      f->jacobi = false;
    }
}

void fact_jacobi(nsmi_ctx* ctx, const std::vector<FactCore*>& fs) {
  unsigned* unconverged = static_cast<unsigned*>(stage_take(ctx, sizeof(unsigned)));
  fact_jacobi_launch(ctx, fs, unconverged);
  NSMI_HIP(hipStreamSynchronize(ctx->stream));
  fact_jacobi_finish(fs, *unconverged);
}

void fact_prepare(nsmi_ctx* ctx, FactCore& f) {
  if (f.route == NSMI_ROUTE_SVD) {
    bool launched = fact_svd_launch(ctx, f);
    if (launched) NSMI_HIP(hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < kRelaunches && launched && reduction_unplaced(f.sr); ++i) {
      launched = fact_svd_launch(ctx, f, true);
      if (launched) NSMI_HIP(hipStreamSynchronize(ctx->stream));
    }
    if (launched) {
      f.sr.xch.reset();  // up to 13 MB over all XCDs; the vectors' solves that follow need the most
      fact_finish(f);
      return;
    }
    f.svd_declined = true;
  }
  fact_gram(ctx, f);
  if (f.jacobi) fact_jacobi(ctx, {&f});
}

// after the caller's closing synchronisation: the orthonormalisation's flag
void fact_emit_check(const FactCore& f) {
  if (f.orth_h && *f.orth_h)
    fail(NSMI_ERR_SOLVER, "factorize: the inverse-iteration vectors are not numerically independent");
}

// U / C for the first k entries of the sorted spectrum (U m x k and C k x nc, or
// U k x nc and C m x k when rows_trailing), columns of the isometry in the
// "largest-magnitude entry positive" gauge.
void fact_emit(nsmi_ctx* ctx, FactCore& f, int64_t k, double* U, double* C) {
  if (k == 0) return;
  const int64_t m = f.m, nc = f.nc, iso = f.iso;
  Scratch d_sgn(ctx, sizeof(double) * size_t(std::max<int64_t>(k, 1)));
  Scratch d_idx(ctx, sizeof(int) * size_t(k));
  // eigenvectors: column-major iso x iso = row-major rows are eigenvectors
  const double* vecs = f.rho ? f.rho->as<double>() : nullptr;  // the svd route has no Gram matrix
  const int* vidx = d_idx.as<int>();
  std::unique_ptr<Scratch> zk;
  {
    int* hidx = static_cast<int*>(stage_take(ctx, sizeof(int) * size_t(k)));
    std::memcpy(hidx, f.order.data(), sizeof(int) * size_t(k));
    NSMI_HIP(hipMemcpyAsync(d_idx.p, hidx, sizeof(int) * k, hipMemcpyHostToDevice, ctx->stream));
    if (f.tri || f.bid) {
      // the kept eigenvalues (tri) or singular values (bid), in the kept order; their
      // vectors by inverse iteration (tridiagonal T, or the Golub-Kahan matrix of B:
      // its odd entries are u, its even ones v), made orthonormal, then back-transformed
      // through the Householder reflectors
      double* hl = static_cast<double*>(stage_take(ctx, sizeof(double) * size_t(k)));
      for (int64_t i = 0; i < k; ++i) hl[i] = f.wh[f.order[size_t(i)]];
      Scratch lamk(ctx, sizeof(double) * size_t(k));
      NSMI_HIP(hipMemcpyAsync(lamk.p, hl, sizeof(double) * k, hipMemcpyHostToDevice, ctx->stream));
      const int64_t len = f.bid ? f.xs : iso;  // length of the vectors of T
      Scratch Y(ctx, sizeof(double) * size_t(len) * k);
      if (f.bid)
        tri_invit(ctx, nullptr, f.gk->as<double>(), int(2 * f.xs), lamk.as<double>(), int(k), Y.as<double>(),
                  f.want_v ? 0 : 1);
      else
        tri_invit(ctx, f.w->as<double>(), f.e->as<double>(), int(iso), lamk.as<double>(), int(k), Y.as<double>(), -1);
      unsigned* ofail = f.sr.flags->as<unsigned>() + kCtlOrthFail;
      orthonormalize_cols(ctx, Y.as<double>(), len, int(k), ofail);
      f.orth_h = static_cast<unsigned*>(stage_take(ctx, sizeof(unsigned)));
      *f.orth_h = 0u;
      NSMI_HIP(hipMemcpyAsync(f.orth_h, ofail, sizeof(unsigned), hipMemcpyDeviceToHost, ctx->stream));
      ProfScope ps2(ctx, NSMI_K_FACT_SOLVE, 2.0 * double(iso) * len * (2.0 * k + len), 0.0);
      zk.reset(new Scratch(ctx, sizeof(double) * size_t(k) * iso));
      hipLaunchKernelGGL(k_transpose_pad, dim3(blocks(k * iso)), dim3(256), 0, ctx->stream, Y.as<double>(), len,
                         int(k), iso, zk->as<double>());
      NSMI_LAUNCH_CHECK();
      if (f.tri) {
        if (iso > 1) apply_q_lower(ctx, f.rho->as<double>(), f.tau->as<double>(), int(iso), zk->as<double>(), int(k));
      } else if (f.want_v) {
        // X's right singular vectors: V = G_0 ... G_{s-2} [v_B]
        if (f.xs > 1) {
          Scratch vt(ctx, sizeof(double) * size_t(f.xs - 1) * f.xs);
          bidiag_reflectors_right(ctx, f.X->as<double>(), int(f.xs), f.tauR->as<double>(), vt.as<double>());
          apply_reflectors(ctx, vt.as<double>(), f.tauR->as<double>(), int(f.xs - 1), f.xs, zk->as<double>(), int(k));
        }
      } else {
        // X's left singular vectors: U = H_0 ... H_{s-1} [u_B; 0]
        Scratch vt(ctx, sizeof(double) * size_t(f.xs) * f.xr);
        bidiag_reflectors_left(ctx, f.X->as<double>(), int(f.xr), int(f.xs), f.tau->as<double>(), vt.as<double>());
        apply_reflectors(ctx, vt.as<double>(), f.tau->as<double>(), int(f.xs), f.xr, zk->as<double>(), int(k));
      }
      vecs = zk->as<double>();
      vidx = nullptr;
    }
  }
  ProfScope ps(ctx, NSMI_K_FACT_GEMM, 2.0 * double(k) * m * nc, 8.0 * (double(m) * nc + double(k) * (m + nc)));
  {
    hipLaunchKernelGGL(k_gauge_sign, dim3(unsigned(k)), dim3(256), 0, ctx->stream, vecs, iso, iso, 1, vidx,
                       d_sgn.as<double>());
    NSMI_LAUNCH_CHECK();
    Scratch Ut(ctx, sizeof(double) * size_t(k) * iso);
    hipLaunchKernelGGL(k_gather_rows, dim3(blocks(k * iso)), dim3(256), 0, ctx->stream, vecs, iso, vidx, int(k), iso,
                       d_sgn.as<double>(), (const double*)nullptr, Ut.as<double>());
    NSMI_LAUNCH_CHECK();
    if (!f.rows_trailing) {
      // U (m x k) = Ut^T ; C (k x nc) = Ut . M
      hipLaunchKernelGGL(k_transpose, dim3(blocks(m, 32), blocks(k, 32)), dim3(32, 8), 0, ctx->stream,
                         Ut.as<double>(), int(k), m, U);
      NSMI_LAUNCH_CHECK();
      gemm_f64(ctx, gdesc(k, nc, m, false, false), 1.0, Ut.as<double>(), f.M, 0.0, C, kRoleFact);
    } else {
      // U (k x nc) = Ut ; C (m x k) = M . Ut^T
      NSMI_HIP(hipMemcpyAsync(U, Ut.p, sizeof(double) * k * nc, hipMemcpyDeviceToDevice, ctx->stream));
      gemm_f64(ctx, gdesc(m, k, nc, false, true), 1.0, f.M, Ut.as<double>(), 0.0, C, kRoleFact);
    }
    // the index copy above reads pinned stage memory, which stays untouched until the
    // next entry point resets the stage after this call's closing synchronisation
  }
}

}  // namespace
}  // namespace nsmi

extern "C" {


int nsmi_factorize(nsmi_ctx* ctx, const nsmi_tensor* theta, int n_row_dims, int rows_trailing,
                   const nsmi_trunc* trunc, nsmi_tensor** Uout, nsmi_tensor** Cout, nsmi_trunc_info* info) {
  if (!ctx || !theta || !trunc || !Uout || !Cout) return NSMI_ERR_INVALID;
  API_BEGIN(ctx)
  stage_reset(ctx);
  *Uout = nullptr;
  *Cout = nullptr;
  require(theta->dtype == NSMI_F64 || theta->dtype == NSMI_C128, "factorize: unknown element type");
  require(n_row_dims >= 1 && n_row_dims < theta->rank, "factorize: n_row_dims must split theta's dims");
  int64_t m = 1, nc = 1;  // M = theta viewed as m x nc (leading dims x trailing dims)
  for (int i = 0; i < n_row_dims; ++i) m *= theta->dims[i];
  for (int i = n_row_dims; i < theta->rank; ++i) nc *= theta->dims[i];
  require(m >= 1 && nc >= 1, "factorize: empty tensor");
  require(m < (int64_t(1) << 31) && nc < (int64_t(1) << 31), "factorize: matrix too large");
  // the isometry side: rows of M (rows_trailing == 0) or columns of M
  const int64_t iso = rows_trailing ? nc : m, oth = rows_trailing ? m : nc;
  const int64_t full = std::min(m, nc);
  int64_t maxdim = trunc->maxdim > 0 ? std::min<int64_t>(trunc->maxdim, full) : full;
  const int64_t mindim = trunc->mindim > 0 ? trunc->mindim : 1;
  int route = trunc->route;
  if (route == NSMI_ROUTE_AUTO) route = (trunc->cutoff <= 1e-12) ? NSMI_ROUTE_SVD : NSMI_ROUTE_EIGEN;
  require(route == NSMI_ROUTE_SVD || route == NSMI_ROUTE_EIGEN, "factorize: unknown route");
  if (theta->dtype == NSMI_C128) {
    int64_t kk = 0;
    double te = 0.0, tot = 0.0;
    zfactorize(ctx, theta, n_row_dims, rows_trailing, trunc, route, maxdim, mindim, Uout, Cout, &kk, &te, &tot,
               truncate_spectrum);
    if (info) {
      info->kept = kk;
      info->full = full;
      info->truncerr = te;
      info->total = tot;
      info->route = route;
    }
    return NSMI_OK;
  }
  FactCore fc(static_cast<const double*>(theta->data), m, nc, rows_trailing != 0, route);
  fact_prepare(ctx, fc);
  double truncerr = 0.0, total = 0.0;
  std::vector<double> P = fc.P;
  const int64_t k = truncate_spectrum(P, mindim, maxdim, trunc->cutoff, &truncerr, &total);
  int64_t udims[8], cdims[8];
  int ur = 0, cr = 0;
  if (!rows_trailing) {
    for (int i = 0; i < n_row_dims; ++i) udims[ur++] = theta->dims[i];
    udims[ur++] = k;
    cdims[cr++] = k;
    for (int i = n_row_dims; i < theta->rank; ++i) cdims[cr++] = theta->dims[i];
  } else {
    udims[ur++] = k;
    for (int i = n_row_dims; i < theta->rank; ++i) udims[ur++] = theta->dims[i];
    for (int i = 0; i < n_row_dims; ++i) cdims[cr++] = theta->dims[i];
    cdims[cr++] = k;
  }
  nsmi_tensor* U = tensor_new(ctx, NSMI_F64, ur, udims);
  nsmi_tensor* C = nullptr;
  try {
    C = tensor_new(ctx, NSMI_F64, cr, cdims);
    fact_emit(ctx, fc, k, static_cast<double*>(U->data), static_cast<double*>(C->data));
  } catch (...) {
    tensor_delete(ctx, U);
    if (C) tensor_delete(ctx, C);
    throw;
  }
  *Uout = U;
  *Cout = C;
  if (info) {
    info->kept = k;
    info->full = full;
    info->truncerr = truncerr;
    info->total = total;
    info->route = fc.svd_declined ? NSMI_ROUTE_EIGEN : route;
  }
  // scratch blocks are returned to the pool in stream order; the host vectors
  // copied above were synchronised already
  NSMI_HIP(hipStreamSynchronize(ctx->stream));
  stage_done(ctx);
  try {
    fact_emit_check(fc);
  } catch (...) {
    tensor_delete(ctx, *Uout);
    tensor_delete(ctx, *Cout);
    *Uout = *Cout = nullptr;
    throw;
  }
  API_END(ctx)
}

int nsmi_qr(nsmi_ctx* ctx, const nsmi_tensor* A, int n_row_dims, int rows_trailing, nsmi_tensor** Qout,
            nsmi_tensor** Rout) {
  if (!ctx || !A || !Qout || !Rout) return NSMI_ERR_INVALID;
  API_BEGIN(ctx)
  *Qout = nullptr;
  *Rout = nullptr;
  require(A->dtype == NSMI_F64 || A->dtype == NSMI_C128, "qr: unknown element type");
  require(n_row_dims >= 1 && n_row_dims < A->rank, "qr: n_row_dims must split A's dims");
  if (A->dtype == NSMI_C128) {
    zqr(ctx, A, n_row_dims, rows_trailing, Qout, Rout);
    return NSMI_OK;
  }
  int64_t m = 1, nc = 1;
  for (int i = 0; i < n_row_dims; ++i) m *= A->dims[i];
  for (int i = n_row_dims; i < A->rank; ++i) nc *= A->dims[i];
  // factor X = Q R where X = M (rows_trailing == 0) or M^T
  const int64_t xr = rows_trailing ? nc : m, xc = rows_trailing ? m : nc;
  const int64_t r = std::min(xr, xc);
  int64_t qd[8], rd[8];
  int qr = 0, rr = 0;
  if (!rows_trailing) {
    for (int i = 0; i < n_row_dims; ++i) qd[qr++] = A->dims[i];
    qd[qr++] = r;
    rd[rr++] = r;
    for (int i = n_row_dims; i < A->rank; ++i) rd[rr++] = A->dims[i];
  } else {
    qd[qr++] = r;
    for (int i = n_row_dims; i < A->rank; ++i) qd[qr++] = A->dims[i];
    for (int i = 0; i < n_row_dims; ++i) rd[rr++] = A->dims[i];
    rd[rr++] = r;
  }
  nsmi_tensor* Q = tensor_new(ctx, NSMI_F64, qr, qd);
  nsmi_tensor* R = tensor_new(ctx, NSMI_F64, rr, rd);
  try {
    // small matrices: the one-workgroup Householder QR (one launch)
    if (qr_one(ctx, static_cast<const double*>(A->data), m, nc, rows_trailing != 0, false,
               static_cast<double*>(Q->data), static_cast<double*>(R->data))) {
      NSMI_HIP(hipStreamSynchronize(ctx->stream));
      *Qout = Q;
      *Rout = R;
      return NSMI_OK;
    }
    Scratch a(ctx, sizeof(double) * size_t(m) * nc);
    Scratch tau(ctx, sizeof(double) * size_t(std::max<int64_t>(r, 1)));
    Scratch sg(ctx, sizeof(double) * size_t(std::max<int64_t>(r, 1)));
    NSMI_HIP(hipMemcpyAsync(a.p, A->data, sizeof(double) * m * nc, hipMemcpyDeviceToDevice, ctx->stream));
    if (!rows_trailing) {
      // row-major M (m x nc) = col-major M^T (nc x m); LQ of M^T: M^T = L Qt -> M = Qt^T L^T
      check_rocsolver(rocsolver_dgelqf(ctx->blas, rocblas_int(nc), rocblas_int(m), a.as<double>(), rocblas_int(nc),
                                       tau.as<double>()),
                      "rocsolver_dgelqf");
      // L (col-major nc x r, lower) read row-major: first r rows of the m x nc buffer, keep j >= i
      hipLaunchKernelGGL(k_diag_sign, dim3(blocks(r)), dim3(256), 0, ctx->stream, a.as<double>(), nc, r,
                         sg.as<double>());
      NSMI_LAUNCH_CHECK();
      hipLaunchKernelGGL(k_extract_tri, dim3(blocks(r * nc)), dim3(256), 0, ctx->stream, a.as<double>(), nc, r, nc,
                         sg.as<double>(), static_cast<double*>(R->data), 0);
      NSMI_LAUNCH_CHECK();
      // Qt (r x m col-major) read row-major = Q (m x r)
      check_rocsolver(rocsolver_dorglq(ctx->blas, rocblas_int(r), rocblas_int(m), rocblas_int(r), a.as<double>(),
                                       rocblas_int(nc), tau.as<double>()),
                      "rocsolver_dorglq");
      // dorglq leaves Qt in the leading r rows (ld = nc) of the col-major buffer;
      // as row-major it is m rows of stride nc, first r columns
      hipLaunchKernelGGL(k_gather_cols, dim3(blocks(r * m)), dim3(256), 0, ctx->stream, a.as<double>(), nc,
                         (const int*)nullptr, int(r), m, sg.as<double>(), (const double*)nullptr,
                         static_cast<double*>(Q->data));
      NSMI_LAUNCH_CHECK();
    } else {
      // X = M^T (nc x m) is col-major M (m x nc) read as... use QR of col-major M^T? The row-major
      // buffer (m x nc) is col-major (nc x m) = M^T = X directly: QR of X.
      check_rocsolver(rocsolver_dgeqrf(ctx->blas, rocblas_int(nc), rocblas_int(m), a.as<double>(), rocblas_int(nc),
                                       tau.as<double>()),
                      "rocsolver_dgeqrf");
      // R (col-major r x m, upper): element (i, j) at a[i + j*nc] = row-major (m x nc)[j][i];
      // we need R^T (m x r row-major): R^T[j][i] = a[j*nc + i] for i <= j
      hipLaunchKernelGGL(k_diag_sign, dim3(blocks(r)), dim3(256), 0, ctx->stream, a.as<double>(), nc, r,
                         sg.as<double>());
      NSMI_LAUNCH_CHECK();
      // rows j of the row-major buffer, entries i <= min(j, r-1); write R^T with sign on column i
      hipLaunchKernelGGL(k_extract_tri_t, dim3(blocks(r * m)), dim3(256), 0, ctx->stream, a.as<double>(), nc, r, m,
                         sg.as<double>(), static_cast<double*>(R->data));
      NSMI_LAUNCH_CHECK();
      check_rocsolver(rocsolver_dorgqr(ctx->blas, rocblas_int(nc), rocblas_int(r), rocblas_int(r), a.as<double>(),
                                       rocblas_int(nc), tau.as<double>()),
                      "rocsolver_dorgqr");
      // Q (col-major nc x r) read row-major = Q^T (r x nc): the site tensor; rows get the signs
      NSMI_HIP(hipMemcpyAsync(Q->data, a.p, sizeof(double) * r * nc, hipMemcpyDeviceToDevice, ctx->stream));
      hipLaunchKernelGGL(k_scale_rows, dim3(blocks(r * nc)), dim3(256), 0, ctx->stream, static_cast<double*>(Q->data),
                         r, nc, sg.as<double>());
      NSMI_LAUNCH_CHECK();
    }
    NSMI_HIP(hipStreamSynchronize(ctx->stream));
  } catch (...) {
    tensor_delete(ctx, Q);
    tensor_delete(ctx, R);
    throw;
  }
  *Qout = Q;
  *Rout = R;
  API_END(ctx)
}

// Block-diagonal (quantum-number) factorisation: every sector matrix M[q] is
// decomposed as nsmi_factorize would, the sector spectra are merged and truncated
// together (NDTensors truncate! on the concatenated, sorted spectrum), and each
// sector keeps the entries above the cut value docut (NDTensors' block-sparse
// svd/eigen): the midpoint between the last kept and first discarded values, moved
// up by 1e-3 of the last kept value when the two are nearly degenerate, so a
// near-degenerate pair is kept or dropped together.
int nsmi_factorize_sectors(nsmi_ctx* ctx, const nsmi_tensor* Mall, int n, const int64_t* offsets, const int64_t* rows,
                           const int64_t* cols, int rows_trailing, const nsmi_trunc* trunc, nsmi_tensor** Uall,
                           nsmi_tensor** Call, int64_t* kept, nsmi_trunc_info* info) {
  if (!ctx || !Mall || n < 0 || (n > 0 && (!offsets || !rows || !cols || !kept)) || !trunc || !Uall || !Call)
    return NSMI_ERR_INVALID;
  std::vector<nsmi_tensor*> made;
  API_BEGIN(ctx)
  stage_reset(ctx);
  *Uall = nullptr;
  *Call = nullptr;
  require(Mall->dtype == NSMI_F64, "factorize_sectors: sector matrices are FP64");
  for (int q = 0; q < n; ++q) {
    kept[q] = 0;
    require(rows[q] >= 1 && cols[q] >= 1 && offsets[q] >= 0 && offsets[q] + rows[q] * cols[q] <= Mall->numel,
            "factorize_sectors: sector matrix outside the buffer");
  }
  int route = trunc->route;
  if (route == NSMI_ROUTE_AUTO) route = (trunc->cutoff <= 1e-12) ? NSMI_ROUTE_SVD : NSMI_ROUTE_EIGEN;
  require(route == NSMI_ROUTE_SVD || route == NSMI_ROUTE_EIGEN, "factorize_sectors: unknown route");
  std::vector<std::unique_ptr<FactCore>> fc;
  int64_t full = 0;
  std::vector<FactCore*> fcp, big, lib;
  for (int q = 0; q < n; ++q) {
    fc.emplace_back(new FactCore(static_cast<const double*>(Mall->data) + offsets[q], rows[q], cols[q],
                                 rows_trailing != 0, route));
    fact_gram_gemm(ctx, *fc.back());
    fcp.push_back(fc.back().get());
    full += fc.back()->full;
    if (!fc.back()->jacobi) big.push_back(fc.back().get());
  }
  // The sectors are independent: every small one goes into one batched Jacobi
  // launch on the main stream, and the reductions and divide-and-conquer solves of
  // the larger ones are spread over auxiliary streams (each solve is a chain of
  // latency-bound launches, so several overlap on the device); a sector whose
  // reduction cannot run takes dsyevd on the main stream.
  const int naux = int(std::min<size_t>(big.size(), kAuxStreams));
  std::unique_ptr<AuxSection> sec;
  if (naux > 1) {
    sec.reset(new AuxSection(ctx, naux));
    sec->fork();
  }
  auto on_stream = [&](size_t t, const std::function<void()>& fn) {
    if (sec) {
      OnAux a(ctx, int(t % size_t(naux)));
      fn();
    } else {
      fn();
    }
  };
  auto sync_all = [&]() {
    if (sec)
      sec->sync();
    else
      NSMI_HIP(hipStreamSynchronize(ctx->stream));
  };
  for (size_t t = 0; t < big.size(); ++t)
    on_stream(t, [&]() {
      if (!fact_tri_launch(ctx, *big[t])) lib.push_back(big[t]);
    });
  unsigned* unconverged = static_cast<unsigned*>(stage_take(ctx, sizeof(unsigned)));
  fact_jacobi_launch(ctx, fcp, unconverged);
  sync_all();
  for (size_t t = 0; t < big.size(); ++t)
    if (big[t]->tri) on_stream(t, [&]() { fact_tri_solve(ctx, *big[t]); });
  for (FactCore* f : lib) fact_syevd(ctx, *f);
  sync_all();
  fact_jacobi_finish(fcp, *unconverged);
  for (FactCore* f : big) fact_finish(*f);
  auto key = [&](double v) { return route == NSMI_ROUTE_EIGEN ? std::fabs(v) : v; };
  struct Entry {
    double key, value;
    int q, i;
  };
  std::vector<Entry> all;
  for (int q = 0; q < n; ++q)
    for (size_t i = 0; i < fc[q]->P.size(); ++i) all.push_back(Entry{key(fc[q]->P[i]), fc[q]->P[i], q, int(i)});
  std::stable_sort(all.begin(), all.end(), [](const Entry& a, const Entry& b) { return a.key > b.key; });
  std::vector<double> P(all.size());
  for (size_t i = 0; i < all.size(); ++i) P[i] = all[i].value;
  const int64_t maxdim = trunc->maxdim > 0 ? std::min<int64_t>(trunc->maxdim, full) : full;
  const int64_t mindim = trunc->mindim > 0 ? trunc->mindim : 1;
  double truncerr = 0.0, total = 0.0;
  const int64_t origm = int64_t(P.size());
  const int64_t nk = truncate_spectrum(P, mindim, maxdim, trunc->cutoff, &truncerr, &total);
  int64_t sum = 0;
  if (nk < origm) {
    double docut = (P[nk - 1] + P[nk]) / 2;
    if (std::fabs(P[nk - 1] - P[nk]) < 1e-3 * P[nk - 1]) docut += 1e-3 * P[nk - 1];
    for (size_t i = 0; i < all.size(); ++i)
      if (P[i] > docut) ++kept[all[i].q];
  } else {
    for (int q = 0; q < n; ++q) kept[q] = int64_t(fc[q]->P.size());
  }
  for (int q = 0; q < n; ++q) sum += kept[q];
  if (sum == 0 && !all.empty()) {  // keep at least the largest entry
    kept[all[0].q] = 1;
    sum = 1;
  }
  // U_q (rows x k, or k x cols when rows_trailing) and C_q concatenated in sector order
  int64_t usz = 0, csz = 0;
  for (int q = 0; q < n; ++q) {
    usz += kept[q] * (rows_trailing ? cols[q] : rows[q]);
    csz += kept[q] * (rows_trailing ? rows[q] : cols[q]);
  }
  const int64_t ud[1] = {std::max<int64_t>(usz, 1)}, cd[1] = {std::max<int64_t>(csz, 1)};
  nsmi_tensor* Ut = tensor_new(ctx, NSMI_F64, 1, ud);
  made.push_back(Ut);
  nsmi_tensor* Ct = tensor_new(ctx, NSMI_F64, 1, cd);
  made.push_back(Ct);
  int64_t uo = 0, co = 0;
  if (sec) sec->fork();  // the outputs were allocated on the main stream
  size_t t = 0;
  for (int q = 0; q < n; ++q) {
    const int64_t k = kept[q];
    if (k == 0) continue;
    double* U = static_cast<double*>(Ut->data) + uo;
    double* C = static_cast<double*>(Ct->data) + co;
    on_stream(t++, [&]() { fact_emit(ctx, *fc[q], k, U, C); });
    uo += k * (rows_trailing ? cols[q] : rows[q]);
    co += k * (rows_trailing ? rows[q] : cols[q]);
  }
  if (sec) sec->join();
  if (info) {
    info->kept = sum;
    info->full = full;
    info->truncerr = truncerr;
    info->total = total;
    info->route = NSMI_ROUTE_EIGEN;  // every sector goes through its Gram matrix
  }
  NSMI_HIP(hipStreamSynchronize(ctx->stream));
  stage_done(ctx);
  for (auto& f : fc) fact_emit_check(*f);
  *Uall = Ut;
  *Call = Ct;
  made.clear();
  }
  catch (const nsmi::Error& e) {
    for (auto* t : made) tensor_delete(ctx, t);
    ctx->err = e.what();
    return e.code;
  }
  catch (const std::exception& e) {
    for (auto* t : made) tensor_delete(ctx, t);
    ctx->err = std::string("internal: ") + e.what();
    return NSMI_ERR_INVALID;
  }
  return NSMI_OK;
}

}  // extern "C"
