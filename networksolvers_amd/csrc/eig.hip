// Symmetric tridiagonalisation of the truncation's Gram matrix rho (n x n) in one launch
// (the eigensolver behind inserter.jl:23 -> ITensors eigen/svd -> LAPACK syevd): the
// kernel is k_sytrd (sytrd.h), its plans and launch below; the batched Jacobi solver for
// small Gram matrices; and the compact-WY back-transformation of the kept vectors.
#include "internal.h"
#include "places.h"
#include "sytrd.h"
#include "wave.h"

namespace nsmi {
namespace {

struct TriPlan {
  const void* fn = nullptr;
  int cl = 1, threads = 0, rows = 0;  // rows per workgroup
  bool spread = false;                // over all XCDs
};
template <int NMAX, int CL, int RW, int NW, bool SHARED>
TriPlan tri_plan_of() {
  constexpr bool kSpread = CL > 8;  // as the kernel's register bound
  static_assert(NMAX <= 64 * CL && (kSpread || NMAX <= XcdPlaces<hipStream_t>::kCusPerXcd * RW * NW),
                "at most one workgroup for each CU of an XCD");
  return {reinterpret_cast<const void*>(k_sytrd<CL, RW, NW, SHARED>), CL, 64 * NW, RW * NW, kSpread};
}

// Measured on gfx950 (us per column; the grid-barrier form on up to 16 spread workgroups
// that these plans replaced: 2.4 at n = 64, 3.4 at 128, 3.9 at 256, 5.2-5.7 at 384-448, 10 at
// 1000): one row per wave 1.05 at n = 64 (2 rows 1.18, 4 rows 1.48) and 1.19 at 128 (1.31,
// 1.61); two rows 1.5 at 154 and 1.56 at 256 (four 1.9; the words shared through LDS 1.67);
// four rows 2.5 at 400 and 512 (two on eight waves 3.3: registers).  Above 512 columns a
// row takes 16 registers a lane and one XCD's 32 workgroups hold the matrix only with
// spills (4.8 at 700, 9 at 1000), so the group spreads over all XCDs: 3.3 at 513, 3.7 at
// 700, 4.3 at 1000.
TriPlan tri_plan(int n) {
  if (n <= 64) return tri_plan_of<64, 1, 1, 4, false>();
  if (n <= 128) return tri_plan_of<128, 2, 1, 4, false>();
  if (n <= 256) return tri_plan_of<256, 4, 2, 4, false>();
  if (n <= 512) return tri_plan_of<512, 8, 4, 4, false>();
  return tri_plan_of<kSytrdMax, 16, 2, 4, true>();
}

// ---- batched Jacobi eigensolver for small Gram matrices ---------------------
//
// One workgroup per symmetric matrix (n <= NP), matrix and eigenvector
// accumulator resident in LDS.  Cyclic two-sided Jacobi in round-robin
// ("chess tournament") order: the m = n + (n odd) indices form m/2 disjoint
// pairs per round (a padded index is a zero row and column, so it never
// rotates), m - 1 rounds cover every pair once per sweep.  The rotations of a
// round commute, so they are applied together: columns of A and V, then rows of
// A.  A pair rotates when |a_pq| > eps ||A||_F (the Frobenius norm is invariant),
// with the classical angle (t = sgn(theta) / (|theta| + sqrt(theta^2 + 1)),
// theta = (a_qq - a_pp) / (2 a_pq)), and its a_pq is then set to zero.  A sweep
// without a rotation ends the solve.  Output in LAPACK dsyevd's layout: the
// eigenvectors overwrite A column-major (column j = vector of eigenvalue w[j]),
// eigenvalues unsorted.
struct JacobiItem {
  double* a;  // n x n, symmetric; overwritten by the eigenvectors
  double* w;  // n eigenvalues
  int n, pad;
};

template <int NP>
__global__ __launch_bounds__(256) void k_jacobi_eig(const JacobiItem* __restrict__ items, int max_sweeps,
                                                    unsigned* __restrict__ unconverged) {
  __shared__ double A[NP][NP + 1];
  __shared__ double V[NP][NP + 1];
  __shared__ double cs[NP / 2], sn[NP / 2];
  __shared__ int pp[NP / 2], qq[NP / 2];
  __shared__ double red[4];
  __shared__ int s_rot;
  const JacobiItem it = items[blockIdx.x];
  const int n = it.n, m = n + (n & 1), half = m / 2, tid = threadIdx.x;
  double nrm = 0.0;
  for (int e = tid; e < m * m; e += 256) {
    const int i = e / m, j = e % m;
    const double v = (i < n && j < n) ? it.a[size_t(i) * n + j] : 0.0;
    A[i][j] = v;
    V[i][j] = (i == j) ? 1.0 : 0.0;
    nrm += v * v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) nrm += __shfl_down(nrm, o, 64);
  if ((tid & 63) == 0) red[tid >> 6] = nrm;
  __syncthreads();
  const double tol = 2.220446049250313e-16 * sqrt(red[0] + red[1] + red[2] + red[3]);
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    if (tid == 0) s_rot = 0;
    __syncthreads();
    for (int r = 0; r + 1 < m; ++r) {
      if (tid < half) {
        const int a = tid == 0 ? r : (r + tid) % (m - 1);
        const int b = tid == 0 ? m - 1 : (r - tid + m - 1) % (m - 1);
        const int p = a < b ? a : b, q = a < b ? b : a;
        const double apq = A[p][q];
        double c = 1.0, s = 0.0;
        if (fabs(apq) > tol) {
          const double theta = (A[q][q] - A[p][p]) / (2.0 * apq);
          double t = fabs(theta) > 1e150 ? 0.5 / fabs(theta) : 1.0 / (fabs(theta) + sqrt(theta * theta + 1.0));
          if (theta < 0.0) t = -t;
          c = 1.0 / sqrt(t * t + 1.0);
          s = t * c;
          s_rot = 1;
        }
        pp[tid] = p;
        qq[tid] = q;
        cs[tid] = c;
        sn[tid] = s;
      }
      __syncthreads();
      // columns p, q of A and V (items: pair k, row i; NP is a power of two)
      for (int e = tid; e < half * NP; e += 256) {
        const int k = e / NP, i = e % NP;
        const double s = sn[k];
        if (i >= m || s == 0.0) continue;
        const double c = cs[k];
        const int p = pp[k], q = qq[k];
        const double aip = A[i][p], aiq = A[i][q];
        A[i][p] = c * aip - s * aiq;
        A[i][q] = s * aip + c * aiq;
        const double vip = V[i][p], viq = V[i][q];
        V[i][p] = c * vip - s * viq;
        V[i][q] = s * vip + c * viq;
      }
      __syncthreads();
      // rows p, q of A (items: pair k, column j); the rotated pair's a_pq, a_qp become 0
      for (int e = tid; e < half * NP; e += 256) {
        const int k = e / NP, j = e % NP;
        const double s = sn[k];
        if (j >= m || s == 0.0) continue;
        const double c = cs[k];
        const int p = pp[k], q = qq[k];
        const double apj = A[p][j], aqj = A[q][j];
        A[p][j] = j == q ? 0.0 : c * apj - s * aqj;
        A[q][j] = j == p ? 0.0 : s * apj + c * aqj;
      }
      __syncthreads();
    }
    const int rot = s_rot;
    __syncthreads();
    if (!rot) break;
  }
  if (sweep == max_sweeps && tid == 0) atomicOr(unconverged, 1u);
  for (int e = tid; e < n * n; e += 256) {
    const int j = e / n, i = e % n;
    it.a[e] = V[i][j];
  }
  for (int i = tid; i < n; i += 256) it.w[i] = A[i][i];
}


// ---- back-transformation Q . Z (Q = H_0 H_1 ... H_{n-2} from the reduction) ---------
// Compact-WY form with the UT transform (Joffrain et al., "Accumulating Householder
// transformations, revisited", ACM TOMS 32, 2006): Q = I - V S^{-1} V^T, with V the
// n x (n-1) matrix of reflector vectors and S upper triangular, S_ii = 1 / tau_i,
// S_ij = v_i . v_j (i < j).  Hence Q Z = Z - V X with S X = V^T Z: two GEMMs for
// V^T Z and V^T V, one triangular solve, one GEMM for the update.  A reflector with
// tau = 0 is the identity: its row of V^T is zero and S_ii = 1, so it drops out.

// Vt (m x n, row-major; m = n - 1): row i is v_i -- zero up to i, 1 at i + 1, then the
// stored A(i+2:n, i), which in the row-major buffer of the column-major view is
// rho[i n + r]
__global__ void k_build_vt(const double* __restrict__ rho, const double* __restrict__ tau, int n,
                           double* __restrict__ Vt) {
  const int64_t m = n - 1;
  const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (e >= m * n) return;
  const int64_t i = e / n, r = e % n;
  double v = 0.0;
  if (tau[i] != 0.0) v = r <= i ? 0.0 : (r == i + 1 ? 1.0 : rho[i * n + r]);
  Vt[e] = v;
}


// X <- S^{-1} X in place (X: m x k row-major), S from G = V^T V (strict upper part
// read; G is symmetric, so G[j][i] is read as G[i][j] wherever that makes the reads
// contiguous across lanes) and tau.  One workgroup per kUtCols columns of X, held in
// LDS with tau; back substitution by blocks of kUtRows rows from the bottom: wave 0
// solves the block's triangle in registers (lane a = row a of the block with its row
// of S, fully unrolled, each pivot broadcast by readlane), then all waves subtract the
// block's contribution from the rows above (one row of X per thread, coalesced reads
// of G, all of a block's loads issued before the first is used).  Wave 0 loads the
// next block's rows of S before that update, so their latency overlaps it.
constexpr int kUtCols = 4, kUtRows = 32, kUtMaxM = 2048;
__global__ __launch_bounds__(256) void k_ut_solve(const double* __restrict__ G, const double* __restrict__ tau,
                                                  double* __restrict__ X, int m, int k) {
  __shared__ double xs[(kUtMaxM + 1) * kUtCols];
  __shared__ double ts[kUtMaxM + 1];
  const int tid = threadIdx.x;
  const int c0 = blockIdx.x * kUtCols;
  const int nc = min(kUtCols, k - c0);
  for (int e = tid; e < m * kUtCols; e += 256) {
    const int i = e / kUtCols, c = e % kUtCols;
    xs[e] = c < nc ? X[int64_t(i) * k + c0 + c] : 0.0;
  }
  for (int i = tid; i < m; i += 256) ts[i] = tau[i];
  // row a = tid of the block's strict upper triangle: S[r0 + a][r0 + b] = G[r0 + b][r0 + a], b > a
  double srow[kUtRows];
  auto load_srow = [&](int r0, int bs) {
#pragma unroll
    for (int b = 0; b < kUtRows; ++b)
      srow[b] = (tid < bs && b < bs && b > tid) ? G[int64_t(r0 + b) * m + r0 + tid] : 0.0;
  };
  int r1 = m, r0 = max(0, m - kUtRows);
  if (tid < 64) load_srow(r0, r1 - r0);
  __syncthreads();
  while (r1 > 0) {
    const int bs = r1 - r0;
    if (tid < 64) {
      const int a = tid;
      double xa[kUtCols];
      const double t = a < bs ? ts[r0 + a] : 1.0;
      const double sc = t == 0.0 ? 1.0 : t;  // x_a / S_aa
#pragma unroll
      for (int c = 0; c < kUtCols; ++c) xa[c] = a < bs ? xs[(r0 + a) * kUtCols + c] : 0.0;
#pragma unroll
      for (int ii = kUtRows - 1; ii >= 0; --ii) {
        if (ii < bs) {
          if (a == ii) {
#pragma unroll
            for (int c = 0; c < kUtCols; ++c) xa[c] *= sc;
          }
          // srow[ii] is zero for every lane a >= ii (strict upper part)
#pragma unroll
          for (int c = 0; c < kUtCols; ++c) xa[c] -= srow[ii] * lane_bcast(xa[c], ii);
        }
      }
      if (a < bs) {
#pragma unroll
        for (int c = 0; c < kUtCols; ++c) xs[(r0 + a) * kUtCols + c] = xa[c];
      }
    }
    __syncthreads();
    const int n1 = r0, n0 = max(0, r0 - kUtRows);
    if (tid < 64 && n1 > 0) load_srow(n0, n1 - n0);
    for (int j = tid; j < r0; j += 256) {
      double g[kUtRows];
#pragma unroll
      for (int b = 0; b < kUtRows; ++b) g[b] = b < bs ? G[int64_t(r0 + b) * m + j] : 0.0;
      double acc[kUtCols] = {};
#pragma unroll
      for (int b = 0; b < kUtRows; ++b)
#pragma unroll
        for (int c = 0; c < kUtCols; ++c) acc[c] += g[b] * xs[(r0 + min(b, bs - 1)) * kUtCols + c];
#pragma unroll
      for (int c = 0; c < kUtCols; ++c) xs[j * kUtCols + c] -= acc[c];
    }
    __syncthreads();
    r1 = n1;
    r0 = n0;
  }
  for (int e = tid; e < m * kUtCols; e += 256) {
    const int i = e / kUtCols, c = e % kUtCols;
    if (c < nc) X[int64_t(i) * k + c0 + c] = xs[e];
  }
}

}  // namespace

void apply_reflectors(nsmi_ctx* ctx, const double* Vt, const double* tau, int m, int64_t len, double* Zr, int k) {
  require(m >= 1 && m <= kUtMaxM && k >= 0, "apply_reflectors: reflector count must be in [1, 2048]");
  if (k == 0) return;
  Scratch g(ctx, sizeof(double) * size_t(m) * m), x(ctx, sizeof(double) * size_t(m) * k);
  GemmDesc dw{};  // X = Vt . Zr^T  (m x k)
  dw.M = m; dw.N = k; dw.K = len; dw.transA = false; dw.transB = true;
  dw.lda = len; dw.ldb = len; dw.ldc = k; dw.batch = 1;
  gemm_f64(ctx, dw, 1.0, Vt, Zr, 0.0, x.as<double>(), kRoleFact);
  GemmDesc dg{};  // G = Vt . Vt^T  (m x m)
  dg.M = m; dg.N = m; dg.K = len; dg.transA = false; dg.transB = true;
  dg.lda = len; dg.ldb = len; dg.ldc = m; dg.batch = 1;
  gemm_f64(ctx, dg, 1.0, Vt, Vt, 0.0, g.as<double>(), kRoleFact);
  hipLaunchKernelGGL(k_ut_solve, dim3(unsigned((k + kUtCols - 1) / kUtCols)), dim3(256), 0, ctx->stream,
                     g.as<double>(), tau, x.as<double>(), m, k);
  NSMI_LAUNCH_CHECK();
  GemmDesc du{};  // Zr -= X^T . Vt  (k x len)
  du.M = k; du.N = len; du.K = m; du.transA = true; du.transB = false;
  du.lda = k; du.ldb = len; du.ldc = len; du.batch = 1;
  gemm_f64(ctx, du, -1.0, x.as<double>(), Vt, 1.0, Zr, kRoleFact);
}

void apply_q_lower(nsmi_ctx* ctx, const double* rho, const double* tau, int n, double* Zr, int k) {
  require(n >= 2 && n <= kUtMaxM && k >= 0, "apply_q_lower: n must be in [2, 2048]");
  if (k == 0) return;
  const int m = n - 1;
  Scratch vt(ctx, sizeof(double) * size_t(m) * n);
  const int64_t nv = int64_t(m) * n;
  hipLaunchKernelGGL(k_build_vt, dim3(unsigned((nv + 255) / 256)), dim3(256), 0, ctx->stream, rho, tau, n,
                     vt.as<double>());
  NSMI_LAUNCH_CHECK();
  apply_reflectors(ctx, vt.as<double>(), tau, m, n, Zr, k);
}

// A: n x n symmetric on the device (row-major == column-major), overwritten with the
// reflectors as k_sytrd leaves them (LAPACK's lower layout without d and e); d (n), e and
// tau (n - 1) on the device.  sytrd_launch enqueues the reduction on ctx->stream and the
// copy of its control words into run.host_flags; it returns false, with nothing
// launched, when n is outside the supported range or the device cannot co-schedule the
// grid (the caller then uses the library path).  Once the stream has passed the copy,
// reduction_unplaced tells whether the group never started (A is then as it was, and the
// caller launches again, spread) and sytrd_check reads the flags.
//
// A group on one XCD goes out as an ordinary launch: a cooperative launch waits for the
// whole device to drain, which would serialise the independent solves that share the
// GPU; that the group becomes resident rests on its place on the XCD
// (launch_on_one_xcd), and its placement ends in a bounded time (group.h).  A spread
// group takes the cooperative launch and its co-residency check.
bool sytrd_launch(nsmi_ctx* ctx, double* A, int n, double* d, double* e, double* tau, SytrdRun& run, bool spread) {
  if (n < 2 || n > kSytrdMax) return false;
  const TriPlan p = tri_plan(n);
  int G = (n + p.rows - 1) / p.rows;
  const size_t words = 6 * 64 * size_t(p.cl);
  run.xch.reset(new Scratch(ctx, sizeof(double) * words));
  run.flags.reset(new Scratch(ctx, sizeof(unsigned) * kCtlWords));
  unsigned* ctl = run.flags->as<unsigned>();
  double* xp = run.xch->as<double>();
  hipLaunchKernelGGL(k_reduction_init, dim3(unsigned((std::max<size_t>(words, kCtlWords) + 255) / 256)), dim3(256), 0,
                     ctx->stream, xp, words, size_t(0), 1u, 1u, 1u, ctl, int(kCtlWords), reduction_fail0(ctx, G),
                     spread && take_misplacement(ctx) ? kNeverArrived : 0u);
  NSMI_LAUNCH_CHECK();
  int nn = n, want = -1;
  void* args[] = {&A, &nn, &d, &e, &tau, &xp, &ctl, &G, &want};
  {
    ProfScope ps(ctx, NSMI_K_FACT_REDUCE, 4.0 / 3.0 * double(n) * n * n, 16.0 * double(n) * n);
    if (p.spread || spread || !one_xcd_groups(ctx)) {
      if (!launch_over_device(ctx, p.fn, G, p.threads, args)) return false;
    } else {
      launch_on_one_xcd(ctx, [&](int xcd) {
        want = take_misplacement(ctx) ? kXcds : xcd;  // kXcds: none has this number
        NSMI_HIP(hipLaunchKernel(p.fn, dim3(unsigned(kXcds * G)), dim3(unsigned(p.threads)), args, 0, ctx->stream));
      });
    }
  }
  reduction_readback(ctx, run, n);
  return true;
}

void sytrd_check(const SytrdRun& run) {
  if (reduction_unplaced(run))
    fail(NSMI_ERR_SOLVER, "factorize: the workgroups of the one-launch reduction found no room on the device");
  // each column's exchange, where every workgroup waits for all the others, is the barrier
  if (run.host_flags[0])
    fail(NSMI_ERR_SOLVER, "factorize: a workgroup of the one-launch reduction timed out at a grid barrier (of " +
                              std::to_string(run.columns) + " columns, in those from " +
                              std::to_string(run.host_flags[kCtlColumn - kCtlFail]) + " on)");
  // the tridiagonal solver is never handed NaN or Inf
  if (run.host_flags[1]) fail(NSMI_ERR_NOT_FINITE, "factorize: non-finite entries in the matrix to be factorized");
}

// Eigen-decomposition of every listed matrix (n <= kJacobiMax) in one launch.
void jacobi_eig_batched(nsmi_ctx* ctx, const std::vector<JacobiJob>& jobs, unsigned* unconverged) {
  *unconverged = 0u;
  if (jobs.empty()) return;
  int nmax = 0;
  std::vector<JacobiItem> h(jobs.size());
  for (size_t i = 0; i < jobs.size(); ++i) {
    require(jobs[i].n >= 1 && jobs[i].n <= kJacobiMax, "jacobi: matrix size outside the batched solver's range");
    h[i] = JacobiItem{jobs[i].a, jobs[i].w, jobs[i].n, 0};
    nmax = std::max(nmax, jobs[i].n);
  }
  Scratch d_items(ctx, sizeof(JacobiItem) * h.size());
  Scratch flag(ctx, 64);
  NSMI_HIP(hipMemcpyAsync(d_items.p, h.data(), sizeof(JacobiItem) * h.size(), hipMemcpyHostToDevice, ctx->stream));
  NSMI_HIP(hipMemsetAsync(flag.p, 0, 64, ctx->stream));
  constexpr int kMaxSweeps = 60;
  double fl = 0.0;
  for (const auto& j : jobs) fl += 9.0 * double(j.n) * j.n * j.n;
  {
    ProfScope ps(ctx, NSMI_K_FACT_SOLVE, fl, 0.0);
    const int m = nmax + (nmax & 1);
    const JacobiItem* it = d_items.as<JacobiItem>();
    unsigned* f = flag.as<unsigned>();
    const dim3 grid(unsigned(h.size())), block(256);
    if (m <= 16)
      hipLaunchKernelGGL(k_jacobi_eig<16>, grid, block, 0, ctx->stream, it, kMaxSweeps, f);
    else if (m <= 32)
      hipLaunchKernelGGL(k_jacobi_eig<32>, grid, block, 0, ctx->stream, it, kMaxSweeps, f);
    else
      hipLaunchKernelGGL(k_jacobi_eig<64>, grid, block, 0, ctx->stream, it, kMaxSweeps, f);
    NSMI_LAUNCH_CHECK();
  }
  NSMI_HIP(hipMemcpyAsync(unconverged, flag.p, sizeof(unsigned), hipMemcpyDeviceToHost, ctx->stream));
}

}  // namespace nsmi
