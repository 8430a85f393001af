/*
 * nsmi.h -- C ABI of libnsmi.so, the MI355X (gfx950) region-step engine for
 * NetworkSolvers.jl's 2-site DMRG / TDVP sweeps.
 *
 * Every entry point returns an int status (NSMI_OK = 0, negative = error);
 * nsmi_last_error(ctx) returns the message of the last failure on that context.
 * No C++ exception crosses this boundary.  Plain pointers and sizes only.
 *
 * Ownership: the context owns all device memory; tensors and operators are
 * freed explicitly (nsmi_tensor_free / nsmi_heff_destroy).  Work is enqueued
 * on the context's HIP stream; calls that return host scalars synchronise.
 * One host thread per context at a time; contexts are independent.
 *
 * Layouts (row-major, last index fastest):
 *   site tensor  A[l, s, r]          chain MPS tensor (left link, site, right link)
 *   MPO tensor   W[wl, wr, s', s]    s' = output (bra) index, s = input (ket) index
 *   environment  E[bra, mpo, ket]    for every directed edge p->q (p's side seen from q)
 *   two-site     theta[l, s1, s2, r]
 *
 * Reference interfaces replaced (paths relative to the NetworkSolvers.jl tree):
 *   operator_map.jl:3-10            optimal_map(P::ProjTTN, psi)  -> nsmi_heff_create/_apply
 *   local_solvers/eigsolve.jl:3-29  eigsolve_solver (KrylovKit)   -> nsmi_lanczos_eig
 *   local_solvers/exponentiate.jl   exponentiate_solver           -> nsmi_krylov_expm
 *   extracter.jl:7                  prod(psi[v] for v in region)  -> nsmi_theta
 *   extracter.jl:14, applyexp.jl:38 itn.position (environments)   -> nsmi_env_update
 *   extracter.jl:6, applyexp.jl:37  orthogonalize / qr            -> nsmi_qr
 *   inserter.jl:23                  it.factorize(theta, inds; trunc...) -> nsmi_factorize
 *   operator_map.jl:3-10 and ProjTTN on trees (up to four environments per
 *   region, multi-neighbour environment updates)  -> nsmi_tensordot,
 *                                   nsmi_permute, nsmi_netop_create
 */
#ifndef NSMI_H
#define NSMI_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define NSMI_OK 0
#define NSMI_ERR_INVALID (-1)     /* bad argument / shape mismatch            */
#define NSMI_ERR_HIP (-2)         /* HIP runtime failure                      */
#define NSMI_ERR_OOM (-3)         /* device pool limit or hipMalloc failure   */
#define NSMI_ERR_SOLVER (-4)      /* solver failure / no convergence          */
#define NSMI_ERR_NOT_FINITE (-5)  /* NaN or Inf met in a checked input        */
#define NSMI_ERR_UNSUPPORTED (-6) /* valid request this build does not serve  */

/* element types */
#define NSMI_F64 0
#define NSMI_C128 1

/* arithmetic of the effective-Hamiltonian contractions (the Krylov vectors,
 * environments handed in and all reductions stay FP64) */
#define NSMI_PREC_FP64 0   /* FP64 MFMA (v_mfma_f64_16x16x4)                      */
#define NSMI_PREC_FP32 1   /* FP32 MFMA on FP32-rounded operands                   */
#define NSMI_PREC_BF16X3 2 /* BF16 MFMA, hi/lo split operands, 3 products, FP32 acc */
#define NSMI_PREC_BF16 3   /* BF16 MFMA, single product, FP32 accumulation          */

/* truncation routes (ITensors factorize) */
#define NSMI_ROUTE_AUTO 0  /* "svd" if cutoff <= 1e-12, else "eigen"        */
#define NSMI_ROUTE_SVD 1
#define NSMI_ROUTE_EIGEN 2

typedef struct nsmi_ctx nsmi_ctx;
typedef struct nsmi_tensor nsmi_tensor;
typedef struct nsmi_heff nsmi_heff;

typedef struct {
  int krylovdim;   /* KrylovKit krylovdim (reference default 3)          */
  int maxiter;     /* only 1 is served (reference default)               */
  double tol;      /* invariant-subspace / convergence tolerance (1e-14) */
  double eta;      /* reorthogonalisation threshold, 1/sqrt(2)           */
} nsmi_lanczos_opts;

typedef struct {
  int numops;       /* H_eff applies performed                */
  int krylov_dim;   /* Krylov dimension reached               */
  double normres;   /* |beta_K * y_K| residual estimate       */
} nsmi_solver_info;

typedef struct {
  double cutoff;   /* relative discarded-weight cutoff            */
  int64_t maxdim;  /* <= 0 means unlimited                        */
  int64_t mindim;  /* reference default 1                         */
  int route;       /* NSMI_ROUTE_*                                */
} nsmi_trunc;

typedef struct {
  int64_t kept;      /* new bond dimension                        */
  int64_t full;      /* spectrum length min(rows, cols)           */
  double truncerr;   /* discarded weight / total weight           */
  double total;      /* sum of the spectrum (= |theta|^2)         */
  int route;         /* route actually taken                      */
} nsmi_trunc_info;

typedef struct {
  int64_t launches;
  double total_ms;   /* summed HIP-event durations                */
  double flops;      /* summed algorithmic flops                  */
  double bytes;      /* summed algorithmic bytes                  */
} nsmi_profile_stats;

/* kernel classes for nsmi_profile_query */
#define NSMI_K_HEFF_GEMM1 0   /* (L . theta) GEMM of the H_eff apply           */
#define NSMI_K_HEFF_GEMM2 1   /* (T . R) GEMM of the H_eff apply               */
#define NSMI_K_HEFF_MIX 2     /* MPO mixing between them                       */
#define NSMI_K_ENV 3          /* environment-update GEMMs + mixing             */
#define NSMI_K_THETA 4        /* theta formation                               */
#define NSMI_K_KRYLOV 5       /* Krylov vector kernels                         */
#define NSMI_K_FACT_GEMM 6    /* Gram / projection GEMMs of factorize          */
#define NSMI_K_FACT_SOLVE 7   /* dense eigensolver / SVD                       */
#define NSMI_K_BLOCK 8        /* block programs of QN (block-sparse) tensors   */
#define NSMI_K_NET 9          /* contraction programs of tree regions          */
#define NSMI_K_FACT_REDUCE 10 /* one-launch bidiagonalisation / tridiagonalisation of factorize */
#define NSMI_K_COUNT 11

/* ---------------------------------------------------------------- context */
int nsmi_version(void);
int nsmi_ctx_create(int device, size_t pool_limit_bytes, nsmi_ctx** out);
int nsmi_ctx_destroy(nsmi_ctx* ctx);
const char* nsmi_last_error(const nsmi_ctx* ctx);
int nsmi_sync(nsmi_ctx* ctx);
int nsmi_pool_stats(nsmi_ctx* ctx, size_t* in_use, size_t* cached, size_t* peak);
int nsmi_pool_trim(nsmi_ctx* ctx);
/* Failure injection for tests (no counterpart in the reference): the next `count`
   one-launch reductions of this context that run on several workgroups (the
   tridiagonalisation and the bidiagonalisation behind nsmi_factorize) start with
   their timeout flag raised: one workgroup leaves before its first column, every
   other one in its first exchange, when it sees the flag, and the call reports
   NSMI_ERR_SOLVER with the column, exactly as when a wait for the other workgroups
   gives up; the context stays usable. */
int nsmi_inject_barrier_timeout(nsmi_ctx* ctx, int count);
/* The same for their placement: the next `count` of them do not get the XCDs that they ask
   for.  A group on one XCD then leaves without having started and is launched again over
   the whole device (with count 2 that placement times out, and it is launched once more);
   a group over all XCDs is formed in the grid's order.  Results are those of the usual
   placement, bit for bit. */
int nsmi_inject_misplacement(nsmi_ctx* ctx, int count);

/* ---------------------------------------------------------------- tensors */
int nsmi_tensor_create(nsmi_ctx* ctx, int dtype, int rank, const int64_t* dims, nsmi_tensor** out);
int nsmi_tensor_upload(nsmi_ctx* ctx, int dtype, int rank, const int64_t* dims, const void* host,
                       nsmi_tensor** out);
int nsmi_tensor_download(nsmi_ctx* ctx, const nsmi_tensor* t, void* host, size_t host_bytes);
int nsmi_tensor_free(nsmi_ctx* ctx, nsmi_tensor* t);
int nsmi_tensor_info(const nsmi_tensor* t, int* dtype, int* rank, int64_t* dims8);
int nsmi_tensor_copy(nsmi_ctx* ctx, const nsmi_tensor* src, nsmi_tensor** out);
int nsmi_tensor_reshape(nsmi_ctx* ctx, nsmi_tensor* t, int rank, const int64_t* dims);
int nsmi_tensor_scale(nsmi_ctx* ctx, nsmi_tensor* t, double re, double im);
int nsmi_tensor_axpy(nsmi_ctx* ctx, double re, double im, const nsmi_tensor* x, nsmi_tensor* y);
int nsmi_tensor_norm(nsmi_ctx* ctx, const nsmi_tensor* t, double* out);
int nsmi_tensor_inner(nsmi_ctx* ctx, const nsmi_tensor* a, const nsmi_tensor* b, double* re, double* im);

/* ----------------------------------------------------------- region step */
/* theta[l,s1,s2,r] = sum_m A[l,s1,m] B[m,s2,r]            (extracter.jl:7) */
int nsmi_theta(nsmi_ctx* ctx, const nsmi_tensor* A, const nsmi_tensor* B, nsmi_tensor** theta);

/* New environment from the previous one (itn.position, extracter.jl:14).
 * side 0: edge i->i+1, E'[b',w',b] = sum conj(A[a',s',b']) E[a',w,a] W[w,w',s',s] A[a,s,b]
 * side 1: edge i->i-1, E'[a',w,a]  = sum conj(A[a',s',b']) E[b',v,b] W[w,v,s',s]  A[a,s,b]
 * precision: NSMI_PREC_* of the contractions (result stored FP64). */
int nsmi_env_update(nsmi_ctx* ctx, const nsmi_tensor* E, const nsmi_tensor* A, const nsmi_tensor* W,
                    int side, int precision, nsmi_tensor** out);

/* Effective Hamiltonian of a 1- or 2-site chain region (optimal_map,
 * operator_map.jl:3-10).  W2 == NULL gives the 1-site operator.  The operator
 * keeps references to L, W1, W2, R (they must outlive it) plus its own
 * workspace and precision-converted copies. */
int nsmi_heff_create(nsmi_ctx* ctx, const nsmi_tensor* L, const nsmi_tensor* W1, const nsmi_tensor* W2,
                     const nsmi_tensor* R, int precision, nsmi_heff** out);
int nsmi_heff_destroy(nsmi_ctx* ctx, nsmi_heff* op);
int nsmi_heff_apply(nsmi_ctx* ctx, nsmi_heff* op, const nsmi_tensor* x, nsmi_tensor* y);
/* The same apply without any device allocation.  No counterpart in the reference:
   it is for callers that cannot allocate (code under HIP graph capture, tight
   serving loops, harnesses that forbid hipMalloc).  The split-K partial sums of
   the GEMMs, the only device memory nsmi_heff_apply takes besides the operator's
   own workspace, come from a per-device array of nsmi_noalloc_scratch_bytes()
   (32 MiB) set up at context creation; an apply that would need more fails with
   NSMI_ERR_INVALID.  Served for real chain operators (1- and 2-site) in the FP64
   and FP32 forms; other operators are rejected with NSMI_ERR_INVALID.  All calls on
   one GPU share its array: calls that overlap on one GPU (other contexts, other
   threads) race and must be serialised by the caller. */
int nsmi_heff_apply_noalloc(nsmi_ctx* ctx, nsmi_heff* op, const nsmi_tensor* x, nsmi_tensor* y);
size_t nsmi_noalloc_scratch_bytes(void);
/* FP64 Rayleigh quotient <x|H|x>/<x|x> with an FP64 apply whatever op's precision */
int nsmi_heff_rayleigh(nsmi_ctx* ctx, nsmi_heff* op, const nsmi_tensor* x, double* e);

/* Lowest Ritz pair (KrylovKit eigsolve with Lanczos, ishermitian, :SR;
 * local_solvers/eigsolve.jl:3-29).  x is the start vector on entry and the
 * Ritz vector on exit. */
int nsmi_lanczos_eig(nsmi_ctx* ctx, nsmi_heff* op, nsmi_tensor* x, const nsmi_lanczos_opts* opts,
                     double* eigval, nsmi_solver_info* info);

/* x <- exp(tau H) x for the Hermitian operator (exponentiate_solver,
 * local_solvers/exponentiate.jl:3-29; tau = -i * weight * dt in TDVP).
 * opts: krylovdim (<= 32, reference default 30), maxiter (sub-steps, 100),
 * tol (error per unit time, 1e-12), eta (re-orthogonalisation threshold).
 * info: numops = H applies, krylov_dim = largest basis used, normres = last
 * error estimate.  A complex tau needs a complex (C128) state. */
int nsmi_krylov_expm(nsmi_ctx* ctx, nsmi_heff* op, double tau_re, double tau_im, nsmi_tensor* x,
                     const nsmi_lanczos_opts* opts, nsmi_solver_info* info);

/* Truncated split of theta (ITensors factorize, ortho="left"; inserter.jl:23).
 * rows = the first n_row_dims dims of theta when rows_trailing == 0, else the
 * remaining trailing dims.  The isometry U carries the row dims:
 *   rows_trailing == 0: U[dims[:n], k],   C[k, dims[n:]]
 *   rows_trailing == 1: U[k, dims[n:]],   C[dims[:n], k]   (U stored transposed)
 * Columns of the isometry get the "largest-magnitude entry real positive" gauge.
 * The svd route (real theta) bidiagonalises the isometry side in one launch; where
 * that cannot run (the shorter side above 2048, the longer above 4096 or, with
 * the shorter above 1024, above 2048, or the device refusing the cooperative
 * launch) the Gram matrix takes its place and
 * info->route reports eigen. */
int nsmi_factorize(nsmi_ctx* ctx, const nsmi_tensor* theta, int n_row_dims, int rows_trailing,
                   const nsmi_trunc* trunc, nsmi_tensor** U, nsmi_tensor** C, nsmi_trunc_info* info);

/* Thin QR with non-negative diag(R) (ITensors qr in the orthogonalize walk,
 * extracter.jl:6).  Same row/transpose conventions as nsmi_factorize. */
int nsmi_qr(nsmi_ctx* ctx, const nsmi_tensor* A, int n_row_dims, int rows_trailing, nsmi_tensor** Q,
            nsmi_tensor** R);

/* ------------------------------------------------- general tree contractions */
/* out = A with its axes permuted: out.dims[k] = A.dims[perm[k]] (rank <= 8).
 * Index relabelling of tree tensors (ITensors' named-index contraction order,
 * extracter.jl:7, inserter.jl:23-29). */
int nsmi_permute(nsmi_ctx* ctx, const nsmi_tensor* A, const int* perm, nsmi_tensor** out);

/* out[free(A)..., free(B)...] = sum over the n axis pairs (axes_a[i], axes_b[i])
 * of op(A) op(B), op = conj when conj_* != 0 (C128); free axes keep their order.
 * A and B share one element type.  One MFMA GEMM (operands permuted into matrix
 * form when needed).  Replaces the ITensor contractions of the tree environment
 * update (ProjTTN position, extracter.jl:14) and theta (extracter.jl:7). */
int nsmi_tensordot(nsmi_ctx* ctx, const nsmi_tensor* A, int conj_a, const nsmi_tensor* B, int conj_b, int n,
                   const int* axes_a, const int* axes_b, nsmi_tensor** out);

/* One step of a contraction program: running = tensordot(running, op(operand),
 * axes_x, axes_o) with op = conj when conj != 0. */
typedef struct nsmi_net_step {
  int operand;    /* index into the operand list            */
  int n;          /* number of contracted axis pairs (<= 8) */
  int axes_x[8];  /* axes of the running tensor             */
  int axes_o[8];  /* axes of the operand                    */
  int conj;
} nsmi_net_step;

/* An effective Hamiltonian given as a contraction program (optimal_map on a tree
 * region, operator_map.jl:3-10, with up to four incident environments): applying
 * it runs the steps on x and permutes the result by out_perm, which must give x's
 * shape.  The returned handle is used like nsmi_heff_create's (apply, rayleigh,
 * Lanczos, Krylov exponential, destroy).  Operands (F64 or C128) must stay alive
 * until nsmi_heff_destroy; they are read in [contracted..., free...] order,
 * permuted once here when needed.  precision NSMI_PREC_FP32 runs the program in
 * FP32 / ComplexF32 on FP32 MFMA (operands converted once here, x and y converted
 * per apply; the Krylov vectors stay F64 / C128); NSMI_PREC_FP64 runs it as given. */
int nsmi_netop_create(nsmi_ctx* ctx, int n_operands, const nsmi_tensor* const* operands, int n_steps,
                      const nsmi_net_step* steps, int x_rank, const int64_t* x_dims, const int* out_perm,
                      int precision, nsmi_heff** out);

/* ------------------------------------------ quantum-number (block-sparse) */
/* A block program: the block operations of one contraction of U(1) block-sparse
 * tensors (ITensors QN ITensors as used by the reference's QN sweeps, README.md
 * QN timings; operator_map.jl:3-10 "per compatible block pair", extracter.jl:7,14,
 * inserter.jl:23).  Buffers: 0 = x, 1 = y, 2.. = operands (FP64 tensors), then
 * n_scratch scratch buffers of scratch_elems[i] doubles.  steps: n_steps rows of
 * (kind, transA, transB, first item, item count, 0); kind 0 = grouped GEMM over
 * gemm_items rows (c_buf, c_off, ldc, M, N, first segment, segment count) whose
 * segments are segs rows (a_buf, a_off, lda, b_buf, b_off, ldb, K) scaled by
 * seg_alpha -- each output block is the sum of its segments, written once; kind 1
 * = linear combinations over lin_items rows (out_buf, out_off, n, first term,
 * term count) of terms rows (src_buf, src_off) times term_coeff; kind 2 = copies
 * over copy_items rows (src_buf, src_off, src_ld, dst_buf, dst_off, dst_ld, rows,
 * cols).  Every block is checked against its buffer here.  With x_elems ==
 * y_elems the handle is an effective Hamiltonian for nsmi_heff_apply/_rayleigh,
 * nsmi_lanczos_eig and nsmi_krylov_expm; any program runs with nsmi_bsop_run.
 * precision NSMI_PREC_FP32 runs the program on FP32 copies of the operands and
 * FP32 scratch (FP32 MFMA GEMMs), x and y converted per run; NSMI_PREC_FP64 as is. */
int nsmi_bsop_create(nsmi_ctx* ctx, int n_operands, const nsmi_tensor* const* operands, int n_scratch,
                     const int64_t* scratch_elems, int64_t x_elems, int64_t y_elems, int n_steps,
                     const int64_t* steps, const int64_t* gemm_items, const int64_t* segs, const double* seg_alpha,
                     const int64_t* lin_items, const int64_t* terms, const double* term_coeff,
                     const int64_t* copy_items, int precision, nsmi_heff** out);
int nsmi_bsop_run(nsmi_ctx* ctx, nsmi_heff* op, const nsmi_tensor* x, nsmi_tensor* y);

/* Tile choice of the block programs' grouped GEMMs (32 x 32 or 64 x 64 output tiles
 * per workgroup; both give bit-identical results).  No counterpart in the reference:
 * ITensors contracts each block pair with BLAS.  NSMI_TUNE_AUTO (the default) times
 * the first launches of each GEMM shape class (transposes, output area, block count,
 * mean K, share of large blocks) with both tiles and keeps the faster;
 * NSMI_TUNE_HEURISTIC takes 64 x 64 when at least half the output area lies in
 * blocks of 48 x 48 or more; NSMI_TUNE_TILE32 / _TILE64 force one tile (64 x 64
 * only where some block exceeds 32 in a dimension). */
#define NSMI_TUNE_HEURISTIC 0
#define NSMI_TUNE_AUTO 1
#define NSMI_TUNE_TILE32 2
#define NSMI_TUNE_TILE64 3
int nsmi_tune_mode(nsmi_ctx* ctx, int mode);
/* The autotuner's table, one row of 8 int64 per shape class: key, launches issued
 * with 32 and with 64 tiles, samples completed with each, best time with each in ns
 * (-1 before a sample), and the chosen tile (32, 64, or -1 while undecided).  Writes
 * at most cap rows; *n_out receives the number of classes.  Synchronises. */
int nsmi_tune_table(nsmi_ctx* ctx, int64_t* rows, int cap, int* n_out);

/* Truncated factorisation of a block-diagonal matrix (ITensors factorize of a QN
 * ITensor, inserter.jl:23): sector q is the rows[q] x cols[q] row-major matrix at
 * offsets[q] of Mall.  Every sector is decomposed through its Gram matrix (the
 * eigen route of nsmi_factorize, also when trunc->route asks for svd, which then
 * only sets the sort key; info->route reports eigen); the
 * spectra are merged and truncated together (truncate! on the sorted union) and
 * each sector keeps its entries above the cut value (NDTensors block-sparse
 * svd/eigen).  kept[q] receives the kept count; Uall / Call hold U_q (rows x k,
 * or k x cols when rows_trailing) and C_q concatenated in sector order. */
int nsmi_factorize_sectors(nsmi_ctx* ctx, const nsmi_tensor* Mall, int n, const int64_t* offsets, const int64_t* rows,
                           const int64_t* cols, int rows_trailing, const nsmi_trunc* trunc, nsmi_tensor** Uall,
                           nsmi_tensor** Call, int64_t* kept, nsmi_trunc_info* info);

/* ------------------------------------------------------------- profiling */
int nsmi_profile_enable(nsmi_ctx* ctx, int on);
/* kernel classes recorded while profiling is on: bit k selects NSMI_K_* class k
 * (default: all), so a timed run can carry events on the classes it reports only */
int nsmi_profile_classes(nsmi_ctx* ctx, unsigned mask);
/* record one launch in `every` of each selected class (default 1: all), which
 * keeps the event overhead out of a timed run while still sampling its kernels;
 * counters restart.  No counterpart in the reference (measurement only). */
int nsmi_profile_sampling(nsmi_ctx* ctx, unsigned every);
int nsmi_profile_reset(nsmi_ctx* ctx);
int nsmi_profile_query(nsmi_ctx* ctx, int kernel_class, nsmi_profile_stats* out);

#ifdef __cplusplus
}
#endif
#endif /* NSMI_H */
