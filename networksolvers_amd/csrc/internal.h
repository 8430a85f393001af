// Internal declarations of libnsmi.so (not part of the C ABI).
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <cstdint>
#include <cstdio>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/nsmi.h"

namespace nsmi {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

[[noreturn]] inline void fail(int code, const std::string& msg) { throw Error(code, msg); }
inline void require(bool ok, const std::string& msg) {
  if (!ok) fail(NSMI_ERR_INVALID, msg);
}

#define NSMI_HIP(call)                                                                        \
  do {                                                                                        \
    hipError_t e_ = (call);                                                                   \
    if (e_ != hipSuccess)                                                                     \
      ::nsmi::fail(NSMI_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_) + " at " + \
                                     __FILE__ + ":" + std::to_string(__LINE__));              \
  } while (0)

#define NSMI_LAUNCH_CHECK() NSMI_HIP(hipGetLastError())

// Body of every extern "C" entry point that takes a context.  The entry point
// holds the context's lock for the whole call: one host thread drives a context,
// but handle frees also come from finalizers on other threads (a garbage
// collection on another worker), and without the lock such a free would change
// the pool's maps, the deferred-release list or the error string while the owner's
// call is using them.  No exception crosses the ABI; the message is kept in ctx->err.
#define API_BEGIN(ctxp)                                                  \
  std::lock_guard<std::recursive_mutex> nsmi_api_lock_((ctxp)->mu);      \
  try {
#define API_END(ctxp)                                                    \
  }                                                                      \
  catch (const nsmi::Error& e) {                                         \
    (ctxp)->err = e.what();                                              \
    return e.code;                                                       \
  }                                                                      \
  catch (const std::exception& e) {                                      \
    (ctxp)->err = std::string("internal: ") + e.what();                  \
    return NSMI_ERR_INVALID;                                             \
  }                                                                      \
  return NSMI_OK;

// Size-class caching allocator.  All work of a context runs on one stream, so a
// block returned to the cache may be handed out again immediately: later work
// using it is ordered after earlier work on the same stream.  trim() returns the
// cached blocks to HIP after waiting for the owning context's own streams (not the
// whole device, which would stall every other context's work).
class Pool {
 public:
  // sync: waits for every stream of the owning context (before blocks are freed)
  Pool(size_t limit, void (*sync)(void*), void* owner) : limit_(limit), sync_(sync), owner_(owner) {}
  ~Pool();
  void* alloc(size_t bytes);
  void release(void* p);
  void trim();
  size_t in_use() const { return in_use_; }
  size_t cached() const { return cached_; }
  size_t peak() const { return peak_; }

 private:
  static size_t round(size_t b);
  size_t limit_;
  void (*sync_)(void*);
  void* owner_;
  size_t in_use_ = 0, cached_ = 0, peak_ = 0;
  std::map<size_t, std::vector<void*>> free_;
  std::map<void*, size_t> live_;
};

struct Tuner;  // tile autotuner of the block-program GEMMs (blocksparse.hip)

struct ProfRec {
  hipEvent_t a, b;
  int cls;
  double flops, bytes;
};

}  // namespace nsmi

struct nsmi_tensor {
  int dtype;
  int rank;
  int64_t dims[8];
  int64_t numel;
  void* data;
  size_t bytes;
};

struct nsmi_ctx {
  int device = 0;
  // held by every entry point for its whole call (API_BEGIN)
  std::recursive_mutex mu;
  hipStream_t stream = nullptr;
  rocblas_handle blas = nullptr;
  nsmi::Pool* pool = nullptr;
  std::string err;
  // reduction scratch
  double* d_partials = nullptr;  // kPartials doubles
  double* d_scal = nullptr;      // 64 result slots
  double* h_scal = nullptr;      // pinned mirror of d_scal
  double* d_mpart = nullptr;     // kMdotPartials doubles: partials of the multi-vector dot products
  double* d_mcoef = nullptr;     // 2 kMdotMax doubles: their coefficients (re, im)
  unsigned* d_count = nullptr;   // 2 arrival counters of the last-workgroup finishes (zero between launches)
  // Host-coherent copies of the Krylov result slots: the kernels that finish a slot
  // write its value, a system-scope fence, then the tag of their pass, so a pass's
  // read-back needs no copy (read_fresh).  64 values and 64 tags in pinned coherent
  // memory; dm_* are the device-side addresses of the same memory.
  double* h_mval = nullptr;
  unsigned* h_mtag = nullptr;
  double* dm_val = nullptr;
  unsigned* dm_tag = nullptr;
  unsigned mseq = 0;  // tag of the latest Krylov pass
  // pinned host chunks for small asynchronous read-backs and uploads of one call
  // (stage_take / stage_reset); never freed before the context
  std::vector<std::pair<void*, size_t>> h_stage;
  size_t h_stage_cur = 0, h_stage_off = 0;
  bool h_stage_busy = false;  // a call took stage memory and has not reached stage_done
  int* d_info = nullptr;
  // auxiliary streams (default priority), each with its own rocBLAS handle and
  // solver status word, for independent sector solves; created on first use
  std::vector<hipStream_t> aux_stream;
  std::vector<rocblas_handle> aux_blas;
  std::vector<int*> aux_info;
  std::vector<hipEvent_t> aux_event;  // [0]: fork from the main stream, [1 + j]: join of aux j
  // while set, released pool blocks are held back (work on several streams may
  // still use them) and returned once every stream has drained
  bool defer_release = false;
  std::vector<void*> deferred;
  // profiling
  bool prof_on = false;
  unsigned prof_mask = ~0u;  // classes recorded while prof_on
  unsigned prof_every = 1;   // record one scope in prof_every per class
  unsigned prof_seen[32] = {};
  // events a kernel-timed ProfScope hands to the next NSMI_LAUNCH_TIMED launch
  hipEvent_t kev_start = nullptr, kev_stop = nullptr;
  bool kev_used = false;
  std::vector<nsmi::ProfRec> recs;
  std::vector<hipEvent_t> spare_events;
  nsmi_profile_stats stats[NSMI_K_COUNT] = {};
  // multi-workgroup reductions still to start with the timeout flag raised (tests)
  int inject_timeouts = 0;
  // placements of multi-workgroup reductions still to fail (tests)
  int inject_misplaced = 0;
  // while set (nsmi_heff_apply_noalloc), split-K GEMMs take their partial sums from
  // this device buffer instead of the pool, and fail when it is too small
  void* fixed_part = nullptr;
  size_t fixed_part_bytes = 0;
  // tile choice of the block-program GEMMs (NSMI_TUNE_*) and the autotuner's table
  int tune_mode = NSMI_TUNE_AUTO;
  nsmi::Tuner* tuner = nullptr;
};

namespace nsmi {

constexpr int kPartials = 1024;  // blocks of the first reduction pass
constexpr int kMdotMax = 32;         // vectors of one classical Gram-Schmidt pass
constexpr int kMdotPartials = 32768; // 2 kMdotMax rows of at most 512 workgroup partials

inline size_t dtype_size(int dt) {
  switch (dt) {
    case NSMI_F64: return 8;
    case NSMI_C128: return 16;
    default: fail(NSMI_ERR_INVALID, "unknown dtype " + std::to_string(dt));
  }
}

nsmi_tensor* tensor_new(nsmi_ctx* ctx, int dtype, int rank, const int64_t* dims);
void tensor_delete(nsmi_ctx* ctx, nsmi_tensor* t);
void* scratch(nsmi_ctx* ctx, size_t bytes);        // pool block, caller releases
// Pinned host memory for a call's small device<->host copies, which then stay
// asynchronous (a copy into pageable memory blocks the host until the stream gets
// there, which would serialise work spread over several streams).  stage_take
// hands out 16-byte aligned slices; stage_reset, at the start of an entry point,
// makes the whole arena reusable, and stage_done, after that entry point's closing
// synchronisation, marks it idle.  A reset after a call that ended early (an error)
// first waits for the main stream, so no copy of that call is still in flight.
void* stage_take(nsmi_ctx* ctx, size_t bytes);
void stage_reset(nsmi_ctx* ctx);
void stage_done(nsmi_ctx* ctx);
void scratch_release(nsmi_ctx* ctx, void* p);

// Work on the auxiliary streams: AuxSection creates them (k at most), holds pool
// releases back for its lifetime and, on exit, waits for every auxiliary stream
// before the held blocks go back to the pool; fork() orders the auxiliary streams
// after everything enqueued so far on the main stream, join() the main stream
// after everything enqueued on them.  OnAux points ctx->stream, ctx->blas and
// ctx->d_info at auxiliary stream j for its scope.
struct AuxSection {
  nsmi_ctx* ctx;
  int k;
  AuxSection(nsmi_ctx* c, int want);
  ~AuxSection();
  void fork();
  void join();
  void sync();  // host wait for the main and every auxiliary stream
};
struct OnAux {
  nsmi_ctx* ctx;
  hipStream_t s;
  rocblas_handle b;
  int* info;
  OnAux(nsmi_ctx* c, int j);
  ~OnAux();
};

// RAII holder for pool scratch
struct Scratch {
  nsmi_ctx* ctx;
  void* p;
  Scratch(nsmi_ctx* c, size_t bytes) : ctx(c), p(scratch(c, bytes)) {}
  ~Scratch() { if (p) scratch_release(ctx, p); }
  template <typename T> T* as() const { return static_cast<T*>(p); }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
};

// profiling brackets (no-ops when profiling is off)
// With kernel_timed, the scope's events are not stream markers around the scope:
// the first NSMI_LAUNCH_TIMED kernel inside it carries them (hipExtLaunchKernelGGL
// records them at that kernel's own start and end), so the duration excludes the
// dispatch gaps that markers around a short kernel would add.
struct ProfScope {
  nsmi_ctx* ctx;
  int cls;
  double flops, bytes;
  bool kernel_timed = false;
  hipEvent_t a = nullptr, b = nullptr;
  ProfScope(nsmi_ctx* c, int k, double f, double by, bool kernel_timed = false);
  ~ProfScope();
};

#define NSMI_LAUNCH_TIMED(ctx, KERNEL, grid, block, ...)                                                  \
  do {                                                                                                    \
    if ((ctx)->kev_start) {                                                                               \
      hipExtLaunchKernelGGL(KERNEL, grid, block, 0, (ctx)->stream, (ctx)->kev_start, (ctx)->kev_stop, 0, \
                            __VA_ARGS__);                                                                 \
      (ctx)->kev_start = (ctx)->kev_stop = nullptr;                                                       \
      (ctx)->kev_used = true;                                                                             \
    } else {                                                                                              \
      hipLaunchKernelGGL(KERNEL, grid, block, 0, (ctx)->stream, __VA_ARGS__);                             \
    }                                                                                                     \
  } while (0)

// An operation of two launches timed as one: the first carries the start event of a
// kernel-timed scope, the last its stop event (each recorded by the kernel itself).
#define NSMI_LAUNCH_TIMED_FIRST(ctx, KERNEL, grid, block, ...)                                      \
  do {                                                                                              \
    if ((ctx)->kev_start) {                                                                         \
      hipExtLaunchKernelGGL(KERNEL, grid, block, 0, (ctx)->stream, (ctx)->kev_start, nullptr, 0,    \
                            __VA_ARGS__);                                                           \
      (ctx)->kev_start = nullptr;                                                                   \
    } else {                                                                                        \
      hipLaunchKernelGGL(KERNEL, grid, block, 0, (ctx)->stream, __VA_ARGS__);                       \
    }                                                                                               \
  } while (0)
#define NSMI_LAUNCH_TIMED_LAST(ctx, KERNEL, grid, block, ...)                                       \
  do {                                                                                              \
    if ((ctx)->kev_stop && !(ctx)->kev_start) {                                                     \
      hipExtLaunchKernelGGL(KERNEL, grid, block, 0, (ctx)->stream, nullptr, (ctx)->kev_stop, 0,     \
                            __VA_ARGS__);                                                           \
      (ctx)->kev_stop = nullptr;                                                                    \
      (ctx)->kev_used = true;                                                                       \
    } else {                                                                                        \
      hipLaunchKernelGGL(KERNEL, grid, block, 0, (ctx)->stream, __VA_ARGS__);                       \
    }                                                                                               \
  } while (0)

// ---- dense kernels (gemm.hip) -------------------------------------------
// Row-major C[b] = alpha * op(A[b]) op(B[b]) + beta * C[b]; op(A) is M x K
// (A stored K x M when transA), op(B) is K x N (B stored N x K when transB).
struct GemmDesc {
  int64_t M, N, K;
  int64_t lda, ldb, ldc;
  int64_t sA, sB, sC;  // batch strides in elements
  int64_t batch;
  bool transA, transB;
  bool tiles_ok() const;
};
void gemm_f64(nsmi_ctx* ctx, const GemmDesc& g, double alpha, const double* A, const double* B,
              double beta, double* C, int role);
// FP32 MFMA on float operands, FP32 result
void gemm_f32(nsmi_ctx* ctx, const GemmDesc& g, const float* A, const float* B, float* C, int role);
// the FP32 H_eff products of a real FP64 vector: GEMM1 reads x (FP64) and GEMM2
// writes y (FP64) directly, rounding / widening inside the kernel
void gemm_f32_heff1_bd(nsmi_ctx* ctx, const GemmDesc& d, const float* A, const double* B, float* C);
void gemm_f32_heff2_cd(nsmi_ctx* ctx, const GemmDesc& d, const float* A, const float* B, double* C);
// BF16 MFMA, C[M x N] = A[M x Kp] . B[N x Kp]^T on pre-split bf16 hi (and lo)
// planes (terms = 1: hi.hi; 3: hi.hi + hi.lo + lo.hi); Kp % 32 == 0 with zero
// padding; C is FP32 or FP64 (c_double)
void gemm_bf16_nt(nsmi_ctx* ctx, int64_t M, int64_t N, int64_t Kp, const uint16_t* Ahi, const uint16_t* Alo,
                  int64_t lda, const uint16_t* Bhi, const uint16_t* Blo, int64_t ldb, void* C, int64_t ldc,
                  bool c_double, int terms, int role);
inline int64_t pad32(int64_t k) { return (k + 31) / 32 * 32; }
// split an FP64 matrix (rows x K, row stride K) into bf16 hi/lo planes of pitch Kp (zero padded);
// transpose != 0 reads the source as K x rows (row stride rows) instead
void split_bf16_pad(nsmi_ctx* ctx, const double* X, int64_t rows, int64_t K, int64_t Kp, uint16_t* hi,
                    uint16_t* lo, int transpose);
// H_eff mixing into GEMM2's bf16 operand: T3[(o*S + srow), v*I + i] for p = srow*D2 + v
void mix_f32_to_bf16_rows(nsmi_ctx* ctx, const float* X, uint16_t* Yhi, uint16_t* Ylo, const double* Mx,
                          int64_t O, int P, int Q, int64_t I, int D2, int64_t Kp, int cls);

// roles select distinct kernel instantiations so each call site is a separate
// kernel name in profiles
enum GemmRole { kRoleHeff1 = 0, kRoleHeff2 = 1, kRoleEnv = 2, kRoleTheta = 3, kRoleFact = 4 };

// ---- elementwise / reduction kernels (vec.hip) -----------------------------
void vec_scale(nsmi_ctx* ctx, double* x, int64_t n, double a);
void vec_axpy(nsmi_ctx* ctx, double* y, const double* x, int64_t n, double a);
void vec_copy(nsmi_ctx* ctx, double* y, const double* x, int64_t n);
// y = a*x  (separate output)
void vec_scaled_copy(nsmi_ctx* ctx, double* y, const double* x, int64_t n, double a);
// slot <- sum x*y (device), returns after enqueue
void vec_dot_dev(nsmi_ctx* ctx, const double* x, const double* y, int64_t n, int slot);
// w += c1*v1 + c2*v2 then slot <- |w|^2  (v2 may be null)
void vec_axpy2_norm2_dev(nsmi_ctx* ctx, double* w, const double* v1, double c1, const double* v2,
                         double c2, int64_t n, int slot);
// out = sum_j c[j] * V[j]
void vec_lincomb(nsmi_ctx* ctx, double* out, const double* const* V, const double* c, int k, int64_t n);
// read result slots [0, count) to host (synchronises)
void read_slots(nsmi_ctx* ctx, int count, double* out);
// The same from the host-coherent copies when every slot in `mask` carries `tag` (the
// kernels of that pass finished it); otherwise, or without the copies, read_slots.
// Slots outside the mask are returned as the copies hold them.
void read_fresh(nsmi_ctx* ctx, int count, double* out, unsigned tag, unsigned mask);
// a fresh tag for the next Krylov pass (never 0)
unsigned next_tag(nsmi_ctx* ctx);
// One classical Gram-Schmidt pass of r against the m <= kMdotMax vectors V + j vstride
// (vstride in doubles), in two launches: optionally r += cprev prev first, then
// c_j = <V_j, r> (conjugated when cplx; n counts complex elements then) for every j
// against the same r, then r -= sum_j c_j V_j and |r|^2.  c_{m-1} goes to slot_dot
// (and slot_dot + 1 when cplx), |r|^2 to slot_norm.
// The start of a Krylov basis from x0 and r = H x0 (n elements, complex when cplx), in
// two launches: slots 4 = |x0|^2, 0 (1) = <x0, r>, 2 = |r|^2; then V0 = x0 / |x0| and
// r <- r / |x0| - alpha V0 with alpha = Re <x0, r> / |x0|^2, slot 3 = the new |r|^2.
// With maxref > 0 (only where vec_start_one_launch holds) the start's refinement
// passes against V0 follow in the same launch while the refinement rule asks for them;
// then, given vnext and once the rule asks for no further pass, vnext = r / |r| and
// slot kRState + 4 = 1 (else 0).
void vec_krylov_start(nsmi_ctx* ctx, const double* x0, double* V0, double* r, int64_t n, bool cplx,
                      unsigned tag = 0, double eta = 0.0, int maxref = 0, double* vnext = nullptr);
bool vec_start_one_launch(int64_t n, bool cplx);
// rmode 1 also starts the refinement state (slots kRState..kRState+3: a = Re c_{m-1},
// |r|^2, the norm before the pass sqrt(|r|^2 + a^2 + rbeta^2), 0 passes); rmode 2 makes
// the pass conditional on that state (it runs only while eps < |r| < eta * the norm
// before the latest pass, then a += Re c_{m-1} and the count rises); the start's second
// launch starts the state too (a = alpha, the norm before = |H x0| / |x0|).
constexpr int kRState = 8;
// With maxref > 0 (rmode 1, only where vec_cgs_one_launch holds) up to maxref
// refinement passes over the mall vectors from Vall follow in the same launch while
// the rule asks for them; then, given vnext and once the rule asks for no further
// pass, vnext = r / |r| and slot kRState + 4 = 1 (else 0).
void vec_cgs_pass(nsmi_ctx* ctx, const double* V, int64_t vstride, int m, double* r, int64_t n, bool cplx,
                  int slot_dot, int slot_norm, const double* prev = nullptr, double cprev = 0.0, unsigned tag = 0,
                  int rmode = 0, double rbeta = 0.0, double eta = 0.0, const double* Vall = nullptr, int mall = 0,
                  int maxref = 0, double* vnext = nullptr);
bool vec_cgs_one_launch(int64_t n);  // a pass over n elements is one workgroup, one launch (n <= 4096)
void vec_to_f32(nsmi_ctx* ctx, float* y, const double* x, int64_t n);
void vec_f32_to_f64(nsmi_ctx* ctx, double* y, const float* x, int64_t n);
void vec_split_bf16(nsmi_ctx* ctx, uint16_t* hi, uint16_t* lo, const double* x, int64_t n);
void vec_split_bf16_f32(nsmi_ctx* ctx, uint16_t* hi, uint16_t* lo, const float* x, int64_t n);
void vec_check_finite(nsmi_ctx* ctx, const double* x, int64_t n, int slot);
// fails with NSMI_ERR_NOT_FINITE when x holds a NaN or Inf (uses slot 0; synchronises)
void require_finite(nsmi_ctx* ctx, const double* x, int64_t n, const char* what);
// complex (interleaved) vectors, n complex elements
void vec_zscale(nsmi_ctx* ctx, double* x, int64_t n, double ar, double ai);
void vec_zaxpy(nsmi_ctx* ctx, double* y, const double* x, int64_t n, double ar, double ai);
// slots [slot, slot+1] <- sum conj(x) y
void vec_zdot_dev(nsmi_ctx* ctx, const double* x, const double* y, int64_t n, int slot);
void vec_zlincomb(nsmi_ctx* ctx, double* out, const double* const* V, const double* cr, const double* ci, int k,
                  int64_t n);
// complex GEMM (zgemm.hip): C = op(A) op(B), interleaved complex, optional conjugation
void gemm_c128(nsmi_ctx* ctx, const GemmDesc& d, const double* A, bool conjA, const double* B, bool conjB,
               double* C, int role);
// complex FP32 (interleaved float pairs) on FP32 MFMA, FP32 accumulation
void gemm_c64(nsmi_ctx* ctx, const GemmDesc& d, const float* A, bool conjA, const float* B, bool conjB, float* C,
              int role);
// One step of a complex network program: C = A B with B row-major K x N (conjugated
// when conjB); A element (m, k) at arow[m] + acol[k] and C element (m, n) at
// crow[m] + ccol[n] (complex elements; device tables) where given, else row-major.
// In the FP32 form (lo) A and C may be complex double (a_f64, c_f64), converted in
// the load and the store.
struct ZNetGemm {
  int64_t M = 0, N = 0, K = 0;
  const void* A = nullptr;
  bool a_f64 = false;
  const int64_t *arow = nullptr, *acol = nullptr;
  const void* B = nullptr;
  bool conjB = false;
  void* C = nullptr;
  bool c_f64 = false;
  const int64_t *crow = nullptr, *ccol = nullptr;
};
void gemm_cplx_net(nsmi_ctx* ctx, bool lo, const ZNetGemm& z);

// ---- MPO mixing (region.hip) --------------------------------------------
// Y[o][p][i] = sum_q Mx[p][q] X[o][q][i]
void mix_f64(nsmi_ctx* ctx, const double* X, double* Y, const double* Mx, int64_t O, int P, int Q,
             int64_t I, int cls);
void mix_f32(nsmi_ctx* ctx, const float* X, float* Y, const double* Mx, int64_t O, int P, int Q,
             int64_t I, int cls);

void small_sym_eigh(int n, const double* A, double* w, double* V);  // host Jacobi, ascending

// ---- tridiagonal reduction (eig.hip) ----------------------------------------
// Householder reduction of a symmetric n x n device matrix to tridiagonal form in
// LAPACK's dsytrd "lower" order, reflectors in place (one launch); false when n is outside
// [2, kSytrdMax] or the device cannot co-schedule the grid.
constexpr int kSytrdMax = 1024;
//
// Control words of a reduction (zero on entry): the words the host reads (an exchange that
// timed out, non-finite d or e, the state of the placement, the first column of the last block
// of 64 in which a workgroup gave up, or the number of columns once the first workgroup has
// finished), then the flag of the orthonormalisation that follows in the same call
// (orthonormalize_cols), then the counters of the placement, each on its own 128-byte line
// (all workgroups, one ticket line per XCD).
constexpr int kXcds = 8;
constexpr int kCtlFail = 32, kCtlNonFinite = 33, kCtlPlaced = 34, kCtlColumn = 35, kCtlHostWords = 4;
constexpr int kCtlOrthFail = 40;
constexpr int kCtlArrived = 64, kCtlTicket = 96;
constexpr int kCtlWords = kCtlTicket + 32 * kXcds;
constexpr unsigned kPlaced = 1, kUnplaced = 2;  // kCtlPlaced once it is decided (group.h)
// one asynchronous reduction: its exchange and control words, and the host copy of
// kCtlHostWords of them from kCtlFail on
struct SytrdRun {
  std::unique_ptr<Scratch> xch, flags;
  unsigned* host_flags = nullptr;  // in pinned stage memory
  int columns = 0;
};
// spread: the workgroups of a group go wherever there is room and not to one XCD
bool sytrd_launch(nsmi_ctx* ctx, double* A, int n, double* d, double* e, double* tau, SytrdRun& run,
                  bool spread = false);
// Whether groups of up to 32 workgroups on one XCD can be asked for on this device
bool one_xcd_groups(nsmi_ctx* ctx);
// runs launch(xcd) for a kernel whose group of at most 32 workgroups (two of them to a CU)
// runs on one XCD: the stream's place among the XCDs, see places.h
void launch_on_one_xcd(nsmi_ctx* ctx, const std::function<void(int)>& launch);
void xcd_places_release(int device, hipStream_t stream);
// whether a placement is to fail, by injection (tests); counts it.  A one-XCD group then asks
// for an XCD that is not there, one launched again starts with an arrival count out of reach
bool take_misplacement(nsmi_ctx* ctx);
constexpr unsigned kNeverArrived = 1u << 31;
// cooperative launch of a group over the device, alone among the groups (places.h); false, with
// nothing launched, when the device cannot hold all of its grid
bool launch_over_device(nsmi_ctx* ctx, const void* fn, int groups, int threads, void** args);
// enqueues the host copy of a launched reduction's control words
void reduction_readback(nsmi_ctx* ctx, SytrdRun& run, int columns);
// once the copy has arrived: whether the group never started (nothing written; launch again,
// spread, kRelaunches times)
constexpr int kRelaunches = 4;
inline bool reduction_unplaced(const SytrdRun& run) { return run.host_flags[kCtlPlaced - kCtlFail] == kUnplaced; }
// start value of a reduction's failure flag: 1 when the context has an injected timeout
// pending and the grid has G > 1 (the first workgroup then gives up before its first column,
// and the others in their first exchange)
unsigned reduction_fail0(nsmi_ctx* ctx, int G);
void sytrd_check(const SytrdRun& run);
// Zr <- (Q Z) with Q = H_0 ... H_{n-2} the reflectors of sytrd_launch's output (rho,
// tau; n <= 1024) and Z = Zr^T (Zr: k x n row-major, i.e. Z column-major n x k): what
// LAPACK dormtr("L", "L", "N") computes, as GEMMs and one triangular solve.
void apply_q_lower(nsmi_ctx* ctx, const double* rho, const double* tau, int n, double* Zr, int k);
// Zr <- rows of (Q Zr^T)^T for Q = H_0 ... H_{m-1}, H_i = I - tau_i v_i v_i^T, v_i the rows
// of Vt (m x len; a row with tau_i == 0 must be zero); m <= 2047.  Compact-WY (UT
// transform): three GEMMs and one triangular solve.
void apply_reflectors(nsmi_ctx* ctx, const double* Vt, const double* tau, int m, int64_t len, double* Zr, int k);

// ---- own dense SVD / tridiagonal eigensolver pieces (svd.hip) -------------------
// One-launch Householder bidiagonalisation of a tall r x s device matrix X (r >= s,
// row-major; reflectors left in place, see bidiag.h), d (s), e, tauR (s - 1), tauL (s).
// Enqueues the launch and the copy of its control words (as sytrd_launch); false
// with nothing launched when the size is outside the kernels' range or the grid cannot
// be co-scheduled.
constexpr int kBidiagMax = 2048, kBidiagRowsMax = 4096;
int bidiag_groups(int r, int s);
bool bidiag_launch(nsmi_ctx* ctx, double* X, int r, int s, double* d, double* e, double* tauL, double* tauR,
                   SytrdRun& run, bool spread = false);
// the Golub-Kahan off-diagonal (d_0, e_0, d_1, ..., d_{s-1}) of the bidiagonal (2 s - 1 entries)
void gk_offdiag(nsmi_ctx* ctx, const double* d, const double* e, int s, double* gk);
// eigenvalues of descending rank i0 .. i0 + count - 1 of the symmetric tridiagonal
// (diagonal a, zero when null; off-diagonal b), N <= kTriSolveMaxN (with a diagonal N <= 4081),
// into lam (device)
constexpr int kTriSolveMaxN = 4096;
void tri_bisect(nsmi_ctx* ctx, const double* a, const double* b, int N, int i0, int count, double* lam);
// eigenvectors for the m eigenvalues lam (device) by inverse iteration, as columns of Y
// (len x m row-major): the whole vector (part < 0, len = N) or its even / odd entries
// (part 0 / 1), normalised
void tri_invit(nsmi_ctx* ctx, const double* a, const double* b, int N, const double* lam, int m, double* Y, int part);
// columns of Y (len x k, row-major) made orthonormal in order (block CGS2 + CholQR2);
// *fail (device word) is raised when they are not numerically independent
void orthonormalize_cols(nsmi_ctx* ctx, double* Y, int64_t len, int k, unsigned* fail);
// the reflector rows of bidiag_launch's output for apply_reflectors: left (s x r) and right ((s - 1) x s)
void bidiag_reflectors_left(nsmi_ctx* ctx, const double* X, int r, int s, const double* tau, double* Vt);
void bidiag_reflectors_right(nsmi_ctx* ctx, const double* X, int s, const double* tau, double* Vt);
// Batched Jacobi eigensolver for small symmetric matrices (one workgroup each, LDS
// resident): eigenvectors overwrite a (column-major, dsyevd layout), eigenvalues
// (unsorted) go to w.  Enqueues only: *unconverged (host memory) receives the
// not-converged flag once the stream reaches it; the caller synchronises.
constexpr int kJacobiMax = 40;
struct JacobiJob {
  double* a;
  double* w;
  int n;
};
void jacobi_eig_batched(nsmi_ctx* ctx, const std::vector<JacobiJob>& jobs, unsigned* unconverged);

// complex factorize / QR (zfactorize.hip); the truncation rule is passed in
void zfactorize(nsmi_ctx* ctx, const nsmi_tensor* theta, int n_row_dims, int rows_trailing, const nsmi_trunc* trunc,
                int route, int64_t maxdim, int64_t mindim, nsmi_tensor** Uout, nsmi_tensor** Cout, int64_t* kept,
                double* truncerr, double* total,
                int64_t (*truncate)(std::vector<double>&, int64_t, int64_t, double, double*, double*));
void zqr(nsmi_ctx* ctx, const nsmi_tensor* A, int n_row_dims, int rows_trailing, nsmi_tensor** Qout,
         nsmi_tensor** Rout);
// Thin QR of a small row-major m x nc matrix A (or of A^T with trailing), real or
// complex, in one launch: writes Q and R in the layouts of nsmi_qr (diag(R) >= 0) and
// returns true; false (nothing launched) when the matrix exceeds 2048 elements or its
// rank bound 64.
bool qr_one(nsmi_ctx* ctx, const double* A, int64_t m, int64_t nc, bool trailing, bool cplx, double* Q, double* R);

// general network contractions (network.hip): a contraction program executed as
// an H_eff (tree regions)
struct NetProgram;
void net_apply(nsmi_ctx* ctx, NetProgram* p, const double* x, double* y);
void net_release(nsmi_ctx* ctx, NetProgram* p);
int64_t net_size(const NetProgram* p);
bool net_is_complex(const NetProgram* p);
nsmi_heff* heff_wrap_net(NetProgram* p);  // region.hip: an nsmi_heff that runs the program

// block-sparse (QN) block programs (blocksparse.hip)
struct BsProgram;
void bs_run(nsmi_ctx* ctx, BsProgram* p, const double* x, double* y);
void bs_release(nsmi_ctx* ctx, BsProgram* p);
void tuner_free(nsmi_ctx* ctx);  // the autotuner's events and table (context teardown)
nsmi_heff* heff_wrap_bs(BsProgram* p, int64_t n);  // region.hip; n < 0: not a square operator
BsProgram* heff_bs_program(nsmi_heff* op);

// the no-allocation entry point (noalloc.hip): per-device set-up at context creation,
// and the operators it serves (real chain operators, FP64 and FP32 forms)
void noalloc_setup(int device);
bool heff_noalloc_ok(const nsmi_heff* op);

// H_eff operator access for the Krylov solvers (krylov.cpp)
void heff_apply_dev(nsmi_ctx* ctx, nsmi_heff* op, const double* x, double* y);
int64_t heff_size(const nsmi_heff* op);
bool heff_is_complex(const nsmi_heff* op);

}  // namespace nsmi
