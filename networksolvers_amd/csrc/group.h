// Exchange between the workgroups of the one-launch reductions (bidiag.h, sytrd.h).
//
// A grid barrier with an agent-scope release and acquire writes back and invalidates
// L2 lines; measured (256 threads per workgroup, in-bounds probe): 1.0 us at 12
// workgroups spread over the XCDs, 1.9 us at 12 on one XCD, 7.3 us at 256; and the data
// still has to be read after it.  Here there is no barrier: a workgroup reads the words
// that the others write until none of them is "empty" (a NaN pattern that no arithmetic
// makes), so one trip through the L2 carries both the value and its readiness.
//
// The words of a vector rotate over three buffers, step j using buffer j mod 3, all of
// them empty at the start.  Once a thread has read step j's words of the others it
// empties its own word of buffer (j - 1) mod 3: everyone it has heard from in step j had
// finished reading step j - 1.  Before it writes its word of step j + 1 it waits for its
// own earlier stores, so whoever sees that word also sees the emptied one, which is
// next polled in step j + 2.  This needs every thread to handle the same word in every
// step and to hear, for that word, from everyone who reads what it empties.
//
// The workgroups that exchange most are placed on one XCD where they fit, so that the
// words stay in that XCD's L2: they are written by relaxed atomic stores of workgroup scope
// (never by plain ones, which the compiler may split, merge or move; they stop in the L2
// that the group shares, as every store that leaves a CU does) and read by relaxed agent-scope
// loads (never from the CU's own cache; 0.16 us inside an XCD, 0.3 us across).  Words that
// cross XCDs are written by relaxed agent-scope stores, which leave nothing in the writer's L2.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "internal.h"
#include "wave.h"

namespace nsmi {
namespace {

// the empty word: a signalling NaN's pattern (arithmetic only makes quiet ones)
constexpr unsigned long long kEmpty = 0x7FF4C0DE5EED0001ull;
__device__ inline bool is_empty(double v) { return (unsigned long long)__double_as_longlong(v) == kEmpty; }
__device__ inline double empty_word() { return __longlong_as_double((long long)kEmpty); }
// input may hold any pattern; what is published as read must not look empty
__device__ inline double not_empty(double v) { return is_empty(v) ? __longlong_as_double(0x7FF8000000000000ll) : v; }

// the XCD this workgroup runs on (0 .. 7)
__device__ inline int xcd_id() {
  unsigned x;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
  return int(x) & (kXcds - 1);
}

template <class T>
__device__ inline T ld_agent(const T* p) {
  return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline void st_agent(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned add_agent(unsigned* p) {
  return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a word for readers inside the group; local: the group shares an L2
__device__ inline void st_group(double* p, double v, bool local) {
  if (local)
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else
    st_agent(p, v);
}
// this wave's stores have reached the level their readers load from
__device__ inline void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Loads N words, addr(i) their addresses, until none is empty: all of them again in every
// round, with a pause of 256 cycles between rounds.  Without the pause the polls keep the L2
// so busy that the awaited stores take 10x longer (394 columns, 14 workgroups of one
// XCD: 36 us per step against 3); loading only what is still missing needs branches and took
// 5.5.  False once it gives up (the failure flag raised) or another workgroup has raised the
// flag.
template <int N, class Addr>
__device__ __forceinline__ bool load_words(double (&v)[N], const Addr& addr, unsigned* fail) {
  for (unsigned spins = 0;;) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = ld_agent(addr(i));
    bool missing = false;
#pragma unroll
    for (int i = 0; i < N; ++i) missing = missing || is_empty(v[i]);
    if (!__any(missing)) return true;
    __builtin_amdgcn_s_sleep(4);
    if ((++spins & 255u) == 0u) {
      if (ld_agent(fail) != 0u) return false;
      if (spins > (1u << 21)) {
        atomicOr(fail, 1u);
        return false;
      }
    }
  }
}

// the host raised the failure flag before the launch (an injected time-out): the first
// workgroup of the group leaves at once, and all the others once their polls see the flag
__device__ inline bool told_to_give_up(const unsigned* ctl, int g) { return g == 0 && ld_agent(ctl + kCtlFail) != 0u; }
// one lane's record of where the reduction ended (the column itself, kept for this, costs the
// register-full plans spills)
__device__ inline void ended_at(unsigned* ctl, int column) { atomicMax(ctl + kCtlColumn, unsigned(column)); }

// ---- placement.  No workgroup of a group does any work before the group's placement is
// decided, once, by a compare-and-swap of kCtlPlaced from 0: placed when all of the group's
// workgroups are on the device, unplaced when that cannot be or takes too long; then all of
// them leave, nothing has been written, and the host launches again.  So a group that is
// only partly resident never holds its CUs for good.
__device__ inline void decide(unsigned* ctl, unsigned state) {
  unsigned undecided = 0u;
  __hip_atomic_compare_exchange_strong(ctl + kCtlPlaced, &undecided, state, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  stores_done();
}
// one lane's wait for the decision: a million polls (about a tenth of a second) at most
__device__ inline bool placed(unsigned* ctl) {
  for (unsigned spins = 0;; ++spins) {
    const unsigned state = ld_agent(ctl + kCtlPlaced);
    if (state != 0u) return state == kPlaced;
    if (spins == (1u << 20)) decide(ctl, kUnplaced);
  }
}

// Placement of a group on XCD `want`: the grid holds 8 G workgroups, of which the first G on
// that XCD (their tickets give the order) form the group.  All the others leave at once:
// they must not keep their CUs, where the members of other groups may be waiting to start.
// The dispatcher hands workgroups out to the XCDs in turn, so the wanted one gets G; if every
// workgroup has arrived and it did not, the last one to arrive says so.  Returns the
// workgroup's index in the group, -1 to leave.
__device__ inline int place_one_xcd(unsigned* ctl, int G, int want, int* s_place) {
  if (threadIdx.x == 0) {
    int place = -1;
    if (xcd_id() == want) {
      const unsigned t = add_agent(ctl + kCtlTicket + 32 * want);
      if (t < unsigned(G)) place = int(t);
      if (t == unsigned(G) - 1u) decide(ctl, kPlaced);
    }
    if (add_agent(ctl + kCtlArrived) == gridDim.x - 1u) decide(ctl, kUnplaced);
    if (place >= 0 && !placed(ctl)) place = -1;
    *s_place = place;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*s_place);
}

// Placement of a group wherever its workgroups are, in the grid's order.
__device__ inline int place_spread(unsigned* ctl, int* s_place) {
  if (threadIdx.x == 0) {
    if (add_agent(ctl + kCtlArrived) == gridDim.x - 1u) decide(ctl, kPlaced);
    *s_place = placed(ctl) ? int(blockIdx.x) : -1;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*s_place);
}

// Placement of a launch over all XCDs, 8 GW workgroups: XCD x and index w inside it.
// Where the dispatcher did not hand GW workgroups to each XCD (or the host asks for it,
// want < 0) the groups are formed by the grid index instead (local = false).
__device__ inline bool place_all_xcds(unsigned* ctl, int GW, int want, int* x, int* w, bool* local, int* s_place) {
  if (threadIdx.x == 0) {
    const int xc = xcd_id();
    const unsigned t = add_agent(ctl + kCtlTicket + 32 * xc);
    stores_done();
    if (add_agent(ctl + kCtlArrived) == gridDim.x - 1u) decide(ctl, kPlaced);
    int p = -1;
    if (placed(ctl)) {
      bool even = want >= 0;
      for (int q = 0; q < kXcds; ++q) even = even && ld_agent(ctl + kCtlTicket + 32 * q) == unsigned(GW);
      p = even ? int(t) * kXcds + xc : (int(blockIdx.x) | (1 << 30));
    }
    *s_place = p;
  }
  __syncthreads();
  const int p = __builtin_amdgcn_readfirstlane(*s_place);
  if (p < 0) return false;
  *local = !(p & (1 << 30));
  *x = (p & ~(1 << 30)) % kXcds;
  *w = (p & ~(1 << 30)) / kXcds;
  return true;
}

// Runs block(CA) for the column blocks at cb = 0, 64, ... below stop, CA the number of blocks
// held by the registers it works on (those from cb to the width, rounded up to a multiple
// of STEP): fewer as the matrix shrinks, every register index a constant.
template <int CA, int STEP, class F>
__device__ __forceinline__ bool column_blocks(int stop, int width, int& cb, const F& block) {
  while (cb < stop && (width - cb + 63) / 64 > CA - STEP) {
    if (!block(std::integral_constant<int, CA>())) return false;
    cb += 64;
  }
  if constexpr (CA > STEP) return column_blocks<CA - STEP, STEP>(stop, width, cb, block);
  return true;
}

// empties the exchange words and zeroes the control words (fail0, arrived0: start values of
// the failure flag and of the arrival count) before a reduction; the first ps words are slots of `slot` words, of
// which every group of `per` fills the first `used`: the others become zeros
__global__ void k_reduction_init(double* __restrict__ xch, size_t n, size_t ps, unsigned slot, unsigned per,
                                 unsigned used, unsigned* __restrict__ ctl, int nctl, unsigned fail0,
                                 unsigned arrived0) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < size_t(nctl)) ctl[i] = int(i) == kCtlFail ? fail0 : int(i) == kCtlArrived ? arrived0 : 0u;
  for (size_t k = i; k < n; k += size_t(gridDim.x) * blockDim.x)
    xch[k] = k < ps && unsigned(k) / slot % per >= used ? 0.0 : empty_word();
}

// A Householder reflector's scalars for [alpha, x] with sigma2 = |x|^2 (LAPACK dlarfg):
// beta = -sign(alpha) sqrt(alpha^2 + sigma2), tau = (beta - alpha) / beta, scal = 1 /
// (alpha - beta).  With n = sqrt(alpha^2 + sigma2): tau = (n + |alpha|) / n, scal =
// sign(alpha) / (n + |alpha|), no cancellation.  1 / n and n by Goldschmidt's iteration
// from the hardware reciprocal square root (g -> n and h -> 1 / (2 n) take the same factor
// 1 + e, e = 1/2 - g h, twice), n corrected by its residual, 1 / (n +
// |alpha|) by the refined reciprocal: each within an ulp or two, on a dependency chain
// less than half as long as a rounded square root and two divisions (450 cycles).
__device__ inline void reflector(double alpha, double sigma2, double* beta, double* tau, double* scal) {
  if (sigma2 == 0.0) {
    *beta = alpha;
    *tau = 0.0;
    *scal = 0.0;
    return;
  }
  const double n2 = fma(alpha, alpha, sigma2);
  if (!(n2 > 1e-280 && n2 < 1e280)) {  // denormals, overflow, NaN: the rounded operations
    const double b = -copysign(sqrt(n2), alpha);
    *beta = b;
    *tau = (b - alpha) / b;
    *scal = 1.0 / (alpha - b);
    return;
  }
  double r = __builtin_amdgcn_rsq(n2);
  double g = n2 * r, h = 0.5 * r;
  double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  g = fma(fma(-g, g, n2), h, g);  // n
  const double a = fabs(alpha), t = g + a;
  double q = __builtin_amdgcn_rcp(t);
  q = fma(fma(-t, q, 1.0), q, q);
  q = fma(fma(-t, q, 1.0), q, q);
  *beta = -copysign(g, alpha);
  *tau = t * (2.0 * h);
  *scal = copysign(q, alpha);
}

// ---- wave-wide sums of R values at once, fewer instructions than wave_totals: two
// values share a register from the first step on (the half-wave and 16-lane swaps
// move value 2 i + 1 into the lanes that value 2 i no longer needs), so R values cost
// R / 2 + R / 4 swap-adds and 4 DPP steps on R / 4 registers.  Every lane gets the totals.
__device__ inline double swap_add32(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(unsigned(__double2loint(a)), unsigned(__double2loint(b)), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(unsigned(__double2hiint(a)), unsigned(__double2hiint(b)), false, false);
  return __hiloint2double(int(hi[0]), int(lo[0])) + __hiloint2double(int(hi[1]), int(lo[1]));
}
__device__ inline double swap_add16(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane16_swap(unsigned(__double2loint(a)), unsigned(__double2loint(b)), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(unsigned(__double2hiint(a)), unsigned(__double2hiint(b)), false, false);
  return __hiloint2double(int(hi[0]), int(lo[0])) + __hiloint2double(int(hi[1]), int(lo[1]));
}
template <int R>
__device__ inline void wave_sums(double (&a)[R]) {
  constexpr int R2 = (R + 1) / 2, R4 = (R2 + 1) / 2;
  double t[R2], u[R4];
#pragma unroll
  for (int i = 0; i < R2; ++i) t[i] = swap_add32(a[2 * i], a[2 * i + 1 < R ? 2 * i + 1 : 2 * i]);
#pragma unroll
  for (int i = 0; i < R4; ++i) u[i] = swap_add16(t[2 * i], t[2 * i + 1 < R2 ? 2 * i + 1 : 2 * i]);
#pragma unroll
  for (int i = 0; i < R4; ++i) u[i] += dpp_mov<0xB1, 0xF>(u[i]);  // quad_perm [1,0,3,2]
#pragma unroll
  for (int i = 0; i < R4; ++i) u[i] += dpp_mov<0x4E, 0xF>(u[i]);  // quad_perm [2,3,0,1]
#pragma unroll
  for (int i = 0; i < R4; ++i) u[i] += dpp_mov<0x141, 0xF>(u[i]);  // row_half_mirror
#pragma unroll
  for (int i = 0; i < R4; ++i) u[i] += dpp_mov<0x140, 0xF>(u[i]);  // row_mirror
  // 16-lane rows of u[i] hold the values 4 i, 4 i + 2, 4 i + 1, 4 i + 3
#pragma unroll
  for (int i = 0; i < R; ++i) a[i] = lane_bcast(u[i / 4], (i & 2 ? 16 : 0) + (i & 1 ? 32 : 0));
}

}  // namespace
}  // namespace nsmi
