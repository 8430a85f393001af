// Plans and launches of the one-launch bidiagonalisation (bidiag.h), and the XCDs that
// its one-XCD groups run on.
#include "bidiag.h"

#include <algorithm>
#include <mutex>

#include "internal.h"

namespace nsmi {
namespace {

// Two groups at a time may hold an XCD (kGroupsPerXcd: their workgroups, at most one for
// each of its CUs, fit two to a CU, and nothing but their members stays on the device, see
// place_one_xcd), so both become resident; with a third one each could have a part of its
// CUs and none enough.  Each stream that launches such groups is given one of the 16 places
// (8 XCDs x 2) for its life, spread over the XCDs first.  With more than 16 streams a place
// is shared: a launch then waits for what the others sharing it have queued (an event per
// stream, under the lock, so that two of them cannot pass each other).
constexpr int kCusPerXcd = 32, kGroupsPerXcd = 2;
struct XcdPlaces {
  std::mutex mu;
  std::vector<hipStream_t> users[kGroupsPerXcd * kXcds];
  hipEvent_t ev = nullptr;
};
XcdPlaces& places_of(int device) {
  static std::mutex mu;
  static std::map<int, XcdPlaces> all;
  std::lock_guard<std::mutex> lock(mu);
  return all[device];
}

}  // namespace

void launch_on_one_xcd(nsmi_ctx* ctx, const std::function<void(int)>& launch) {
  XcdPlaces& p = places_of(ctx->device);
  std::lock_guard<std::mutex> lock(p.mu);
  int at = -1, best = 0;
  for (int i = 0; i < kGroupsPerXcd * kXcds; ++i) {
    for (hipStream_t s : p.users[i])
      if (s == ctx->stream) at = i;
    if (p.users[i].size() < p.users[best].size()) best = i;
  }
  if (at < 0) {
    p.users[best].push_back(ctx->stream);
    at = best;
  }
  for (hipStream_t s : p.users[at]) {
    if (s == ctx->stream) continue;
    if (!p.ev) NSMI_HIP(hipEventCreateWithFlags(&p.ev, hipEventDisableTiming));
    NSMI_HIP(hipEventRecord(p.ev, s));
    NSMI_HIP(hipStreamWaitEvent(ctx->stream, p.ev, 0));
  }
  launch(at % kXcds);
}

void xcd_places_release(int device, hipStream_t stream) {
  XcdPlaces& p = places_of(device);
  std::lock_guard<std::mutex> lock(p.mu);
  for (auto& u : p.users) u.erase(std::remove(u.begin(), u.end(), stream), u.end());
}

unsigned reduction_fail0(nsmi_ctx* ctx, int G) {
  if (G <= 1 || ctx->inject_timeouts <= 0) return 0u;
  --ctx->inject_timeouts;
  return 1u;
}

bool take_misplacement(nsmi_ctx* ctx) {
  if (ctx->inject_misplaced <= 0) return false;
  --ctx->inject_misplaced;
  return true;
}

bool one_xcd_groups(nsmi_ctx* ctx) {
  int xcds = 0, ncu = 0;
  NSMI_HIP(hipDeviceGetAttribute(&xcds, hipDeviceAttributeNumberOfXccs, ctx->device));
  NSMI_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device));
  return xcds == kXcds && ncu >= kXcds * kCusPerXcd;
}

bool launch_cooperative(nsmi_ctx* ctx, const void* fn, int groups, int threads, void** args) {
  int coop = 0, ncu = 0, per_cu = 0;
  NSMI_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, ctx->device));
  NSMI_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device));
  NSMI_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, 0));
  if (!coop || per_cu < 1 || groups > ncu * per_cu) return false;
  const hipError_t st = hipLaunchCooperativeKernel(fn, dim3(unsigned(groups)), dim3(unsigned(threads)), args, 0,
                                                   ctx->stream);
  if (st != hipSuccess) (void)hipGetLastError();
  return st == hipSuccess;
}

void reduction_readback(nsmi_ctx* ctx, SytrdRun& run) {
  run.host_flags = static_cast<unsigned*>(stage_take(ctx, kCtlHostWords * sizeof(unsigned)));
  for (int i = 0; i < kCtlHostWords; ++i) run.host_flags[i] = 0u;
  NSMI_HIP(hipMemcpyAsync(run.host_flags, run.flags->as<unsigned>() + kCtlFail, kCtlHostWords * sizeof(unsigned),
                          hipMemcpyDeviceToHost, ctx->stream));
}

namespace {

struct BidiagPlan {
  const void* fn = nullptr;
  BidiagMode mode = kOneGroup;
  int cl = 1, threads = 0, gmax = 1;
  int rows = 0;  // rows per workgroup
};
template <int CL, int RW, int NW, BidiagMode MODE, int GMAX>
BidiagPlan plan_of() {
  static_assert(MODE == kOneGroup || GMAX <= kCusPerXcd, "at most one workgroup for each CU of an XCD");
  return {reinterpret_cast<const void*>(k_bidiag<CL, RW, NW, MODE, GMAX>), MODE, CL, 64 * NW, GMAX, RW * NW};
}

// Measured on gfx950 (us per column; the barrier form with 32-row workgroups spread over
// the XCDs that these plans replaced: 7.1 at 384 x 384, 17.5 at 1024 x 1024, 28.6 at
// 2048 x 2048):
//   one workgroup: 1.4 at 32 x 32 (1.7 on 8 workgroups), 1.95 at 64 x 64 (1.7 on 8
//   workgroups of one XCD), 3.7 at 128 x 128 (1.8 on 16);
//   one XCD, everyone reading everyone's sums: 1.9 at 128 x 60, 1.8 at 128 x 128, 2.1 at 256 x
//   128; 2.26 at 256 x 256 against 2.21 with the columns sliced, 4.0 against 2.5 at 422 x 394;
//   one XCD, sliced, as few rows per workgroup as 32 workgroups allow: 2.6 at 512 x 512 (3.0
//   with 16 workgroups of twice the rows), 2.9 at 1000 x 256, 3.7 at 2000 x 128;
//   all XCDs: 3.7 at 512 x 512, 4.2 at 700 x 700, 4.5 at 1000 x 1000 (5.2 on one XCD), 5.9 at
//   2048 x 2048, 5.8 at 4000 x 1000.
// One-XCD groups go out as ordinary launches (at most 32 workgroups, places_of); the
// others need up to one workgroup on every CU and take the cooperative launch, and so does a
// one-XCD group that was not placed or that the device has no XCDs for.
BidiagPlan bidiag_plan(int r, int s) {
  if (s <= 64) {
    if (r <= 32) return plan_of<1, 4, 8, kOneGroup, 1>();
    if (r <= 64) return plan_of<1, 2, 4, kOneXcd, 8>();
    if (r <= 128) return plan_of<1, 4, 4, kOneXcd, 8>();
    if (r <= 256) return plan_of<1, 4, 8, kOneXcd, 8>();
    if (r <= 2048) return plan_of<1, 8, 8, kOneXcdSliced, 32>();
    return plan_of<1, 8, 4, kAllXcds, 32>();
  }
  if (s <= 128) {
    if (r <= 128) return plan_of<2, 2, 4, kOneXcd, 16>();
    if (r <= 256) return plan_of<2, 4, 4, kOneXcd, 16>();
    if (r <= 1024) return plan_of<2, 4, 8, kOneXcdSliced, 32>();
    if (r <= 2048) return plan_of<2, 8, 8, kOneXcdSliced, 32>();
    return plan_of<2, 8, 4, kAllXcds, 32>();
  }
  if (s <= 256) {
    if (r <= 256) return plan_of<4, 2, 4, kOneXcdSliced, 32>();
    if (r <= 512) return plan_of<4, 2, 8, kOneXcdSliced, 32>();
    if (r <= 1024) return plan_of<4, 4, 8, kOneXcdSliced, 32>();
    return plan_of<4, 4, 4, kAllXcds, 32>();
  }
  if (s <= 512) return r <= 512 ? plan_of<8, 2, 8, kOneXcdSliced, 32>() : plan_of<8, 4, 4, kAllXcds, 32>();
  if (s <= 1024) return r <= 2048 ? plan_of<16, 2, 4, kAllXcds, 32>() : plan_of<16, 2, 8, kAllXcds, 32>();
  return plan_of<32, 2, 4, kAllXcds, 32>();
}

// workgroups of a group (of an XCD): enough for the rows, and for slices of at most 64
// columns; 0 when the plan has no room
int plan_groups(const BidiagPlan& p, int r, int s) {
  int g = (r + p.rows - 1) / p.rows;
  if (p.mode == kAllXcds) g = (g + kXcds - 1) / kXcds;
  if (p.mode == kAllXcds || p.mode == kOneXcdSliced) g = std::max(g, (s + 63) / 64);
  return g <= (p.mode == kOneGroup ? 1 : p.gmax) ? g : 0;
}

}  // namespace

int bidiag_groups(int r, int s) {
  if (s < 1 || r < s || s > kBidiagMax || r > kBidiagRowsMax) return 0;
  const BidiagPlan p = bidiag_plan(r, s);
  const int g = plan_groups(p, r, s);
  return p.mode == kAllXcds ? kXcds * g : g;
}

bool bidiag_launch(nsmi_ctx* ctx, double* X, int r, int s, double* d, double* e, double* tauL, double* tauR,
                   SytrdRun& run, bool spread) {
  const int G = bidiag_groups(r, s);
  if (G == 0) return false;
  const BidiagPlan p = bidiag_plan(r, s);
  int groups = plan_groups(p, r, s);
  BidiagExchange x{};
  if (p.mode != kOneGroup) x = bidiag_exchange(p.cl, p.gmax, groups, p.mode == kAllXcds);
  run.xch.reset(new Scratch(ctx, sizeof(double) * std::max<size_t>(x.words, 1)));
  run.flags.reset(new Scratch(ctx, sizeof(unsigned) * kCtlWords));
  unsigned* ctl = run.flags->as<unsigned>();
  double* xp = run.xch->as<double>();
  const unsigned nblk = unsigned(std::min<size_t>(1024, (std::max<size_t>(x.words, kCtlWords) + 255) / 256));
  hipLaunchKernelGGL(k_reduction_init, dim3(nblk), dim3(256), 0, ctx->stream, xp, x.words, x.ps_words,
                     unsigned(3 * 64 * p.cl), unsigned(std::max(x.per, 1)), unsigned(x.used), ctl, int(kCtlWords),
                     reduction_fail0(ctx, G));
  NSMI_LAUNCH_CHECK();
  int rr = r, ss = s, want = -1;
  void* args[] = {&X, &rr, &ss, &d, &e, &tauL, &tauR, &xp, &ctl, &groups, &want};
  {
    // algorithmic work of a Householder bidiagonalisation: 4 s^2 (r - s / 3) flops
    ProfScope ps(ctx, NSMI_K_FACT_REDUCE, 4.0 * double(s) * s * (double(r) - double(s) / 3.0),
                 16.0 * double(r) * s);
    if (p.mode == kOneGroup) {
      NSMI_HIP(hipLaunchKernel(p.fn, dim3(1), dim3(unsigned(p.threads)), args, 0, ctx->stream));
    } else if (p.mode == kAllXcds || spread || !one_xcd_groups(ctx)) {
      if (p.mode == kAllXcds && !take_misplacement(ctx)) want = 0;
      if (!launch_cooperative(ctx, p.fn, G, p.threads, args)) return false;
    } else {
      launch_on_one_xcd(ctx, [&](int xcd) {
        want = take_misplacement(ctx) ? kXcds : xcd;  // kXcds: none has this number
        NSMI_HIP(hipLaunchKernel(p.fn, dim3(unsigned(kXcds * G)), dim3(unsigned(p.threads)), args, 0, ctx->stream));
      });
    }
  }
  reduction_readback(ctx, run);
  return true;
}

}  // namespace nsmi
