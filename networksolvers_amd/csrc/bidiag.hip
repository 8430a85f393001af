// Plans and launches of the one-launch bidiagonalisation (bidiag.h), and the XCDs that
// its one-XCD groups run on.
#include "bidiag.h"

#include <unistd.h>

#include <algorithm>
#include <mutex>

#include "internal.h"
#include "places.h"

namespace nsmi {
namespace {

struct DevicePlaces {
  std::mutex mu;
  XcdPlaces<hipStream_t> places{unsigned(getpid())};
  hipEvent_t ev = nullptr;         // for the waits on streams
  hipEvent_t device_ev = nullptr;  // the last group over the device
};
DevicePlaces& places_of(int device) {
  static std::mutex mu;
  static std::map<int, DevicePlaces> all;
  std::lock_guard<std::mutex> lock(mu);
  return all[device];
}

void wait_in_order(nsmi_ctx* ctx, DevicePlaces& p, const XcdPlaces<hipStream_t>::Order& o) {
  for (hipStream_t s : o.streams) {
    if (!p.ev) NSMI_HIP(hipEventCreateWithFlags(&p.ev, hipEventDisableTiming));
    NSMI_HIP(hipEventRecord(p.ev, s));
    NSMI_HIP(hipStreamWaitEvent(ctx->stream, p.ev, 0));
  }
  if (o.device && p.device_ev) NSMI_HIP(hipStreamWaitEvent(ctx->stream, p.device_ev, 0));
}

}  // namespace

void launch_on_one_xcd(nsmi_ctx* ctx, const std::function<void(int)>& launch) {
  DevicePlaces& p = places_of(ctx->device);
  std::lock_guard<std::mutex> lock(p.mu);
  const auto o = p.places.one_xcd(ctx->stream);
  wait_in_order(ctx, p, o);
  launch(o.xcd);
}

bool launch_over_device(nsmi_ctx* ctx, const void* fn, int groups, int threads, void** args) {
  int coop = 0, ncu = 0, per_cu = 0;
  NSMI_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, ctx->device));
  NSMI_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device));
  NSMI_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, 0));
  if (!coop || per_cu < 1 || groups > ncu * per_cu) return false;
  DevicePlaces& p = places_of(ctx->device);
  std::lock_guard<std::mutex> lock(p.mu);
  if (!p.device_ev) NSMI_HIP(hipEventCreateWithFlags(&p.device_ev, hipEventDisableTiming));
  wait_in_order(ctx, p, p.places.over_device(ctx->stream));
  const hipError_t st = hipLaunchCooperativeKernel(fn, dim3(unsigned(groups)), dim3(unsigned(threads)), args, 0,
                                                   ctx->stream);
  if (st != hipSuccess) (void)hipGetLastError();
  NSMI_HIP(hipEventRecord(p.device_ev, ctx->stream));
  return st == hipSuccess;
}

void xcd_places_release(int device, hipStream_t stream) {
  DevicePlaces& p = places_of(device);
  std::lock_guard<std::mutex> lock(p.mu);
  p.places.release(stream);
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
  return xcds == kXcds && ncu >= kXcds * XcdPlaces<hipStream_t>::kCusPerXcd;
}

void reduction_readback(nsmi_ctx* ctx, SytrdRun& run, int columns) {
  run.columns = columns;
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
  static_assert(MODE == kOneGroup || GMAX <= XcdPlaces<hipStream_t>::kCusPerXcd,
                "at most one workgroup for each CU of an XCD");
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
// One-XCD groups go out as ordinary launches (at most 32 workgroups, places.h); the
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
                     reduction_fail0(ctx, G), spread && take_misplacement(ctx) ? kNeverArrived : 0u);
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
      if (!launch_over_device(ctx, p.fn, G, p.threads, args)) return false;
    } else {
      launch_on_one_xcd(ctx, [&](int xcd) {
        want = take_misplacement(ctx) ? kXcds : xcd;  // kXcds: none has this number
        NSMI_HIP(hipLaunchKernel(p.fn, dim3(unsigned(kXcds * G)), dim3(unsigned(p.threads)), args, 0, ctx->stream));
      });
    }
  }
  reduction_readback(ctx, run, s);
  return true;
}

}  // namespace nsmi
