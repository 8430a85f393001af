// Which of the reductions' launches may be on the device together.
//
// A group whose workgroups wait for each other must not share the device with so many others
// that each of them has a part of its CUs and none enough.  Two kinds:
//   * a group on one XCD: at most one workgroup for each of its 32 CUs, each of at most half
//     a CU's registers and less than a third of its LDS, so two groups fit an XCD (kPerXcd);
//   * a group over the device (all XCDs, or spread): up to a whole CU each on all 256, so it is
//     alone among the groups.
// Kernels without waits come and go beside them.
//
// Each stream that launches one-XCD groups has one of the 16 places (8 XCDs x 2) for its
// life, spread over the XCDs first; with more than 16 streams places are shared.  A launch is
// told which streams it must wait for (whatever they have queued) and whether for the last
// group over the device:
//   * one-XCD: for the other streams of its place, and for the last group over the device;
//   * over the device: for every stream that launched a one-XCD group since the last group
//     over the device, and for that one.
// Other processes on the device are not seen.  Each starts its places at an XCD of its own
// (first), so that a few processes of few streams each stay apart; where too many groups meet all
// the same, the placement ends without a group having started and it is launched again
// (group.h).
//
// The caller holds a lock from the question to its launch, so launches are ordered as they
// asked and never wait in a circle.  Host code without HIP, tested as such.
#pragma once
#include <algorithm>
#include <vector>

namespace nsmi {

template <class Stream>
class XcdPlaces {
 public:
  static constexpr int kXcdCount = 8, kCusPerXcd = 32, kPerXcd = 2, kPlaces = kXcdCount * kPerXcd;
  struct Order {
    int xcd = -1;
    std::vector<Stream> streams;  // wait for what these have queued
    bool device = false;          // wait for the last group over the device
  };

  explicit XcdPlaces(unsigned first = 0) : first_(first) {}

  Order one_xcd(Stream s) {
    int at = -1, best = 0;
    for (int i = 0; i < kPlaces; ++i) {
      for (const User& u : users_[i])
        if (u.s == s) at = i;
      if (users_[i].size() < users_[best].size()) best = i;
    }
    if (at < 0) {
      at = best;
      users_[at].push_back(User{s, false});
    }
    Order o;
    o.xcd = int((unsigned(at) + first_) % kXcdCount);
    for (User& u : users_[at]) {
      if (u.s == s)
        u.active = true;
      else
        o.streams.push_back(u.s);
    }
    o.device = device_busy_ && device_stream_ != s;
    return o;
  }

  Order over_device(Stream s) {
    Order o;
    for (auto& place : users_)
      for (User& u : place) {
        if (u.active && u.s != s) o.streams.push_back(u.s);
        u.active = false;
      }
    o.device = device_busy_ && device_stream_ != s;
    device_stream_ = s;
    device_busy_ = true;
    return o;
  }

  // a stream that has drained and launches no more
  void release(Stream s) {
    for (auto& place : users_)
      place.erase(std::remove_if(place.begin(), place.end(), [&](const User& u) { return u.s == s; }), place.end());
    if (device_busy_ && device_stream_ == s) device_busy_ = false;
  }

 private:
  struct User {
    Stream s;
    bool active;  // a one-XCD group launched since the last group over the device
  };
  unsigned first_;
  std::vector<User> users_[kPlaces];
  Stream device_stream_{};
  bool device_busy_ = false;
};

}  // namespace nsmi
