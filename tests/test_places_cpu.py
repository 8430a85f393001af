"""The order of the reductions' launches (csrc/places.h), in random programs of up to 40 streams:
at no time can three one-XCD groups be on one XCD, or a group over the device beside another
group.  The harness follows what each launch is told to wait for and derives which launches
are unordered, that is, may be on the device together."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "networksolvers_amd", "csrc")

HARNESS = r"""
#include <bitset>
#include <cstdio>
#include <cstdlib>
#include <random>
#include "places.h"
constexpr int N = 400;                       // launches
using Past = std::bitset<N>;                 // launches that have ended before something
int main(int argc, char** argv) {
  const int seed = std::atoi(argv[1]), streams = std::atoi(argv[2]), percent = std::atoi(argv[3]);
  std::mt19937 rng(seed);
  const unsigned first = rng();
  nsmi::XcdPlaces<int> places(first);
  if (nsmi::XcdPlaces<int>(first).one_xcd(1).xcd != int(first % 8)) return std::printf("first XCD\n"), 1;
  Past past[N], queued[64], device_past;     // before launch i; on a stream so far; the last group over the device
  int xcd[N];                                // -1: over the device
  for (int i = 0; i < N; ++i) {
    const int s = 1 + int(rng() % streams);
    if (rng() % 20 == 0) {                   // the stream drains, is destroyed, and its number used again
      places.release(s);
      for (int t = 0; t <= streams; ++t) queued[t] |= queued[s];
      device_past |= queued[s];
      queued[s] = queued[0];
      for (int t = 0; t <= streams; ++t) queued[t] |= queued[0];
    }
    const bool all = int(rng() % 100) < percent;
    const auto o = all ? places.over_device(s) : places.one_xcd(s);
    xcd[i] = o.xcd;
    if (all != (o.xcd < 0) || o.xcd >= 8) return std::printf("launch %d: XCD %d\n", i, o.xcd), 1;
    for (int t : o.streams) queued[s] |= queued[t];
    if (o.device) queued[s] |= device_past;
    past[i] = queued[s];
    queued[s].set(i);
    if (all) device_past = queued[s];
    std::vector<int> with;                   // earlier launches that may still be on the device
    for (int k = 0; k < i; ++k)
      if (!past[i][k]) with.push_back(k);
    for (int k : with) {
      if (all || xcd[k] < 0) return std::printf("launches %d and %d, one over the device\n", k, i), 1;
      if (xcd[k] != xcd[i]) continue;
      for (int l : with)
        if (l < k && xcd[l] == xcd[i] && !past[k][l]) return std::printf("%d, %d, %d on one XCD\n", l, k, i), 1;
    }
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    d = tmp_path_factory.mktemp("places")
    (d / "h.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(d / "h.cpp"), "-o", str(d / "h")],
                   check=True)
    return str(d / "h")


@pytest.mark.parametrize("percent", [0, 3, 30, 100])
@pytest.mark.parametrize("streams", [1, 2, 16, 17, 40])
def test_launch_order(harness, streams, percent):
    for seed in range(10):
        r = subprocess.run([harness, str(seed), str(streams), str(percent)], capture_output=True, text=True)
        assert r.returncode == 0, (seed, r.stdout)
