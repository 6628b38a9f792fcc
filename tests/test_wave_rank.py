"""wave_rank (csrc/moe_route.h) on the CPU, 64 threads standing for a wavefront's lanes: ranks and counts
against their definition, with every lane given a copy of the LDS counts of its own. Without a fence
a lane may rely on its own stores alone, so a caller that reads cnt[lane] back at once has to
find there what the lane itself stored."""
import re
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "mlsys26-flashinfer-moe_amd" / "csrc"

HOST = r"""
#include <barrier>
#include <cstdint>
#include <cstdio>
#include <thread>
#include <vector>
static std::barrier<> lanes(64);
static int value[64];
static thread_local int my_lane;
static int lane_id() { return my_lane; }
static uint64_t lanemask_lt() { return (1ull << my_lane) - 1; }
static int __popcll(uint64_t m) { return __builtin_popcountll(m); }
static uint64_t __ballot(bool b) {
  value[my_lane] = b;
  lanes.arrive_and_wait();
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l) m |= (uint64_t)value[l] << l;
  lanes.arrive_and_wait();
  return m;
}
static int __builtin_amdgcn_readlane(int v, int from) {
  value[my_lane] = v;
  lanes.arrive_and_wait();
  const int r = value[from];
  lanes.arrive_and_wait();
  return r;
}
constexpr int kExpertsLocal = 32;
#define __device__
#define __forceinline__ inline
//FUNCTION
int main() {
  static int le[64], rank[64], cnt[64][kExpertsLocal];
  for (;;) {
    for (int l = 0; l < 64; ++l)
      if (scanf("%d", &le[l]) != 1) return 0;
    std::vector<std::thread> t;
    for (int l = 0; l < 64; ++l)
      t.emplace_back([l] {
        my_lane = l;
        for (int& c : cnt[l]) c = -7;
        rank[l] = wave_rank(le[l], cnt[l]);
      });
    for (auto& x : t) x.join();
    for (int l = 0; l < 64; ++l) printf("%d ", le[l] >= 0 ? rank[l] : -1);
    for (int e = 0; e < kExpertsLocal; ++e) printf("%d ", cnt[e][e]);
    printf("\n");
  }
}
"""


def test_ranks_and_counts(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    fn = re.search(r"^__device__ __forceinline__ int wave_rank\(.*?^}$", (CSRC / "moe_route.h").read_text(), re.M | re.S)
    (tmp_path / "wave.cpp").write_text(HOST.replace("//FUNCTION", fn.group(0)))
    exe = tmp_path / "wave"
    subprocess.run(["g++", "-std=c++20", "-O1", "-pthread", str(tmp_path / "wave.cpp"), "-o", str(exe)], check=True)
    rng = np.random.default_rng(5)
    none = np.full(64, -1)
    cases = [none, np.full(64, 31), np.arange(64) % 32, np.where(np.arange(64) == 63, 0, -1),
             np.where(np.arange(64) < 32, rng.integers(-1, 32, 64), -1)]
    cases += [rng.integers(-hi, hi, 64).clip(-1) for hi in (2, 8, 32)]
    text = "\n".join(" ".join(map(str, c)) for c in cases)
    res = subprocess.run([str(exe)], input=text, capture_output=True, text=True, timeout=60, check=True)
    got = np.array([line.split() for line in res.stdout.splitlines()], dtype=int)
    for le, row in zip(cases, got, strict=True):
        rank = [int(np.sum(le[:l] == le[l])) if le[l] >= 0 else -1 for l in range(64)]
        assert list(row[:64]) == rank
        assert list(row[64:]) == [int(np.sum(le == e)) for e in range(32)]
