"""The queue that spreads the end of a failing 2-D substep (grid.hip,
bounds_body<true>) on the host: the source is compiled as C++ with the passes
replaced by ones that record when they ran, a block is a thread, and no more
blocks run at a time than a chip would hold.  Every item runs once, no phase
starts before the one ahead of it is over, the waits end, the queue is empty
again afterwards, and the work does not pile up in one block."""
import ctypes
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "harm_harm_amd", "csrc", "hip", "grid.hip")

STUBS = r"""
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <thread>
#include <vector>
#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__ static thread_local
using std::max;
using std::min;
static const int kBlock = 256;
static thread_local struct { int x; } threadIdx;
#define __builtin_amdgcn_readfirstlane(x) (x)
static inline void __syncthreads() {}
static inline void __threadfence() { std::atomic_thread_fence(std::memory_order_seq_cst); }
static unsigned long long atomicAdd(unsigned long long* p, unsigned long long v) { return __atomic_fetch_add(p, v, __ATOMIC_RELAXED); }
static void wait_count(unsigned long long* p, int n)
{
  while (__atomic_load_n(p, __ATOMIC_RELAXED) < (unsigned long long)n) std::this_thread::yield();
}
enum { DI_FIX, DI_DRAWN, DI_DONE, DI_LEFT, DI_N };
struct Dims { int n1, n2, n3; int nA, nB, nD; };
struct Params { double safe; int bc; };
struct BoundPlan {
  int nA, nB, nC, nD;
  int total() const { return nA + nB + nC + nD; }
};
static BoundPlan bound_plan(const Dims& d, bool flags) { return {d.nA, d.nB, 0, flags ? d.nD : 0}; }
static void scal_end_step(double*, unsigned long long*, double) {}

// one record per item, four phases; an item takes a while
static std::atomic<int> over[4], started[4], early, work_of[4096];
static std::vector<std::atomic<int>> ran[4];
static thread_local int self;
static int phase_size[4], nfail;
static void item(int phase, int v)
{
  if (v < 0 || v >= phase_size[phase]) {
    early++;
    return;
  }
  for (int q = 0; q < phase; q++)
    if (over[q] != phase_size[q]) early++;
  started[phase]++;
  std::this_thread::sleep_for(std::chrono::microseconds(100));
  ran[phase][v]++;
  work_of[self]++;
  over[phase]++;
}
static void bounds_prims(const Dims& d, const Params&, const BoundPlan& b, double*, const double*, const double*, int v)
{
  item(over[0] == phase_size[0] && nfail ? 3 : 0, v);
}
static void bounds_flags(const Dims& d, int, int32_t*, long t) { item(0, d.nA + d.nB + (int)(t / kBlock)); }
// (the list holds the zones backwards; thread 0 stands for its run of 256)
static void post_fixup_body(const Dims&, const Params&, double*, int32_t*, double*, const double*, int, long z)
{
  item(1, (int)(nfail - 1 - z) / kBlock);
}
static void fixup_apply_body(const Dims&, double*, int32_t*, double*, int, long z) { item(2, (int)(nfail - 1 - z) / kBlock); }
"""

RUN = r"""
// A launch with `resident` blocks at a time: 0, or what is wrong.  most: items
// of the block that did most.
extern "C" int launch(int n1, int n2, int nA, int nB, int nD, int resident, int fail, int* most)
{
  const Dims d{n1, n2, 1, nA, nB, nD};
  const Params P{};
  const int runs = (fail + kBlock - 1) / kBlock, n[4] = {nA + nB + nD, runs, runs, nA + nB};
  for (int q = 0; q < 4; q++) {
    phase_size[q] = n[q];
    over[q] = started[q] = 0;
    ran[q] = std::vector<std::atomic<int>>(n[q]);
  }
  for (auto& w : work_of) w = 0;
  early = 0;
  nfail = fail;
  static unsigned long long di[DI_N + 300 * 290];
  for (int z = 0; z < fail; z++) ((int32_t*)(di + DI_N))[z] = fail - 1 - z;
  di[DI_FIX] = fail;
  std::atomic<int> next{0};
  const int nblk = finish_blocks(d);
  std::vector<std::thread> slots;
  for (int s = 0; s < resident; s++)
    slots.emplace_back([&] {
      threadIdx.x = 0;
      for (int b; (b = next++) < nblk;) {
        self = b;
        bounds_body<true>(d, P, nullptr, nullptr, nullptr, nullptr, nullptr, di, 0, true, false, b, nullptr);
      }
    });
  for (auto& t : slots) t.join();
  *most = 0;
  for (auto& w : work_of) *most = std::max(*most, w.load());
  if (early) return 1;
  for (int q = 0; q < 4; q++)
    for (auto& r : ran[q])
      if (r != (q == 0 || fail ? 1 : 0)) return 2;
  return di[DI_DRAWN] || di[DI_DONE] || di[DI_LEFT] ? 3 : 0;
}
"""


@pytest.fixture(scope="module")
def launch(tmp_path_factory):
    text = open(SRC).read()
    body = text[text.index("__host__ __device__ __forceinline__ int finish_blocks("):
                text.index("template <bool FIX2D>\n__global__ __launch_bounds__(kBlock) void k_bounds(")]
    d = tmp_path_factory.mktemp("queue")
    cc, so = str(d / "queue.cc"), str(d / "queue.so")
    with open(cc, "w") as f:
        f.write(STUBS + body + RUN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", cc, "-o", so], check=True)
    L = ctypes.CDLL(so)
    return lambda *a: (lambda m: (L.launch(*a, ctypes.byref(m)), m.value))(ctypes.c_int())


@pytest.mark.timeout(60)
@pytest.mark.parametrize("resident", [1, 2, 8])
@pytest.mark.parametrize("n", [(8, 5, 2, 1, 1), (64, 64, 2, 3, 1), (256, 256, 8, 10, 3), (300, 290, 10, 12, 4)])
def test_every_item_once_and_in_order(launch, n, resident):
    for fail in (1, 0, 256, 257, n[0] * n[1]):  # a launch leaves the queue as the next one needs it
        if fail <= n[0] * n[1]:
            assert launch(*n, resident, fail)[0] == 0, fail


def test_items_are_shared(launch):
    # 256 x 256 zones, all failed, on 8 slots: 551 items, so a block that took more than a third of them held the others up
    status, most = launch(256, 256, 8, 10, 3, 8, 65536)
    assert status == 0 and most <= 184
