"""The plan of the one-launch boundary pass (grid.hip, bound_plan and the block
bodies behind it) on the host: the source between its two markers is compiled
as C++ with the zone functions replaced by ones that mark the zone they would
fill, and every block of every size that takes the pass is walked.  No block
count may be negative, no zone outside the storage box may be touched, and
every zone of the box must be active or filled.  Grids without an x2 direction
have no polar rows to rebuild: they must not take this pass."""
import ctypes
import itertools
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "harm_harm_amd", "csrc", "hip", "grid.hip")

STUBS = r"""
#include <cmath>
#include <cstdint>
#include <vector>
#include <algorithm>
#include "harmstep.h"
#define __device__
#define __host__
#define __forceinline__ inline
#define __restrict__
static const int kBlock = 256;
static struct { int x; } threadIdx;
static inline void __syncthreads() {}
static inline long min(long a, long b) { return std::min(a, b); }
struct Dims { int n1, n2, n3, ng1, ng2, ng3, ns1, ns2, ns3, ps1; long nplane, ncell; };
struct Params { int bc; };
static long bad;
namespace hd {
static long cidx(const Dims& d, int i, int j, int k)
{
  if (i < -d.ng1 || i >= d.n1 + d.ng1 || j < -d.ng2 || j >= d.n2 + d.ng2 || k < -d.ng3 || k >= d.n3 + d.ng3) {
    bad++;
    return 0;
  }
  return ((long)(k + d.ng3) * d.ns2 + j + d.ng2) * d.ps1 + i + d.ng1;
}
}
static void fill(const Dims& d, double* p, int i, int j, int k, long img)
{
  const long o = hd::cidx(d, i, j, k);
  for (long at : {o, o + img})
    if (at < 0 || at >= d.ncell) bad++;
    else p[at] = 1.0;
}
static void extrap_line(const Dims& d, const Params&, double* p, const double*, int up, int j, int k, int g, long img)
{
  fill(d, p, up ? d.n1 + g : -1 - g, j, k, img);
}
static void bondi_line(const Dims& d, const Params&, double* p, const double*, int up, int j, int k, int g)
{
  fill(d, p, up ? d.n1 + g : -1 - g, j, k, 0);
}
static void x2_reflect_zone(const Dims& d, double* p, int side, int g, long col, long img = 0)
{
  const int i = (int)(col % d.ns1) - d.ng1, k = (int)(col / d.ns1), j = side == 0 ? -d.ng2 + g : d.n2 + g;
  hd::cidx(d, i, side == 0 ? -1 - j : 2 * d.n2 - 1 - j, d.n3 > 1 ? (k + d.n3 / 2) % d.n3 : k);  // the row it reads
  fill(d, p, i, j, k, img);
}
static void x2_poledeath_row(const Dims& d, const Params&, double* p, const double*, const double*, int side, bool ghost,
                             long col, bool, long img)
{
  const int i = (int)(col % d.ns1) - d.ng1, k = (int)(col / d.ns1);
  hd::cidx(d, i, side == 0 ? 1 : d.n2 - 2, k);
  fill(d, p, i, ghost ? (side == 0 ? -1 : d.n2) : (side == 0 ? 0 : d.n2 - 1), k, img);
}
"""

WALK = r"""
// 0: the grid does not take the pass; 1: sound; -1: negative block counts; -2:
// a zone outside the box; -3: a zone that is not filled
extern "C" int walk(int n1, int n2, int n3, int ng, int bc)
{
  Dims d{n1, n2, n3, n1 > 1 ? ng : 0, n2 > 1 ? ng : 0, n3 > 1 ? ng : 0};
  d.ns1 = n1 + 2 * d.ng1;
  d.ns2 = n2 + 2 * d.ng2;
  d.ns3 = n3 + 2 * d.ng3;
  d.ps1 = (d.ns1 + 15) & ~15;
  d.nplane = (long)d.ps1 * d.ns2;
  d.ncell = d.nplane * d.ns3;
  if (!bounds_merge(d)) return 0;
  const Params P{bc};
  for (int flags = 0; flags < 2; flags++) {
    const BoundPlan b = bound_plan(d, flags);
    if (b.nchunk < 1 || b.nA < 0 || b.nB < 0 || b.nC < 0 || b.nD < 0) return -1;
    bad = 0;
    std::vector<double> p((size_t)d.ncell * HARM_NPR, 0.0);
    std::vector<int32_t> fl(d.ncell, 0);
    for (int k = 0; k < n3; k++)
      for (int j = 0; j < n2; j++)
        for (int i = 0; i < n1; i++) p[hd::cidx(d, i, j, k)] = 1.0;
    for (int blk = 0; blk < b.total(); blk++)
      for (threadIdx.x = 0; threadIdx.x < kBlock; threadIdx.x++) {
        if (blk < b.nA + b.nB + b.nC) bounds_prims(d, P, b, p.data(), nullptr, nullptr, blk);
        else bounds_flags(d, bc, fl.data(), (long)(blk - b.nA - b.nB - b.nC) * kBlock + threadIdx.x);
      }
    if (bad) return -2;
    for (int k = -d.ng3; k < n3 + d.ng3; k++)
      for (int j = -d.ng2; j < n2 + d.ng2; j++)
        for (int i = -d.ng1; i < n1 + d.ng1; i++)
          if (p[hd::cidx(d, i, j, k)] != 1.0) return -3;
  }
  return 1;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    text = open(SRC).read()
    body = text[text.index("struct BoundPlan {"):text.index("// cond: the second pass, only where")]
    d = tmp_path_factory.mktemp("plan")
    cc, so = str(d / "plan.cc"), str(d / "plan.so")
    with open(cc, "w") as f:
        f.write(STUBS + body + WALK)
    inc = os.path.join(os.path.dirname(SRC), "..", "..", "..", "include")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", inc, cc, "-o", so], check=True)
    return ctypes.CDLL(so).walk


@pytest.mark.parametrize("ng", [3, 4])
def test_every_block_stays_in_the_box_and_every_zone_is_filled(walk, ng):
    taken = 0
    for n1, n2, n3 in itertools.product([1, 3, 7, 8, 9, 16, 65], [1, 4, 5, 6, 9, 33, 64, 130], [1, 6, 8, 10, 16]):
        if n3 > 1 and n3 // 2 < ng:
            continue
        for bc in (0, 1) if n3 == 1 else (0,):
            r = walk(n1, n2, n3, ng, bc)
            assert r in (0, 1), (n1, n2, n3, ng, bc, r)
            taken += r
    assert taken > 50


@pytest.mark.parametrize("n", [(8, 1, 1), (16, 1, 1), (16, 1, 8), (64, 1, 16)])
def test_grids_without_polar_rows_do_not_take_the_pass(walk, n):
    for bc in (0, 1) if n[2] == 1 else (0,):
        assert walk(*n, 4, bc) == 0
