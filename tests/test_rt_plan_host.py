"""Launch shapes of the passes of any smooth length (fh_rt_plan.hip), evaluated on the host over grids up to the
limits: every index split exact where the kernels use it, lanes without work outside of every buffer resource
and without wrapping, workgroups within their threads and LDS, more components than the plan's in groups
below 2 GiB; and the split that flat grids need (quot_any in fh_rt.hpp)."""
import os
import random
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'ffthompy_amd', 'csrc')

MAIN = r'''
#include <cstdio>
#include "fh_rt_launch.hpp"
using namespace fh::rt;
static long long bad = 0, ok = 0;
#define CHECK(x) do { if (!(x)) { if (++bad < 20) std::printf("%s: %d x %d x %d, %d components, %d bytes\n", #x, n0, n1, n2, nc, (int)rb); } } while (0)
static bool exact(long long x, Div d) {  // x / d by quot() for every argument up to x
  if (d.d == 1) return true;
  for (long long q : {x, x - 1, x / d.d * d.d, x / d.d * d.d - 1, (long long)d.d - 1})
    if (q >= 0 && q <= x && (long long)(((unsigned long long)q * d.m) >> 32) != q / d.d) return false;
  return true;
}
static void axis(const Axis& ax, int tpp, int n0, int n1, int n2, int nc, size_t rb) {
  int p = 1;
  for (int s = 0; s < ax.nst; ++s) {
    const Stage& g = ax.st[s];
    CHECK(g.p == p && g.R * g.LR == ax.L && g.R <= 16 && g.R >= 2);
    CHECK(g.LR <= tpp * max_m(rb, g.R));  // a thread's butterflies fit its registers
    for (int i : {0, g.p - 1, g.LR - 1}) CHECK((long long)(((unsigned long long)i * g.mp) >> 20) == i / g.p || g.p == 1);
    p *= g.R;
  }
  CHECK(p == ax.L);
}
static void grid(int n0, int n1, int n2, int nc, size_t rb, bool fixed) {
  const Config c = make_config(rb, n0, n1, n2, nc, fixed);
  if (!c.ok) return;
  ++ok;
  const Geo& g = c.g;
  const long long cs = 2 * rb, nh = g.nh;
  CHECK(nh == (long long)n0 * n1 * (n2 / 2 + 1));
  CHECK(nc * nh * cs < kSpan);                       // dead lanes: offsets from kSpan on ...
  CHECK(kSpan + nc * nh * cs < (1LL << 32));         // ... plus any step do not wrap
  // components per launch of a forward transform of more than the plan's
  const long long group = (kSpan - 1) / (nh * cs) < 36 ? (kSpan - 1) / (nh * cs) : 36;
  CHECK(group >= nc && group * nh * cs < kSpan);
  CHECK(exact((long long)c.nblk / nc * group - 1, make_div(group)));
  CHECK(exact((long long)c.nblk - 1, g.dnc));
  CHECK(c.lds <= kLdsUse && c.nthr <= 1024 && c.nthr >= 64);
  CHECK(g.rbe / 2 * g.tpp2 <= c.nthr && g.tpp2 >= 1);
  CHECK(exact(c.nthr - 1, g.dpr) && exact(c.nthr - 1, g.dn2) && exact(c.nthr - 1, g.dn2h));
  axis(g.a2, g.tpp2, n0, n1, n2, nc, rb);
  CHECK((long long)((g.nrows + g.rb - 1) / g.rb) * nc == c.nblk);
  if (g.plane) {
    CHECK(n0 > 1 && g.rb == n1 && g.n2h * g.tpp1 <= c.nthr);
    axis(g.a1, g.tpp1, n0, n1, n2, nc, rb);
    if (n1 == n2 && compiled_length(n2)) CHECK(const_plane_threads(n2, rb) == c.nthr);
  } else if (n0 > 1) {
    CHECK((1 << c.lp1) * c.tpp_1 <= c.nthr_1 && c.lds_1 <= kLdsUse && c.nthr_1 <= 512);
    axis(g.a1, c.tpp_1, n0, n1, n2, nc, rb);
  }
  CHECK(((long long)nc << c.lf) * c.tpp_g <= c.nthr_g && c.lds_g <= kLdsUse && c.nthr_g <= 512);
  CHECK((1 << c.lp0) * c.tpp_0 <= c.nthr_0 && c.lds_0 <= kLdsUse && c.nthr_0 <= 512);
  axis(c.a0, c.tpp_g, n0, n1, n2, nc, rb);
  axis(c.a0, c.tpp_0, n0, n1, n2, nc, rb);
  CHECK(exact(c.nthr_g - 1, make_div((long long)nc << c.lf)));
  if (n0 > 1) CHECK(exact((long long)n1 * g.n2h - 1, g.dn2h));  // frequencies of the projection pass
}
int main() {
  const int L[] = {2, 3, 4, 5, 7, 9, 11, 13, 15, 16, 20, 25, 27, 33, 45, 63, 66, 75, 81, 90, 98, 99, 100, 105, 125, 126, 128, 135,
                   140, 143, 144, 169, 200, 225, 243, 256, 300, 512, 600, 729, 1000, 1001, 1024, 1100, 1200, 1500, 2000, 2048, 2187, 4000, 4096};
  for (size_t rb : {(size_t)4, (size_t)8})
    for (int n2 : L)
      for (int n1 : L) {
        for (int nc : {2, 3}) grid(1, n1, n2, nc, rb, false);
        for (int n0 : L)
          if ((long long)n0 * n1 * n2 < 400000000LL)
            for (int nc : {3, 6})
              for (bool fixed : {false, true}) grid(n0, n1, n2, nc, rb, fixed);
      }
  std::printf("%lld shapes, %lld violations\n", ok, bad);
  return bad != 0 || ok < 10000;
}
'''


@pytest.mark.skipif(shutil.which('hipcc') is None, reason='no hipcc')
def test_launch_shapes(tmp_path):
    src = tmp_path / 'shapes.hip'
    src.write_text(MAIN)
    exe = str(tmp_path / 'shapes')
    subprocess.run(['hipcc', '--offload-arch=gfx950', '-O1', '-std=c++17', '-Xclang', '-target-feature', '-Xclang',
                    '-packed-fp32-ops', '-I', CSRC, '-o', exe, str(src), os.path.join(CSRC, 'fh_rt_plan.hip')], check=True,
                   capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout


def test_split_of_any_index():
    """quot_any: the multiply-high by ceil(2^32 / d) is the quotient or one more for indexes below 2^31, the product
    with d does not wrap, and one comparison corrects it; without it, 2 x 2000 x 2000 fails."""
    def estimate(x, d):
        return x if d == 1 else (x * -(-(1 << 32) // d)) >> 32

    rng = random.Random(71)
    cases = [(int(2 ** rng.uniform(0, 30.99)), rng.randrange(1 << 31)) for _ in range(100000)]
    cases += [(d, min((1 << 31) - 1, max(0, x // d * d + k))) for d, x in cases[:50000] for k in (-1, 0, 1)]
    for d, x in cases:
        q = estimate(x, d)
        assert q in (x // d, x // d + 1) and q * d < 1 << 32
        assert q - (q * d > x) == x // d
    assert any(estimate(x, 125125) != x // 125125 for x in range(125124, 3 * 125125, 125125))
