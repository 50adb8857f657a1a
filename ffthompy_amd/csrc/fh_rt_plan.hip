// Host side of the runtime-radix passes: radix schedules and launch shapes.
#include <algorithm>

#include "fh_rt_launch.hpp"

namespace fh {
namespace rt {

static bool div_exact(long long x, long long d) { return x * d < (1LL << 32); }

// Points per tile (2^lf) of a strided pass of nc components: up to 2^most of nf, fewer until `blocks`
// workgroups exist (256 CUs, about two workgroups each) and the tile leaves room for other workgroups
// in LDS. Each butterfly of the longest stage gets a thread where 512 threads allow it.
static bool pick_cols(const Axis& ax, int nc, size_t rb, long long nf, long long outer, int most, int least,
                      long long blocks, size_t lds_max, int* lf, int* nthr, int* tpp, size_t* lds) {
  const int need = threads_need(ax, rb), want = threads_want(ax);
  for (int l = most; l >= 0; --l) {
    const long long f = 1LL << l, P = f * nc;
    *lds = ((size_t)ax.L * P + ax.L) * 2 * rb;
    const bool fits = P * need <= 512 && *lds <= kLdsUse;
    const bool small = *lds <= lds_max && ((nf + f - 1) / f * outer >= blocks || l <= least);
    if (!fits || (!small && l > 0)) continue;
    *lf = l;
    *tpp = (int)std::min<long long>(want, 512 / P);
    *nthr = roundw(P * *tpp);
    return true;
  }
  return false;
}

bool compiled_length(int L) {
  switch (L) {
#define FH_RT_CASE(X) case X:
    FH_RT_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
    return true;
    default: return false;
  }
}

// Too few planes to fill the chip, each long to transform (see make_config).
static bool thin_planes(const Geo& g, int n1, int planes) {
  const long long points = (long long)n1 * g.n2;
  if (n1 == g.n2 && compiled_length(n1)) return points * (g.a2.nst > 2 ? 3 : 2) > 2 * (220LL * planes + 3300);
  return std::min(n1, g.n2) >= 25 && planes < 128 && points > (long long)planes * planes;
}

Config make_config(size_t rb, int n0, int n1, int n2, int nc, bool fixed) {
  Config c;
  const bool three = n0 > 1;
  if (n1 < 2 || n2 < 2 || n2 > 4096 || n1 > 4096 || n0 > 4096) return c;
  Geo& g = c.g;
  g.nc = nc;
  g.n2 = n2;
  g.n2h = n2 / 2 + 1;
  g.nrows = (long long)n0 * n1;
  g.n = g.nrows * n2;
  g.nh = g.nrows * g.n2h;
  g.a2 = plan_axis(n2);
  if (three) g.a1 = plan_axis(n1);
  c.a0 = plan_axis(three ? n0 : n1);
  if (!g.a2.nst || !c.a0.nst || (three && !g.a1.nst)) return c;
  if (!div_exact((long long)n1 * g.n2h, g.n2h)) return c;
  g.dn2 = make_div(n2);
  g.dn2h = make_div(g.n2h);
  if (nc * g.nh * 2 * (long long)rb >= kSpan) return c;
  // Plane mode (the whole plane of one component in LDS) for every compiled plane (135^3: 114 us against
  // 130 us of row mode in double, 71 against 85 in single precision). A plane of other lengths runs the
  // schedule-driven kernel: it wins while one round of workgroups covers the chip (63 x 81 x 105, 189
  // workgroups: 52 against 59 us) and loses beyond (90 x 100 x 77, 270: 70 against 62 us; 105 x 63 x 45
  // elasticity, 630: 76 against 64 us).
  g.plane = 0;
  if (three && div_exact((long long)(n1 + 1) * n2, n2)) set_plane(g, n1, rb, &c.nthr, &c.lds);
  if (g.plane && !(n1 == n2 && compiled_length(n2)) && n0 * nc > 256) g.plane = 0;
  // Grids of fixed lengths have five passes with many workgroups of their own. A thin one loses by a few
  // workgroups with a plane each and takes rows here (passes of fixed lengths / planes / rows, per application:
  // 5 x 225 x 75 double 44 / 62 / 46 us, its 40 CG iterations 2018 / 2564 / 1771; 15 x 99 x 135 single 45 / 53 / 46;
  // 27 x 243 x 45 single 47 / 54 / 47; 5 x 135 x 135 double 49 / 55 / 45; but 27 x 27 x 45 single 38 / 38 / 37,
  // 15 x 99 x 99 double 49 / 48 / 49, 27 x 135 x 135 double 76 / 68 / 76, 45 x 225 x 75 double 83 / 77 / 82). The time
  // of the planes does not depend on their number while they fit the chip, that of the rows does, hence lines
  // between the two; 125 x 125 with its three stages costs half as much again. Planes of more than half of the LDS
  // with three stages stay on the passes of fixed lengths (the caller's rule).
  const bool slow = c.lds > kLdsBytes / 2 && g.a2.nst > 2;
  c.thin = g.plane && fixed && !slow && thin_planes(g, n1, n0 * nc);
  if (c.thin) g.plane = 0;
  if (g.plane) c.nblk = (unsigned)(n0 * nc);
  if (!g.plane) {
    // row mode: more rows per workgroup while the chip stays covered
    int rows = 2;
    auto blocks = [&](int r) { return (g.nrows + r - 1) / r * nc; };
    while (2 * rows <= 32 && blocks(2 * rows) >= 1024 && (size_t)(n2 + 2) * (rows | 1) * 2 * rb <= 40 * 1024 &&
           rows * threads_need(g.a2, rb) <= 512)
      rows *= 2;
    set_rows(g, rows);
    g.tw1_off = 0;
    c.lds = ((size_t)g.tile + n2) * 2 * rb;
    const int npr = g.rbe / 2;
    if (c.lds > kLdsUse || npr * threads_need(g.a2, rb) > 512) return c;
    g.tpp2 = std::min(threads_want(g.a2), 512 / npr);
    g.tpp1 = 1;
    c.nthr = round64(npr * g.tpp2);
    c.nblk = (unsigned)blocks(rows);
    if (three && !pick_cols(g.a1, 1, rb, g.n2h, (long long)n0 * nc, rb == 4 ? 5 : 4, rb == 4 ? 3 : 2, 1024, 40 * 1024,
                            &c.lp1, &c.nthr_1, &c.tpp_1, &c.lds_1))
      return c;
  }
  // Tiles of a strided pass read segments of 64 bytes; 128 where the spectrum exceeds the Infinity Cache
  // by far (in cache the shorter segments win by 2-6 %: more workgroups, less LDS each).
  const int seg = (rb == 4 ? 3 : 2) + ((size_t)nc * g.nh * 2 * rb > ((size_t)192 << 20));
  const long long nf = three ? (long long)n1 * g.n2h : g.n2h;
  if (!pick_cols(c.a0, nc, rb, nf, 1, seg, 0, 256, 64 * 1024, &c.lf, &c.nthr_g, &c.tpp_g, &c.lds_g)) return c;
  if (!pick_cols(c.a0, 1, rb, nf, 1, rb == 4 ? 5 : 4, 0, 512, 48 * 1024, &c.lp0, &c.nthr_0, &c.tpp_0, &c.lds_0)) return c;
  g.dnc = make_div(nc);
  g.dx = c.nthr % n2;
  g.drow = c.nthr / n2;
  g.dk = c.nthr % g.n2h;
  g.dq = c.nthr / g.n2h;
  if (!div_exact((long long)c.nblk, nc)) return c;
  c.ok = true;
  return c;
}

bool pad_config(int L, int es, long long outer, PadArgs* a, unsigned* nblk, int* nthr, size_t* lds) {
  a->ax = plan_axis(L);
  a->es = es;
  if (!a->ax.nst || (long long)L * es * 16 >= kSpan) return false;
  if (!pick_cols(a->ax, 1, 8, es, outer, 3, 2, 1024, 48 * 1024, &a->lf, nthr, &a->tpp, lds)) return false;
  a->ntiles = (es + (1 << a->lf) - 1) >> a->lf;
  a->dtiles = make_div(a->ntiles);
  const long long nb = outer * a->ntiles;
  if (nb > 0x7fffffffLL || !div_exact(nb, a->ntiles)) return false;
  *nblk = (unsigned)nb;
  return true;
}

bool ga_rows_config(int L, int npencils, GaRowArgs* a, int* nthr, size_t* lds) {
  a->ax = plan_axis(L);
  const int need = npencils * threads_need(a->ax, 8);
  if (!a->ax.nst || need > 512) return false;
  // About a thread per point of a row (the energies' loop), in whole rounds of the four SIMDs: of
  // workgroups of five waves at 160 registers a CU held one at a time (270 points: 755 us against 490 us
  // of four waves).
  *nthr = round64(std::max(need, std::min(L, 256)));
  if (*nthr > 256) *nthr = 512;
  a->tpp = std::min(threads_want(a->ax), *nthr / npencils);
  *lds = ((size_t)L * (npencils | 1) + L) * 16;
  return *lds <= kLdsUse;
}

}  // namespace rt
}  // namespace fh
