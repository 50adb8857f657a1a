// Host-visible side of the runtime-radix passes (fh_rt.hpp): radix schedules, geometry, launchers.
#pragma once
#include <hip/hip_runtime.h>

#include "fh_kernels.hpp"
#include "fh_pot.hpp"

namespace fh {
namespace rt {

// Radices of the butterflies. Composite ones keep most axes below 256 points at two stages (a stage
// is a round trip through LDS with two barriers).
#define FH_RT_RADICES(X) \
  X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(15) X(16)

// Butterflies a thread may hold in one stage: 20 single- or 10 double-precision complex values and
// what rounds up to whole butterflies, so a tile of the whole LDS fits 1024 threads.
__host__ __device__ constexpr int max_m(size_t real_bytes, int R) {
  return ((real_bytes == 4 ? 20 : 10) + R - 1) / R;
}

// x / d by a multiply-high with m = ceil(2^32 / d): exact while x * d < 2^32 (checked where built).
struct Div {
  unsigned d, m;
};

struct Stage {
  int R, p, LR, tws;  // radix, product of the radices before, L / R, twiddle stride L / (p R)
  unsigned mp;        // i / p = (i * mp) >> 20 with 24-bit operands: mp = ceil(2^20 / p), i * p < 2^20
};

constexpr int kMaxSt = 4;  // radices up to 16: lengths up to 4096

struct Axis {
  int L, nst;
  Stage st[kMaxSt];
};

constexpr int kRadices[] = {16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
constexpr int kNumRadices = sizeof(kRadices) / sizeof(int);

// Cost of one stage per element: a round trip through LDS with two barriers (kStage) and the
// butterfly's arithmetic.
constexpr int kStage = 12;
constexpr int radix_cost(int R) {
  constexpr int c[17] = {0, 0, 2, 4, 4, 7, 6, 10, 6, 8, 9, 16, 8, 19, 0, 12, 9};
  return c[R];
}

// Cheapest factorisation of rem into at most `left` non-increasing radices from index `from` on.
constexpr int search_radices(int rem, int from, int left, int* pick, int depth, int* best, int* nbest, int cost,
                             int bound) {
  if (rem == 1) {
    if (cost < bound) {
      for (int i = 0; i < depth; ++i) best[i] = pick[i];
      *nbest = depth;
      return cost;
    }
    return bound;
  }
  if (left == 0) return bound;
  for (int i = from; i < kNumRadices; ++i) {
    const int R = kRadices[i];
    if (rem % R) continue;
    const int c = cost + kStage + radix_cost(R);
    if (c >= bound) continue;
    pick[depth] = R;
    bound = search_radices(rem / R, i, left - 1, pick, depth + 1, best, nbest, c, bound);
  }
  return bound;
}

// Lengths with compiled-in passes: planes of L x L points, rows of L points, strided passes along an axis
// of L points. Every constant stride becomes an immediate offset of an LDS instruction: at 128^3 (double)
// the projection pass takes 30 us against 49 us of the schedule-driven kernel, a plane pass 39 against
// 47 us. The odd lengths of the method, powers of two and round numbers; others run the same code
// with the schedule as data.
#define FH_RT_LENGTHS(X)                                                                                    \
  X(9) X(15) X(16) X(20) X(21) X(24) X(25) X(27) X(30) X(32) X(33) X(35) X(36) X(39) X(40) X(45) X(48) X(49) \
  X(50) X(54) X(55) X(60) X(63) X(64) X(65) X(72) X(75) X(77) X(80) X(81) X(90) X(91) X(96) X(99) X(100)     \
  X(105) X(108) X(117) X(120) X(121) X(125) X(128) X(135) X(144) X(150) X(160) X(180) X(192) X(200) X(216)   \
  X(225) X(240) X(243) X(250) X(256)

// Radix schedule of length L; nst = 0 where it has a prime factor above 13 or needs too many stages.
constexpr Axis plan_axis(int L) {
  Axis ax{};
  ax.L = L;
  if (L < 2) return ax;
  int pick[kMaxSt] = {}, best[kMaxSt] = {}, n = 0;
  if (search_radices(L, 0, kMaxSt, pick, 0, best, &n, 0, 1 << 30) == (1 << 30)) return ax;
  int p = 1;
  for (int s = 0; s < n; ++s) {
    Stage& g = ax.st[s];
    g.R = best[s];
    g.p = p;
    g.LR = L / g.R;
    g.tws = L / (p * g.R);
    g.mp = (unsigned)(((1 << 20) + p - 1) / p);
    if ((long long)g.LR * p >= (1 << 20)) return ax;
    p *= g.R;
  }
  ax.nst = n;
  return ax;
}

constexpr Div make_div(long long d) {
  return Div{(unsigned)d, d <= 1 ? 0u : (unsigned)(((1ULL << 32) + (unsigned long long)d - 1) / (unsigned long long)d)};
}

// Geometry of the contiguous-axis passes of one precision.
struct Geo {
  int nc, n2, n2h;
  long long n, nh, nrows;  // voxels, half-spectrum points (one component), grid rows
  int rb, rbe;             // rows per workgroup, the same rounded up to even
  int plane;               // 1: rb = n1 and axis 1 is transformed too
  int S;                   // LDS stride of a pencil element (row pairs, odd)
  int tile;                // complex values of the tile
  int tpp2, tpp1;          // threads per pencil along axis 2 and axis 1
  int tw1_off;             // twiddles of axis 1 after those of axis 2 (0: the same table)
  Div dn2, dn2h, dpr, dnc; // by n2, n2h, rbe / 2, nc
  int dx, drow, dk, dq;    // threads modulo and over n2, modulo and over n2h
  Axis a2, a1;
};

// Threads per pencil that hold every stage in registers (need), and that give each butterfly of the
// longest stage a thread (want).
constexpr int threads_need(const Axis& ax, size_t rb) {
  int n = 1;
  for (int s = 0; s < ax.nst; ++s) {
    const int m = max_m(rb, ax.st[s].R), k = (ax.st[s].LR + m - 1) / m;
    n = k > n ? k : n;
  }
  return n;
}
constexpr int threads_want(const Axis& ax) {
  int n = 1;
  for (int s = 0; s < ax.nst; ++s) n = ax.st[s].LR > n ? ax.st[s].LR : n;
  return n;
}
constexpr int round64(long long n) { return (int)((n + 63) / 64 * 64); }
// Threads of a workgroup: whole rounds of the CU's four SIMDs, which a workgroup of, say, five waves fills
// unevenly so that fewer fit (81^3 elasticity single 42.2 -> 41.3 us, double 60.4 -> 58.8, 64^3 double 29.9
// -> 28.4, 60^3 single 22.0 -> 21.1; no grid measured slower).
constexpr int roundw(long long n) { return n <= 128 ? round64(n) : (int)((n + 255) / 256 * 256); }

// What a pass reaches through one buffer resource stays below this: lanes without work take byte offsets from
// kDead = 2^31 on, which a larger resource would hold.
constexpr long long kSpan = 1LL << 31;

constexpr size_t kLdsBytes = 160 * 1024;
constexpr size_t kLdsUse = kLdsBytes - 2048;  // static LDS of the kernels and rounding

// Rows per workgroup of the contiguous-axis passes and what follows from it.
constexpr void set_rows(Geo& g, int rows) {
  g.rb = rows;
  g.rbe = (rows + 1) / 2 * 2;
  g.S = (g.rbe / 2) | 1;
  g.tile = (g.n2 + 1 + (g.n2 % 2 == 0)) * g.S;
  g.dpr = make_div(g.rbe / 2);
}

// Plane geometry of n1 x n2 planes: *nthr threads and *lds bytes; plane = 0 where a plane does not fit.
// 1024 threads only for a plane of more than half of the LDS (its workgroup has the CU to itself).
constexpr void set_plane(Geo& g, int n1, size_t rb, int* nthr, size_t* lds) {
  set_rows(g, n1);
  const bool same = n1 == g.n2;
  g.tw1_off = same ? 0 : g.n2;
  *lds = ((size_t)g.tile + g.n2 + (same ? 0 : n1)) * 2 * rb;
  const int npr = g.rbe / 2, cap = *lds > kLdsBytes / 2 ? 1024 : 512;
  g.plane = *lds <= kLdsUse && npr * threads_need(g.a2, rb) <= cap && g.n2h * threads_need(g.a1, rb) <= cap;
  if (!g.plane) return;
  const int w2 = threads_want(g.a2), w1 = threads_want(g.a1);
  g.tpp2 = w2 < cap / npr ? w2 : cap / npr;
  g.tpp1 = w1 < cap / g.n2h ? w1 : cap / g.n2h;
  *nthr = roundw(npr * g.tpp2 > g.n2h * g.tpp1 ? npr * g.tpp2 : g.n2h * g.tpp1);
}

// Geometry of a plane of n x n points without the grid's own fields (nc, n, nh, nrows).
constexpr Geo const_plane(int n, size_t rb) {
  Geo r{};
  r.n2 = n;
  r.n2h = n / 2 + 1;
  r.a2 = plan_axis(n);
  r.a1 = r.a2;
  r.dn2 = make_div(r.n2);
  r.dn2h = make_div(r.n2h);
  int nthr = 0;
  size_t lds = 0;
  set_plane(r, n, rb, &nthr, &lds);
  return r;
}
// Threads of its workgroup (0: the plane does not fit).
constexpr int const_plane_threads(int n, size_t rb) {
  Geo r = const_plane(n, rb);
  int nthr = 0;
  size_t lds = 0;
  set_plane(r, n, rb, &nthr, &lds);
  return r.plane ? nthr : 0;
}

template <typename T>
struct FwdArgs {
  Geo g;
  const T* in;
  T* pout;
  const T* coef;
  int kind;
  const T* r;
  T* xc;
  cpx<T>* out;
  const CGState* st;
  double* partial;
  const double* bpart;
  int bnp;
  const int* halt;
  const cpx<T>*tw2, *tw1;
};

template <typename T>
struct InvArgs {
  Geo g;
  const cpx<T>* in;
  T* out;
  T scale;
  int epi;
  const T* w;
  float* r32;
  double* partial;
  CGState* st;
  int defer_beta;
  const int* halt;
  const cpx<T>*tw2, *tw1;
};

template <typename T>
struct ColArgs {
  const cpx<T>* src;
  cpx<T>* dst;
  long long ostride, total;  // slab stride, values of the whole array
  int cs, es, nf, lf, ntiles, n2h, tpp;  // component and element stride, points, log2 F
  Div dP, dn2h, dtiles;
  Axis ax;
  GParams g;
  const cpx<T>* tw;
  CgFin fin;
  const int* halt;
};

// Launch shapes of one plan in one precision.
struct Config {
  bool ok = false;
  bool thin = false;   // rows although the planes fit: too few of them
  Geo g{};
  int nthr = 0;        // contiguous-axis passes
  unsigned nblk = 0;
  size_t lds = 0;
  Axis a0{};           // axis of the projection pass (0 in 3-D, 1 in 2-D)
  int lf = 0, nthr_g = 0, tpp_g = 1;  // log2 of the tile's points, threads, threads per pencil
  size_t lds_g = 0;
  int lp1 = 0, nthr_1 = 0, tpp_1 = 1;  // axis 1 of a 3-D grid in row mode: columns per tile
  size_t lds_1 = 0;
  int lp0 = 0, nthr_0 = 0, tpp_0 = 1;  // the projection axis without G (transforms of single components)
  size_t lds_0 = 0;
};

// Potential formulation: the strided pass along the outermost axis fused with the scalar <-> gradient
// spectra. dir +1: p = r + beta p (r set), gradient of P p, inverse transform into data; dir -1: forward
// transform of data, o = sgn P div. The operator form stores o in out and sums the weighted <o, w>.
// A CG iteration (x set / upd_r set) adds the pending alpha p to x in dir +1 and takes r -= alpha o with
// the weighted <r, r> in dir -1, where every workgroup forms alpha from the round trip's np1 partials p1
// (0: it is final in *st) and block 0 finalises it; bpart/bnp: the deferred beta, as in FwdArgs.
struct PotArgs {
  int dir;
  cpx<double>* data;
  cpx<double>* p;
  const cpx<double>* r;
  cpx<double>* x;
  CGState* st;
  double sgn;
  cpx<double>* out;
  const cpx<double>* w;
  cpx<double>* upd_r;
  double* partial;
  const double *p1, *bpart;
  int np1, bnp, defer_beta;
  pot::PotParams g;
  int cs, es, lf, ntiles, tpp;  // component and axis stride (points), log2 of the tile's points
  Div dP, dn2h;
  Axis ax;
  const cpx<double>* tw;
  const int* halt;
};

// Round trip in place on a component-major spectrum: C2R (axis 1 too in plane mode) times scale, times
// a(x), and back. With partial set it also sums n <e, a e> of its field e; block 0 finalises a
// deferred beta.
struct TripArgs {
  Geo g;
  cpx<double>* spec;
  const double* coef;
  double scale;
  double* partial;
  CGState* st;
  const double* bpart;
  int bnp;
  const int* halt;
  const cpx<double>*tw2, *tw1;
};

// Quadrature lengths with compiled-in passes of the Ga energies: about twice the method's odd lengths.
#define FH_GA_LENGTHS(X) \
  X(18) X(30) X(42) X(50) X(54) X(66) X(70) X(78) X(90) X(98) X(110) X(126) X(130) X(150) X(162) X(198) X(210) X(234) \
  X(250) X(270)

// Zero-padded inverse transform along one axis (see k_pad): outer slabs of n x es -> L x es points.
struct PadArgs {
  const cpx<double>* src;
  cpx<double>* dst;
  int n, es, lf, ntiles, tpp;
  double scale;
  Div dtiles;
  Axis ax;
  const cpx<double>* tw;
};

// Last transform of the interpolation (see k_ga_rows): components cs points apart.
struct GaRowArgs {
  const cpx<double>* src;
  long long cs, nrows, ngroups, nvox;
  int n2, n2h, tpp, kind;
  Div dn2h;
  Axis ax;
  const cpx<double>* tw;
  const double* coef;
  double* partial;
  double* out;
};

// Launch shapes of the two; false where a pass does not exist for the length.
bool pad_config(int L, int es, long long outer, PadArgs* a, unsigned* nblk, int* nthr, size_t* lds);
bool ga_rows_config(int L, int npencils, GaRowArgs* a, int* nthr, size_t* lds);

// Whether length L is in FH_RT_LENGTHS.
bool compiled_length(int L);

// Shapes for a grid (3-D view n0, n1, n2; 2-D: n0 = 1) of nc components; ok = false where these passes
// do not cover it. fixed: a 3-D grid that the passes of fixed lengths cover too.
Config make_config(size_t real_bytes, int n0, int n1, int n2, int nc, bool fixed);

// Stream of a launch and, if set, the events that take its start and stop times.
struct Launch {
  hipStream_t stream;
  hipEvent_t t0, t1;
};

// Launchers; nc <= the configuration's component count is passed where a transform handles fewer.
template <typename T>
hipError_t launch_fwd(const Config& c, const FwdArgs<T>& a, bool upd, unsigned nblk, const Launch& s);
template <typename T>
hipError_t launch_inv(const Config& c, const InvArgs<T>& a, unsigned nblk, const Launch& s);
// mode 0 / 1: nslab slabs of axis length L (axis 1 of a 3-D grid, or the projection axis of single
// components); mode 2: the projection.
template <typename T>
hipError_t launch_cols(int nc, int mode, const ColArgs<T>& a, unsigned nblk, int nthr, size_t lds, const Launch& s);

hipError_t launch_pad(PadArgs a, unsigned nblk, int nthr, size_t lds, const Launch& s);
hipError_t launch_ga_rows(int nc, bool store, GaRowArgs a, unsigned nblk, int nthr, size_t lds, const Launch& s);
hipError_t launch_pot(int nc, const PotArgs& a, int nthr, size_t lds, const Launch& s);
hipError_t launch_trip(const Config& c, const TripArgs& a, unsigned nblk, const Launch& s);

#define FH_RT_EXTERN(T)                                                                                           \
  extern template hipError_t launch_fwd<T>(const Config&, const FwdArgs<T>&, bool, unsigned, const Launch&);     \
  extern template hipError_t launch_inv<T>(const Config&, const InvArgs<T>&, unsigned, const Launch&);           \
  extern template hipError_t launch_cols<T>(int, int, const ColArgs<T>&, unsigned, int, size_t, const Launch&);
FH_RT_EXTERN(float)
FH_RT_EXTERN(double)
#undef FH_RT_EXTERN

}  // namespace rt
}  // namespace fh
