// Passes for grids of any smooth size (prime factors <= 13), on a half spectrum that is component-major:
// spec[c][k0][k1][k2], each component in the reference's 'r' layout. The radix schedule of an axis is
// data, or compiled in for the lengths of FH_RT_LENGTHS.
//
// Why these exist beside the fixed-length passes: the fixed kernels are compiled per length and need
// five launches per 3-D operator application. Here the radix schedule of an axis is data (so every
// smooth length runs the same code), a workgroup owns one component, and on grids whose plane fits
// LDS the two inner axes are transformed in one kernel: three launches and half of the spectrum
// traffic (4 sweeps of the half spectrum instead of 8). Measured per operator application against the
// kernels that served the grid before: 128^3 double 409 -> 99 us (0.32 GB, 3.2 TB/s), 90 x 100 x 77 double
// 161 -> 62 us, 135^3 single 80 -> 71 us, 81^3 elasticity single 58 -> 42 us, 45^2 double 17 -> 15 us.
// Bounds: small grids are latency (about 5 us a kernel: one dependent trip to memory each way and two LDS
// stages); planes in double precision at 100 points and more own their CU alone, so their loads do not
// overlap another workgroup's transforms (128^3: k_fwd 39 us for 0.12 GB); smaller planes are bound by
// VALU issue and LDS.
//
// Kernels
//  k_fwd : A(x) v of one component (with the CG direction update), R2C along axis 2 and, in plane
//          mode, the forward transform along axis 1. A workgroup owns the rows of one plane (or, in row
//          mode, rb consecutive rows).
//  k_cols: transform along a strided axis, forward, inverse, or forward + G(xi) + inverse.
//  k_inv : the inverse of k_fwd, then the epilogue of the operator (store, dot product, CG residual
//          update, or single-precision residual of a right-hand side).
//
// LDS: one complex tile. Two real rows make one complex pencil; pencil q, element e sits at e*S + q
// (S = pencils, odd), so the lanes of a wavefront, which run over q, touch consecutive words. After
// the row transform the pair is untangled in place: row 2q of frequency k replaces element k, row
// 2q+1 replaces element L-k (two extra elements take row 2q+1 at k = 0 and at the Nyquist frequency),
// so the plane needs no second buffer; the transform along axis 1 then runs over pencils k with
// element row at slot(k, row & 1) * S + (row >> 1).
//
// A stage keeps its butterflies in registers between its loads and its stores (in place, two
// barriers). Thread (t, q) = (tid / npen, tid % npen) owns butterflies t, t + TPP, ... of pencil q; every
// address of a butterfly is one origin plus a uniform step, HBM goes through buffer resources (32-bit
// offsets, out-of-range lanes read 0 and store nothing), and index splits are 24-bit multiplies or
// running remainders: an earlier form with 64-bit addresses, a branch per guarded load and 32-bit
// multiply-highs ran the same passes 2-3 times slower.
#pragma once
#include "fh_fixed.hpp"
#include "fh_rt_launch.hpp"

namespace fh {
namespace rt {

// ---- composite butterflies ------------------------------------------------------------------
// R = A * B: input n = n2 + B n1, A-point transforms over n1, twiddles W_R^{n2 k1} (cos / sin of
// 2 pi m / R), B-point transforms over n2, output k = k1 + A k2.
template <int R>
struct MixTab {
  static constexpr int A = 0, B = 0;
};
template <>
struct MixTab<6> {
  static constexpr int A = 3, B = 2;
  static constexpr double c[3] = {1.0, 0.5, -0.5};
  static constexpr double s[3] = {0.0, 0.866025403784438646764, 0.866025403784438646764};
};
template <>
struct MixTab<8> {
  static constexpr int A = 2, B = 4;
  static constexpr double c[4] = {1.0, 0.707106781186547524401, 0.0, -0.707106781186547524401};
  static constexpr double s[4] = {0.0, 0.707106781186547524401, 1.0, 0.707106781186547524401};
};
template <>
struct MixTab<10> {
  static constexpr int A = 5, B = 2;
  static constexpr double c[5] = {1.0, 0.809016994374947424102, 0.309016994374947424102, -0.309016994374947424102, -0.809016994374947424102};
  static constexpr double s[5] = {0.0, 0.587785252292473129169, 0.951056516295153572116, 0.951056516295153572116, 0.587785252292473129169};
};
template <>
struct MixTab<12> {
  static constexpr int A = 4, B = 3;
  static constexpr double c[7] = {1.0, 0.866025403784438646764, 0.5, 0.0, -0.5, -0.866025403784438646764, -1.0};
  static constexpr double s[7] = {0.0, 0.5, 0.866025403784438646764, 1.0, 0.866025403784438646764, 0.5, 0.0};
};
template <>
struct MixTab<15> {
  static constexpr int A = 5, B = 3;
  static constexpr double c[9] = {1.0, 0.913545457642600895502, 0.669130606358858213826, 0.309016994374947424102, -0.1045284632676534714, -0.5, -0.809016994374947424102, -0.978147600733805637929, -0.978147600733805637929};
  static constexpr double s[9] = {0.0, 0.406736643075800207754, 0.743144825477394235015, 0.951056516295153572116, 0.994521895368273336923, 0.866025403784438646764, 0.587785252292473129169, 0.207911690817759337102, -0.207911690817759337102};
};
template <>
struct MixTab<16> {
  static constexpr int A = 4, B = 4;
  static constexpr double c[10] = {1.0, 0.923879532511286756128, 0.707106781186547524401, 0.382683432365089771728, 0.0, -0.382683432365089771728, -0.707106781186547524401, -0.923879532511286756128, -1.0, -0.923879532511286756128};
  static constexpr double s[10] = {0.0, 0.382683432365089771728, 0.707106781186547524401, 0.923879532511286756128, 1.0, 0.923879532511286756128, 0.707106781186547524401, 0.382683432365089771728, 0.0, -0.382683432365089771728};
};

template <typename T, int R, int DIR>
__device__ __forceinline__ void dft_mix(cpx<T> (&v)[R]);

template <typename T, int R, int DIR>
__device__ __forceinline__ void dft_rt(cpx<T> (&v)[R]) {
  if constexpr (R == 9)
    dft9<T, DIR>(v);
  else if constexpr (MixTab<R>::A != 0)
    dft_mix<T, R, DIR>(v);
  else
    dft<T, R, DIR>(v);
}

template <typename T, int R, int DIR>
__device__ __forceinline__ void dft_mix(cpx<T> (&v)[R]) {
  using Tab = MixTab<R>;
  constexpr int A = Tab::A, B = Tab::B;
  cpx<T> a[B][A];
#pragma unroll
  for (int n2 = 0; n2 < B; ++n2) {
    cpx<T> t[A];
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) t[n1] = v[n2 + B * n1];
    dft<T, A, DIR>(t);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      const int m = n2 * k1;
      if (m == 0) {
        a[n2][k1] = t[k1];
      } else if (4 * m == R) {
        a[n2][k1] = DIR < 0 ? mk(t[k1].y, -t[k1].x) : mk(-t[k1].y, t[k1].x);
      } else {
        a[n2][k1] = cmul(t[k1], mk(T(Tab::c[m]), T(DIR < 0 ? -Tab::s[m] : Tab::s[m])));
      }
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    cpx<T> t[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) t[n2] = a[n2][k1];
    dft<T, B, DIR>(t);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = t[k2];
  }
}

// x / d for the thread's start index (once per phase)
__device__ __forceinline__ int quot(int x, const Div d) {
  return d.d == 1 ? x : (int)__umulhi((unsigned)x, d.m);
}

// x / d for any x, d below 2^31, where the multiply-high alone is one too large at times (x * d >= 2^32).
__device__ __forceinline__ int quot_any(int x, const Div d) {
  const int q = quot(x, d);
  return q - ((unsigned)q * d.d > (unsigned)x);
}

// ---- accessors: at(q, e, de) is element e of pencil q; get(j) / put(j, v) element e + j de -----------

// LDS tile, element e of pencil q at e * es + q
template <typename T>
struct LdsAcc {
  cpx<T>* s;
  int es;
  struct H {
    cpx<T>* p;
    int step;
    __device__ __forceinline__ cpx<T> get(int j) const { return p[j * step]; }
    __device__ __forceinline__ void put(int j, cpx<T> v) const { p[j * step] = v; }
  };
  __device__ __forceinline__ H at(int q, int e, int de) const { return H{s + (int)__umul24(e, es) + q, de * es}; }
};

// untangled plane (see the header): pencil k, element = row
__device__ __forceinline__ int tangle_slot1(int k, int L) { return k == 0 ? L : (2 * k == L ? L + 1 : L - k); }

// Row r = e + j de of pencil k sits at slot(k, r & 1) * S + (r >> 1). An even step keeps the parity of e,
// an odd one flips it for odd j only, so two origins serve every j (chosen by j & 1 at compile time) and
// the rest is the uniform (j de) >> 1.
template <typename T>
struct TangleAcc {
  cpx<T>* s;
  int S, L;
  struct H {
    cpx<T>* p[2];
    int de;
    __device__ __forceinline__ cpx<T> get(int j) const { return p[j & 1][(j * de) >> 1]; }
    __device__ __forceinline__ void put(int j, cpx<T> v) const { p[j & 1][(j * de) >> 1] = v; }
  };
  __device__ __forceinline__ H at(int k, int e, int de) const {
    const int b0 = (int)__umul24(k, S), b1 = (int)__umul24(tangle_slot1(k, L), S);
    const int h = e & 1, r = e >> 1;
    cpx<T>* pe = s + (h ? b1 : b0) + r;
    cpx<T>* po = s + (h ? b0 : b1) + r + h;
    return H{{pe, (de & 1) ? po : pe}, de};
  }
};

// HBM through a buffer resource: element e of pencil q at byte e * es + qoff, qoff given by the kernel
// (kDead for a pencil outside the tile). The resource is below 2 GiB (kSpan, checked by the host), so kDead
// plus any step is out of range and does not wrap.
constexpr unsigned kDead = 0x80000000u;
static_assert(kDead == kSpan, "dead lanes sit past every resource");

template <typename T>
struct BufAcc {
  __amdgpu_buffer_rsrc_t r;
  unsigned es, qoff;
  struct H {
    __amdgpu_buffer_rsrc_t r;
    unsigned o, step;
    __device__ __forceinline__ cpx<T> get(int j) const { return bload_c<T>(r, o + (unsigned)j * step); }
    __device__ __forceinline__ void put(int j, cpx<T> v) const { bstore_c<T>(r, o + (unsigned)j * step, v); }
  };
  __device__ __forceinline__ H at(int, int e, int de) const {
    return H{r, qoff + (unsigned)e * es, (unsigned)de * es};
  }
};

// ---- one Stockham stage --------------------------------------------------------------------
// Thread (t, q) of TPP threads per pencil; on = the thread owns a pencil. MID: barrier between the
// loads and the stores (in place in LDS); END: barrier after the stores (a following stage reads them).
template <typename T, int R, int DIR, bool MID, bool END, class Ld, class St>
__device__ __forceinline__ void stage_r(const Stage g, const cpx<T>* tw, int t, int q, int TPP, bool on, const Ld ld,
                                        const St st) {
  constexpr int M = max_m(sizeof(T), R);
  cpx<T> v[M][R];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (m * TPP < g.LR) {
      const int i = t + m * TPP;
      if (on && i < g.LR) {
        const auto h = ld.at(q, i, g.LR);
#pragma unroll
        for (int j = 0; j < R; ++j) v[m][j] = h.get(j);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (m * TPP < g.LR) {
      const int i = t + m * TPP;
      if (on && i < g.LR) {
        if (g.p > 1) {
          const int k = i - (int)__umul24(__umul24(i, g.mp) >> 20, g.p);
          const int b = (int)__umul24(k, g.tws);
          int x = b;
#pragma unroll
          for (int j = 1; j < R; ++j, x += b) {
            cpx<T> w = tw[x];
            if (DIR > 0) w.y = -w.y;
            v[m][j] = cmul(v[m][j], w);
          }
        }
        dft_rt<T, R, DIR>(v[m]);
      }
    }
  }
  if constexpr (MID) __syncthreads();
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (m * TPP < g.LR) {
      const int i = t + m * TPP;
      if (on && i < g.LR) {
        const int k = i - (int)__umul24(__umul24(i, g.mp) >> 20, g.p);
        const auto h = st.at(q, (int)__umul24(i - k, R) + k, g.p);
#pragma unroll
        for (int j = 0; j < R; ++j) h.put(j, v[m][j]);
      }
    }
  }
  if constexpr (END) __syncthreads();
}

template <typename T, int DIR, bool MID, bool END, class Ld, class St>
__device__ __forceinline__ void run_stage(const Stage g, const cpx<T>* tw, int t, int q, int TPP, bool on, const Ld ld,
                                          const St st) {
  switch (g.R) {
#define FH_RT_CASE(RR) \
  case RR: stage_r<T, RR, DIR, MID, END>(g, tw, t, q, TPP, on, ld, st); break;
    FH_RT_RADICES(FH_RT_CASE)
#undef FH_RT_CASE
    default: break;  // no other radix is planned
  }
}

// The passes are compiled with the schedule of one length (CL > 0: every radix, index split and LDS
// address is a constant) or for the schedule that the launch carries (CL 0).
template <int CL>
struct CtAxis {
  static constexpr Axis ax = plan_axis(CL);
};

// First (LAST 0) or last (LAST 1) stage of an axis.
template <typename T, int DIR, int CL, int LAST, bool MID, bool END, class Ld, class St>
__device__ __forceinline__ void end_stage(const Axis& ax, const cpx<T>* tw, int t, int q, int TPP, bool on, const Ld ld,
                                          const St st) {
  if constexpr (CL > 0) {
    constexpr Stage g = CtAxis<CL>::ax.st[LAST ? CtAxis<CL>::ax.nst - 1 : 0];
    stage_r<T, g.R, DIR, MID, END>(g, tw, t, q, TPP, on, ld, st);
  } else {
    run_stage<T, DIR, MID, END>(ax.st[LAST ? ax.nst - 1 : 0], tw, t, q, TPP, on, ld, st);
  }
}

// Stages FROM .. nst - 1 - DROP in place in LDS.
template <typename T, int DIR, int CL, int FROM, int DROP, class Acc>
__device__ __forceinline__ void lds_stages(const Axis& ax, const cpx<T>* tw, int t, int q, int TPP, bool on,
                                           const Acc acc) {
  if constexpr (CL > 0) {
    if constexpr (FROM < CtAxis<CL>::ax.nst - DROP) {
      constexpr Stage g = CtAxis<CL>::ax.st[FROM];
      stage_r<T, g.R, DIR, true, true>(g, tw, t, q, TPP, on, acc, acc);
      lds_stages<T, DIR, CL, FROM + 1, DROP>(ax, tw, t, q, TPP, on, acc);
    }
  } else {
    for (int s = FROM; s < ax.nst - DROP; ++s) run_stage<T, DIR, true, true>(ax.st[s], tw, t, q, TPP, on, acc, acc);
  }
}

// Geometry of the contiguous-axis passes: the launch's (CL 0), the constants of CL x CL planes (PL 1), or
// rows of CL points with the row count of the launch (PL 0).
template <typename T, int CL, int PL>
struct View {
  static constexpr Geo k = const_plane(CL, sizeof(T));
  static constexpr int n2 = k.n2, n2h = k.n2h, S = k.S, rbe = k.rbe, tile = k.tile, tpp2 = k.tpp2, tpp1 = k.tpp1;
  static constexpr int tw1_off = k.tw1_off, plane = 1;
  static constexpr Div dn2 = k.dn2, dn2h = k.dn2h, dpr = k.dpr;
  __device__ __forceinline__ View(const Geo&) {}
};
template <typename T, int CL>
struct View<T, CL, 0> {
  static constexpr int n2 = CL, n2h = CL / 2 + 1, tpp1 = 1, tw1_off = 0, plane = 0;
  static constexpr Div dn2 = make_div(CL), dn2h = make_div(CL / 2 + 1);
  int S, rbe, tile, tpp2;
  Div dpr;
  __device__ __forceinline__ View(const Geo& g) : S(g.S), rbe(g.rbe), tile(g.tile), tpp2(g.tpp2), dpr(g.dpr) {}
};
template <typename T, int PL>
struct View<T, 0, PL> {
  static constexpr int plane = PL;
  int n2, n2h, S, rbe, tile, tpp2, tpp1, tw1_off;
  Div dn2, dn2h, dpr;
  __device__ __forceinline__ View(const Geo& g)
      : n2(g.n2), n2h(g.n2h), S(g.S), rbe(g.rbe), tile(g.tile), tpp2(g.tpp2), tpp1(g.tpp1), tw1_off(g.tw1_off),
        dn2(g.dn2), dn2h(g.dn2h), dpr(g.dpr) {}
};
template <typename T>
struct View<T, 0, 0> {
  static constexpr int plane = 0, tpp1 = 1, tw1_off = 0;
  int n2, n2h, S, rbe, tile, tpp2;
  Div dn2, dn2h, dpr;
  __device__ __forceinline__ View(const Geo& g)
      : n2(g.n2), n2h(g.n2h), S(g.S), rbe(g.rbe), tile(g.tile), tpp2(g.tpp2), dn2(g.dn2), dn2h(g.dn2h), dpr(g.dpr) {}
};

// Values of a run that a thread loads before it uses the first: all of a compiled plane's share in as
// few rounds as `most` allows (each round waits once for memory), `most` / 2 otherwise.
constexpr int load_batch(int ne, int nthr, int most) {
  const int per = (ne + nthr - 1) / nthr, rounds = (per + most - 1) / most;
  return (per + rounds - 1) / rounds;
}

template <typename T, class V>
__device__ __forceinline__ void load_tw(const V& v, cpx<T>* twl, const cpx<T>* tw2, const cpx<T>* tw1, int n1, int tid,
                                        int nthr) {
  for (int e = tid; e < v.n2; e += nthr) twl[e] = tw2[e];
  if (V::plane && v.tw1_off)
    for (int e = tid; e < n1; e += nthr) twl[v.tw1_off + e] = tw1[e];
}

// Rows of the tile (real pairs) -> half spectrum: R2C along axis 2 and, in plane mode, the forward
// transform along axis 1, written to `ro` (the rows' run of one component).
template <typename T, int CL, int PL>
__device__ __forceinline__ void forward_rows(const View<T, CL, PL>& vw, const Geo& g, __amdgpu_buffer_rsrc_t ro,
                                             cpx<T>* s, const cpx<T>* twl, int tid, int nthr) {
  constexpr unsigned CS = sizeof(cpx<T>);
  const int n2h = vw.n2h, S = vw.S, L = vw.n2, npr = vw.rbe >> 1;
  {
    const int t = quot(tid, vw.dpr), q = tid - t * npr;
    lds_stages<T, -1, CL, 0, 0>(g.a2, twl, t, q, vw.tpp2, t < vw.tpp2, LdsAcc<T>{s, S});
  }
  // untangle the paired rows: in place for the transform along axis 1, else straight to HBM
  {
    const int dk = g.dk, dq = g.dq;
    int q = quot(tid, vw.dn2h), k = tid - q * n2h;
    while (q < npr) {
      const cpx<T> Z = s[(int)__umul24(k, S) + q];
      const cpx<T> Zc = conj(s[(int)__umul24(k ? L - k : 0, S) + q]);
      const cpx<T> d = Z - Zc;
      const cpx<T> Ya = T(0.5) * (Z + Zc), Yb = mk(T(0.5) * d.y, T(-0.5) * d.x);
      if constexpr (PL) {
        s[(int)__umul24(k, S) + q] = Ya;
        s[(int)__umul24(tangle_slot1(k, L), S) + q] = Yb;
      } else {
        // rows past nr lie outside of the resource (the last workgroup may own fewer)
        const unsigned o = ((unsigned)(2 * q) * n2h + k) * CS;
        bstore_c<T>(ro, o, Ya);
        bstore_c<T>(ro, o + (unsigned)n2h * CS, Yb);
      }
      k += dk;
      q += dq;
      if (k >= n2h) {
        k -= n2h;
        ++q;
      }
    }
  }
  if constexpr (PL) {
    __syncthreads();
    const cpx<T>* tw1 = twl + vw.tw1_off;
    const int t = quot(tid, vw.dn2h), k = tid - t * n2h;
    const bool on = t < vw.tpp1;
    const TangleAcc<T> at{s, S, L};
    lds_stages<T, -1, CL, 0, 1>(g.a1, tw1, t, k, vw.tpp1, on, at);
    end_stage<T, -1, CL, 1, false, false>(g.a1, tw1, t, k, vw.tpp1, on, at,
                                          BufAcc<T>{ro, (unsigned)n2h * CS, (unsigned)k * CS});
  }
}

// The inverse: half spectrum `ri` (nr rows) -> rows of the tile.
template <typename T, int CL, int PL>
__device__ __forceinline__ void inverse_rows(const View<T, CL, PL>& vw, const Geo& g, __amdgpu_buffer_rsrc_t ri,
                                             cpx<T>* s, const cpx<T>* twl, int tid, int nthr, int nr) {
  constexpr unsigned CS = sizeof(cpx<T>);
  const int n2h = vw.n2h, S = vw.S, L = vw.n2, npr = vw.rbe >> 1;
  if constexpr (PL) {
    const cpx<T>* tw1 = twl + vw.tw1_off;
    const int t = quot(tid, vw.dn2h), k = tid - t * n2h;
    const bool on = t < vw.tpp1;
    const TangleAcc<T> at{s, S, L};
    end_stage<T, +1, CL, 0, false, true>(g.a1, tw1, t, k, vw.tpp1, on,
                                         BufAcc<T>{ri, (unsigned)n2h * CS, (unsigned)k * CS}, at);
    lds_stages<T, +1, CL, 1, 0>(g.a1, tw1, t, k, vw.tpp1, on, at);
  }
  // Hermitian completion into pencils of two real rows; a row past the end is zero
  {
    const int dk = g.dk, dq = g.dq;
    int q = quot(tid, vw.dn2h), k = tid - q * n2h;
    while (q < npr) {
      cpx<T> Ya, Yb;
      if constexpr (PL) {
        Ya = s[(int)__umul24(k, S) + q];
        Yb = s[(int)__umul24(tangle_slot1(k, L), S) + q];
        if (2 * q + 1 >= nr) Yb = mk(T(0), T(0));
      } else {
        const unsigned o = ((unsigned)(2 * q) * n2h + k) * CS;
        Ya = bload_c<T>(ri, o);
        Yb = bload_c<T>(ri, o + (unsigned)n2h * CS);
      }
      if (k == 0 || 2 * k == L) {
        s[(int)__umul24(k, S) + q] = mk(Ya.x, Yb.x);
      } else {
        s[(int)__umul24(k, S) + q] = mk(Ya.x - Yb.y, Ya.y + Yb.x);
        s[(int)__umul24(L - k, S) + q] = mk(Ya.x + Yb.y, Yb.x - Ya.y);
      }
      k += dk;
      q += dq;
      if (k >= n2h) {
        k -= n2h;
        ++q;
      }
    }
  }
  __syncthreads();
  const int t = quot(tid, vw.dpr), q = tid - t * npr;
  lds_stages<T, +1, CL, 0, 0>(g.a2, twl, t, q, vw.tpp2, t < vw.tpp2, LdsAcc<T>{s, S});
}

// ---- forward: A(x) v, R2C along axis 2 (and axis 1) -------------------------------------------
// UPD 0: v = in. UPD 2 (fused CG): first xc += alpha p_old when a step is pending (xc = alpha p_old
// while it holds no value), p = r + beta p_old written to pout, v = p, partial sums of <p, A p>.
// (beta = 0, a (re)start: p = r, whatever the old direction's buffer holds.)
// pout may be `in` where a workgroup reads only its own component (none / isotropic coefficient);
// coupled coefficients (Lame, full) read the other components' p_old, so pout is another buffer.
template <typename T, int UPD, int NT, int CL, int PL>
__global__ void __launch_bounds__(NT) k_fwd(FwdArgs<T> A) {
  if (A.halt && *A.halt) return;
  const Geo& g = A.g;
  const View<T, CL, PL> vw(g);
  constexpr unsigned SR = sizeof(T), CS = sizeof(cpx<T>);
  extern __shared__ __align__(16) unsigned char fh_rt_smem[];
  cpx<T>* s = reinterpret_cast<cpx<T>*>(fh_rt_smem);
  T* sr = reinterpret_cast<T*>(fh_rt_smem);
  cpx<T>* twl = s + vw.tile;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int rblk = quot(lin, g.dnc), c = lin - rblk * g.nc;  // a plane's components follow each other
  const long long row0 = (long long)rblk * g.rb;
  const int nr = (int)min((long long)g.rb, g.nrows - row0);
  const int n2 = vw.n2, n2h = vw.n2h, S = vw.S;
  const long long v0 = row0 * n2, n = g.n;
  T bta = T(0), alp = T(0);
  bool fold = false, fresh = false;
  if constexpr (UPD == 2) {
    bta = T(A.st->beta);
    fold = A.st->pend != 0;
    fresh = A.st->xfresh != 0;
    alp = T(A.st->alpha);
    if (A.bpart && A.st->bpend) {
      // small grids: the previous beta from the inverse pass's partials, as k_rows_fwd_st
      const BetaStep b = beta_step(A.st, fixed_sum_partials(A.bpart, A.bnp));
      if (A.st->mixed ? b.pause_mixed : (b.conv || b.maxed)) return;
      bta = T(b.beta);
    }
  }
  load_tw<T>(vw, twl, A.tw2, A.tw1, g.a1.L, tid, nthr);
  double acc = 0.0;
  // the rows -> LDS, U values per thread in flight; a resource spans the block's run of one component,
  // so the padding row of an odd count reads 0
  const unsigned run = (unsigned)(nr * n2) * SR;
  auto res = [&](const T* base, long long comp) { return make_rsrc(base + comp * n + v0, run); };
  const __amdgpu_buffer_rsrc_t rin = res(A.in, c);
  const __amdgpu_buffer_rsrc_t rr = UPD == 2 ? res(A.r, c) : rin;
  const __amdgpu_buffer_rsrc_t rx = UPD == 2 ? res(A.xc, c) : rin;
  const __amdgpu_buffer_rsrc_t rp = UPD == 2 ? res(A.pout, c) : rin;
  constexpr int UMAX = (sizeof(T) == 4 ? 16 : 8) / (UPD == 2 ? 2 : 1);
  constexpr int U = CL > 0 && PL ? load_batch((CL + 1) / 2 * 2 * CL, NT, UMAX) : UMAX / 2;
  const int ne = vw.rbe * n2, dx = g.dx, drow = g.drow, dn = g.nc == 6 ? 3 : 2;
  const bool rst = UPD == 2 && bta == T(0);
  int row = quot(tid, vw.dn2), x = tid - row * n2;
  for (int e0 = tid; e0 < ne; e0 += U * nthr) {
    T po[U], rv[U], xv[U], pn[U], y[U];
    unsigned o[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      o[u] = (unsigned)(e0 + u * nthr) * SR;
      po[u] = bload_r<T>(rin, o[u]);
      if constexpr (UPD == 2) {
        rv[u] = bload_r<T>(rr, o[u]);
        if (fold && !fresh) xv[u] = bload_r<T>(rx, o[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) pn[u] = UPD == 2 ? (rst ? rv[u] : rv[u] + bta * po[u]) : po[u];
    // p of component d at the thread's values
    auto comp = [&](int d, T(&z)[U]) {
      const __amdgpu_buffer_rsrc_t rd = res(A.in, d);
#pragma unroll
      for (int u = 0; u < U; ++u) z[u] = bload_r<T>(rd, o[u]);
      if constexpr (UPD == 2) {
        const __amdgpu_buffer_rsrc_t qd = res(A.r, d);
        T w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = bload_r<T>(qd, o[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) z[u] = rst ? w[u] : w[u] + bta * z[u];
      }
    };
    if (A.kind == COEF_ISO) {
      const __amdgpu_buffer_rsrc_t ra = res(A.coef, 0);
#pragma unroll
      for (int u = 0; u < U; ++u) y[u] = bload_r<T>(ra, o[u]) * pn[u];
    } else if (A.kind == COEF_LAME) {
      const __amdgpu_buffer_rsrc_t rl = res(A.coef, 0), rm = res(A.coef, 1);
      T mu[U], lam[U], tr[U], z[U];
#pragma unroll
      for (int u = 0; u < U; ++u) mu[u] = bload_r<T>(rm, o[u]);
      if (c < dn) {
#pragma unroll
        for (int u = 0; u < U; ++u) lam[u] = bload_r<T>(rl, o[u]);
        comp(0, tr);
        for (int d = 1; d < dn; ++d) {
          comp(d, z);
#pragma unroll
          for (int u = 0; u < U; ++u) tr[u] += z[u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) y[u] = T(2) * mu[u] * pn[u] + lam[u] * tr[u];
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) y[u] = T(2) * mu[u] * pn[u];
      }
    } else if (A.kind == COEF_FULL) {
#pragma unroll
      for (int u = 0; u < U; ++u) y[u] = T(0);
      for (int d = 0; d < g.nc; ++d) {
        const __amdgpu_buffer_rsrc_t ra = res(A.coef, c * g.nc + d);
        T a[U], z[U];
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = bload_r<T>(ra, o[u]);
        comp(d, z);
#pragma unroll
        for (int u = 0; u < U; ++u) y[u] += a[u] * z[u];
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) y[u] = pn[u];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (UPD == 2) {
        if (fold) bstore_r<T>(rx, o[u], (fresh ? T(0) : xv[u]) + alp * po[u]);
        bstore_r<T>(rp, o[u], pn[u]);
        acc += (double)y[u] * (double)pn[u];
      }
      if (e0 + u * nthr < ne) sr[(((int)__umul24(x, S) + (row >> 1)) << 1) | (row & 1)] = y[u];
      x += dx;
      row += drow;
      if (x >= n2) {
        x -= n2;
        ++row;
      }
    }
  }
  __syncthreads();
  forward_rows<T, CL, PL>(vw, g, make_rsrc(A.out + (long long)c * g.nh + row0 * n2h, (unsigned long long)nr * n2h * CS),
                          s, twl, tid, nthr);
  if constexpr (UPD == 2) {
    const double bs = block_sum(acc);
    if (tid == 0) A.partial[blockIdx.x] = bs;
  }
}

// ---- inverse: (axis 1,) C2R along axis 2, epilogue ----------------------------------------------
// epi 0: out = y. epi 1: also partial sums of <y, w>. epi 2: out is r, r -= alpha y, partial sums of
// <r, r>. epi 3 (double): r32 = float(w - y), partial sums of <w - y, w - y> in double.
template <typename T, int NT, int CL, int PL>
__global__ void __launch_bounds__(NT) k_inv(InvArgs<T> A) {
  if (A.halt && *A.halt) return;
  const Geo& g = A.g;
  const View<T, CL, PL> vw(g);
  constexpr unsigned SR = sizeof(T), CS = sizeof(cpx<T>);
  extern __shared__ __align__(16) unsigned char fh_rt_smem[];
  cpx<T>* s = reinterpret_cast<cpx<T>*>(fh_rt_smem);
  const T* sr = reinterpret_cast<const T*>(fh_rt_smem);
  cpx<T>* twl = s + vw.tile;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int rblk = quot(lin, g.dnc), c = lin - rblk * g.nc;
  const long long row0 = (long long)rblk * g.rb;
  const int nr = (int)min((long long)g.rb, g.nrows - row0);
  const int n2 = vw.n2, n2h = vw.n2h, S = vw.S;
  load_tw<T>(vw, twl, A.tw2, A.tw1, g.a1.L, tid, nthr);
  const __amdgpu_buffer_rsrc_t ri =
      make_rsrc(A.in + (long long)c * g.nh + row0 * n2h, (unsigned long long)nr * n2h * CS);
  inverse_rows<T, CL, PL>(vw, g, ri, s, twl, tid, nthr, nr);
  const T scale = A.scale;
  const T alp = A.epi == 2 ? T(A.st->alpha) : T(0);
  const long long o0 = (long long)c * g.n + row0 * n2;
  const int nv = nr * n2;
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(A.out + o0, (unsigned)nv * SR);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc((A.epi == 2 ? A.out : A.w) + o0, (unsigned)nv * SR);
  double acc = 0.0;
  constexpr int U = CL > 0 && PL ? load_batch(CL * CL, NT, sizeof(T) == 4 ? 16 : 8) : 4;
  const int dx = g.dx, drow = g.drow;
  int row = quot(tid, vw.dn2), x = tid - row * n2;
  for (int e0 = tid; e0 < nv; e0 += U * nthr) {
    T wv[U];
    if (A.epi) {
#pragma unroll
      for (int u = 0; u < U; ++u) wv[u] = bload_r<T>(rw, (unsigned)(e0 + u * nthr) * SR);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned e = (unsigned)(e0 + u * nthr);
      const bool ok = (int)e < nv;
      const int l = ok ? (((int)__umul24(x, S) + (row >> 1)) << 1) | (row & 1) : 0;
      const T y = scale * sr[l];
      x += dx;
      row += drow;
      if (x >= n2) {
        x -= n2;
        ++row;
      }
      if (A.epi <= 1) {
        bstore_r<T>(ro, e * SR, y);
        if (A.epi == 1 && ok) acc += (double)y * (double)wv[u];
      } else if (A.epi == 2) {
        const T rn = wv[u] - alp * y;
        bstore_r<T>(ro, e * SR, rn);
        if (ok) acc += (double)rn * (double)rn;
      } else if (ok) {
        const T d = wv[u] - y;
        A.r32[o0 + e] = (float)d;
        acc += (double)d * (double)d;
      }
    }
  }
  if (A.epi) {
    const double bs = block_sum(acc);
    if (tid == 0) A.partial[blockIdx.x] = bs;
  }
  if (A.defer_beta && blockIdx.x == 0 && tid == 0) A.st->bpend = 1;
}

// ---- strided axis: forward (MODE 0), inverse (1), forward + G(xi) + inverse (2) --------------------
// The array is viewed as `outer` slabs of L x nf complex values (element stride es); a tile is F
// (a power of two) consecutive points of the nf, in MODE 2 with all NC components (stride cs apart),
// so G reads every component of a frequency from LDS.
template <typename T, int NC, int MODE, int CL>
__global__ void __launch_bounds__(512) k_cols(ColArgs<T> A) {
  if (A.halt && *A.halt) return;
  if (A.fin.st && blockIdx.x == 0) cg_fin_block(A.fin);
  constexpr unsigned CS = sizeof(cpx<T>);
  extern __shared__ __align__(16) unsigned char fh_rt_smem[];
  cpx<T>* s = reinterpret_cast<cpx<T>*>(fh_rt_smem);
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int lf = A.lf, F = 1 << lf, P = F * NC, TPP = A.tpp;
  const Axis& ax = A.ax;
  const int L = CL > 0 ? CL : ax.L;
  cpx<T>* twl = s + L * P;
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  // a flat grid's tiles along the outermost axis, times its slabs, pass the range of quot()
  const int o = MODE == 2 ? 0 : quot_any(lin, A.dtiles), tile = lin - o * A.ntiles;
  const int f0 = tile << lf;
  const int nf = min(F, A.nf - f0);
  for (int e = tid; e < L; e += nthr) twl[e] = A.tw[e];
  const int t = NC == 1 ? tid >> lf : quot(tid, A.dP), q = tid - t * P;
  const bool on = t < TPP;
  const int c = q >> lf, f = q & (F - 1);
  const unsigned qoff = f < nf ? ((unsigned)c * (unsigned)A.cs + (unsigned)f) * CS : kDead;
  const long long base = (long long)o * A.ostride + f0;
  const unsigned long long span = (unsigned long long)(A.total - base) * CS;
  const BufAcc<T> src{make_rsrc(A.src + base, span), (unsigned)A.es * CS, qoff};
  const BufAcc<T> dst{make_rsrc(A.dst + base, span), (unsigned)A.es * CS, qoff};
  const LdsAcc<T> at{s, P};
  constexpr int DIR = MODE == 1 ? +1 : -1;
  if constexpr (MODE != 2) {
    if (A.ax.nst == 1) {
      end_stage<T, DIR, CL, 0, false, false>(ax, twl, t, q, TPP, on, src, dst);
      return;
    }
  }
  end_stage<T, DIR, CL, 0, false, true>(ax, twl, t, q, TPP, on, src, at);
  if constexpr (MODE != 2) {
    lds_stages<T, DIR, CL, 1, 1>(ax, twl, t, q, TPP, on, at);
    end_stage<T, DIR, CL, 1, false, false>(ax, twl, t, q, TPP, on, at, dst);
  } else {
    lds_stages<T, -1, CL, 1, 0>(ax, twl, t, q, TPP, on, at);
    {
      const int fs = tid & (F - 1), fp = f0 + fs;
      int k1 = 0, k2 = fp;
      if (A.g.n0 > 1) {
        k1 = quot(fp, A.dn2h);
        k2 = fp - k1 * A.n2h;
      }
      if (fs < nf) {
        for (int e = tid >> lf; e < L; e += nthr >> lf) {
          cpx<T> v[NC];
          cpx<T>* sp = s + e * P + fs;
#pragma unroll
          for (int d = 0; d < NC; ++d) v[d] = sp[d << lf];
          if (A.g.n0 > 1)
            apply_G_fx<T, NC>(v, e, k1, k2, A.g);
          else
            apply_G_fx<T, NC>(v, 0, e, fp, A.g);
#pragma unroll
          for (int d = 0; d < NC; ++d) sp[d << lf] = v[d];
        }
      }
    }
    __syncthreads();
    lds_stages<T, +1, CL, 0, 1>(ax, twl, t, q, TPP, on, at);
    end_stage<T, +1, CL, 1, false, false>(ax, twl, t, q, TPP, on, at, dst);
  }
}

}  // namespace rt
}  // namespace fh
