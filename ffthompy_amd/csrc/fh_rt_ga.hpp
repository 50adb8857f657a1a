// Ga energies on the passes of any smooth length: a coarse spectrum (n0, n1, n2/2+1) is interpolated onto
// the quadrature grid (m0, m1, m2) axis by axis, so that the zeros of the enlarged spectrum (3/4 of it and
// more) are neither stored nor transformed along the other axes, and the last transform's rows meet the
// coefficient in LDS: the interpolated fields of the unit loads never reach HBM.
//   k_pad     (.., n, es) -> (.., m, es): zero-padded inverse transform along a strided axis
//   k_ga_rows rows of n2/2+1 -> m2 real values: stored (STORE), or the energies of all unit loads
// Double precision only. 135^3 on 270^3, three loads: 2.5 GB of traffic against 20 GB with the padded
// spectrum stored and transformed whole, component by component (6.2 ms -> 1.1 ms): k_pad 58 us a launch
// (268 MB, 4.6 TB/s), k_ga_rows 490 us (0.9 GB; LDS busy 45 % of the cycles, fp64 arithmetic 37 %).
#pragma once
#include "fh_rt.hpp"

namespace fh {
namespace rt {

// element e of the fine axis (m points) read from the coarse axis (n points): frequencies |k| <= n / 2, the
// Nyquist coefficient of an even n in halves at +n/2 and -n/2, zero elsewhere
struct PadAcc {
  __amdgpu_buffer_rsrc_t r;
  unsigned es, qoff;
  int n, m;
  double scale;
  struct H {
    const PadAcc& a;
    int e, de;
    __device__ __forceinline__ cpx<double> get(int j) const {
      const int i = e + j * de, neg = a.m - i;
      const bool lo = 2 * i <= a.n, hi = 2 * neg <= a.n;
      const int src = lo ? i : a.n - neg;
      const cpx<double> v = bload_c<double>(a.r, lo || hi ? a.qoff + (unsigned)src * a.es : kDead);
      const double f = 2 * src == a.n ? 0.5 * a.scale : a.scale;
      return mk(f * v.x, f * v.y);
    }
  };
  __device__ __forceinline__ H at(int, int e, int de) const { return H{*this, e, de}; }
};

template <int CL>
__global__ void __launch_bounds__(512) k_pad(PadArgs A) {
  constexpr unsigned CS = sizeof(cpx<double>);
  extern __shared__ __align__(16) unsigned char fh_rt_smem[];
  cpx<double>* s = reinterpret_cast<cpx<double>*>(fh_rt_smem);
  const int tid = threadIdx.x, F = 1 << A.lf, TPP = A.tpp;
  const Axis& ax = A.ax;
  const int L = CL > 0 ? CL : ax.L;
  cpx<double>* twl = s + L * F;
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int o = quot(lin, A.dtiles), f0 = (lin - o * A.ntiles) << A.lf;
  const int nf = min(F, A.es - f0);
  for (int e = tid; e < L; e += blockDim.x) twl[e] = A.tw[e];
  const int t = tid >> A.lf, q = tid & (F - 1);
  const bool on = t < TPP;
  const unsigned qoff = q < nf ? (unsigned)q * CS : kDead;
  const PadAcc src{make_rsrc(A.src + (long long)o * A.n * A.es + f0, ((unsigned long long)A.n * A.es - f0) * CS),
                   (unsigned)A.es * CS, qoff, A.n, L, A.scale};
  const BufAcc<double> dst{make_rsrc(A.dst + (long long)o * L * A.es + f0, ((unsigned long long)L * A.es - f0) * CS),
                           (unsigned)A.es * CS, qoff};
  const LdsAcc<double> at{s, F};
  if (ax.nst == 1) {
    end_stage<double, +1, CL, 0, false, false>(ax, twl, t, q, TPP, on, src, dst);
    return;
  }
  end_stage<double, +1, CL, 0, false, true>(ax, twl, t, q, TPP, on, src, at);
  lds_stages<double, +1, CL, 1, 1>(ax, twl, t, q, TPP, on, at);
  end_stage<double, +1, CL, 1, false, false>(ax, twl, t, q, TPP, on, at, dst);
}

// What k_ga_rows does with its rows: stores them, or the energies with an isotropic or a full coefficient.
enum GaMode { GA_STORE = 0, GA_ISO = 1, GA_FULL = 2 };

// A workgroup owns pairs of grid rows of every component (a pencil: component c of both rows) and goes on to
// the next pair; energies: component i NC + c is component c of unit load i. A pass over one pair is a
// chain of short phases, so the next pair's spectrum (PF values per thread) and the isotropic coefficient
// are in flight during the transform, and three workgroups share a CU (270 points, three loads: 47 KB).
template <int NC, int CL, int MODE>
__global__ void __launch_bounds__(512) k_ga_rows(GaRowArgs A) {
  constexpr int NP = MODE == GA_STORE ? NC : NC * NC;  // pencils
  constexpr int S = NP | 1, PF = 2;
  extern __shared__ __align__(16) unsigned char fh_rt_smem[];
  cpx<double>* s = reinterpret_cast<cpx<double>*>(fh_rt_smem);
  const int tid = threadIdx.x, nthr = blockDim.x;
  const Axis& ax = A.ax;
  const int L = CL > 0 ? CL : ax.L, n2h = A.n2h;
  cpx<double>* twl = s + L * S;
  for (int e = tid; e < L; e += nthr) twl[e] = A.tw[e];
  double acc[MODE == GA_STORE ? 1 : NC * NC] = {};
  const int ne = NP * n2h, nz = (L - 2 * n2h + 1) * NP;
  struct Pair {
    cpx<double> a, b;
  };
  auto load = [&](long long grp, int e) {
    const long long row0 = 2 * grp;
    const int p = quot(e, A.dn2h);
    const cpx<double>* y = A.src + (long long)p * A.cs + row0 * n2h + (e - p * n2h);
    Pair v;
    v.a = y[0];
    v.b = row0 + 1 < A.nrows ? y[n2h] : mk(0.0, 0.0);
    return v;
  };
  auto fill = [&](int e, Pair v) {
    const int p = quot(e, A.dn2h), k = e - p * n2h;
    if (2 * k == A.n2) {
      v.a = mk(0.5 * v.a.x, 0.5 * v.a.y);
      v.b = mk(0.5 * v.b.x, 0.5 * v.b.y);
    }
    if (k == 0) {
      s[p] = mk(v.a.x, v.b.x);
    } else {
      s[k * S + p] = mk(v.a.x - v.b.y, v.a.y + v.b.x);
      s[(L - k) * S + p] = mk(v.a.x + v.b.y, v.b.x - v.a.y);
    }
  };
  Pair pre[PF];
  auto prefetch = [&](long long grp, int tid) {
#pragma unroll
    for (int i = 0; i < PF; ++i)
      if (tid + i * nthr < ne) pre[i] = load(grp, tid + i * nthr);
  };
  prefetch(blockIdx.x, tid);  // the grid has no more workgroups than pairs
  for (long long grp = blockIdx.x; grp < A.ngroups; grp += gridDim.x) {
    // the thread's indices opaque: the addresses of every stage, kept in registers over the pairs, would
    // halve the number of workgroups that a CU holds (200 registers against 128)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int t = tid / NP, q = tid - t * NP;
    const long long row0 = 2 * grp;
    const bool two = row0 + 1 < A.nrows;
#pragma unroll
    for (int i = 0; i < PF; ++i)
      if (tid + i * nthr < ne) fill(tid + i * nthr, pre[i]);
    for (int e = tid + PF * nthr; e < ne; e += nthr) fill(e, load(grp, e));
    for (int e = tid; e < nz; e += nthr) s[(n2h + e / NP) * S + e % NP] = mk(0.0, 0.0);
    if (grp + gridDim.x < A.ngroups) prefetch(grp + gridDim.x, tid);
    double a0 = 0.0, a1 = 0.0;
    if (MODE == GA_ISO && tid < L) {
      a0 = A.coef[row0 * L + tid];
      if (two) a1 = A.coef[row0 * L + L + tid];
    }
    __syncthreads();
    lds_stages<double, +1, CL, 0, 0>(ax, twl, t, q, A.tpp, t < A.tpp, LdsAcc<double>{s, S});
    for (int x = tid; x < L; x += nthr) {
      const long long vox = row0 * L + x;
      if constexpr (MODE == GA_STORE) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const cpx<double> v = s[x * S + c];
          A.out[c * A.nvox + vox] = v.x;
          if (two) A.out[c * A.nvox + vox + L] = v.y;
        }
      } else {
        if (MODE == GA_ISO && x != tid) {
          a0 = A.coef[vox];
          if (two) a1 = A.coef[vox + L];
        }
        cpx<double> v[NC][NC];
#pragma unroll
        for (int i = 0; i < NC; ++i)
#pragma unroll
          for (int c = 0; c < NC; ++c) v[i][c] = s[x * S + i * NC + c];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          if (r && !two) break;
          const double a = r ? a1 : a0;
#pragma unroll
          for (int i = 0; i < NC; ++i) {
            double Ae[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
              if constexpr (MODE == GA_ISO) {
                Ae[c] = a * (r ? v[i][c].y : v[i][c].x);
              } else {
                double m = 0.0;
#pragma unroll
                for (int d = 0; d < NC; ++d)
                  m += A.coef[(long long)(c * NC + d) * A.nvox + vox + (r ? L : 0)] * (r ? v[i][d].y : v[i][d].x);
                Ae[c] = m;
              }
            }
#pragma unroll
            for (int j = 0; j < NC; ++j) {
              double m = 0.0;
#pragma unroll
              for (int c = 0; c < NC; ++c) m += Ae[c] * (r ? v[j][c].y : v[j][c].x);
              acc[i * NC + j] += m;
            }
          }
        }
      }
    }
    __syncthreads();
  }
  if constexpr (MODE != GA_STORE) {
    for (int k = 0; k < NC * NC; ++k) {
      dd u;
      u.hi = acc[k];
      u.lo = 0.0;
      u = block_sum_dd(u);
      if (tid == 0) {
        A.partial[(2 * (long long)blockIdx.x) * NC * NC + k] = u.hi;
        A.partial[(2 * (long long)blockIdx.x + 1) * NC * NC + k] = u.lo;
      }
    }
  }
}

}  // namespace rt
}  // namespace fh
