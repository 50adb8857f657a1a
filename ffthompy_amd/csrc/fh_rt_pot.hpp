// Potential formulation on the passes of any smooth length (fh_rt.hpp): the gradient spectrum is component
// -major, the strided passes along the outermost axis expand and contract the scalar potential, and the
// middle of the operator (axis 1 inverse, C2R, a(x), R2C, axis 1 forward) is one kernel per plane.
// Traffic per application in scalar spectra S (3-D): 3 S + 3 S in, 3 S + 3 S + coefficient in the round
// trip, 3 S + 2 S out; with separate passes along axis 1 (planes larger than LDS) 12 S more.
#pragma once
#include "fh_rt.hpp"

namespace fh {
namespace rt {

// view frequencies of point fp of the inner axes at index i of the transformed (outermost) axis
__device__ __forceinline__ void pot_freq(int i, int fp, const Div& dn2h, const pot::PotParams& g, int (&k)[3]) {
  int i1 = i, i2 = fp;
  k[0] = 0;
  if (g.n0 > 1) {
    i1 = quot(fp, dn2h);
    i2 = fp - i1 * g.n2h;
    k[0] = (2 * i >= g.n0) ? i - g.n0 : i;
  }
  k[1] = (2 * i1 >= g.n1) ? i1 - g.n1 : i1;
  k[2] = ((g.n2 & 1) == 0 && 2 * i2 == g.n2) ? -i2 : i2;
}

template <int NC, int DIR, int CL>
__global__ void __launch_bounds__(512) k_pot(PotArgs A) {
  using T = double;
  if (A.halt && *A.halt) return;
  constexpr unsigned CS = sizeof(cpx<T>);
  constexpr int U = 4;  // points of a sweep in flight per thread
  extern __shared__ __align__(16) unsigned char fh_rt_smem[];
  cpx<T>* s = reinterpret_cast<cpx<T>*>(fh_rt_smem);
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int lf = A.lf, F = 1 << lf, P = F * NC, TPP = A.tpp;
  const Axis& ax = A.ax;
  const int L = CL > 0 ? CL : ax.L;
  cpx<T>* twl = s + L * P;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  const int f0 = tile << lf;
  const int nf = min(F, A.es - f0);
  for (int e = tid; e < L; e += nthr) twl[e] = A.tw[e];
  const int t = quot(tid, A.dP), q = tid - t * P;
  const bool on = t < TPP;
  const int c = q >> lf, f = q & (F - 1);
  const unsigned qoff = f < nf ? ((unsigned)c * (unsigned)A.cs + (unsigned)f) * CS : kDead;
  const BufAcc<T> mem{make_rsrc(A.data + f0, ((unsigned long long)A.cs * NC - f0) * CS), (unsigned)A.es * CS, qoff};
  const LdsAcc<T> at{s, P};
  // sweep over the tile's points: thread -> point fs, axis indices e, e + step, ...
  const int fs = tid & (F - 1), fp = f0 + fs, step = nthr >> lf;
  const unsigned es = (unsigned)A.es * CS, fo = fs < nf ? (unsigned)fp * CS : kDead;
  const unsigned long long span = (unsigned long long)A.cs * CS;
  if constexpr (DIR > 0) {
    const bool upd = A.r != nullptr;
    T bta = upd ? T(A.st->beta) : T(0), alp = T(0);
    bool fold = false, fresh = false;
    if (A.x) {
      fold = A.st->pend != 0;
      fresh = A.st->xfresh != 0;
      alp = T(A.st->alpha);
      if (A.bpart && A.st->bpend) {
        const BetaStep b = beta_step(A.st, fixed_sum_partials(A.bpart, A.bnp));
        if (A.st->mixed ? b.pause_mixed : (b.conv || b.maxed)) return;
        bta = T(b.beta);
      }
    }
    const bool rst = bta == T(0);
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(A.p, span), rr = make_rsrc(upd ? A.r : A.p, span);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(fold ? A.x : A.p, span);
    for (int e0 = tid >> lf; e0 < L; e0 += U * step) {
      cpx<T> u[U], rv[U], xv[U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int e = e0 + i * step;
        const unsigned o = e < L ? fo + (unsigned)e * es : kDead;
        u[i] = bload_c<T>(rp, o);
        if (upd) rv[i] = bload_c<T>(rr, o);
        xv[i] = mk(T(0), T(0));
        if (fold && !fresh) xv[i] = bload_c<T>(rx, o);
      }
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int e = e0 + i * step;
        if (e >= L) continue;
        if (fold) bstore_c<T>(rx, fo + (unsigned)e * es, mk(xv[i].x + alp * u[i].x, xv[i].y + alp * u[i].y));
        if (upd) {
          u[i] = rst ? rv[i] : mk(rv[i].x + bta * u[i].x, rv[i].y + bta * u[i].y);
          bstore_c<T>(rp, fo + (unsigned)e * es, u[i]);
        }
        cpx<T> v[NC];
#pragma unroll
        for (int d = 0; d < NC; ++d) v[d] = mk(T(0), T(0));
        int k[3];
        pot_freq(e, fp, A.dn2h, A.g, k);
        T qv[3] = {T(0), T(0), T(0)}, Pw = T(1);
        if (fs < nf && pot::grad_symbol<T>(k, A.g, qv, Pw)) {
          const cpx<T> w = mk(Pw * u[i].x, Pw * u[i].y);
#pragma unroll
          for (int d = 0; d < NC; ++d) v[d] = mk(-qv[d] * w.y, qv[d] * w.x);
        }
#pragma unroll
        for (int d = 0; d < NC; ++d) s[e * P + (d << lf) + fs] = v[d];
      }
    }
    __syncthreads();
    lds_stages<T, +1, CL, 0, 1>(ax, twl, t, q, TPP, on, at);
    end_stage<T, +1, CL, 1, false, false>(ax, twl, t, q, TPP, on, at, mem);
  } else {
    double ps = 0.0;
    T alp = T(0);
    if (A.upd_r) {
      if (A.np1) {
        ps = fixed_sum_partials(A.p1, A.np1);
        const double pAp = ps * A.st->inv_nvox;
        if (!(pAp > 0.0) || !isfinite(pAp)) {  // breakdown: no workgroup changes r
          if (blockIdx.x == 0 && tid == 0) cg_step_known(A.st, ps);
          return;
        }
        alp = T(A.st->rr / pAp);
      } else {
        alp = T(A.st->alpha);
      }
    }
    end_stage<T, -1, CL, 0, false, true>(ax, twl, t, q, TPP, on, mem, at);
    lds_stages<T, -1, CL, 1, 0>(ax, twl, t, q, TPP, on, at);
    const bool step_r = A.upd_r != nullptr, dot = A.w != nullptr || step_r;
    cpx<T>* dst = step_r ? A.upd_r : A.out;
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(dst, span);
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(step_r || !A.w ? dst : A.w, span);
    double acc = 0.0;
    for (int e0 = tid >> lf; e0 < L; e0 += U * step) {
      cpx<T> wv[U];
      if (dot) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const int e = e0 + i * step;
          wv[i] = bload_c<T>(rw, e < L ? fo + (unsigned)e * es : kDead);
        }
      }
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int e = e0 + i * step;
        if (e >= L || fs >= nf) continue;
        int k[3];
        pot_freq(e, fp, A.dn2h, A.g, k);
        T qv[3] = {T(0), T(0), T(0)}, Pw = T(1);
        cpx<T> o = mk(T(0), T(0));
        if (pot::grad_symbol<T>(k, A.g, qv, Pw)) {
          T re = T(0), im = T(0);
#pragma unroll
          for (int d = 0; d < NC; ++d) {
            const cpx<T> v = s[e * P + (d << lf) + fs];
            re += -qv[d] * v.y;
            im += qv[d] * v.x;
          }
          const T sc = A.sgn * Pw;
          o = mk(sc * re, sc * im);
        }
        cpx<T> w = o;
        if (step_r)
          w = o = mk(wv[i].x - alp * o.x, wv[i].y - alp * o.y);
        else if (dot)
          w = wv[i];
        bstore_c<T>(ro, fo + (unsigned)e * es, o);
        if (dot) {
          const double wt = (k[2] == 0 || ((A.g.n2 & 1) == 0 && 2 * k[2] == -A.g.n2)) ? 1.0 : 2.0;
          acc += wt * ((double)o.x * (double)w.x + (double)o.y * (double)w.y);
        }
      }
    }
    if (dot) {
      const double bs = block_sum(acc);
      if (tid == 0) A.partial[blockIdx.x] = bs;
    }
    if (step_r && blockIdx.x == 0 && tid == 0) {
      // the other workgroups read none of these
      CGState* st = A.st;
      if (A.np1) cg_step_known(st, ps);
      if (A.defer_beta) st->bpend = 1;
    }
  }
}

// C2R, a(x), R2C of one component's rows (PL 0) or plane (PL 1) in place: the real field never leaves LDS.
template <int NT, int CL, int PL>
__global__ void __launch_bounds__(NT) k_trip(TripArgs A) {
  using T = double;
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
  const int rblk = quot(lin, g.dnc), c = lin - rblk * g.nc;
  const long long row0 = (long long)rblk * g.rb;
  const int nr = (int)min((long long)g.rb, g.nrows - row0);
  const int n2 = vw.n2, n2h = vw.n2h, S = vw.S;
  if (A.bpart && blockIdx.x == 0 && A.st->bpend) {
    // the other workgroups read only the halt flag, and on a stop their results are not used
    const double rs = fixed_sum_partials(A.bpart, A.bnp);
    if (tid == 0) {
      finalize_beta(A.st, rs);
      A.st->bpend = 0;
    }
  }
  load_tw<T>(vw, twl, A.tw2, A.tw1, g.a1.L, tid, nthr);
  const __amdgpu_buffer_rsrc_t ri =
      make_rsrc(A.spec + (long long)c * g.nh + row0 * n2h, (unsigned long long)nr * n2h * CS);
  inverse_rows<T, CL, PL>(vw, g, ri, s, twl, tid, nthr, nr);
  double acc = 0.0;
  {
    // a(x) times the scaled rows; a padding row stays as it is (its spectrum is not kept)
    constexpr int UM = 8;
    constexpr int U = CL > 0 && PL ? load_batch(CL * CL, NT, UM) : UM / 2;
    const int nv = nr * n2;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(A.coef + row0 * n2, (unsigned)nv * SR);
    const T scale = A.scale;
    int row = quot(tid, vw.dn2), x = tid - row * n2;
    for (int e0 = tid; e0 < nv; e0 += U * nthr) {
      T a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = bload_r<T>(ra, (unsigned)(e0 + u * nthr) * SR);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (e0 + u * nthr < nv) {
          T* y = sr + ((((int)__umul24(x, S) + (row >> 1)) << 1) | (row & 1));
          const T v = scale * *y, w = a[u] * v;
          *y = w;
          acc += (double)v * (double)w;
        }
        x += g.dx;
        row += g.drow;
        if (x >= n2) {
          x -= n2;
          ++row;
        }
      }
    }
  }
  __syncthreads();
  forward_rows<T, CL, PL>(vw, g, ri, s, twl, tid, nthr);
  if (A.partial) {
    const double bs = block_sum(acc);
    if (tid == 0) A.partial[blockIdx.x] = bs * (double)g.n;
  }
}

}  // namespace rt
}  // namespace fh
