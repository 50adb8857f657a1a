// Launchers of the runtime-radix passes for one precision (included by the translation units of each pass).
#pragma once
#include <hip/hip_ext.h>

#include "fh_rt.hpp"

namespace fh {
namespace rt {

constexpr int kLdsLimit = 160 * 1024;

// The kernels use more than 64 KiB of dynamic LDS on large planes: raise each kernel's limit once.
inline hipError_t launch(const void* kernel, unsigned nblk, int nthr, size_t lds, const Launch& s, void* args) {
  void* p[] = {args};
  return hipExtLaunchKernel(kernel, dim3(nblk), dim3(nthr), p, lds, s.stream, s.t0, s.t1, 0);
}

template <class K>
inline bool allow(K kernel) {
  return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit - 1024) ==
         hipSuccess;
}

#define FH_RT_GO(...)                                                            \
  do {                                                                           \
    static const bool ok = allow(__VA_ARGS__);                                   \
    (void)ok;                                                                    \
    return launch((const void*)(__VA_ARGS__), nblk, c.nthr, c.lds, s, &x);       \
  } while (0)

// The compiled length of a configuration's planes or rows (0: none).
inline int ct_length(const Config& c) { return !c.g.plane || c.g.rb == c.g.n2 ? c.g.n2 : 0; }

// 512 threads leave a thread 128 registers; only a plane of more than half of the LDS takes 1024
template <typename T, int UPD, int CL>
hipError_t fwd_go(const Config& c, FwdArgs<T>& x, unsigned nblk, const Launch& s) {
  if (!c.g.plane) FH_RT_GO(k_fwd<T, UPD, 512, CL, 0>);
  if constexpr (CL > 0) {
    constexpr int NT = const_plane_threads(CL, sizeof(T));
    if constexpr (NT > 0) FH_RT_GO(k_fwd<T, UPD, NT, CL, 1>);
  } else {
    if (c.nthr > 512) FH_RT_GO(k_fwd<T, UPD, 1024, CL, 1>);
    FH_RT_GO(k_fwd<T, UPD, 512, CL, 1>);
  }
  return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_fwd(const Config& c, const FwdArgs<T>& a, bool upd, unsigned nblk, const Launch& s) {
  FwdArgs<T> x = a;
  switch (ct_length(c)) {
#define FH_RT_CASE(L) \
  case L: return upd ? fwd_go<T, 2, L>(c, x, nblk, s) : fwd_go<T, 0, L>(c, x, nblk, s);
    FH_RT_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
    default: return upd ? fwd_go<T, 2, 0>(c, x, nblk, s) : fwd_go<T, 0, 0>(c, x, nblk, s);
  }
}

template <typename T, int CL>
hipError_t inv_go(const Config& c, InvArgs<T>& x, unsigned nblk, const Launch& s) {
  if (!c.g.plane) FH_RT_GO(k_inv<T, 512, CL, 0>);
  if constexpr (CL > 0) {
    constexpr int NT = const_plane_threads(CL, sizeof(T));
    if constexpr (NT > 0) FH_RT_GO(k_inv<T, NT, CL, 1>);
  } else {
    if (c.nthr > 512) FH_RT_GO(k_inv<T, 1024, CL, 1>);
    FH_RT_GO(k_inv<T, 512, CL, 1>);
  }
  return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_inv(const Config& c, const InvArgs<T>& a, unsigned nblk, const Launch& s) {
  InvArgs<T> x = a;
  switch (ct_length(c)) {
#define FH_RT_CASE(L) \
  case L: return inv_go<T, L>(c, x, nblk, s);
    FH_RT_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
    default: return inv_go<T, 0>(c, x, nblk, s);
  }
}


template <typename T, int CL>
hipError_t cols_go(int nc, int mode, ColArgs<T>& x, unsigned nblk, int nthr, size_t lds, const Launch& s) {
#define FH_RT_COLS(NCC, MODE)                                                                 \
  do {                                                                                        \
    static const bool ok = allow(k_cols<T, NCC, MODE, CL>);                                   \
    (void)ok;                                                                                 \
    return launch((const void*)(k_cols<T, NCC, MODE, CL>), nblk, nthr, lds, s, &x);           \
  } while (0)
  if (mode == 0) FH_RT_COLS(1, 0);
  if (mode == 1) FH_RT_COLS(1, 1);
  switch (nc) {
    case 2: FH_RT_COLS(2, 2);
    case 3: FH_RT_COLS(3, 2);
    case 6: FH_RT_COLS(6, 2);
    default: return hipErrorInvalidValue;
  }
#undef FH_RT_COLS
}

template <typename T>
hipError_t launch_cols(int nc, int mode, const ColArgs<T>& a, unsigned nblk, int nthr, size_t lds, const Launch& s) {
  ColArgs<T> x = a;
  switch (a.ax.L) {
#define FH_RT_CASE(L) \
  case L: return cols_go<T, L>(nc, mode, x, nblk, nthr, lds, s);
    FH_RT_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
    default: return cols_go<T, 0>(nc, mode, x, nblk, nthr, lds, s);
  }
}

}  // namespace rt
}  // namespace fh
