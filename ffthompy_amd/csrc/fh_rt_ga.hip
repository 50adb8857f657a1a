// Launchers of the Ga energies' passes (fh_rt_ga.hpp).
#include "fh_rt_ga.hpp"

#include "fh_rt_impl.hpp"

namespace fh {
namespace rt {

hipError_t launch_pad(PadArgs x, unsigned nblk, int nthr, size_t lds, const Launch& s) {
#define FH_RT_PAD(CL)                                                             \
  {                                                                               \
    static const bool ok = allow(k_pad<CL>);                                      \
    (void)ok;                                                                     \
    return launch((const void*)k_pad<CL>, nblk, nthr, lds, s, &x);                \
  }
  switch (x.ax.L) {
#define FH_RT_CASE(L) case L: FH_RT_PAD(L)
    FH_GA_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
    default: FH_RT_PAD(0)
  }
#undef FH_RT_PAD
}

template <int NC, int MODE>
static hipError_t rows_go(GaRowArgs& x, unsigned nblk, int nthr, size_t lds, const Launch& s) {
#define FH_RT_ROWS(CL)                                                                   \
  {                                                                                      \
    static const bool ok = allow(k_ga_rows<NC, CL, MODE>);                              \
    (void)ok;                                                                            \
    return launch((const void*)(k_ga_rows<NC, CL, MODE>), nblk, nthr, lds, s, &x);      \
  }
  if constexpr (NC == 3 && MODE != GA_STORE) {
    switch (x.ax.L) {
#define FH_RT_CASE(L) case L: FH_RT_ROWS(L)
      FH_GA_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
      default: break;
    }
  }
  FH_RT_ROWS(0)
#undef FH_RT_ROWS
}

hipError_t launch_ga_rows(int nc, bool store, GaRowArgs x, unsigned nblk, int nthr, size_t lds, const Launch& s) {
  const bool iso = x.kind == COEF_ISO;
  if (nc == 2 && store) return rows_go<2, GA_STORE>(x, nblk, nthr, lds, s);
  if (nc == 3 && store) return rows_go<3, GA_STORE>(x, nblk, nthr, lds, s);
  if (nc == 6 && store) return rows_go<6, GA_STORE>(x, nblk, nthr, lds, s);
  if (nc == 2) return iso ? rows_go<2, GA_ISO>(x, nblk, nthr, lds, s) : rows_go<2, GA_FULL>(x, nblk, nthr, lds, s);
  if (nc == 3) return iso ? rows_go<3, GA_ISO>(x, nblk, nthr, lds, s) : rows_go<3, GA_FULL>(x, nblk, nthr, lds, s);
  return hipErrorInvalidValue;
}

}  // namespace rt
}  // namespace fh
