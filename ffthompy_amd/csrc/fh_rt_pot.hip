// Launchers of the potential formulation's passes of any smooth length.
#include "fh_rt_pot.hpp"

#include "fh_rt_impl.hpp"

namespace fh {
namespace rt {

template <int CL>
hipError_t trip_go(const Config& c, TripArgs& x, unsigned nblk, const Launch& s) {
  if (!c.g.plane) FH_RT_GO(k_trip<512, CL, 0>);
  if constexpr (CL > 0) {
    constexpr int NT = const_plane_threads(CL, sizeof(double));
    if constexpr (NT > 0) FH_RT_GO(k_trip<NT, CL, 1>);
  } else {
    if (c.nthr > 512) FH_RT_GO(k_trip<1024, CL, 1>);
    FH_RT_GO(k_trip<512, CL, 1>);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_trip(const Config& c, const TripArgs& a, unsigned nblk, const Launch& s) {
  TripArgs x = a;
  switch (ct_length(c)) {
#define FH_RT_CASE(L) \
  case L: return trip_go<L>(c, x, nblk, s);
    FH_RT_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
    default: return trip_go<0>(c, x, nblk, s);
  }
}
template <int CL>
hipError_t pot_go(int nc, PotArgs& x, int nthr, size_t lds, const Launch& s) {
#define FH_RT_POT(NCC, DIR)                                                                        \
  do {                                                                                             \
    static const bool ok = allow(k_pot<NCC, DIR, CL>);                                          \
    (void)ok;                                                                                      \
    return launch((const void*)(k_pot<NCC, DIR, CL>), (unsigned)x.ntiles, nthr, lds, s, &x);    \
  } while (0)
  if (nc == 2 && x.dir > 0) FH_RT_POT(2, 1);
  if (nc == 2) FH_RT_POT(2, -1);
  if (nc == 3 && x.dir > 0) FH_RT_POT(3, 1);
  if (nc == 3) FH_RT_POT(3, -1);
#undef FH_RT_POT
  return hipErrorInvalidValue;
}

hipError_t launch_pot(int nc, const PotArgs& a, int nthr, size_t lds, const Launch& s) {
  PotArgs x = a;
  switch (a.ax.L) {
#define FH_RT_CASE(L) \
  case L: return pot_go<L>(nc, x, nthr, lds, s);
    FH_RT_LENGTHS(FH_RT_CASE)
#undef FH_RT_CASE
    default: return pot_go<0>(nc, x, nthr, lds, s);
  }
}

}  // namespace rt
}  // namespace fh
