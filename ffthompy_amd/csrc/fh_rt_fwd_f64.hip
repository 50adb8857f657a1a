// Forward contiguous-axis (plane) pass of any smooth length, double precision (a translation unit of its own, so that
// the build compiles the passes in parallel).
#include "fh_rt_impl.hpp"

namespace fh {
namespace rt {
template hipError_t launch_fwd<double>(const Config&, const FwdArgs<double>&, bool, unsigned, const Launch&);
}  // namespace rt
}  // namespace fh
