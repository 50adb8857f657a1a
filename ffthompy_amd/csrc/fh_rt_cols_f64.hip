// Strided and projection passes of any smooth length, double precision (a translation unit of its own, so that
// the build compiles the passes in parallel).
#include "fh_rt_impl.hpp"

namespace fh {
namespace rt {
template hipError_t launch_cols<double>(int, int, const ColArgs<double>&, unsigned, int, size_t, const Launch&);
}  // namespace rt
}  // namespace fh
