#include "design_cone.hpp"

namespace lbmx {
hipError_t launch_cone_3d_small(const ConeArgs& a, hipStream_t s) { return cone_3d<1, 3>(a, s); }
}  // namespace lbmx
