#include "design_cone.hpp"

namespace lbmx {
hipError_t launch_cone_2d_small(const ConeArgs& a, hipStream_t s) { return cone_2d<1, 8>(a, s); }
}  // namespace lbmx
