#include "design_cone.hpp"

namespace lbmx {
hipError_t launch_cone_2d_large(const ConeArgs& a, hipStream_t s) { return cone_2d<9, 12>(a, s); }
}  // namespace lbmx
