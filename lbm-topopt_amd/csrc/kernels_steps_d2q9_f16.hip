// Several steps per launch for D2Q9: incompressible BGK / MRT (forward + adjoint), cascaded and
// standard BGK (forward); storage f16.
#include "lbmx_steps.hpp"
#include "lbmx_launch.h"
#define LAT LatD2Q9
#define PREC PrecF16
#define SUFFIX d2q9_f16
#define FWD_OPS X(C_BGK) X(C_MRT) X(C_CASC) X(C_BGK_STD)
#define ADJ_OPS X(C_BGK) X(C_MRT)
#include "lbmx_steps_dispatch.inc"
