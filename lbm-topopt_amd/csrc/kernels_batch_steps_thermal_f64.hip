// Batched sweeps, several steps per launch (every instance of a batch in one launch) for the thermal D2Q9 + D2Q5 lattice,
// incompressible BGK / MRT flow part; storage f64.
#include "lbmx_steps.hpp"
#include "lbmx_launch.h"
#define LAT LatD2Q9D2Q5
#define PREC PrecF64
#define SUFFIX thermal_f64
#define BATCH_OPS X(C_BGK) X(C_MRT)
#include "lbmx_batch_steps_dispatch.inc"
