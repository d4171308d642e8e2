// Batched sweeps, several steps per launch (every instance of a batch in one launch) for D2Q9 incompressible BGK / MRT / cascaded;
// shifted bf16 storage, FP32 arithmetic.
#include "lbmx_steps.hpp"
#include "lbmx_launch.h"
#define LAT LatD2Q9
#define PREC PrecBF16
#define SUFFIX d2q9_bf16
#define BATCH_OPS X(C_BGK) X(C_MRT) X(C_CASC)
#include "lbmx_batch_steps_dispatch.inc"
