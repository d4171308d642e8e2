// Host entry points of the sweep kernels, one instantiation set per (lattice, storage type).
#pragma once
#include <hip/hip_runtime.h>

#include "lbmx_common.h"

namespace lbmx {

// Each returns hipErrorInvalidValue for an operator/coupling combination that is not built.
#define LBMX_DECLARE_LAUNCHERS(SUFFIX)                                                                   \
  hipError_t launch_fwd_##SUFFIX(int coll, int des, const FwdArgs& a, hipStream_t s);                    \
  hipError_t launch_init_##SUFFIX(int coll, int des, const FwdArgs& a, const double* macros,             \
                                  const double* u, double rho0, double T0, hipStream_t s);               \
  hipError_t launch_adj_##SUFFIX(int coll, int des, const AdjArgs& a, hipStream_t s);                    \
  hipError_t launch_neumann_fix_##SUFFIX(const DevBC& e, void* lam, const Layout& ll, const double* nside,  \
                                         hipStream_t s);
#define LBMX_DECLARE_LATTICE(LAT) \
  LBMX_DECLARE_LAUNCHERS(LAT##_f64) LBMX_DECLARE_LAUNCHERS(LAT##_f32) LBMX_DECLARE_LAUNCHERS(LAT##_f16) LBMX_DECLARE_LAUNCHERS(LAT##_bf16)
LBMX_DECLARE_LATTICE(d2q9)
LBMX_DECLARE_LATTICE(d3q19)
LBMX_DECLARE_LATTICE(thermal)
#undef LBMX_DECLARE_LATTICE
#undef LBMX_DECLARE_LAUNCHERS

// Several steps per launch (2D lattices): single lattices and batches (kind 0 forward, 1 reverse).
#define LBMX_DECLARE_STEPS(SUFFIX)                                                              \
  hipError_t launch_fwd_steps_##SUFFIX(int coll, int des, const FwdSteps& a, hipStream_t s);    \
  hipError_t launch_adj_steps_##SUFFIX(int coll, int des, const AdjSteps& a, hipStream_t s);    \
  hipError_t launch_batch_steps_##SUFFIX(int coll, int des, int kind, const BatchSteps& st, hipStream_t s);
LBMX_DECLARE_STEPS(d2q9_f64) LBMX_DECLARE_STEPS(d2q9_f32) LBMX_DECLARE_STEPS(d2q9_f16) LBMX_DECLARE_STEPS(d2q9_bf16)
LBMX_DECLARE_STEPS(thermal_f64) LBMX_DECLARE_STEPS(thermal_f32) LBMX_DECLARE_STEPS(thermal_f16) LBMX_DECLARE_STEPS(thermal_bf16)
#undef LBMX_DECLARE_STEPS

// Zero fill of a device range (bytes a multiple of 4) by a kernel.
hipError_t fill_zero(void* p, size_t bytes, hipStream_t s);

// FP64 -> FP32 conversion of n values (design fields of the reduced-storage forms).
hipError_t convert_f64_f32(float* out, const double* in, long long n, hipStream_t s);

// Design pipeline kernels (natural-order FP64 fields on the full grid).
// Projection of one stage: (tb + tanh(beta (x - eta))) / tsum with tb = tanh(beta eta) and
// tsum = tb + tanh(beta (1 - eta)); with a per-node eta field (etaf != nullptr) eta, tb and
// tsum are those of etaf[i].
struct ProjectArgs {
  int on;              // 0: the stage does not project
  double beta, eta, tb, tsum;
  const double* etaf;
};
struct ConeArgs {
  // input: the full field `in`, or with design != nullptr the mapped field (inside dbox
  // design[box-local i], elsewhere background[i])
  const double* in;
  const double* design;
  const double* background;
  double* out;         // full field: the filtered field (forward), W^T in (transposed)
  const double* den;   // forward: divide by den inside the box (nullptr: no division)
  const double* wt;    // weights [(dz+R)(2R+1) + dy+R][dx+R], (2R+1)^3 entries (2D: dz = 0 only)
  const double* wd2;   // the same weights by squared offset: R - sqrt(d2), d2 = 0 .. R^2
  const int* rx;       // per (dz, dy): largest |dx| with dx^2+dy^2+dz^2 <= R^2, or -1
  int nx, ny, nz, R;
  int box[6];          // filter box, inclusive, clipped to the grid
  int dbox[6];         // design box
  int transposed;      // 0: out = W in (rows in the box), 1: out = W^T in
  // forward: projected field and a copy of the stage's output (either may be nullptr)
  ProjectArgs proj;
  double* proj_out;
  double* copy_out;
  // transposed, one of: design_out != nullptr: only the design box's entries, box-local;
  // scale_den != nullptr: out = the result scaled for the stage before (its projection `proj`
  // at its filtered field scale_x, divided by scale_den), see launch_sens_scale
  double* design_out;
  const double* scale_x;
  const double* scale_den;
};
hipError_t launch_cone(const ConeArgs& a, hipStream_t s);
// (its kernels of one radius: 2D radii 1..8 and 9..12, 3D radii 1..3)
hipError_t launch_cone_2d_small(const ConeArgs& a, hipStream_t s);
hipError_t launch_cone_2d_large(const ConeArgs& a, hipStream_t s);
hipError_t launch_cone_3d_small(const ConeArgs& a, hipStream_t s);
// out = (inside box && project ? sens * (1 - tanh(beta (x - eta))^2) beta / tsum : sens) / den
hipError_t launch_sens_scale(double* out, const double* sens, const double* x, const double* den, int nx, int ny,
                             int nz, const int box[6], const ProjectArgs& p, hipStream_t s);

// Method of moving asymptotes: one update's per-variable inputs (n variables, m <= 8
// constraints) and the dual iteration's state on the device.
constexpr int kMmaMaxM = 8;
struct MmaArgs {
  long long n;
  int m, k, con_mod, asym_type;
  double movlim, asyminit, asymdec, asyminc;
  const double* x;                 // the design the subproblem is built around
  const double* dfdx;
  const double* dgdx[kMmaMaxM];    // constraint sensitivities, one row each
  double *L, *U;                   // asymptotes (in: of the last update, out: of this one)
};
struct MmaConsts {
  double a[kMmaMaxM], c[kMmaMaxM], gx[kMmaMaxM];
  double tol;                      // the iteration ends when epsi falls to this
};
struct MmaState {
  double lam[kMmaMaxM], mu[kMmaMaxM], y[kMmaMaxM], b[kMmaMaxM];
  double z, epsi, err;
  int loop, newton_iters, done, started;
};
int mma_blocks(long long n);  // blocks of the reductions (partials per block)
// The subproblem at a.x: asymptotes into a.L, a.U, the design into xkeep (which may be xo2), and
// the state of a dual iteration that starts there.
hipError_t launch_mma_gensub(const MmaArgs& a, const double* xo1, const double* xo2, double* xkeep, const MmaConsts& c,
                             double* part, MmaState* state, hipStream_t s);
// One Newton iteration of the dual (nothing once state->done is set): the sums at x(lam), the
// residual they leave, and the next multipliers.
hipError_t launch_mma_newton(const MmaArgs& a, const MmaConsts& c, double* part, MmaState* state, hipStream_t s);
// xnew (and xnew2 unless nullptr) = x(lam)
hipError_t launch_mma_primal(const MmaArgs& a, const MmaState* state, double* xnew, double* xnew2, hipStream_t s);
// out[0] = max |xnew - xo1|
hipError_t launch_mma_change(const double* xnew, const double* xo1, long long n, double* part, double* out,
                             hipStream_t s);

// Batched sweeps (kind 0 forward, 1 adjoint) over every instance of a batch; ty = tile rows,
// pair = the forward of a 2- or 4-row tile takes two nodes per thread.
#define LBMX_DECLARE_BATCH(SUFFIX) \
  hipError_t launch_batch_##SUFFIX(int coll, int des, int ty, bool pair, int kind, const BatchStep& st, hipStream_t s);
LBMX_DECLARE_BATCH(d2q9_f64) LBMX_DECLARE_BATCH(d2q9_f32) LBMX_DECLARE_BATCH(d2q9_f16) LBMX_DECLARE_BATCH(d2q9_bf16)
LBMX_DECLARE_BATCH(d3q19_f64) LBMX_DECLARE_BATCH(d3q19_f32) LBMX_DECLARE_BATCH(d3q19_f16) LBMX_DECLARE_BATCH(d3q19_bf16)
LBMX_DECLARE_BATCH(thermal_f64) LBMX_DECLARE_BATCH(thermal_f32) LBMX_DECLARE_BATCH(thermal_f16) LBMX_DECLARE_BATCH(thermal_bf16)
#undef LBMX_DECLARE_BATCH

}  // namespace lbmx
