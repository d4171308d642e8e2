// Method of moving asymptotes on the device: the per-variable work of one update (move limits,
// asymptotes, the convex separable approximation, the primal point of the dual multipliers),
// the sums over the design variables that the dual Newton iteration needs, and the iteration
// itself on its m multipliers. Sums are reduced in a fixed order (per-block partials, then one
// block over the partials), so an update is deterministic. Arithmetic is separately rounded, as
// in the reference's loops.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "lbmx_launch.h"

namespace lbmx {

namespace {

constexpr int kMmaThreads = 256;

__device__ inline double dmax(double a, double b) { return a > b ? a : b; }
__device__ inline double dmin(double a, double b) { return a < b ? a : b; }

// v of lane (this + D) for the lanes whose partner lies in the same group of 2 D lanes: the
// halves of the wave and its pairs of rows change places in registers, within a row of 16 lanes
// the value is shifted (no trip through LDS, as a shuffle takes).
template <int D>
__device__ __forceinline__ unsigned int lane_down(unsigned int v) {
  if constexpr (D == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];
  else if constexpr (D == 16) return __builtin_amdgcn_permlane16_swap(v, v, false, false)[1];
  else return __builtin_amdgcn_update_dpp(0u, v, 0x100 | D, 0xf, 0xf, true);
}
template <int D>
__device__ __forceinline__ double lane_down(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned long long lo = lane_down<D>((unsigned int)u), hi = lane_down<D>((unsigned int)(u >> 32));
  return __builtin_bit_cast(double, (hi << 32) | lo);
}

// Tree over 256 values (t with t + 128, + 64, .. + 1), by one wave: lane l holds v[j], the value
// of thread l + 64 j. The sum is lane 0's.
__device__ inline double tree_256(const double (&v)[4]) {
  double s = (v[0] + v[2]) + (v[1] + v[3]);
  s = s + lane_down<32>(s);
  s = s + lane_down<16>(s);
  s = s + lane_down<8>(s);
  s = s + lane_down<4>(s);
  s = s + lane_down<2>(s);
  return s + lane_down<1>(s);
}

// Sums `val[0..K)` of every thread of the block into part[k * nblocks + blockIdx.x] (a fixed
// tree over the 256 threads). The values pass through LDS kChunk at a time and each wave sums
// its share of them, so a block of many sums waits at two barriers per chunk.
template <int K>
__device__ inline void block_sums(const double (&val)[K], double* part, int nblocks) {
  constexpr int kChunk = K < 8 ? K : 8;
  __shared__ double red[kChunk][kMmaThreads];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += kChunk) {
    if (k0 > 0) __syncthreads();
#pragma unroll
    for (int k = 0; k < kChunk; ++k)
      if (k0 + k < K) red[k][threadIdx.x] = val[k0 + k];
    __syncthreads();
    for (int k = wave; k < kChunk && k0 + k < K; k += kMmaThreads / 64) {
      const double v[4] = {red[k][lane], red[k][lane + 64], red[k][lane + 128], red[k][lane + 192]};
      const double s = tree_256(v);
      if (lane == 0) part[(size_t)(k0 + k) * nblocks + blockIdx.x] = s;
    }
  }
}

constexpr int kMmaMaxBlocks = 2048;

// out[k] = sum over blocks b of part[k * nblocks + b], by wave `wave` of `waves`: thread t of
// 256 adds the partials t, t + 256, ... in order, then the fixed tree over the 256 threads. All
// of a sum's partials are loaded before the first addition.
__device__ inline void sum_partials(const double* part, int nblocks, int K, double* out, int wave, int waves) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x % 64;
  constexpr int NB = kMmaMaxBlocks / kMmaThreads;
  for (int k = wave; k < K; k += waves) {
    double t[4][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int b = lane + 64 * j + kMmaThreads * i;
        t[j][i] = b < nblocks ? part[(size_t)k * nblocks + b] : 0.0;
      }
    double v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = 0.0;
#pragma unroll
      for (int i = 0; i < NB; ++i) v[j] = v[j] + t[j][i];
    }
    const double s = tree_256(v);
    if (lane == 0) out[k] = s;
  }
}

// The subproblem's per-variable numbers at design x with asymptotes Li, Ui (GenSub). They are
// functions of the update's inputs alone, so every evaluation forms them anew from 4 + m values
// per variable instead of reading the 6 + 2m that they are.
template <int M>
struct SubVar {
  double alpha, beta, p0, q0, p[M], q[M];
};
template <int M>
__device__ inline void subproblem(const MmaArgs& a, long long i, double x, double Li, double Ui, SubVar<M>& v) {
#pragma clang fp contract(off)
  const double up = dmin(1.0, x + a.movlim);
  const double lo = dmax(0.0, x - a.movlim);
  v.alpha = dmax(lo, 0.9 * Li + 0.1 * x);
  v.beta = dmin(up, 0.9 * Ui + 0.1 * x);
  const double ux = Ui - x, xl = x - Li, ul = Ui - Li;
  const double feps = 1.0e-6;
  const double df = a.dfdx[i];
  v.p0 = (ux * ux) * (dmax(0.0, df) + 0.001 * fabs(df) + 0.5 * feps / ul);
  v.q0 = (xl * xl) * (dmax(0.0, -df) + 0.001 * fabs(df) + 0.5 * feps / ul);
#pragma unroll
  for (int j = 0; j < M; ++j) {
    const double g = a.dgdx[j][i];
    if (a.con_mod) {
      v.p[j] = (ux * ux) * (dmax(0.0, g) + 0.001 * fabs(g) + 0.5 * feps / ul);
      v.q[j] = (xl * xl) * (dmax(0.0, -g) + 0.001 * fabs(g) + 0.5 * feps / ul);
    } else {
      v.p[j] = (ux * ux) * dmax(0.0, g);
      v.q[j] = (xl * xl) * dmax(0.0, -g);
    }
  }
}

// p_j / du + q_j / dl and p_j / du - q_j / dl (du, dl > 0). Without the constraint modification
// one of p_j, q_j is zero (g_j has one sign), so one division gives both; adding or subtracting
// the other's exact zero changes nothing.
template <int M>
__device__ inline double pq_sum(const MmaArgs& a, const SubVar<M>& v, int j, double du, double dl) {
#pragma clang fp contract(off)
  if (a.con_mod) return v.p[j] / du + v.q[j] / dl;
  const bool up = v.p[j] > 0.0;
  return (up ? v.p[j] : v.q[j]) / (up ? du : dl);
}
template <int M>
__device__ inline double pq_difference(const MmaArgs& a, const SubVar<M>& v, int j, double du, double dl) {
#pragma clang fp contract(off)
  if (a.con_mod) return v.p[j] / du - v.q[j] / dl;
  const bool up = v.p[j] > 0.0;
  return (up ? v.p[j] : -v.q[j]) / (up ? du : dl);
}

// The primal point of the multipliers, before its bounds; pl, ql: the objective's and
// constraints' coefficients weighted by lam.
template <int M>
__device__ inline double primal_point(const SubVar<M>& v, const double (&lam)[M], double Li, double Ui, double& pl,
                                      double& ql) {
#pragma clang fp contract(off)
  pl = v.p0;
  ql = v.q0;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    pl = pl + v.p[j] * lam[j];
    ql = ql + v.q[j] * lam[j];
  }
  const double sp = sqrt(pl), sq = sqrt(ql);
  return (sp * Li + sq * Ui) / (sp + sq);
}
__device__ inline double clamped(double xp, double alpha, double beta) {
  double x = xp;
  if (x < alpha) x = alpha;
  if (x > beta) x = beta;
  return x;
}

// x^3 to about half a unit of the last place (the products' rounding errors added back)
__device__ inline double cube(double x) {
#pragma clang fp contract(off)
  const double h = x * x, l = __builtin_fma(x, x, -h);
  const double c = h * x;
  return c + (__builtin_fma(h, x, -c) + l * x);
}

// GenSub: move limits clipped to [0, 1], asymptotes, and the partial sums of
// pij / (U - x) + qij / (x - L) for b. The design is kept in xkeep, which may be the buffer of
// xo2 (each entry is read before it is written, by the same thread).
template <int M>
__global__ __launch_bounds__(kMmaThreads) void k_mma_gensub(MmaArgs a, const double* xo1, const double* xo2,
                                                            double* xkeep, double* part) {
#pragma clang fp contract(off)
  double acc[M];
  for (int j = 0; j < M; ++j) acc[j] = 0.0;
  const long long n = a.n;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const double x = a.x[i];
    const double up = dmin(1.0, x + a.movlim);
    const double lo = dmax(0.0, x - a.movlim);
    double Li, Ui;
    if (a.k < 3) {
      Li = (x - a.asyminit * up) + a.asyminit * lo;
      Ui = (x + a.asyminit * up) - a.asyminit * lo;
    } else {
      const double x1 = xo1[i], x2 = xo2[i];
      const double trend = (x - x1) * (x1 - x2);
      const double g = trend < 0.0 ? a.asymdec : (trend > 0.0 ? a.asyminc : 1.0);
      Li = x - g * (x1 - a.L[i]);
      Ui = x + g * (a.U[i] - x1);
      const double span = dmax(1.0e-5, up - lo);
      if (a.asym_type == 0) {
        Li = dmin(dmax(Li, x - 10.0 * span), x - 0.01 * span);
        Ui = dmin(dmax(Ui, x + 0.01 * span), x + 10.0 * span);
      } else {
        Li = dmin(dmax(Li, x - 100.0 * span), x - 1.0e-4 * span);
        Ui = dmin(dmax(Ui, x + 1.0e-4 * span), x + 100.0 * span);
        const double l2 = lo - 1.0e-5, h2 = up + 1.0e-5;
        if (x < l2) {
          Li = x - (h2 - x) / 0.9;
          Ui = x + (h2 - x) / 0.9;
        }
        if (x > h2) {
          Li = x - (x - l2) / 0.9;
          Ui = x + (x - l2) / 0.9;
        }
      }
    }
    a.L[i] = Li;
    a.U[i] = Ui;
    xkeep[i] = x;
    SubVar<M> v;
    subproblem<M>(a, i, x, Li, Ui, v);
    const double ux = Ui - x, xl = x - Li;
#pragma unroll
    for (int j = 0; j < M; ++j) acc[j] = acc[j] + pq_sum<M>(a, v, j, ux, xl);
  }
  block_sums<M>(acc, part, gridDim.x);
}

// At the primal point x(lam): the constraint approximations sum_i pij / (U - x) + qij / (x - L)
// (sums 0 .. M-1) and the Gauss-Newton part of the dual Hessian sum_i PQ_ij d2_i PQ_il (sums
// M + j M + l). Bound by FP64 issue (divisions and square roots) while the inputs fit the
// last-level cache: 15.5 us for 524288 variables and 4 constraints, 42 us when it read stored
// coefficients, called pow and summed through barriers; the step after it takes 9 us of one
// workgroup, against 25 us for the sums alone and a trip to the host.
template <int M>
__global__ __launch_bounds__(kMmaThreads) void k_mma_dual(MmaArgs a, const MmaState* st, double* part) {
#pragma clang fp contract(off)
  if (st->done) return;  // (uniform)
  constexpr int K = M + M * M;
  double acc[K];
#pragma unroll
  for (int j = 0; j < K; ++j) acc[j] = 0.0;
  double lam[M];
#pragma unroll
  for (int j = 0; j < M; ++j) lam[j] = st->lam[j];
  const long long n = a.n;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const double Li = a.L[i], Ui = a.U[i];
    SubVar<M> v;
    subproblem<M>(a, i, a.x[i], Li, Ui, v);
    double pl, ql;
    const double xp = primal_point<M>(v, lam, Li, Ui, pl, ql);
    const double x = clamped(xp, v.alpha, v.beta);
    const double ux = Ui - x, xl = x - Li;
#pragma unroll
    for (int j = 0; j < M; ++j) acc[j] = acc[j] + pq_sum<M>(a, v, j, ux, xl);
    double d2 = -1.0 / (2.0 * pl / cube(ux) + 2.0 * ql / cube(xl));
    if (xp < v.alpha || xp > v.beta) d2 = 0.0;
    double pq[M];
#pragma unroll
    for (int j = 0; j < M; ++j) pq[j] = pq_difference<M>(a, v, j, ux * ux, xl * xl);
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const double t = pq[j] * d2;
#pragma unroll
      for (int l = 0; l < M; ++l) acc[M + j * M + l] = acc[M + j * M + l] + t * pq[l];
    }
  }
  block_sums<K>(acc, part, gridDim.x);
}

template <int M>
__global__ __launch_bounds__(kMmaThreads) void k_mma_primal(MmaArgs a, const MmaState* st, double* xnew, double* xnew2) {
#pragma clang fp contract(off)
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  double lam[M];
#pragma unroll
  for (int j = 0; j < M; ++j) lam[j] = st->lam[j];
  const double Li = a.L[i], Ui = a.U[i];
  SubVar<M> v;
  subproblem<M>(a, i, a.x[i], Li, Ui, v);
  double pl, ql;
  const double x = clamped(primal_point<M>(v, lam, Li, Ui, pl, ql), v.alpha, v.beta);
  xnew[i] = x;
  if (xnew2) xnew2[i] = x;
}

// y, z of the current multipliers (the scalar part of XYZofLAMBDA, MMA.cc:697-716)
template <int M>
__device__ void primal_scalars(MmaState& s, const MmaConsts& c) {
#pragma clang fp contract(off)
  double la = 0.0;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    if (s.lam[j] < 0.0) s.lam[j] = 0.0;
    s.y[j] = dmax(0.0, s.lam[j] - c.c[j]);
    la += s.lam[j] * c.a[j];
  }
  s.z = dmax(0.0, 10.0 * (la - 1.0));
}

// One step of SolveDIP (MMA.cc:655-950) by one thread, from the sums at x(lam): the residual of
// the multipliers reached last, the continuation in epsi, and then the Newton direction
// (DualGrad, DualHess, LU without pivoting) and the step to the next multipliers. The sums that
// give a residual are those that the next direction needs, at the same multipliers.
template <int M>
__device__ void newton_step(MmaState& s, const MmaConsts& c, const double* sums) {
#pragma clang fp contract(off)
  if (s.started) {  // DualResidual
    double nr = 0.0;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const double r1 = sums[j] + (-s.b[j] - c.a[j] * s.z - s.y[j] + s.mu[j]);
      const double r2 = s.mu[j] * s.lam[j] - s.epsi;
      const double f1 = fabs(r1), f2 = fabs(r2);
      const double f = f1 < f2 ? f2 : f1;
      nr = nr < f ? f : nr;
    }
    s.err = nr;
  }
  s.started = 1;
  bool step = s.err > 0.9 * s.epsi && s.loop < 100;
  while (!step && s.epsi > c.tol) {
    s.epsi = s.epsi * 0.1;
    s.loop = 0;
    step = s.err > 0.9 * s.epsi;
  }
  s.done = s.epsi > c.tol ? 0 : 1;
  if (s.done) return;
  s.loop += 1;
  s.newton_iters += 1;
  double grad[M], h[M][M];
  double la = 0.0;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    double g = sums[j];
    g += -s.b[j] - c.a[j] * s.z - s.y[j];
    grad[j] = -1.0 * g - s.epsi / s.lam[j];
#pragma unroll
    for (int l = 0; l < M; ++l) h[j][l] = sums[M + j * M + l];
  }
#pragma unroll
  for (int j = 0; j < M; ++j) {
    la += s.lam[j] * c.a[j];
    if (s.lam[j] > c.c[j]) h[j][j] += -1.0;
    h[j][j] += -s.mu[j] / s.lam[j];
  }
  if (la > 0.0) {
#pragma unroll
    for (int j = 0; j < M; ++j)
#pragma unroll
      for (int l = 0; l < M; ++l) h[j][l] += -10.0 * c.a[j] * c.a[l];
  }
  double tr = 0.0;
#pragma unroll
  for (int j = 0; j < M; ++j) tr += h[j][j];
  double corr = 1e-4 * tr / M;
  if (-corr < 1.0e-7) corr = -1.0e-7;
#pragma unroll
  for (int j = 0; j < M; ++j) h[j][j] += corr;
  // LU without pivoting and the solve (MMA.cc:952-986)
#pragma unroll
  for (int p = 0; p < M - 1; ++p)
#pragma unroll
    for (int i = p + 1; i < M; ++i) {
      h[i][p] = h[i][p] / h[p][p];
#pragma unroll
      for (int j = p + 1; j < M; ++j) h[i][j] = h[i][j] - h[i][p] * h[p][j];
    }
#pragma unroll
  for (int i = 1; i < M; ++i) {
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < i; ++j) acc = acc - h[i][j] * grad[j];
    grad[i] = grad[i] + acc;
  }
  grad[M - 1] = grad[M - 1] / h[M - 1][M - 1];
#pragma unroll
  for (int i = M - 2; i >= 0; --i) {
    double acc = grad[i];
#pragma unroll
    for (int j = i + 1; j < M; ++j) acc = acc - h[i][j] * grad[j];
    grad[i] = acc / h[i][i];
  }
  double sm[M];
  double theta = 1.005;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    sm[j] = -s.mu[j] + s.epsi / s.lam[j] - grad[j] * s.mu[j] / s.lam[j];
    if (theta < -1.01 * grad[j] / s.lam[j]) theta = -1.01 * grad[j] / s.lam[j];
    if (theta < -1.01 * sm[j] / s.mu[j]) theta = -1.01 * sm[j] / s.mu[j];
  }
  theta = 1.0 / theta;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    s.lam[j] = s.lam[j] + theta * grad[j];
    s.mu[j] = s.mu[j] + theta * sm[j];
  }
  primal_scalars<M>(s, c);
}

constexpr int kFinishThreads = 1024;

// The sums of k_mma_gensub's partials and the dual iteration's state to begin with.
template <int M>
__global__ __launch_bounds__(kFinishThreads) void k_mma_begin(const double* part, int nblocks, MmaConsts c,
                                                              MmaState* st) {
#pragma clang fp contract(off)
  __shared__ double sums[M];
  sum_partials(part, nblocks, M, sums, threadIdx.x / 64, kFinishThreads / 64);
  __syncthreads();
  if (threadIdx.x != 0) return;
  MmaState s;
#pragma unroll
  for (int j = 0; j < kMmaMaxM; ++j) s.lam[j] = s.mu[j] = s.y[j] = s.b[j] = 0.0;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    s.b[j] = sums[j] - c.gx[j];
    s.lam[j] = c.c[j] / 2.0;
    s.mu[j] = 1.0;
  }
  s.epsi = 1.0;
  s.err = 1.0;
  s.loop = s.newton_iters = s.done = s.started = 0;
  primal_scalars<M>(s, c);
  *st = s;
}

// The sums of k_mma_dual's partials and one step of the iteration. One workgroup: its 16 waves
// share the sums, its first thread takes the step.
template <int M>
__global__ __launch_bounds__(kFinishThreads) void k_mma_step(const double* part, int nblocks, MmaConsts c,
                                                             MmaState* st) {
  if (st->done) return;  // (uniform)
  constexpr int K = M + M * M;
  __shared__ double sums[K];
  sum_partials(part, nblocks, K, sums, threadIdx.x / 64, kFinishThreads / 64);
  __syncthreads();
  if (threadIdx.x != 0) return;
  MmaState s = *st;
  newton_step<M>(s, c, sums);
  *st = s;
}

// per-block max |xnew - xo1|
__global__ __launch_bounds__(kMmaThreads) void k_mma_change(const double* xnew, const double* xo1, long long n,
                                                              double* part) {
  __shared__ double red[kMmaThreads];
  double v = 0.0;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    v = dmax(v, fabs(xnew[i] - xo1[i]));
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = kMmaThreads / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = dmax(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// maximum of the per-block maxima (one thread over 2048 of them took 154 us, one block 4 us)
__global__ __launch_bounds__(kMmaThreads) void k_mma_max(const double* part, int nblocks, double* out) {
  __shared__ double red[kMmaThreads];
  double v = 0.0;
  for (int b = threadIdx.x; b < nblocks; b += kMmaThreads) v = dmax(v, part[b]);
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = kMmaThreads / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = dmax(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// calls f with m as a compile-time number
template <int M, class F>
hipError_t with_m(int m, F&& f) {
  if constexpr (M <= kMmaMaxM) {
    if (m == M) {
      f(std::integral_constant<int, M>{});
      return hipGetLastError();
    }
    return with_m<M + 1>(m, f);
  }
  return hipErrorInvalidValue;
}

}  // namespace

int mma_blocks(long long n) {
  const long long b = (n + kMmaThreads - 1) / kMmaThreads;
  return (int)(b < kMmaMaxBlocks ? (b < 1 ? 1 : b) : kMmaMaxBlocks);
}

hipError_t launch_mma_gensub(const MmaArgs& a, const double* xo1, const double* xo2, double* xkeep, const MmaConsts& c,
                             double* part, MmaState* state, hipStream_t s) {
  const int nb = mma_blocks(a.n);
  return with_m<1>(a.m, [&](auto mc) {
    constexpr int M = decltype(mc)::value;
    hipLaunchKernelGGL(k_mma_gensub<M>, dim3(nb), dim3(kMmaThreads), 0, s, a, xo1, xo2, xkeep, part);
    hipLaunchKernelGGL(k_mma_begin<M>, dim3(1), dim3(kFinishThreads), 0, s, (const double*)part, nb, c, state);
  });
}

hipError_t launch_mma_newton(const MmaArgs& a, const MmaConsts& c, double* part, MmaState* state, hipStream_t s) {
  const int nb = mma_blocks(a.n);
  return with_m<1>(a.m, [&](auto mc) {
    constexpr int M = decltype(mc)::value;
    hipLaunchKernelGGL(k_mma_dual<M>, dim3(nb), dim3(kMmaThreads), 0, s, a, (const MmaState*)state, part);
    hipLaunchKernelGGL(k_mma_step<M>, dim3(1), dim3(kFinishThreads), 0, s, (const double*)part, nb, c, state);
  });
}

hipError_t launch_mma_primal(const MmaArgs& a, const MmaState* state, double* xnew, double* xnew2, hipStream_t s) {
  const unsigned blocks = (unsigned)((a.n + kMmaThreads - 1) / kMmaThreads);
  return with_m<1>(a.m, [&](auto mc) {
    constexpr int M = decltype(mc)::value;
    hipLaunchKernelGGL(k_mma_primal<M>, dim3(blocks), dim3(kMmaThreads), 0, s, a, state, xnew, xnew2);
  });
}

hipError_t launch_mma_change(const double* xnew, const double* xo1, long long n, double* part, double* out,
                             hipStream_t s) {
  const int nb = mma_blocks(n);
  hipLaunchKernelGGL(k_mma_change, dim3(nb), dim3(kMmaThreads), 0, s, xnew, xo1, n, part);
  hipLaunchKernelGGL(k_mma_max, dim3(1), dim3(kMmaThreads), 0, s, (const double*)part, nb, out);
  return hipGetLastError();
}

}  // namespace lbmx
