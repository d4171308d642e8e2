// Method of moving asymptotes behind the lbmx_mma_* entry points (src/topOpt/MMA.cc, the
// reference's PETSc MMA with robust constants). Per-variable arrays and the dual Newton
// iteration live on the device; the host queues the iteration's launches and looks at its state
// once per batch of them.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "host_common.hpp"
#include "lbmx.h"
#include "lbmx_launch.h"

namespace lbmx {

struct Mma {
  long long n = 0;
  int m = 0, k = 0;
  double asyminit = 0.5, asymdec = 0.7, asyminc = 1.2;
  int con_mod = 0, asym_type = 0;
  std::vector<double> a, c, lam;
  int newton_iters = 0;
  double last_ms = 0.0;
  hipStream_t st = nullptr;
  MmaState* state_host = nullptr;  // pinned: where the iteration's state is read back to
  DeviceBuffer x, xin, dfdx, dgdx, xo1, xo2, L, U, part, out, tmp, state;

  Mma(long long nn, int mm) : n(nn), m(mm) {
    if (n < 1) throw Error{LBMX_ERR_ARG, "MMA needs at least one design variable"};
    if (m < 1 || m > LBMX_MMA_MAX_CONSTRAINTS) throw Error{LBMX_ERR_ARG, "MMA constraints out of range 1..8"};
    a.assign(m, 0.0);
    c.assign(m, 1000.0);
    lam.assign(m, 0.0);
    const size_t nb = (size_t)n * 8;
    for (DeviceBuffer* d : {&x, &xo1, &xo2, &L, &U}) d->ensure(nb);
    part.ensure((size_t)mma_blocks(n) * (m + m * m) * 8);
    out.ensure(8);
    state.ensure(sizeof(MmaState));
    HIP_OK(hipStreamCreate(&st));
    if (hipHostMalloc(reinterpret_cast<void**>(&state_host), sizeof(MmaState), hipHostMallocDefault) != hipSuccess) {
      (void)hipStreamDestroy(st);
      throw Error{LBMX_ERR_MEM, "hipHostMalloc of the MMA state failed"};
    }
  }
  ~Mma() {
    if (st) {
      (void)hipStreamSynchronize(st);
      (void)hipStreamDestroy(st);
    }
    if (state_host) (void)hipHostFree(state_host);
  }

  MmaArgs args(double movlim) {
    MmaArgs r{};
    r.n = n;
    r.m = m;
    r.k = k;
    r.con_mod = con_mod;
    r.asym_type = asym_type;
    r.movlim = movlim;
    r.asyminit = asyminit;
    r.asymdec = asymdec;
    r.asyminc = asyminc;
    r.L = L.as<double>();
    r.U = U.as<double>();
    return r;
  }

  // whether the n values at p share memory with the n at q without being the same array (the
  // kernels read entry i of every input before they write entry i of the design)
  bool overlaps(const double* p, const double* q) const { return p != q && p < q + n && q < p + n; }

  // Update (MMA.cc:485-524): GenSub, history shift, dual interior-point solve. The caller's
  // arrays are host arrays, or device arrays when dev is set, which are then read in place.
  void update(double* xh, const double* dfdxh, const double* gx, const double* const* dgdxh, double movlim,
              bool dev) {
    auto t0 = std::chrono::steady_clock::now();
    const size_t nb = (size_t)n * 8;
    bool in_place = dev;
    if (dev) {
      in_place = !overlaps(xh, dfdxh);
      for (int j = 0; j < m; ++j) in_place = in_place && !overlaps(xh, dgdxh[j]);
    }
    k += 1;
    MmaArgs ar = args(movlim);
    if (in_place) {
      ar.x = xh;
      ar.dfdx = dfdxh;
      for (int j = 0; j < m; ++j) ar.dgdx[j] = dgdxh[j];
    } else {
      const hipMemcpyKind in = dev ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
      xin.ensure(nb);
      dfdx.ensure(nb);
      dgdx.ensure(nb * m);
      HIP_OK(hipMemcpyAsync(xin.p, xh, nb, in, st));
      HIP_OK(hipMemcpyAsync(dfdx.p, dfdxh, nb, in, st));
      ar.x = xin.as<double>();
      ar.dfdx = dfdx.as<double>();
      for (int j = 0; j < m; ++j) {
        HIP_OK(hipMemcpyAsync(dgdx.as<double>() + (size_t)j * n, dgdxh[j], nb, in, st));
        ar.dgdx[j] = dgdx.as<double>() + (size_t)j * n;
      }
    }
    MmaConsts co{};
    for (int j = 0; j < m; ++j) {
      co.a[j] = a[j];
      co.c[j] = c[j];
      co.gx[j] = gx[j];
    }
    co.tol = 1.0e-9 * std::sqrt((double)(m + n));
    // xo2 <- xo1, xo1 <- the design (the old xo2 buffer is reused)
    HIP_OK(launch_mma_gensub(ar, xo1.as<double>(), xo2.as<double>(), xo2.as<double>(), co, part.as<double>(),
                             state.as<MmaState>(), st));
    std::swap(xo1.p, xo2.p);
    ar.x = xo1.as<double>();
    solve_dual(ar, co);
    const bool direct = dev && in_place;
    HIP_OK(launch_mma_primal(ar, state.as<MmaState>(), x.as<double>(), direct ? xh : nullptr, st));
    if (!direct) HIP_OK(hipMemcpyAsync(xh, x.p, nb, dev ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    last_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }

  // The dual iteration: the host queues a batch of iterations, then reads the state back;
  // iterations queued past the end leave at once. epsi falls from 1 to the tolerance by tenths
  // and mostly takes two iterations at each, which is what the first batch covers.
  void solve_dual(const MmaArgs& ar, const MmaConsts& co) {
    int batch = 6;
    for (double e = 1.0; e > co.tol; e *= 0.1) batch += 2;
    for (;;) {
      for (int i = 0; i < batch; ++i) HIP_OK(launch_mma_newton(ar, co, part.as<double>(), state.as<MmaState>(), st));
      HIP_OK(hipMemcpyAsync(state_host, state.p, sizeof(MmaState), hipMemcpyDeviceToHost, st));
      HIP_OK(hipStreamSynchronize(st));
      if (state_host->done) break;
      batch = 8;
    }
    for (int j = 0; j < m; ++j) lam[j] = state_host->lam[j];
    newton_iters = state_host->newton_iters;
  }

  double design_change(const double* xnew, bool dev) {
    const double* xn = x.as<double>();
    if (xnew && dev) {
      xn = xnew;
    } else if (xnew) {
      tmp.ensure((size_t)n * 8);
      HIP_OK(hipMemcpyAsync(tmp.p, xnew, (size_t)n * 8, hipMemcpyHostToDevice, st));
      xn = tmp.as<double>();
    }
    HIP_OK(launch_mma_change(xn, xo1.as<double>(), n, part.as<double>(), out.as<double>(), st));
    double ch = 0.0;
    HIP_OK(hipMemcpyAsync(&ch, out.p, sizeof(double), hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    return ch;
  }
};

}  // namespace lbmx

struct lbmx_mma {
  std::unique_ptr<lbmx::Mma> o;
};

// Scratch of lbmx_design_change_noalloc: the per-block partial maxima of the change reduction
// (mma_blocks() launches at most kNoAllocPartials blocks). Each device holds its own copy for
// the life of the process; its address on the current device comes from hipGetSymbolAddress
// (the array's name is a host-side stand-in, never a device address).
static constexpr int kNoAllocPartials = 2048;
static __device__ __align__(256) double scratch[kNoAllocPartials];

namespace {
std::mutex g_scratch_mu;
std::vector<double*> g_scratch_ptr;  // per device, filled on the first call there

double* scratch_on_current_device() {
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if ((size_t)dev >= g_scratch_ptr.size()) g_scratch_ptr.resize((size_t)dev + 1, nullptr);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      throw lbmx::Error{LBMX_ERR_DEVICE, std::string("hipGetSymbolAddress of the scratch array failed: ") +
                                            hipGetErrorString(e)};
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  return g_scratch_ptr[dev];
}
}  // namespace

using lbmx::Error;
using lbmx::guarded;

#define CHECK_MMA(h)                                    \
  if (!(h) || !(h)->o) {                                \
    lbmx::g_last_error = "null MMA handle";             \
    return LBMX_ERR_ARG;                                \
  }

extern "C" {

lbmx_status lbmx_mma_create(long long n, int m, lbmx_mma** out) {
  if (!out) {
    lbmx::g_last_error = "null argument";
    return LBMX_ERR_ARG;
  }
  return guarded([&] {
    auto h = std::make_unique<lbmx_mma>();
    h->o = std::make_unique<lbmx::Mma>(n, m);
    *out = h.release();
  });
}

lbmx_status lbmx_mma_destroy(lbmx_mma* h) {
  delete h;
  return LBMX_OK;
}

lbmx_status lbmx_mma_set_robust_constants(lbmx_mma* h, const double* a) {
  CHECK_MMA(h);
  if (!a) { lbmx::g_last_error = "null argument"; return LBMX_ERR_ARG; }
  for (int j = 0; j < h->o->m; ++j) h->o->a[j] = a[j];
  return LBMX_OK;
}

lbmx_status lbmx_mma_set_asymptotes(lbmx_mma* h, double init, double decrease, double increase) {
  CHECK_MMA(h);
  h->o->asyminit = init;
  h->o->asymdec = decrease;
  h->o->asyminc = increase;
  return LBMX_OK;
}

lbmx_status lbmx_mma_set_options(lbmx_mma* h, int constraint_modification, int robust_asymptotes_type) {
  CHECK_MMA(h);
  if (robust_asymptotes_type != 0 && robust_asymptotes_type != 1) {
    lbmx::g_last_error = "robust asymptotes type must be 0 or 1";
    return LBMX_ERR_ARG;
  }
  h->o->con_mod = constraint_modification != 0;
  h->o->asym_type = robust_asymptotes_type;
  return LBMX_OK;
}

lbmx_status lbmx_mma_update(lbmx_mma* h, double* x, const double* dfdx, const double* gx, const double* const* dgdx,
                            double movlim) {
  CHECK_MMA(h);
  if (!x || !dfdx || !gx || !dgdx) { lbmx::g_last_error = "null argument"; return LBMX_ERR_ARG; }
  for (int j = 0; j < h->o->m; ++j)
    if (!dgdx[j]) { lbmx::g_last_error = "null constraint sensitivity"; return LBMX_ERR_ARG; }
  return guarded([&] { h->o->update(x, dfdx, gx, dgdx, movlim, false); });
}

lbmx_status lbmx_mma_update_device(lbmx_mma* h, double* x, const double* dfdx, const double* gx,
                                   const double* const* dgdx, double movlim) {
  CHECK_MMA(h);
  if (!x || !dfdx || !gx || !dgdx) { lbmx::g_last_error = "null argument"; return LBMX_ERR_ARG; }
  for (int j = 0; j < h->o->m; ++j)
    if (!dgdx[j]) { lbmx::g_last_error = "null constraint sensitivity"; return LBMX_ERR_ARG; }
  return guarded([&] { h->o->update(x, dfdx, gx, dgdx, movlim, true); });
}

lbmx_status lbmx_mma_design_change(lbmx_mma* h, const double* xnew, double* ch) {
  CHECK_MMA(h);
  if (!ch) { lbmx::g_last_error = "null argument"; return LBMX_ERR_ARG; }
  return guarded([&] { *ch = h->o->design_change(xnew, false); });
}

lbmx_status lbmx_mma_design_change_device(lbmx_mma* h, const double* xnew, double* ch) {
  CHECK_MMA(h);
  if (!ch) { lbmx::g_last_error = "null argument"; return LBMX_ERR_ARG; }
  return guarded([&] { *ch = h->o->design_change(xnew, true); });
}

lbmx_status lbmx_design_change_noalloc(const double* xnew, const double* xold, long long n, double* ch,
                                       void* hip_stream) {
  if (!xnew || !xold || !ch) { lbmx::g_last_error = "null argument"; return LBMX_ERR_ARG; }
  if (n < 1 || n > LBMX_NOALLOC_MAX_N) {
    lbmx::g_last_error = "design length " + std::to_string(n) + " outside 1.." + std::to_string(LBMX_NOALLOC_MAX_N);
    return LBMX_ERR_ARG;
  }
  return guarded([&] {
    static_assert(kNoAllocPartials >= 2048, "the scratch must hold mma_blocks() partials");
    if (lbmx::mma_blocks(n) > kNoAllocPartials) throw Error{LBMX_ERR_ARG, "too many reduction blocks"};
    double* part = scratch_on_current_device();
    HIP_OK(lbmx::launch_mma_change(xnew, xold, n, part, ch, static_cast<hipStream_t>(hip_stream)));
  });
}

lbmx_status lbmx_mma_get_state(lbmx_mma* h, double* L, double* U, double* lam, int* newton_iters, double* ms) {
  CHECK_MMA(h);
  return guarded([&] {
    lbmx::Mma& o = *h->o;
    if (L) HIP_OK(hipMemcpy(L, o.L.p, (size_t)o.n * 8, hipMemcpyDeviceToHost));
    if (U) HIP_OK(hipMemcpy(U, o.U.p, (size_t)o.n * 8, hipMemcpyDeviceToHost));
    if (lam)
      for (int j = 0; j < o.m; ++j) lam[j] = o.lam[j];
    if (newton_iters) *newton_iters = o.newton_iters;
    if (ms) *ms = o.last_ms;
  });
}

}  // extern "C"
