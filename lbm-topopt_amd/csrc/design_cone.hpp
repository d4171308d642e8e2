// Device code of the cone filter, shared by the kernel of any radius (design_kernels.hip) and
// the kernels of one radius each (design_cone_*.hip).
//
// The cone filter sums its taps in ascending (dz, dy, dx) order with separately rounded
// multiplies and adds. That is the order in which a compressed-row MatMult visits the columns
// of a row, and the order in which MatMultTranspose accumulates into an entry, so the results
// equal a plain row loop (and a scatter-form transpose) bit for bit.
#pragma once
#include <hip/hip_runtime.h>

#include "design_cone_shape.hpp"
#include "lbmx_device.hpp"
#include "lbmx_launch.h"

namespace lbmx {

namespace {

__device__ inline bool in_box(int x, int y, int z, const int* b) { return lbmx::in_box(b, x, y, z); }

__device__ __forceinline__ size_t node(const ConeArgs& a, int x, int y, int z) {
  return ((size_t)z * a.ny + y) * a.nx + x;
}

// the input field at an in-grid node
__device__ __forceinline__ double cone_input(const ConeArgs& a, int x, int y, int z) {
  if (a.design) {
    const int* b = a.dbox;
    if (in_box(x, y, z, b)) {
      const int nxd = b[1] - b[0] + 1, nyd = b[3] - b[2] + 1;
      return a.design[((size_t)(z - b[4]) * nyd + (y - b[2])) * nxd + (x - b[0])];
    }
    return a.background[node(a, x, y, z)];
  }
  return a.in[node(a, x, y, z)];
}

// the input as the cone reads it: 0 outside the grid and, transposed, outside the box (only
// rows inside the box carry cone weights); MAPPED: the input is the mapped design
template <bool MAPPED, bool TR>
__device__ __forceinline__ double cone_tile_value(const ConeArgs& a, int x, int y, int z) {
  if (x < 0 || x >= a.nx || y < 0 || y >= a.ny) return 0.0;
  if (TR && !in_box(x, y, z, a.box)) return 0.0;
  return MAPPED ? cone_input(a, x, y, z) : a.in[node(a, x, y, z)];
}

// tanh(x) = E / (E + 2) with E = exp(2|x|) - 1: 2|x| = n ln 2 + r in two parts, E on r from
// its Taylor series (degree 14, |r| <= ln(2)/2), scaled back as 2^n E_r + (2^n - 1), each step
// with its rounding error carried, and one correction of the quotient by its remainder. Less
// than one unit of the last place from the exact value (host transcription against 113-bit
// arithmetic over 1e8 arguments: 0.82 at most, near |x| = 0.174; rms 0.27 to 0.30, where correct
// rounding gives 0.29). The library's tanh takes about 250 FP64 instructions, which bound the
// projecting kernels of large grids; this one takes about 60.
__device__ __forceinline__ double tanh64(double x) {
#pragma clang fp contract(off)
  const double ax = __builtin_fabs(x);
  const double y = 2.0 * ax < 40.0 ? 2.0 * ax : 40.0;  // tanh(20) rounds to 1
  const double n = __builtin_rint(y * 1.4426950408889634);
  constexpr double ln2_hi = 0x1.62e42fefa0000p-1, ln2_lo = 0x1.cf79abc9e3b39p-40;
  const double r0 = __builtin_fma(-n, ln2_hi, y);  // exact
  const double c0 = n * ln2_lo;
  const double r = r0 - c0;
  const double rl = (r0 - r) - c0;
  double q = 1.0 / 87178291200.0;
  q = __builtin_fma(q, r, 1.0 / 6227020800.0);
  q = __builtin_fma(q, r, 1.0 / 479001600.0);
  q = __builtin_fma(q, r, 1.0 / 39916800.0);
  q = __builtin_fma(q, r, 1.0 / 3628800.0);
  q = __builtin_fma(q, r, 1.0 / 362880.0);
  q = __builtin_fma(q, r, 1.0 / 40320.0);
  q = __builtin_fma(q, r, 1.0 / 5040.0);
  q = __builtin_fma(q, r, 1.0 / 720.0);
  q = __builtin_fma(q, r, 1.0 / 120.0);
  q = __builtin_fma(q, r, 1.0 / 24.0);
  q = __builtin_fma(q, r, 1.0 / 6.0);
  const double c = r * r * __builtin_fma(r, q, 0.5) + __builtin_fma(rl, r, rl);
  const double s = r + c, lo = c - (s - r);
  const double two = __builtin_ldexp(1.0, (int)n);
  const double a = two - 1.0, b = two * s;
  const double h = a + b, l = __builtin_fma(two, lo, b - (h - a));
  const double d = h + 2.0, bb = d - h;
  const double dl = ((h - (d - bb)) + (2.0 - bb)) + l;
  double rc = __builtin_amdgcn_rcp(d);
  rc = __builtin_fma(rc, __builtin_fma(-d, rc, 1.0), rc);
  rc = __builtin_fma(rc, __builtin_fma(-d, rc, 1.0), rc);
  double t = h * rc;
  t = __builtin_fma(__builtin_fma(-t, d, h) + (l - t * dl), rc, t);
  return __builtin_copysign(ax != ax ? ax : t, x);
}

// threshold of node i: the stage constant, or a per-node value with its own tanh terms
__device__ inline void node_eta(const ProjectArgs& p, size_t i, double& eta, double& tb, double& tsum) {
#pragma clang fp contract(off)
  eta = p.eta;
  tb = p.tb;
  tsum = p.tsum;
  if (p.etaf) {
    eta = p.etaf[i];
    tb = tanh64(p.beta * eta);
    tsum = tb + tanh64(p.beta * (1.0 - eta));
  }
}

__device__ __forceinline__ double projected(const ProjectArgs& p, size_t i, double v) {
#pragma clang fp contract(off)
  double eta, tb, tsum;
  node_eta(p, i, eta, tb, tsum);
  return (tb + tanh64(p.beta * (v - eta))) / tsum;
}

// the sensitivity s of a stage's output at node i, taken through its projection (inside the
// box) and divided by its denominators
__device__ __forceinline__ double scaled(const ProjectArgs& p, bool mine, size_t i, double s, const double* x,
                                         const double* den) {
#pragma clang fp contract(off)
  if (p.on && mine) {
    double eta, tb, tsum;
    node_eta(p, i, eta, tb, tsum);
    const double t = tanh64(p.beta * (x[i] - eta));
    s = s * (((1.0 - t * t) * p.beta) / tsum);
  }
  return s / den[i];
}

// What an output needs besides its sum: forward, its denominator (1 where there is none), or
// its own input outside the box.
__device__ __forceinline__ double cone_second(const ConeArgs& a, int x, int y, int z) {
  if (!in_box(x, y, z, a.box)) return cone_input(a, x, y, z);
  return a.den ? a.den[node(a, x, y, z)] : 1.0;
}

// What follows the sum `acc` of an output: forward, `v` is the filtered value and `p` the
// projected one (second: cone_second); transposed, the scaling for the stage before.
__device__ __forceinline__ void cone_finish(const ConeArgs& a, int x, int y, int z, double acc, double second, double& v,
                                            double& p) {
#pragma clang fp contract(off)
  const size_t i = node(a, x, y, z);
  const bool mine = in_box(x, y, z, a.box);
  if (a.transposed) {
    v = a.scale_den ? scaled(a.proj, mine, i, acc, a.scale_x, a.scale_den) : acc;
  } else {
    v = mine ? (a.den ? acc / second : acc) : second;
    p = v;
    if (a.proj.on && mine) p = projected(a.proj, i, v);
  }
}

// Stores of one output, or of the outputs at x and x + 1 at once.
using Double2 = double __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void cone_store(const ConeArgs& a, int x, int y, int z, double v, double p) {
  const size_t i = node(a, x, y, z);
  if (a.transposed && a.design_out) {
    const int* b = a.dbox;
    if (in_box(x, y, z, b)) {
      const int nxd = b[1] - b[0] + 1, nyd = b[3] - b[2] + 1;
      a.design_out[((size_t)(z - b[4]) * nyd + (y - b[2])) * nxd + (x - b[0])] = v;
    }
    return;
  }
  a.out[i] = v;
  if (a.transposed) return;
  if (a.proj.on) a.proj_out[i] = p;
  if (a.copy_out) a.copy_out[i] = p;
}
__device__ __forceinline__ void cone_store2(const ConeArgs& a, int x, int y, int z, const double (&v)[2],
                                            const double (&p)[2]) {
  const size_t i = node(a, x, y, z);
  auto put = [](double* to, const double(&q)[2]) { *reinterpret_cast<Double2*>(to) = Double2{q[0], q[1]}; };
  if (a.transposed && a.design_out) {
    const int* b = a.dbox;
    const int nxd = b[1] - b[0] + 1, nyd = b[3] - b[2] + 1;
    if (in_box(x, y, z, b) && in_box(x + 1, y, z, b)) {
      put(a.design_out + ((size_t)(z - b[4]) * nyd + (y - b[2])) * nxd + (x - b[0]), v);
    } else {
      cone_store(a, x, y, z, v[0], p[0]);
      cone_store(a, x + 1, y, z, v[1], p[1]);
    }
    return;
  }
  put(a.out + i, v);
  if (a.transposed) return;
  if (a.proj.on) put(a.proj_out + i, p);
  if (a.copy_out) put(a.copy_out + i, p);
}

// ---- cone with the radius known to the compiler ----
// A lane sums 2 (x) by KY (y) by KZ (z) adjacent outputs in registers; a wave covers 128 x KY
// outputs of KZ slices, and kConeWaves waves are stacked along y. The input planes z0 - R ..
// z0 + KZ - 1 + R pass through LDS one after another. Each value a lane reads (a 16-byte pair
// of neighbours, conflict-free) serves every output of the lane within the radius, and the
// product of a value with a weight is shared by the outputs at mirrored offsets; which outputs
// those are is decided while compiling, so the inner code is multiplies and adds alone, with
// the weights (one per squared distance) in scalar registers. Every output still adds its taps
// in ascending (dz, dy, dx) order, since planes, rows and columns are visited ascending.
constexpr int kConeWaves = 4;
template <int R, int KY, int KZ>
struct ConeTile {
  static constexpr int TX = 128, TY = kConeWaves * KY;
  static constexpr int W = TX + 2 * R, H = TY + 2 * R;
};

using ConstDouble = const __attribute__((address_space(4))) double;

template <int R, int KY, int KZ, bool D3, bool TR>
__global__ __launch_bounds__(64 * kConeWaves, KZ > 1 && TR ? 3 : 4) void k_cone_fixed(ConeArgs a) {
#pragma clang fp contract(off)
  using Tile = ConeTile<R, KY, KZ>;
  constexpr int W = Tile::W, H = Tile::H;
  constexpr int RZ = D3 ? R : 0;
  __shared__ __align__(16) double tile[W * H];
  // transposed: the slice's own values, which identity rows (outputs outside the box) take in
  // place of their masked tile entry
  __shared__ __align__(16) double own[TR ? Tile::TX * Tile::TY : 1];
  const ConstDouble* w = (const ConstDouble*)a.wd2;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int x0 = blockIdx.x * Tile::TX, y0 = blockIdx.y * Tile::TY, z0 = blockIdx.z * KZ;
  const int x = x0 + 2 * lane, y = y0 + wave * KY;
  const int* bx = a.box;
  double acc[KZ][KY][2];
#pragma unroll
  for (int kz = 0; kz < KZ; ++kz)
#pragma unroll
    for (int k = 0; k < KY; ++k) acc[kz][k][0] = acc[kz][k][1] = 0.0;

  // A plane's values on their way to LDS, loaded before the plane ahead of it is summed. A
  // wave takes every kConeWaves-th row (its y tests and row addresses are the wave's, on the
  // scalar unit), each lane columns lane and lane + 64 of it; the 2 R columns past 128 of all
  // rows are shared out over the workgroup.
  constexpr int NR = (H + kConeWaves - 1) / kConeWaves, TAIL = 2 * R * H;
  constexpr int NT = (TAIL + 64 * kConeWaves - 1) / (64 * kConeWaves);
  double staged[NR][2], tail[NT];
  const int swave = __builtin_amdgcn_readfirstlane(wave);
  // (out-of-grid columns load an in-grid one and then count as 0)
  const int gx0 = x0 - R + lane, gx1 = gx0 + 64;
  const int cx0 = min(max(gx0, 0), a.nx - 1), cx1 = min(max(gx1, 0), a.nx - 1);
  auto at = [&](int gx, int gy, int zz) __attribute__((always_inline)) {
    const double* p;
    if (a.design) {
      const int* b = a.dbox;
      const int nxd = b[1] - b[0] + 1, nyd = b[3] - b[2] + 1;
      const double* d = a.design + (((long long)(zz - b[4]) * nyd + (gy - b[2])) * nxd + (gx - b[0]));
      p = in_box(gx, gy, zz, b) ? d : a.background + node(a, gx, gy, zz);
    } else {
      p = a.in + node(a, gx, gy, zz);
    }
    return *p;
  };
  auto load_plane = [&](int zz) __attribute__((always_inline)) {
    if (zz < 0 || zz >= a.nz) return;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int gy = y0 - R + swave + kConeWaves * i;
      staged[i][0] = staged[i][1] = 0.0;
      if (gy >= 0 && gy < a.ny && swave + kConeWaves * i < H) {
        staged[i][0] = at(cx0, gy, zz);
        staged[i][1] = at(cx1, gy, zz);
      }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int t = threadIdx.x + i * 64 * kConeWaves;
      const int gx = x0 - R + 128 + t % (2 * R), gy = y0 - R + t / (2 * R);
      tail[i] = 0.0;
      if (t < TAIL && gx >= 0 && gx < a.nx && gy >= 0 && gy < a.ny) tail[i] = at(gx, gy, zz);
    }
  };
  auto place_plane = [&](int zz) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int row = swave + kConeWaves * i, gy = y0 - R + row;
      if (row < H) {
        double v0 = gx0 >= 0 && gx0 < a.nx ? staged[i][0] : 0.0;
        double v1 = gx1 >= 0 && gx1 < a.nx ? staged[i][1] : 0.0;
        if constexpr (TR) {
          if (row >= R && row < R + Tile::TY) {
            double* o = own + (row - R) * Tile::TX - R;
            if (lane >= R) o[lane] = v0;
            o[lane + 64] = v1;
          }
          // only rows inside the box carry cone weights
          if (!in_box(gx0, gy, zz, bx)) v0 = 0.0;
          if (!in_box(gx1, gy, zz, bx)) v1 = 0.0;
        }
        tile[row * W + lane] = v0;
        tile[row * W + lane + 64] = v1;
      }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int t = threadIdx.x + i * 64 * kConeWaves, col = 128 + t % (2 * R), row = t / (2 * R);
      if (t < TAIL) {
        double v = tail[i];
        if constexpr (TR) {
          if (row >= R && row < R + Tile::TY && col - R < Tile::TX) own[(row - R) * Tile::TX + col - R] = v;
          if (!in_box(x0 - R + col, y0 - R + row, zz, bx)) v = 0.0;
        }
        tile[row * W + col] = v;
      }
    }
  };
  load_plane(z0 - RZ);
  static_for<0, KZ + 2 * RZ>([&](auto pc) __attribute__((always_inline)) {
#pragma clang fp contract(off)
    constexpr int pz = decltype(pc)::value;
    const int zz = z0 - RZ + pz;
    const bool in_grid = zz >= 0 && zz < a.nz;  // uniform over the workgroup
    if (in_grid) {
      if (pz > 0) __syncthreads();
      place_plane(zz);
      __syncthreads();
    }
    if (pz + 1 < KZ + 2 * RZ) load_plane(zz + 1);
    if (in_grid) {
      const double* base = tile + wave * KY * W + 2 * lane;
      static_for<0, KY + 2 * R>([&](auto rc) __attribute__((always_inline)) {
#pragma clang fp contract(off)
        constexpr int r = decltype(rc)::value;
        double v[2 * R + 2];
#pragma unroll
        for (int c = 0; c < R + 1; ++c) {
          const double2 d = *reinterpret_cast<const double2*>(base + r * W + 2 * c);
          v[2 * c] = d.x;
          v[2 * c + 1] = d.y;
        }
        // (all of it is decided while compiling, down to the multiplies and adds)
        static_for<0, 2 * R + 2>([&](auto cc) __attribute__((always_inline)) {
#pragma clang fp contract(off)
          constexpr int c = decltype(cc)::value;
#pragma unroll
          for (int o = 0; o < 2 * KY * KZ; ++o) {
            const int e = o % 2, k = o / 2 % KY, kz = o / (2 * KY);
            const int dz = pz - RZ - kz, dy = r - R - k, dx = c - R - e;
            const int d2 = dx * dx + dy * dy + dz * dz;
            if (d2 <= R * R) {
              double t = w[d2] * v[c];
              if (TR && d2 == 0) {
                // the diagonal entry: cone weight for a row in the box, 1 for an identity row
                const bool row_in = lbmx::in_box(bx, x + e, y + k, z0 + kz);
                t = bsel(row_in, t, own[(wave * KY + k) * Tile::TX + 2 * lane + e]);
              }
              acc[kz][k][e] = acc[kz][k][e] + t;
            }
          }
        });
        // one row's values live at a time: neither the next row's loads nor this row's sums move
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      });
    }
  });

  // A pair of outputs at a time, the rest moved down a pair after each: the sums stay in
  // registers while the code of what follows them (division, tanh) exists once. What the next
  // pair needs besides is loaded ahead.
  constexpr int NP = KY * KZ;
  const bool in0 = x < a.nx, in1 = x + 1 < a.nx;
  auto seconds = [&](int o, double(&d)[2]) __attribute__((always_inline)) {
    const int yo = y + o % KY, zo = z0 + o / KY;
    d[0] = d[1] = 1.0;
    if (TR || o >= NP || yo >= a.ny || zo >= a.nz) return;
    if (in0) d[0] = cone_second(a, x, yo, zo);
    if (in1) d[1] = cone_second(a, x + 1, yo, zo);
  };
  double den[2];
  seconds(0, den);
#pragma unroll 1
  for (int o = 0; o < NP; ++o) {
    double next[2];
    seconds(o + 1, next);
    const int yo = y + o % KY, zo = z0 + o / KY;
    if (yo < a.ny && zo < a.nz && in0) {
      double v[2] = {0.0, 0.0}, p[2] = {0.0, 0.0};
      cone_finish(a, x, yo, zo, acc[0][0][0], den[0], v[0], p[0]);
      if (in1) {
        cone_finish(a, x + 1, yo, zo, acc[0][0][1], den[1], v[1], p[1]);
        cone_store2(a, x, yo, zo, v, p);
      } else {
        cone_store(a, x, yo, zo, v[0], p[0]);
      }
    }
    den[0] = next[0];
    den[1] = next[1];
#pragma unroll
    for (int i = 1; i < NP; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) acc[(i - 1) / KY][(i - 1) % KY][e] = acc[i / KY][i % KY][e];
  }
}

template <int R, int KY, int KZ, bool D3>
hipError_t cone_fixed(const ConeArgs& a, hipStream_t s) {
  using Tile = ConeTile<R, KY, KZ>;
  dim3 grid((a.nx + Tile::TX - 1) / Tile::TX, (a.ny + Tile::TY - 1) / Tile::TY, (a.nz + KZ - 1) / KZ);
  if (a.transposed)
    hipLaunchKernelGGL((k_cone_fixed<R, KY, KZ, D3, true>), grid, dim3(64 * kConeWaves), 0, s, a);
  else
    hipLaunchKernelGGL((k_cone_fixed<R, KY, KZ, D3, false>), grid, dim3(64 * kConeWaves), 0, s, a);
  return hipGetLastError();
}

// the 2D kernel of radius a.R, searched from R0 to R1
template <int R0, int R1>
hipError_t cone_2d(const ConeArgs& a, hipStream_t s) {
  static_assert(ConeTile<R0, 2, 1>::TY == kConeFixedTY2D, "cone_fixed_radius counts workgroups of this height");
  if constexpr (R0 <= R1) {
    if (a.R == R0) return cone_fixed<R0, 2, 1, false>(a, s);
    return cone_2d<R0 + 1, R1>(a, s);
  }
  return hipErrorInvalidValue;
}
template <int R0, int R1>
hipError_t cone_3d(const ConeArgs& a, hipStream_t s) {
  if constexpr (R0 <= R1) {
    if (a.R == R0) return cone_fixed<R0, 4, 4, true>(a, s);
    return cone_3d<R0 + 1, R1>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace
}  // namespace lbmx
