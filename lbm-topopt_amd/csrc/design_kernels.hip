// Design pipeline kernels: design-box mapping, cone density filter (forward and transposed),
// tanh projection and its sensitivity scaling. All fields are FP64 in natural order
// (z*ny + y)*nx + x on the full grid.
#include <hip/hip_runtime.h>

#include "design_cone.hpp"
#include "design_cone_shape.hpp"
#include "lbmx_launch.h"

namespace lbmx {

namespace {

constexpr int kMaxR = 16;

// LDS bytes of one workgroup: the input region of one plane and that plane's cone weights
inline size_t cone_lds_bytes(int R) {
  const size_t W = kConeTX + 2 * R, H = kConeTY + 2 * R, S = 2 * R + 1;
  return (W * H + S * S) * sizeof(double);
}

// One workgroup: a 64 x 16 tile of outputs in one z plane. For each in-grid plane z + dz the
// (64 + 2R) x (16 + 2R) input region and the plane's (2R + 1)^2 weights are staged in LDS;
// then for each tap row (dy) and tap (dx) one weight is read and applied to the thread's four
// outputs (four independent sums, each in ascending (dz, dy, dx) order). MAPPED: the input is the
// mapped design (a.design); a test of that per staged value costs 2 to 4% of a call (101x47x53,
// radius 4, transposed: 87 us with it, 82 us without).
template <bool MAPPED, bool TR>
__global__ __launch_bounds__(256) void k_cone(ConeArgs a) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  const int R = a.R;
  const int W = kConeTX + 2 * R;
  const int H = kConeTY + 2 * R;
  const int S = 2 * R + 1;
  double* tile = lds;
  double* wl = lds + W * H;
  const int tx = threadIdx.x % kConeTX;
  const int ty = threadIdx.x / kConeTX;
  const int x0 = blockIdx.x * kConeTX;
  const int y0 = blockIdx.y * kConeTY;
  const int z = blockIdx.z;
  const int x = x0 + tx;

  double acc[kConeKY];
  double own[kConeKY];  // transposed: this output's own input (identity rows outside the box)
  bool mine[kConeKY];   // output inside the filter box
#pragma unroll
  for (int k = 0; k < kConeKY; ++k) {
    const int y = y0 + ty + kConeWY * k;
    acc[k] = 0.0;
    const bool valid = x < a.nx && y < a.ny;
    mine[k] = valid && in_box(x, y, z, a.box);
    own[k] = TR && valid ? a.in[node(a, x, y, z)] : 0.0;
  }

  for (int dz = -R; dz <= R; ++dz) {
    const int zz = z + dz;
    if (zz < 0 || zz >= a.nz) continue;  // uniform over the workgroup
    __syncthreads();
    for (int idx = threadIdx.x; idx < W * H; idx += blockDim.x)
      tile[idx] = cone_tile_value<MAPPED, TR>(a, x0 - R + idx % W, y0 - R + idx / W, zz);
    const double* wz = a.wt + (size_t)(dz + R) * S * S;
    for (int idx = threadIdx.x; idx < S * S; idx += blockDim.x) wl[idx] = wz[idx];
    __syncthreads();
    const int* rxz = a.rx + (dz + R) * S;
    for (int dy = -R; dy <= R; ++dy) {
      const int r = rxz[dy + R];
      if (r < 0) continue;
      const double* w = wl + (dy + R) * S + R;  // w[dx], dx in [-R, R]
      const double* row = tile + (ty + dy + R) * W + tx + R;
      constexpr int kStep = kConeWY;           // rows between this thread's outputs
      const double* r1 = row + kStep * W;
      const double* r2 = row + 2 * kStep * W;
      const double* r3 = row + 3 * kStep * W;
      double s0 = acc[0], s1 = acc[1], s2 = acc[2], s3 = acc[3];
      // taps [lo, hi) of this row, two at a time with all loads issued first
      auto taps = [&](int lo, int hi) {
        int dx = lo;
        for (; dx + 1 < hi; dx += 2) {
          const double wa = w[dx], wb = w[dx + 1];
          const double a0 = row[dx], b0 = row[dx + 1], a1 = r1[dx], b1 = r1[dx + 1];
          const double a2 = r2[dx], b2 = r2[dx + 1], a3 = r3[dx], b3 = r3[dx + 1];
          s0 = s0 + wa * a0;
          s1 = s1 + wa * a1;
          s2 = s2 + wa * a2;
          s3 = s3 + wa * a3;
          s0 = s0 + wb * b0;
          s1 = s1 + wb * b1;
          s2 = s2 + wb * b2;
          s3 = s3 + wb * b3;
        }
        if (dx < hi) {
          const double wa = w[dx];
          const double a0 = row[dx], a1 = r1[dx], a2 = r2[dx], a3 = r3[dx];
          s0 = s0 + wa * a0;
          s1 = s1 + wa * a1;
          s2 = s2 + wa * a2;
          s3 = s3 + wa * a3;
        }
      };
      if (!(dz == 0 && dy == 0)) {
        taps(-r, r + 1);
      } else {
        taps(-r, 0);
        // the diagonal entry: cone weight for a row in the box, 1 for an identity row
        const double wv = w[0];
        if constexpr (TR) {
          s0 = s0 + (mine[0] ? wv : 1.0) * own[0];
          s1 = s1 + (mine[1] ? wv : 1.0) * own[1];
          s2 = s2 + (mine[2] ? wv : 1.0) * own[2];
          s3 = s3 + (mine[3] ? wv : 1.0) * own[3];
        } else {
          s0 = s0 + wv * row[0];
          s1 = s1 + wv * r1[0];
          s2 = s2 + wv * r2[0];
          s3 = s3 + wv * r3[0];
        }
        taps(1, r + 1);
      }
      acc[0] = s0;
      acc[1] = s1;
      acc[2] = s2;
      acc[3] = s3;
    }
  }

  // (the sums move down one by one, so that the code after them exists once)
#pragma unroll 1
  for (int k = 0; k < kConeKY; ++k) {
    const int y = y0 + ty + kConeWY * k;
    if (x < a.nx && y < a.ny) {
      double v = 0.0, p = 0.0;
      cone_finish(a, x, y, z, acc[0], TR ? 1.0 : cone_second(a, x, y, z), v, p);
      cone_store(a, x, y, z, v, p);
    }
    for (int i = 1; i < kConeKY; ++i) acc[i - 1] = acc[i];
  }
}

struct Grid3 {
  int nx, ny, nz;
  __device__ bool locate(long long i, int& x, int& y, int& z) const {
    if (i >= (long long)nx * ny * nz) return false;
    x = (int)(i % nx);
    const long long r = i / nx;
    y = (int)(r % ny);
    z = (int)(r / ny);
    return true;
  }
};

struct Box6 {
  int b[6];
};

__global__ __launch_bounds__(256) void k_sens_scale(double* out, const double* sens, const double* xin,
                                                     const double* den, Grid3 g, Box6 bx, ProjectArgs p) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  int x, y, z;
  if (!g.locate(i, x, y, z)) return;
  out[i] = scaled(p, in_box(x, y, z, bx.b), (size_t)i, sens[i], xin, den);
}

__global__ __launch_bounds__(256) void k_convert_f64_f32(float* out, const double* in, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (float)in[i];
}

inline unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

inline Box6 box6(const int b[6]) {
  Box6 r;
  for (int k = 0; k < 6; ++k) r.b[k] = b[k];
  return r;
}

}  // namespace

hipError_t launch_cone(const ConeArgs& a, hipStream_t s) {
  if (a.R < 1 || a.R > kMaxR || a.nx < 1 || a.ny < 1 || a.nz < 1) return hipErrorInvalidValue;
  if (cone_fixed_radius(a.nx, a.ny, a.nz, a.R, a.transposed != 0)) {
    if (a.nz > 1) return launch_cone_3d_small(a, s);
    return a.R <= 8 ? launch_cone_2d_small(a, s) : launch_cone_2d_large(a, s);
  }
  dim3 grid((a.nx + kConeTX - 1) / kConeTX, (a.ny + kConeTY - 1) / kConeTY, a.nz);
  const dim3 block(kConeTX * kConeWY);
  if (a.transposed) hipLaunchKernelGGL((k_cone<false, true>), grid, block, cone_lds_bytes(a.R), s, a);
  else if (a.design) hipLaunchKernelGGL((k_cone<true, false>), grid, block, cone_lds_bytes(a.R), s, a);
  else hipLaunchKernelGGL((k_cone<false, false>), grid, block, cone_lds_bytes(a.R), s, a);
  return hipGetLastError();
}

hipError_t launch_sens_scale(double* out, const double* sens, const double* x, const double* den, int nx, int ny,
                             int nz, const int box[6], const ProjectArgs& p, hipStream_t s) {
  const long long n = (long long)nx * ny * nz;
  hipLaunchKernelGGL(k_sens_scale, dim3(blocks_for(n)), dim3(256), 0, s, out, sens, x, den, Grid3{nx, ny, nz},
                     box6(box), p);
  return hipGetLastError();
}

hipError_t convert_f64_f32(float* out, const double* in, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_convert_f64_f32, dim3(blocks_for(n)), dim3(256), 0, s, out, in, n);
  return hipGetLastError();
}

}  // namespace lbmx
