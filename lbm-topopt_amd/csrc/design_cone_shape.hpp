// Which cone filter kernel a grid takes: the kernel of its radius (design_cone.hpp) or the one of
// any radius (design_kernels.hip). Both give the same bits.
#pragma once

namespace lbmx {

// ---- cone of any radius ----
constexpr int kConeTX = 64;   // outputs along x per workgroup (one wave wide)
constexpr int kConeWY = 4;    // waves per workgroup, stacked along y
constexpr int kConeKY = 4;    // outputs per thread along y (four named sums in k_cone)
constexpr int kConeTY = kConeWY * kConeKY;  // outputs along y per workgroup

// Radii up to these have a kernel of their own (2D: 2 x 2 outputs per lane, 3D: 2 x 4 x 4): those
// that filters of the usual widths have. In 3D the unrolled taps of radius 3 fill the
// instruction cache (32 x 123 taps per lane).
constexpr int kConeFixed2D = 12;
constexpr int kConeFixed3D = 3;
constexpr int kConeFixedTY2D = 8;  // outputs along y per workgroup of the 2D kernel
constexpr int kMaxGridY = 65535;   // most workgroups along y of a launch

// Whether the kernel of the radius runs. In 2D it does on every grid (0.74 to 0.97 of the other's
// time from 48x24 to 2049x1025, also on grids 30 and 70 wide). A 3D lane sums 32 outputs one plane
// after another, so a small grid leaves most CUs idle while the kernel of any radius has eight
// times the workgroups (radius 3 at 64^3: 74 and 59 us a call; at 128^3 84 and 121 us). Where
// the two meet, in workgroups of the latter, over 17 grids from 16^3 to 256x128x128: forward
// (plain and projecting) near 3500, 1500 and 1100 for radii 1, 2 and 3, transposed near 1600, 900
// and 700.
constexpr bool cone_fixed_radius(int nx, int ny, int nz, int R, bool transposed) {
  // (a 2D grid of more than 524280 rows has too many workgroups along y for the low tile)
  if (nz == 1) return R <= kConeFixed2D && (ny + kConeFixedTY2D - 1) / kConeFixedTY2D <= kMaxGridY;
  if (R > kConeFixed3D) return false;
  constexpr long long least[2][kConeFixed3D] = {{3500, 1500, 1100}, {1600, 900, 700}};
  const long long blocks = (long long)((nx + kConeTX - 1) / kConeTX) * ((ny + kConeTY - 1) / kConeTY) * nz;
  return blocks >= least[transposed ? 1 : 0][R - 1];
}

}  // namespace lbmx
