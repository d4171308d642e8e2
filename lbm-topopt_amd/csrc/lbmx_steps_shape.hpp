// Shape of a launch that takes tiles of a 2D field through several steps (lbmx_steps.hpp): the
// steps K and the tile's rows H, by what such a workgroup takes and by how many there are. No
// device code: the functions are constant expressions, which the kernels use too.
#pragma once
#include "lbmx.h"
#include "lbmx_common.h"

namespace lbmx {

// dynamic LDS of a launch: boundary pieces, their K time factors, then the field(s)
constexpr size_t steps_pieces_bytes(int nbc, int K) {
  return ((size_t)nbc * (sizeof(DevBC) + (size_t)K * sizeof(double)) + 15) & ~(size_t)15;
}
constexpr int steps_cells(int K, int H) { return (kTileX + 2 * (K - 1)) * (H + 2 * (K - 1)); }
constexpr size_t steps_field_bytes(int K, int H, int Q, int elem) {
  return (((size_t)steps_cells(K, H) * Q * elem + 15) & ~(size_t)15) * (K > 2 ? 2 : 1);
}
// waves of a workgroup: the region's rows, and the columns beside the 64
constexpr int steps_waves(int K, int H) {
  const int rows = H + 2 * (K - 1), side = 2 * (K - 1) * rows;
  return rows + (side + kTileX - 1) / kTileX;
}
// Most waves of a workgroup. The FP64 reverse steps need more than the 128 registers that a
// workgroup of 16 waves leaves each lane (they spill up to 200 of them, and at 1024 x 512 a
// reverse step takes 30 us instead of the single-step sweep's 27); with 12 waves they have 168
// and it takes 21.
constexpr int steps_max_waves(int dir, bool fp64) { return dir == 1 && fp64 ? 12 : 16; }

struct StepsShape {
  int K, H;  // K = 1: the single-step sweeps
};

// dir: 0 forward, 1 reverse; nodes, blocks(H): of all fields that a launch covers; cus: CUs of the
// device (256, or an eighth of them where it is partitioned).
//
// A workgroup of this kind fills a CU, so what counts first is whether all of them run at once
// (at most one per CU). Then a launch's time hardly depends on the tile and more steps per launch
// are always better: the deepest K that the waves and the LDS allow with the fewest rows that
// still fit one round. Single-step sweeps and these, us per step (reverse incl. its share of a
// gradient pass): D2Q9 FP64 forward 256x128 7.6 and 4.1 (4 steps, 2 rows), 512x256 8.8 and 4.9
// (4, 8); thermal FP64 384x192 9.7 and 6.1 (3, 5); D2Q9 FP32 reverse 256x128 16.9 and 12.2.
//
// Fields of several rounds are bound by memory or arithmetic; every step of a launch saves one
// read and one write of the field and pays for the tile's ring, most where the tile is low. So
// the tile takes all rows that fit, and K is the best of those measured (at 2048x1024, forward
// us per step, single step / K = 2 / 3 / 4): D2Q9 FP64 58.9 / 42.8 / 39.1 / 39.4, thermal FP64 (3
// steps leave only 6 rows in the LDS) 91.7 / 62.3 / 64.7, D2Q9 FP32 33.7 / 29.2 / 28.7 / 28.5; in
// reverse, per step of a gradient pass, D2Q9 FP64 175 / 161 / 157, thermal FP64 260 / 235 / 232.
// The single-step sweeps stay where the arithmetic of the rings costs more than the saved
// passes: the 16-bit forward sweeps, which compute two nodes per lane (D2Q9 1024x512, in a gradient
// pass 8.4 and 9.5, 1536x512 12.2 and 13.9), the cascaded FP32 forward sweep above 2^21 nodes
// (1024x512 14.4 and 12.4, 2048x2048 66.3 and 65.5, a batch of 5.9e6 nodes 99 and 115), and the
// thermal FP64 reverse sweep with Brinkman's term, which spills (640x300 21.4 and 23.0).
//
// The cascaded reverse sweep stays with one step per launch everywhere: it has the most
// arithmetic of all (FP64 at 1024x512 34.9 and 36.8), and its long polynomials, left to the
// compiler's fusing, do not come out with the same bits in both kernels.
template <class Blocks>
inline StepsShape steps_shape(const lbmx_desc& d, int dir, int nbc, long long nodes, int cus, Blocks&& blocks) {
  constexpr size_t kLds = 160 * 1024;
  const bool fp64 = d.precision == LBMX_FP64, fp32 = d.precision == LBMX_FP32;
  const bool thermal = d.lattice == LBMX_D2Q9_D2Q5, cascaded = d.collision == LBMX_CASCADED;
  if (dir == 1 && cascaded) return {1, 1};
  const int elem = fp64 ? 8 : (fp32 || dir == 1 ? 4 : 2);
  auto fits = [&](int K, int H) {
    return steps_waves(K, H) <= steps_max_waves(dir, fp64) &&
           steps_pieces_bytes(nbc, K) + steps_field_bytes(K, H, thermal ? 14 : 9, elem) <= kLds;
  };
  for (int K = kMaxSteps; K > 1; --K)
    for (int H = 2; fits(K, H); ++H)
      if (blocks(H) <= cus) return {K, H};
  if (dir == 0 && !fp64 && !fp32) return {1, 1};
  if (dir == 0 && fp32 && cascaded && nodes > (1ll << 21)) return {1, 1};
  if (dir == 1 && fp64 && thermal && d.design == LBMX_DESIGN_BRINKMAN) return {1, 1};
  const int K = cascaded || (dir == 0 && fp64 && thermal) ? 2 : 3;
  int H = 2;
  while (fits(K, H + 1)) ++H;
  return {K, H};
}

}  // namespace lbmx
