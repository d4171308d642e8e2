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
// Where a lane's node lies: offsets from the tile's first node, distance from the tile (0 inside)
// and LDS cell. One wave holds one row of the region, x0 .. x0 + 63; the ring's columns beside
// those 64 are packed into further waves, whose last lanes hold nothing.
struct StepsPlace {
  int dx, dy, ring, cell;
  bool row;   // the wave holds a row of the tile (not of its ring)
  bool side;  // the wave holds columns beside the 64
  bool held;
};
constexpr StepsPlace steps_place(int K, int H, int wave, int lane) {
  const int h = K - 1, rows = H + 2 * h, pitch = kTileX + 2 * h;
  StepsPlace p{lane, wave - h, 0, 0, wave >= h && wave < h + H, wave >= rows, true};
  if (p.side) {
    const int i = (wave - rows) * kTileX + lane, r = i / (2 * h), k = i - r * (2 * h);
    p.dx = k < h ? k - h : kTileX + k - h;
    p.dy = r - h;
    p.held = r < rows;
  }
  const int ox = p.dx < 0 ? -p.dx : (p.dx >= kTileX ? p.dx - kTileX + 1 : 0);
  const int oy = p.dy < 0 ? -p.dy : (p.dy >= H ? p.dy - H + 1 : 0);
  p.ring = ox > oy ? ox : oy;
  p.cell = (p.dy + h) * pitch + p.dx + h;
  return p;
}
// Most waves of a workgroup. The FP64 reverse steps need more than the 128 registers that a
// workgroup of 16 waves leaves each lane (they spill up to 200 of them, and at 1024 x 512 a
// reverse step takes 30 us instead of the single-step sweep's 27); with 12 waves they have 168
// and it takes 21.
constexpr int steps_max_waves(int dir, bool fp64) { return dir == 1 && fp64 ? 12 : 16; }

struct StepsShape {
  int K, H;  // K = 1: the single-step sweeps
};

// The fields that a launch covers: nodes, rows, and 64-node segments of rows.
struct StepsFields {
  long long nodes = 0, rows = 0, segments = 0;
  void add(int nx, int ny) {
    nodes += (long long)nx * ny;
    rows += ny;
    segments += (long long)((nx + kTileX - 1) / kTileX) * ny;
  }
};

// dir: 0 forward, 1 reverse; blocks(H): workgroups with tiles of H rows; cus: CUs of the device
// (256, or an eighth of them where it is partitioned).
//
// What counts first is whether all workgroups run at once, one per CU. Then a launch's time
// hardly depends on the tile and more steps per launch are always better: the deepest K that the
// waves and the LDS allow with the fewest rows that still fit one round. Single-step sweeps and
// these, us per step (reverse incl. its share of a gradient pass): D2Q9 FP64 forward 256x128 7.6
// and 4.1 (4 steps, 2 rows), 512x256 8.8 and 4.9 (4, 8); thermal FP64 384x192 9.7 and 6.1 (3, 5);
// D2Q9 FP32 reverse 256x128 16.9 and 12.2. From 24x12 to 640x320 no form took more than 0.89 of its
// single-step time.
//
// Fields of several rounds are bound by memory or arithmetic; every step of a launch saves one
// read and one write of the field and pays for the tile's ring, most where the tile is low. K and
// H are the best of those measured over 17 fields from 65x2400 to 2048x1024 (time over that of
// single steps at 2048x1024, forward runs and reverse passes, K/H):
//   D2Q9 FP64 forward 3/11 0.66 (2/13 0.73, 4/8 0.67), cascaded 0.75 (2/13 0.77; at 200x1600, two
//   rounds of 2/13, 0.95 and 0.81); thermal FP64 forward 2/13 0.69 (3/6 0.72); D2Q9 FP64 reverse 3/7 0.80 (2/9 0.86); D2Q9 FP32 reverse 3/11 0.80 (2/13 0.88),
//   16-bit 0.86, thermal FP32 0.81, 16-bit 0.92.
// All rows that fit are not always the best: 12 waves of the D2Q9 FP32 forward sweep leave room
// for a second workgroup on the CU, which runs while the first one waits at its barriers. 3/7
// takes 0.81 (3/11 0.86), cascaded 0.89 (2/13 0.97); at 200x1600 0.77 and 0.83 (0.93 and 0.89).
//
// Narrow fields waste lanes (65 nodes fill half of two segments) and most of their tiles hold
// boundary nodes, the longer path: `waste` is lanes per node times 1 + 0.26 of the tile columns
// at the domain's sides. Where it is high, fields of several rounds take fewer steps or one per
// launch. 3 steps and single steps, us per step: thermal FP64 reverse 65x16000 (waste 2.5) 158 and
// 122, 200x1600 (1.45) 36 and 34, where 2/9 takes 31 (so up to six columns; 512x300, eight, 15.7, 2/9
// 17.1); D2Q9 FP64 reverse 200x6000 58 and 49, 260x4000 (1.36) 0.87 of it; 16-bit reverse 128x8000
// (1.26) 1.02 of single steps; thermal FP32 forward 200x6000 3/11 1.06 of them, 2/9 0.90. Fields of
// few rounds still gain (D2Q9 FP32 reverse 64x4000 0.91) unless one column leaves much of the last
// round empty (64x4000: D2Q9 FP64 reverse 1.2, thermal and cascaded FP64 forward 1.17) or it is
// the thermal FP64 reverse sweep (64x3000 1.16).
// The single-step sweeps also stay where the arithmetic of the rings costs more than the saved
// passes: the 16-bit forward sweeps, which compute two nodes per lane (D2Q9 1024x512, in a gradient
// pass that keeps every state, wall time of one box, 8.4 and 9.5, 1536x512 12.2 and 13.9; a kernel
// trace of passes that recompute gives 9.4 for the former), the cascaded FP32 forward
// sweep above 2^20 nodes (a gradient pass that keeps every state: 330x3600 1.12 of single steps,
// 2048x1024 1.04, 1280x640 0.93), and the thermal FP64 reverse sweep with Brinkman's term, which
// spills (640x300 21.4 and 23.0).
//
// The cascaded reverse sweep stays with one step per launch everywhere: it has the most
// arithmetic of all (FP64 at 1024x512 34.9 and 36.8), and its long polynomials, left to the
// compiler's fusing, do not come out with the same bits in both kernels.
template <class Blocks>
inline StepsShape steps_shape(const lbmx_desc& d, int dir, int nbc, const StepsFields& f, int cus, Blocks&& blocks) {
  constexpr size_t kLds = 160 * 1024;
  constexpr StepsShape one{1, 1};
  const bool fp64 = d.precision == LBMX_FP64, fp32 = d.precision == LBMX_FP32;
  const bool thermal = d.lattice == LBMX_D2Q9_D2Q5, cascaded = d.collision == LBMX_CASCADED;
  if (dir == 1 && cascaded) return one;
  const int elem = fp64 ? 8 : (fp32 || dir == 1 ? 4 : 2);
  auto fits = [&](int K, int H) {
    return steps_waves(K, H) <= steps_max_waves(dir, fp64) &&
           steps_pieces_bytes(nbc, K) + steps_field_bytes(K, H, thermal ? 14 : 9, elem) <= kLds;
  };
  for (int K = kMaxSteps; K > 1; --K)
    for (int H = 2; fits(K, H); ++H)
      if (blocks(H) <= cus) return {K, H};

  if (dir == 0 && !fp64 && !fp32) return one;
  if (dir == 0 && fp32 && cascaded && f.nodes > (1ll << 20)) return one;
  if (dir == 1 && fp64 && thermal && d.design == LBMX_DESIGN_BRINKMAN) return one;
  const double columns = (double)f.segments / f.rows;
  const double waste = (1.0 + 0.52 / columns) * (double)f.segments * kTileX / f.nodes;
  auto shape = [&](int K, int most) {  // the tile takes the rows that fit, at most `most`
    int H = 2;
    while (H < most && fits(K, H + 1)) ++H;
    return StepsShape{K, H};
  };
  auto rounds = [&](StepsShape s) { return (blocks(s.H) + cus - 1) / cus; };
  // FP64 fields of one column whose two or three rounds would be less than four fifths full
  auto thin = [&](StepsShape s) {
    return fp64 && columns < 2.0 && rounds(s) > 1 && rounds(s) <= 3 && 5 * blocks(s.H) < 4 * rounds(s) * cus;
  };
  constexpr int kAll = 64;
  StepsShape s = shape(3, kAll);
  if (dir == 0) {
    const StepsShape two = shape(2, kAll);
    if (fp64 && (thermal || (cascaded && rounds(two) <= 2))) return thin(two) ? one : two;
    if (fp64) return s;
    if (thermal) return waste <= 1.2 || rounds(s) <= 2 ? s : waste > 2.0 ? one : shape(2, 9);
    s = shape(3, 7);
    return waste > 1.4 && rounds(s) > 8 ? one : s;
  }
  if (fp64 && thermal && columns <= 6.0) s = shape(2, kAll);
  const int few = fp64 && thermal && columns < 2.0 ? 1 : fp64 && waste < 2.2 ? 4 : 2;
  return thin(s) || (waste > (fp64 || fp32 ? 1.4 : 1.25) && rounds(s) > few) ? one : s;
}

}  // namespace lbmx
