// Shapes of the launches that take several steps (lbmx_steps_shape.hpp): every one stays within a
// workgroup's waves and LDS, and the rule. Prints "RESULT OK" at the end.
#include <cstdio>
#include <vector>

#include "lbmx_steps_shape.hpp"

using namespace lbmx;

static int fails = 0;

struct Form {
  int lattice, collision, design, precision;
};

static StepsShape shape(const Form& f, int dir, int nx, int ny, int nbc = 7, int cus = 256) {
  lbmx_desc d{};
  d.lattice = f.lattice;
  d.collision = f.collision;
  d.design = f.design;
  d.precision = f.precision;
  StepsFields fields;
  fields.add(nx, ny);
  return steps_shape(d, dir, nbc, fields, cus, [&](int H) {
    return (long long)((nx + kTileX - 1) / kTileX) * ((ny + H - 1) / H);
  });
}

static void expect(const Form& f, int dir, int nx, int ny, int K, int H, int cus = 256) {
  const StepsShape s = shape(f, dir, nx, ny, 7, cus);
  if (s.K == K && (s.H == H || K == 1)) return;
  std::printf("lattice %d collision %d design %d precision %d dir %d %d x %d on %d CUs: %d steps of %d rows, not %d of %d\n",
              f.lattice, f.collision, f.design, f.precision, dir, nx, ny, cus, s.K, s.H, K, H);
  ++fails;
}

// Every LDS access of a launch of K steps on tiles of H rows lies inside its region, and every
// cell of the region has one lane.
static void check_places(int K, int H) {
  const int h = K - 1, rows = H + 2 * h, pitch = kTileX + 2 * h, cells = steps_cells(K, H);
  std::vector<int> held(cells, 0), ring(cells, -1);
  auto fail = [&](const char* what, int wave, int lane) {
    std::printf("K %d H %d wave %d lane %d: %s\n", K, H, wave, lane, what);
    ++fails;
  };
  for (int wave = 0; wave < steps_waves(K, H); ++wave)
    for (int lane = 0; lane < kTileX; ++lane) {
      const StepsPlace p = steps_place(K, H, wave, lane);
      if (!p.held) {
        if (!p.side || wave + 1 != steps_waves(K, H)) fail("holds nothing", wave, lane);
        continue;
      }
      if (p.cell < 0 || p.cell >= cells) {
        fail("cell out of range", wave, lane);
        continue;
      }
      if (p.ring < 0 || p.ring > h) fail("beyond the ring", wave, lane);
      if (p.row && (p.side || p.dx != lane || p.dy < 0 || p.dy >= H)) fail("not a row of the tile", wave, lane);
      ++held[p.cell];
      ring[p.cell] = p.ring;
      // step j is taken by ring <= K - j; it reads the cells around its own from step j - 1, and
      // writes reflections around it for step j + 1 where ring <= K - j - 1
      if (p.ring < h)
        for (int y = p.dy - 1; y <= p.dy + 1; ++y)
          for (int x = p.dx - 1; x <= p.dx + 1; ++x) {
            if (x < -h || x >= kTileX + h || y < -h || y >= H + h) fail("neighbour outside the region", wave, lane);
            const int at = p.cell + (x - p.dx) + (y - p.dy) * pitch;
            if (at != (y + h) * pitch + x + h || at < 0 || at >= cells) fail("neighbour's cell", wave, lane);
          }
    }
  for (int c = 0; c < cells; ++c)
    if (held[c] != 1) fail("a cell without one lane", c / pitch, c % pitch);
  for (int y = 0; y < rows; ++y)  // a node of ring r finds its neighbours' values of the step before
    for (int x = 0; x < pitch; ++x)
      for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx)
          if (ring[y * pitch + x] < h && ring[(y + dy) * pitch + x + dx] > ring[y * pitch + x] + 1)
            fail("a neighbour two rings out", y, x);
  for (int nbc = 0; nbc <= kMaxBC; ++nbc) {
    const size_t bytes = steps_pieces_bytes(nbc, K);
    if (bytes % 16 || (size_t)nbc * sizeof(DevBC) % sizeof(double) ||
        (size_t)nbc * sizeof(DevBC) + (size_t)K * nbc * sizeof(double) > bytes)
      fail("pieces and time factors", nbc, 0);
  }
  for (int Q : {9, 14})
    for (int elem : {2, 4, 8}) {
      const size_t field = ((size_t)cells * Q * elem + 15) & ~(size_t)15;  // the second field's offset
      if (field % elem || (K > 2 ? 2 : 1) * field > steps_field_bytes(K, H, Q, elem)) fail("fields", Q, elem);
    }
}

int main() {
  for (int K = 2; K <= kMaxSteps; ++K)
    for (int H = 2; steps_waves(K, H) <= 16; ++H) check_places(K, H);
  std::vector<Form> forms;
  for (int lat : {LBMX_D2Q9, LBMX_D2Q9_D2Q5})
    for (int coll : {LBMX_BGK, LBMX_MRT, LBMX_CASCADED})
      for (int des : {LBMX_DESIGN_NONE, LBMX_DESIGN_PBB, LBMX_DESIGN_BRINKMAN})
        for (int prec : {LBMX_FP64, LBMX_FP32, LBMX_FP16_SHIFTED, LBMX_BF16_SHIFTED})
          if (lat == LBMX_D2Q9 || coll != LBMX_CASCADED) forms.push_back({lat, coll, des, prec});
  for (const Form& f : forms)
    for (int dir : {0, 1})
      for (int nx : {1, 2, 12, 48, 64, 65, 100, 128, 200, 330, 640, 1024, 2048, 4100})
        for (int ny : {1, 2, 5, 24, 128, 301, 512, 1024, 4000, 16000})
          for (int nbc : {0, 1, 4, 7, kMaxBC})
            for (int cus : {32, 256}) {
              const StepsShape s = shape(f, dir, nx, ny, nbc, cus);
              const bool fp64 = f.precision == LBMX_FP64;
              const int elem = fp64 ? 8 : (f.precision == LBMX_FP32 || dir == 1 ? 4 : 2);
              const bool ok = s.K == 1 ||
                              (s.K <= kMaxSteps && s.H >= 2 && steps_waves(s.K, s.H) <= steps_max_waves(dir, fp64) &&
                               steps_pieces_bytes(nbc, s.K) +
                                       steps_field_bytes(s.K, s.H, f.lattice == LBMX_D2Q9 ? 9 : 14, elem) <=
                                   160 * 1024);
              if (!ok || s.K < 1) {
                std::printf("%d x %d dir %d, %d pieces: %d steps of %d rows do not fit\n", nx, ny, dir, nbc, s.K, s.H);
                ++fails;
              }
            }
  const Form mrt64{LBMX_D2Q9, LBMX_MRT, LBMX_DESIGN_BRINKMAN, LBMX_FP64};
  const Form casc32{LBMX_D2Q9, LBMX_CASCADED, LBMX_DESIGN_PBB, LBMX_FP32};
  // one round of workgroups: the deepest launch with the fewest rows
  expect(mrt64, 0, 256, 128, 4, 2);
  expect(mrt64, 0, 512, 256, 4, 8);
  expect(mrt64, 1, 512, 256, 2, 8);
  expect(casc32, 1, 256, 128, 1, 1);
  // the round is that of the device's CUs
  expect(mrt64, 0, 256, 128, 3, 11, 32);
  expect(mrt64, 0, 64, 64, 4, 2, 32);
  // several rounds: two workgroups of the D2Q9 FP32 forward sweep share a CU
  const Form casc64{LBMX_D2Q9, LBMX_CASCADED, LBMX_DESIGN_PBB, LBMX_FP64};
  expect(casc64, 0, 1024, 512, 3, 11);
  expect(casc64, 0, 200, 1600, 2, 13);
  const Form mrt32{LBMX_D2Q9, LBMX_MRT, LBMX_DESIGN_BRINKMAN, LBMX_FP32};
  const Form mrt16{LBMX_D2Q9, LBMX_MRT, LBMX_DESIGN_PBB, LBMX_BF16_SHIFTED};
  const Form th64{LBMX_D2Q9_D2Q5, LBMX_MRT, LBMX_DESIGN_PBB, LBMX_FP64};
  const Form th32{LBMX_D2Q9_D2Q5, LBMX_MRT, LBMX_DESIGN_BRINKMAN, LBMX_FP32};
  expect(mrt64, 0, 1024, 512, 3, 11);
  expect(mrt64, 1, 1024, 512, 3, 7);
  expect(mrt32, 0, 1024, 512, 3, 7);
  expect(mrt32, 1, 1024, 512, 3, 11);
  expect(th64, 0, 1024, 512, 2, 13);
  expect(th64, 1, 1024, 512, 3, 6);
  expect(casc32, 0, 600, 400, 3, 7);
  expect(casc32, 0, 1280, 640, 3, 7);
  expect(casc32, 0, 2048, 1024, 1, 1);
  // narrow fields: fewer steps or one, unless there are few rounds
  expect(th32, 0, 2048, 1024, 3, 11);
  expect(th32, 0, 128, 8000, 2, 9);
  expect(th32, 0, 65, 2400, 3, 11);
  expect(mrt32, 0, 200, 6000, 1, 1);
  expect(mrt32, 0, 200, 1600, 3, 7);
  expect(mrt32, 1, 200, 1600, 1, 1);
  expect(mrt32, 1, 100, 2400, 3, 11);
  expect(mrt64, 0, 65, 16000, 3, 11);
  expect(mrt64, 1, 65, 16000, 1, 1);
  expect(mrt64, 1, 200, 1600, 3, 7);
  expect(mrt16, 1, 128, 8000, 1, 1);
  expect(mrt16, 1, 520, 2200, 3, 11);
  expect(th64, 1, 128, 8000, 2, 9);
  expect(th64, 1, 65, 2400, 1, 1);
  expect(th64, 1, 64, 3000, 1, 1);
  expect(mrt32, 1, 64, 4000, 3, 11);
  expect(th64, 1, 512, 300, 3, 6);
  expect(th64, 0, 64, 4000, 1, 1);
  expect(th64, 0, 64, 6000, 2, 13);
  expect(mrt64, 1, 64, 4000, 1, 1);
  expect(mrt64, 0, 64, 4000, 3, 11);
  expect(mrt32, 1, 64, 16000, 1, 1);
  if (!fails) std::printf("RESULT OK\n");
  return fails != 0;
}
