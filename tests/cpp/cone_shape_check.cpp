// Which cone kernel a grid takes. Prints "RESULT OK" at the end.
#include <cstdio>
#include <initializer_list>

#include "design_cone_shape.hpp"

using namespace lbmx;

static int fails = 0;
static void expect(bool want, int nx, int ny, int nz, int R, bool tr) {
  if (cone_fixed_radius(nx, ny, nz, R, tr) == want) return;
  std::printf("%d x %d x %d radius %d %s: expected %s\n", nx, ny, nz, R, tr ? "transposed" : "forward",
              want ? "the kernel of its radius" : "the kernel of any radius");
  ++fails;
}

int main() {
  for (bool tr : {false, true})
    for (int R = 1; R <= 3; ++R) {
      // small grids, where the kernel of the radius is slower, and large ones, where it is faster
      for (int n : {2, 16, 25, 48, 64}) expect(false, n, n, n, R, tr);
      expect(false, 101, 47, 53, R, tr);
      expect(true, 256, 128, 128, R, tr);
      expect(true, 384, 192, 192, R, tr);
      expect(false, 384, 192, 192, R + 3, tr);
      for (int r = R; r <= 12; r += 3) expect(true, 48, 24, 1, r, tr);
    }
  expect(false, 48, 24, 1, 13, false);
  // a launch has at most 65535 workgroups along y
  expect(true, 3, 524280, 1, 2, false);
  expect(false, 3, 524281, 1, 2, false);
  expect(false, 3, 1048560, 1, 12, true);
  if (!fails) std::printf("RESULT OK\n");
  return fails != 0;
}
