// Launch shapes of the row x/y flux kernel (row_launch, fused_kernels.hpp) over
// boxes of all proportions: within the device's grid limits, every row or
// window covered.  tests/test_launch_shapes.py builds and runs it.
#include <cstdio>
#include <random>

#include "fused_kernels.hpp"

static int g_seg = 0;
namespace pgpu {
int flux_xy_kind() { return 1; }
int flux_xy_seg() { return g_seg; }
}  // namespace pgpu

using namespace pgpu;

int main()
{
  constexpr int GRID = 65535;   // workgroups along the grid's y and z
  std::mt19937 rng(5);
  auto size = [&](int lo, int hi) {   // by the logarithm
    std::uniform_real_distribution<double> u(std::log((double)lo), std::log((double)hi + 1.0));
    const int n = (int)std::exp(u(rng));
    return n < lo ? lo : (n > hi ? hi : n);
  };
  int bad = 0, tiles = 0, rows = 0, windows = 0;
  const int fixed[][4] = {{1000, 8, 60000, 0},  {300, 3, 65000, 0},  {257, 3, 65535, 0}, {256, 3, 65535, 0},
                          {3, 3, 65535, 0},     {60000, 3, 1000, 0}, {3, 60000, 1000, 0}, {100000, 100, 1, 0},
                          {16, 16, 65536, 16},  {8, 8, 80000, 8},    {256, 256, 1024, 256}};
  for (int q = 0; q < 200000; q++) {
    Geo g{};
    if (q < (int)(sizeof fixed / sizeof fixed[0])) {
      g.nx = fixed[q][0];
      g.ny = fixed[q][1];
      g.nz = fixed[q][2];
      g.pz = fixed[q][3];
    } else if (q % 4 == 0) {   // a stack of patches
      g.nx = g.ny = g.pz = size(4, 256);
      g.nz = g.pz * size(1, 4096);
    } else {
      g.nx = size(3, 70000);
      g.ny = size(3, 70000);
      g.nz = q % 4 == 1 ? 1 : size(3, 65535);
    }
    g.dims = g.nz > 1 ? 3 : 2;
    g.n = (long)g.nx * g.ny * g.nz;
    if (g.n * 8 >= (1l << 32)) continue;
    for (int seg : {0, 1, 7, 40})
      for (int real : {8, 4}) {
        g_seg = seg;
        const RowLaunch r = row_launch(g, real);
        bool ok = true;
        if (!r.nt) {
          tiles++;
          // the tiles' planes go along z; a stack has no tiles
          ok = g.pz <= 0 && g.nz <= GRID;
        } else {
          const int deep = g.pz > 0 ? g.pz : g.nz;
          ok = r.nt % 64 == 0 && r.nt <= 256 && r.seg >= 1 && (g.pz > 0 || r.wgs <= GRID);
          if (r.rows > 0) {
            rows++;
            ok = ok && r.rows * g.nx <= r.nt && (long)r.wgs * r.rows >= g.nz && r.rows <= deep &&
                 (g.pz <= 0 || g.pz % r.rows == 0);
          } else {
            windows++;
            // the owned cells of the last window end past the last row
            ok = ok && g.pz <= 0 && (long)r.wgs * (r.nt - 4) + 4 >= (long)g.nz * (g.nx + 4);
          }
        }
        if (!ok && bad++ < 20)
          printf("%d x %d x %d (pz %d) seg %d real %d: nt %d wgs %d rows %d seg %d\n", g.nx, g.ny, g.nz, g.pz, seg,
                 real, r.nt, r.wgs, r.rows, r.seg);
      }
  }
  printf("%d as tiles, %d as rows, %d as windows, %d bad\n", tiles, rows, windows, bad);
  return bad || !tiles || !rows || !windows;
}
