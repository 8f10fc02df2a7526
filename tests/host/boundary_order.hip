// The ghost fill's copies on the host (pluto_amd/csrc/boundary_kernels.hip):
// both sides of an axis in one launch, whose lines may run in any order,
// against one side after the other.  tests/test_boundary_order.py builds and
// runs it.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "boundary_kernels.hip"

using namespace pgpu;

struct Arrays {
  std::vector<double> a[11];
  double *vc[8], *vs[3];
  Arrays(const GhostBox& b, unsigned seed)
  {
    std::mt19937 r(seed);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    for (int q = 0; q < 11; q++) {
      long n = 1;
      for (int x = 0; x < 3; x++) n *= b.t[x] + (b.uni || x == q - 8);
      a[q].resize(n);
      for (auto& v : a[q]) v = u(r);
      if (q < 8) vc[q] = a[q].data();
      else vs[q - 8] = a[q].data();
    }
  }
};

static void run(const GhostBox& b, const FillSides& f, int sides, long most, int order, unsigned seed)
{
  struct Line { int side, op; long t; };
  std::vector<Line> all;
  for (int q = 0; q < sides; q++)
    for (int o = 0; o < f.side[q].nop; o++)
      for (long t = 0; t < most; t++) all.push_back({q, o, t});
  if (order == 1) std::reverse(all.begin(), all.end());
  if (order == 2) std::shuffle(all.begin(), all.end(), std::mt19937(seed));
  for (const auto& l : all) fill_line(b, f.side[l.side], f.side[l.side].op[l.op], l.t);
}

int main()
{
  const int pairs[][2] = {{BOUND_PERIODIC, BOUND_PERIODIC},   {BOUND_OUTFLOW, BOUND_OUTFLOW},
                          {BOUND_REFLECTIVE, BOUND_OUTFLOW},  {BOUND_OUTFLOW, BOUND_EQTSYMMETRIC},
                          {BOUND_AXISYMMETRIC, BOUND_REFLECTIVE}};
  const int boxes[][4] = {{5, 4, 7, 2}, {3, 3, 3, 3}, {2, 6, 3, 2}, {9, 4, 5, 4}};   // cells, ghost zones
  int bad = 0, runs = 0;
  for (const auto& x : boxes)
    for (int uni = 0; uni < 2; uni++) {
      GhostBox b;
      for (int a = 0; a < 3; a++) {
        b.n[a] = x[a];
        b.t[a] = x[a] + 2 * x[3];
        b.beg[a] = x[3];
        b.end[a] = x[3] + x[a] - 1;
      }
      b.uni = uni;
      for (int axis = 0; axis < 3; axis++)
        for (const auto& type : pairs)
          for (int order = 0; order < 5; order++) {   // 2 and up: shuffled
            if (b.n[axis] < x[3]) continue;
            Arrays one(b, 7), two(b, 7);
            for (int q = 0; q < 2; q++) {
              FillSides f{};
              long most = 0;
              if (fill_sides(b, 2 * axis + q, &type[q], 1, one.vc, one.vs, f, most)) return 2;
              run(b, f, 1, most, 0, 0);
            }
            FillSides f{};
            long most = 0;
            if (fill_sides(b, 2 * axis, type, 2, two.vc, two.vs, f, most)) return 2;
            run(b, f, 2, most, std::min(order, 2), 100 + order);
            runs++;
            for (int q = 0; q < 11; q++)
              if (one.a[q] != two.a[q]) {
                bad++;
                printf("box %d %d %d ghosts %d uni %d axis %d types %d %d order %d: array %d differs\n", x[0], x[1],
                       x[2], x[3], uni, axis, type[0], type[1], order, q);
              }
          }
    }
  printf("%d runs, %d arrays differ\n", runs, bad);
  return bad ? 1 : 0;
}
