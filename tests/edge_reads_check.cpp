// Host check of every array index the boundary stencils read in global memory
// (EdgeEnv in nr-amssncku_amd/csrc/bssn_env.h), from the index functions of
// bssn_edge_tiles.h that it calls; built by test_edge_read_indexes.py.
//
// Over all shapes of 5 to 9 points per axis (3 to 9 with a symmetry plane), every
// set of planes and every point of the three shells: the upwind stencil's seven
// samples per axis, the centred stencils of the shell's order (two axes at a
// time) and the dissipation where it is taken must fold to an index of the array.
#include <cstdio>

#include "bssn_edge_tiles.h"

using namespace amss;

static long reads = 0;
static bool inside(int q, int n) {
  ++reads;
  const int f = edge_fold(q);
  return f >= 0 && f < n;
}

static bool check_point(int ord, const int q[3], const int n[3], const int mlo[3]) {
  bool room3 = true;
  for (int a = 0; a < 3; ++a) {
    for (int m = -3; m <= 3; ++m)
      if (!inside(q[a] + edge_clamp(q[a], m, n[a]), n[a])) return false;
    for (int m = -ord; m <= ord; ++m)
      if (q[a] + m < mlo[a] || !inside(q[a] + m, n[a])) return false;
    room3 = room3 && q[a] - 3 >= mlo[a] && q[a] + 3 <= n[a] - 1;
  }
  if (ord == 2 && room3)
    for (int a = 0; a < 3; ++a)
      if (!inside(q[a] - 3, n[a]) || !inside(q[a] + 3, n[a])) return false;
  return true;
}

int main() {
  long points = 0;
  for (int planes = 0; planes < 8; ++planes) {
    int mlo[3], lo[3];
    for (int a = 0; a < 3; ++a) {
      mlo[a] = (planes >> a) & 1 ? -3 : 0;
      lo[a] = mlo[a] < 0 ? 3 : 5;
    }
    for (int nx = lo[0]; nx <= 9; ++nx)
      for (int ny = lo[1]; ny <= 9; ++ny)
        for (int nz = lo[2]; nz <= 9; ++nz) {
          const int n[3] = {nx, ny, nz}, bl[3] = {3, 3, 3}, bh[3] = {nx - 3, ny - 3, nz - 3};
          const EdgeShells S = edge_shells_of(n, bl, bh, mlo);
          for (int o = 0; o < 3; ++o)
            for (long t = 0; t < S.s[o].size(); ++t, ++points) {
              int q[3];
              S.s[o].point(t, q[0], q[1], q[2]);
              if (!check_point(o, q, n, mlo)) {
                std::printf("n %d %d %d planes %d order %d point %d %d %d\n", nx, ny, nz, planes, o, q[0], q[1], q[2]);
                return 1;
              }
            }
        }
  }
  std::printf("ok %ld points, %ld reads\n", points, reads);
  return 0;
}
