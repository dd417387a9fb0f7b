// Host check of the LDS windows of the boundary tiles
// (nr-amssncku_amd/csrc/bssn_edge_tiles.h), built by test_edge_windows.py.
//
// For every array shape in the sweep (odd and even pitches, arrays that start
// on and off 16 bytes, with and without symmetry planes) the window of every
// tile is filled as the kernel fills it: chunk c of a buffer takes the two
// array elements from the (clamped) index that EdgeWindow::element gives for
// LDS index 2c.  Then every chunk must be 16-byte aligned and hold an element of
// the array (an even-pitched one only such), and every array index a boundary stencil may read at a live point -- within
// +-3 along each axis or within +-2 along two -- must be found at
// EdgeWindow::index of its place in the window.
#include <cstdio>
#include <vector>

#include "bssn_edge_tiles.h"

using namespace amss;

template <int NRM, bool ODD>
static bool check_tile(const EdgeTile& t, const int n[3], int base) {
  using W = EdgeWindow<NRM, ODD>;
  const int sy = n[0], sz = n[0] * n[1], N = n[0] * n[1] * n[2];
  const int gbase = t.wlo[0] + t.wlo[1] * sy + t.wlo[2] * sz;
  const int ob = ODD ? (base + gbase) & 1 : 0;
  std::vector<int> lds(W::PAD, -1);
  for (int c = 0; c < W::ROUNDS * kEdgeThreads; ++c) {
    int x, y, z;
    W::element(2 * c, sz, ob, x, y, z);
    const int gi = W::clamp(gbase + x + y * sy + z * sz, N);
    if ((gi + base) % 2 != 0 || gi < -1 || gi > N - 1 || (!ODD && (gi < 0 || gi + 1 >= N))) return false;
    lds[2 * c] = gi;
    lds[2 * c + 1] = gi + 1;
  }
  for (int tid = 0; tid < kEdgeThreads; ++tid) {
    int q[3];
    bool live;
    edge_tile_point(t, tid, q, live);
    if (!live) continue;
    for (int a = 0; a < 3; ++a)
      for (int b = a; b < 3; ++b)
        for (int d = (a == b ? -3 : -2); d <= (a == b ? 3 : 2); ++d)
          for (int e = (a == b ? 0 : -2); e <= (a == b ? 0 : 2); ++e) {
            int r[3] = {q[0], q[1], q[2]};
            r[a] += d;
            r[b] += e;
            bool in = true;
            for (int m = 0; m < 3; ++m) in = in && r[m] >= 0 && r[m] < n[m];
            if (!in) continue;
            const int li = W::index(r[0] - t.wlo[0], r[1] - t.wlo[1], r[2] - t.wlo[2], sz, ob);
            if (li < 0 || li >= W::PAD || lds[li] != r[0] + r[1] * sy + r[2] * sz) return false;
          }
  }
  return true;
}

template <bool ODD>
static bool check_set(const int n[3], const int mlo[3], int base) {
  const int lo[3] = {3, 3, 3}, hi[3] = {n[0] - 3, n[1] - 3, n[2] - 3};
  const EdgeTileSet S = edge_tile_set(edge_shells_of(n, lo, hi, mlo));
  for (int s = 0; s < 6; ++s)
    for (int b = 0; b < S.t[s].tiles(); ++b) {
      const EdgeTile t = edge_tile(S.t[s], b);
      const bool ok = s % 3 == 0 ? check_tile<0, ODD>(t, n, base)
                                 : (s % 3 == 1 ? check_tile<1, ODD>(t, n, base) : check_tile<2, ODD>(t, n, base));
      if (!ok) {
        std::printf("FAIL n %d %d %d base %d set %d tile %d\n", n[0], n[1], n[2], base, s, b);
        return false;
      }
    }
  return true;
}

int main() {
  int shapes = 0;
  for (int nx : {5, 6, 7, 8, 9, 13, 14, 15, 21, 22, 23, 24, 37, 54})
    for (int ny : {5, 6, 7, 9, 16, 21, 38})
      for (int nz : {5, 6, 8, 11, 20, 37})
        for (int sym = 0; sym < 3; ++sym) {
          const int n[3] = {nx, ny, nz};
          const int mlo[3] = {sym == 2 ? -3 : 0, sym == 2 ? -3 : 0, sym >= 1 ? -3 : 0};
          if (nx % 2 == 0) {
            if (!check_set<false>(n, mlo, 0)) return 1;
          } else {
            if (!check_set<true>(n, mlo, 0) || !check_set<true>(n, mlo, 1)) return 1;
          }
          ++shapes;
        }
  std::printf("ok %d shapes\n", shapes);
  return 0;
}
