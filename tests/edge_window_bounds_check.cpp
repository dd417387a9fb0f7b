// Host check of what the boundary tiles' windows read, and of their mirror
// image (nr-amssncku_amd/csrc/bssn_edge_tiles.h), built by
// test_edge_window_bounds.py.
//
// For every array shape in the sweep (odd and even pitches, arrays on and off
// 16 bytes, no, one and three symmetry planes) every tile's window is filled as
// the kernel fills it, by 16-byte chunks.  Every chunk must lie inside the array;
// with symmetry planes the first may start one element before an array that
// starts off 16 bytes (another field of the slab ends there).  The mirror pass
// then runs: every source must be a cell of the window that the pass does not write.  Last,
// every read of a boundary stencil -- within +-3 along one axis or within +-2
// along two, below the planes included -- must find the right element, mirrored
// along the right axes.
#include <cstdio>
#include <vector>

#include "bssn_edge_tiles.h"

using namespace amss;

struct Cell {
  int gi, axes;  // array element, axes it was mirrored along
};

template <int NRM, bool ODD>
static const char* check_tile(const EdgeTile& t, const int n[3], const int mlo[3], int base) {
  using W = EdgeWindow<NRM, ODD>;
  const int sy = n[0], sz = n[0] * n[1], N = n[0] * n[1] * n[2];
  const int gbase = t.wlo[0] + t.wlo[1] * sy + t.wlo[2] * sz;
  const int ob = ODD ? (base + gbase) & 1 : 0;
  const bool planes = mlo[0] < 0 || mlo[1] < 0 || mlo[2] < 0;
  std::vector<Cell> lds(W::PAD, Cell{-9, 0});
  for (int c = 0; c < W::ROUNDS * kEdgeThreads; ++c) {
    int x, y, z;
    W::element(2 * c, sz, ob, x, y, z);
    const int gi = W::clamp(gbase + x + y * sy + z * sz, N, planes);
    if ((gi + base) % 2 != 0) return "a chunk off 16 bytes";
    if (gi + 1 >= N) return "a chunk past the array";
    if (gi < 0 && !(planes && base == 1 && gi == -1)) return "a chunk before the array";
    lds[2 * c] = Cell{gi, 0};
    lds[2 * c + 1] = Cell{gi + 1, 0};
  }
  int mir = 0;
  for (int a = 0; a < 3; ++a)
    if (mlo[a] < 0 && t.wlo[a] < 0) mir |= 1 << a;
  if (mir) {
    const int ext[3] = {W::W0, W::W1, W::W2};
    std::vector<Cell> next = lds;
    for (int c = 0; c < W::W0 * W::W1 * W::W2; ++c) {
      int x[3], m[3], y[3], k[3];
      const int im = W::image(c, t.wlo, mir, x, m);
      if (im == 0) continue;
      for (int a = 0; a < 3; ++a) {
        y[a] = m[a] - t.wlo[a];
        if (y[a] < 0 || y[a] >= ext[a]) return "a mirror source outside the window";
      }
      if (W::image(y[0] + W::W0 * (y[1] + W::W1 * y[2]), t.wlo, mir, y, k) != 0) return "a mirror source that the pass writes";
      next[W::index(x[0], x[1], x[2], sz, ob)] = Cell{lds[W::index(y[0], y[1], y[2], sz, ob)].gi, im};
    }
    lds = next;
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
            int r[3] = {q[0], q[1], q[2]}, f[3], axes = 0;
            r[a] += d;
            r[b] += e;
            bool in = true;
            for (int m = 0; m < 3; ++m) {
              in = in && r[m] >= mlo[m] && r[m] < n[m];
              f[m] = r[m] < 0 ? -r[m] - 1 : r[m];
              in = in && f[m] < n[m];
              axes |= r[m] < 0 ? 1 << m : 0;
            }
            if (!in) continue;
            const int li = W::index(r[0] - t.wlo[0], r[1] - t.wlo[1], r[2] - t.wlo[2], sz, ob);
            if (li < 0 || li >= W::PAD) return "a read outside the window";
            if (lds[li].gi != f[0] + f[1] * sy + f[2] * sz || lds[li].axes != axes) return "a read of the wrong element";
          }
  }
  return nullptr;
}

template <bool ODD>
static bool check_set(const int n[3], const int mlo[3], int base) {
  const int lo[3] = {3, 3, 3}, hi[3] = {n[0] - 3, n[1] - 3, n[2] - 3};
  const EdgeTileSet S = edge_tile_set(edge_shells_of(n, lo, hi, mlo));
  for (int s = 0; s < 6; ++s)
    for (int b = 0; b < S.t[s].tiles(); ++b) {
      const EdgeTile t = edge_tile(S.t[s], b);
      const char* bad = s % 3 == 0 ? check_tile<0, ODD>(t, n, mlo, base)
                                   : (s % 3 == 1 ? check_tile<1, ODD>(t, n, mlo, base) : check_tile<2, ODD>(t, n, mlo, base));
      if (bad) {
        std::printf("%s: n %d %d %d mlo %d %d %d base %d set %d tile %d\n", bad, n[0], n[1], n[2], mlo[0], mlo[1], mlo[2],
                    base, s, b);
        return false;
      }
    }
  return true;
}

int main() {
  int shapes = 0;
  for (int nx : {5, 6, 7, 8, 9, 14, 15, 21, 22, 37, 54})
    for (int ny : {5, 6, 7, 9, 16, 21, 38})
      for (int nz : {5, 6, 8, 11, 20, 37})
        for (int sym = 0; sym < 5; ++sym) {  // none, z, x y z, x, y
          const int n[3] = {nx, ny, nz};
          const int mlo[3] = {sym == 2 || sym == 3 ? -3 : 0, sym == 2 || sym == 4 ? -3 : 0, sym == 1 || sym == 2 ? -3 : 0};
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
