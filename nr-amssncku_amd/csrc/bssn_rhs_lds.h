// bssn_rhs_lds.h -- the plain right-hand side (the compute_rhs_bssn outputs)
// of a whole array without symmetry planes in one launch: every workgroup takes an LDS tile of the
// order-1 and order-2 shells, 256 points of the outermost layer, or an LDS
// tile of the interior, by its block index.
//
// A call is bound by the latency of a tile's chain of field groups (one load
// and barrier after another) while the array is small, by the 55 output arrays
// while it is large.  As launches of their own the interior and the three
// shells ran one after the other, each with such a chain: a 54^3 block took
// 188 + 103 + 149 + 211 us.  In one launch the chains run side by side, the
// boundary tiles, whose chains are longest, first: 172 us, and 1.58 ms for
// 134^3 with matter (2.9 ms before: the interior read its stencils through L1
// and L2).
#pragma once
#include "bssn_edge_lds.h"

namespace amss {

// The reference ABI's outputs at one point, masked as IO masks.
template <class IO>
struct RhsIoSink {
  const FieldsOut& O;
  const AuxOut& X;
  IO io;
  __device__ __forceinline__ void put(int v, double k) { io.st(O.p[v], k); }
  __device__ __forceinline__ void gam(int a, double x) { io.st(X.gam[a], x); }
  __device__ __forceinline__ void ric(int a, double x) { io.st(X.ric[a], x); }
  __device__ __forceinline__ void res(int a, double x) { io.st(X.res[a], x); }
};

// Blocks of each kind: [0, edge) shell tiles, [edge, edge + face) outermost
// layer, then the interior's tiles.
struct RhsBlocks {
  int edge, face, tiles;
};

template <int GAUGE, bool CO, int ORD, int NRM, bool ODD>
__device__ __forceinline__ void rhs_edge_tile(const FieldsIn& in, const FieldsIn& mat, const FieldsOut& out,
                                              const AuxOut& aux, const Box& box, const EdgeTiles& T, int lb,
                                              const Coef& C, int* flag, lds_double* win) {
  const EdgeTile t = edge_tile(T, lb);
  int q[3];
  bool live;
  edge_tile_point(t, (int)threadIdx.x, q, live);
  EdgeLdsEnv<ORD, NRM, ODD, false> E(in, mat, C, q, box, t, win, (int)threadIdx.x, live);
  const unsigned vo = (unsigned)E.p * 8u;
  RhsIoSink<BufIo> S{out, aux, {vo, live ? vo : kDropStore, (unsigned)E.gmax * 8u}};
  E.prologue();
  bssn_rhs_point<GAUGE, CO, true, true>(E, S);
  if (E.bad) *flag = 1;
}

template <int GAUGE, bool CO, bool ODD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
rhs_lds_kernel(FieldsIn in, FieldsIn mat, FieldsOut out, AuxOut aux, Box box, EdgeTileSet T, Shell face, RhsBlocks nb,
               Coef C, int* flag) {
  using Tl = LdsTile<kLdsTX, kLdsTY, kLdsTZ, ODD>;
  constexpr int kWin = edge_lds_doubles<ODD>(), kTile = kLdsBuffers * Tl::NPAD;
  __shared__ __attribute__((aligned(16))) double lds[kWin > kTile ? kWin : kTile];
  lds_double* w = (lds_double*)lds;
  int b = (int)blockIdx.x;
  if (b < nb.edge) {
    const int s = T.set_of(b), lb = b - T.first[s];
#define AMSS_TILE(S, ORD, NRM) \
  case S: rhs_edge_tile<GAUGE, CO, ORD, NRM, ODD>(in, mat, out, aux, box, T.t[S], lb, C, flag, w); break
    switch (s) {
      AMSS_TILE(0, 1, 0);
      AMSS_TILE(1, 1, 1);
      AMSS_TILE(2, 1, 2);
      AMSS_TILE(3, 2, 0);
      AMSS_TILE(4, 2, 1);
      AMSS_TILE(5, 2, 2);
    }
#undef AMSS_TILE
    return;
  }
  b -= nb.edge;
  if (b < nb.face) {
    const long t = b * 256L + threadIdx.x;
    if (t >= face.size()) return;
    int i, j, k;
    face.point(t, i, j, k);
    const long p = i + j * box.sy + k * box.sz;
    if (bad_input(in, p)) *flag = 1;
    EdgeEnv<0> E(in, mat, C, i, j, k, box.n, box.mlo, box.sy, box.sz);
    RhsIoSink<PtrIo> S{out, aux, {p}};
    bssn_rhs_point<GAUGE, CO, true, true>(E, S);
    return;
  }
  b = xcd_spread(b - nb.face, nb.tiles);
  int tx, ty, tz;
  Tl::point((int)threadIdx.x, tx, ty, tz);
  const int gx = (box.hi[0] - box.lo[0] + kLdsTX - 1) / kLdsTX, gy = (box.hi[1] - box.lo[1] + kLdsTY - 1) / kLdsTY;
  const int i0 = box.lo[0] + (b % gx) * kLdsTX, j0 = box.lo[1] + ((b / gx) % gy) * kLdsTY;
  const int k0 = box.lo[2] + (b / (gx * gy)) * kLdsTZ;
  const int N = box.n[0] * box.n[1] * box.n[2];
  bool live;
  const BufIo io = tile_io(i0 + tx, j0 + ty, k0 + tz, box.hi[0], box.hi[1], box.hi[2], (int)box.sy, (int)box.sz, N, live);
  LdsEnv<kLdsTX, kLdsTY, kLdsTZ, FieldsIn, void, ODD> E{
      in, mat, C, w, w + (kLdsBuffers / 2) * Tl::NPAD, io, Tl::lds_index(tx, ty, tz, (int)box.sz),
      (int)((i0 - 3) + (j0 - 3) * box.sy + (k0 - 3) * box.sz), (int)box.sy, (int)box.sz, N, (int)threadIdx.x, tz + 3};
  RhsIoSink<BufIo> S{out, aux, io};
  E.prologue();
  bssn_rhs_point<GAUGE, CO, true, true>(E, S);
  if (E.bad && live) *flag = 1;
}

template <int G, bool CO, bool ODD>
void launch_rhs_lds(const FieldsIn& in, const FieldsIn& mat, const FieldsOut& out, const AuxOut& aux, const Box& box,
                    const Coef& C, int* flag, hipStream_t s) {
  const EdgeShells es = edge_shells(box);
  const EdgeTileSet T = edge_tile_set(es);
  RhsBlocks nb{T.tiles(), (int)blocks_for(es.s[0].size(), 256), 1};
  const int Td[3] = {kLdsTX, kLdsTY, kLdsTZ};
  for (int a = 0; a < 3; ++a) nb.tiles *= box.hi[a] > box.lo[a] ? (box.hi[a] - box.lo[a] + Td[a] - 1) / Td[a] : 0;
  rhs_lds_kernel<G, CO, ODD><<<(unsigned)(nb.edge + nb.face + nb.tiles), 256, 0, s>>>(in, mat, out, aux, box, T,
                                                                                         es.s[0], nb, C, flag);
}

}  // namespace amss
