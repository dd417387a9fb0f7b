// bssn_kernels_impl.h -- kernel templates of the BSSN RHS + RK4 path.
// Instantiated once per gauge in bssn_gauge0.hip / bssn_gauge2.hip so the
// heavy point kernels compile in parallel translation units.
#pragma once
#include "bssn_batch.h"
#include "bssn_edge_tiles.h"
#include "bssn_lds.h"

namespace amss {

#define AMSS_POINT_KERNEL __global__ void __launch_bounds__(kRhsThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))

template <class FI>
__device__ __forceinline__ bool bad_input(const FI& F, long p) {
  // the reference's NaN test covers the first 21 fields (bssn_rhs.f90:110-113)
  bool b = false;
#pragma unroll
  for (int v = 0; v < 21; ++v) {
    const double x = ((const gdouble*)F.ptr(v))[p];
    b |= !(x == x);
  }
  return b;
}

// The frozen-ghost fill of point p after an RK4 sub-step: the sub-step's
// base state U0, the NaN test on it, enforce_ga the next RHS applies to its
// input (sub-steps 0-2) and the lower bound on chi -- the sequence rk4 ->
// copy -> lowerboundset -> enforce_ga the reference runs on such points
// (bssn_class.C:3119-3156, 3415-3525).
__device__ __forceinline__ void ghost_fill_point(const FieldsIn& u0, const FieldsOut& out, long p, int stage,
                                                 double tinny, int* flag) {
  double u[NFIELD];
#pragma unroll
  for (int v = 0; v < NFIELD; ++v) u[v] = u0.p[v][p];
  bool bad = false;
#pragma unroll
  for (int v = 0; v < 21; ++v) bad |= !(u[v] == u[v]);  // bssn_rhs.f90:110-113
  if (bad) *flag = 1;
  if (stage < 3) enforce_point(u + DXX, u + AXX);
  u[CHI] = u[CHI] < tinny ? tinny : u[CHI];
#pragma unroll
  for (int v = 0; v < NFIELD; ++v) out.p[v][p] = u[v];
}

__device__ __forceinline__ bool interior_index(const Box& box, int& i, int& j, int& k) {
  i = box.lo[0] + blockIdx.x * kTileX + (threadIdx.x % kTileX);
  j = box.lo[1] + blockIdx.y * kTileY + (threadIdx.x / kTileX);
  k = box.lo[2] + blockIdx.z;
  return i < box.hi[0] && j < box.hi[1];
}
inline EdgeShells edge_shells(const Box& b) { return edge_shells_of(b.n, b.lo, b.hi, b.mlo); }

// Every point of the shell lies on the outermost layer of a face in mask
// (the on_faces bits): each of its slabs is one point deep along its axis,
// at index 0 of a lower face or n - 1 of an upper one in mask.
inline bool shell_on_faces(const Shell& sh, const int n[3], int mask) {
  // slab s: axis 2 - s / 2 (z, z, y, y, x, x), lower slab for even s
  for (int s = 0; s < 6; ++s) {
    if (sh.cnt[s] == 0) continue;
    const int a = 2 - s / 2;
    const int lo = (s & 1) ? sh.IH[a] : sh.OL[a], hi = (s & 1) ? sh.OH[a] : sh.IL[a];
    if (hi - lo != 1) return false;
    const bool on = (s & 1) ? (lo == n[a] - 1 && ((mask >> a) & 1)) : (lo == 0 && ((mask >> (3 + a)) & 1));
    if (!on) return false;
  }
  return true;
}

// Whether the LDS boundary kernels may take the order-1 and order-2 shells
// of this box: no Sommerfeld or copy face on them (a physical lower face has
// no mirrored halo, so its index 0 is an outermost-layer point; upper faces
// are at n - 1), and room for their tiles in the right-hand-side buffer.
inline bool edge_lds_ok(const Box& box, const SommerGeom& sg, const EdgeTileSet& T, const Rk4Param& R) {
  if (!R.edge_k || T.tiles() > R.edge_k_tiles) return false;
  const int mask = sg.faces | sg.copy;
  for (int a = 0; a < 3; ++a)
    if (((mask >> (3 + a)) & 1) && box.mlo[a] != 0) return false;
  return true;
}

// The right-hand side on the tiles of the order-1 and order-2 shells
// (bssn_edge_lds.h; instantiated in bssn_edge_inst.hip; ODD: an odd row
// pitch; MIRROR: the array has a symmetry plane), and the RK4 update of their
// points.
template <int G, bool CO, bool ODD, bool MIRROR>
void launch_edge_lds_rhs(const FieldsIn& in, const AuxOut& aux, const Box& box, const EdgeTileSet& T,
                         const Coef& C, double* K, int* flag, hipStream_t s);
template <int G, bool CO>
auto* edge_lds_launcher(bool odd, bool mirror) {
  return odd ? (mirror ? launch_edge_lds_rhs<G, CO, true, true> : launch_edge_lds_rhs<G, CO, true, false>)
             : (mirror ? launch_edge_lds_rhs<G, CO, false, true> : launch_edge_lds_rhs<G, CO, false, false>);
}
void launch_edge_lds_update(const FieldsIn& u0, const FieldsOut& acc, const FieldsOut& out, const AuxOut& aux,
                            const Box& box, const EdgeTileSet& T, const double* K, const Rk4Param& R,
                            hipStream_t s);

__device__ __forceinline__ bool edge_index(const Shell& sh, int& i, int& j, int& k) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t >= sh.size()) return false;
  sh.point(t, i, j, k);
  return true;
}

// ---- plain RHS (the compute_rhs_bssn outputs) ------------------------------
template <int GAUGE, bool CO>
AMSS_POINT_KERNEL rhs_interior_kernel(FieldsIn in, FieldsIn mat, FieldsOut out, AuxOut aux, Box box, Coef C,
                                      int* flag) {
  int i, j, k;
  if (!interior_index(box, i, j, k)) return;
  const long p = i + j * box.sy + k * box.sz;
  if (bad_input(in, p)) *flag = 1;
  InteriorEnv E{in, mat, C, p, box.sy, box.sz};
  RhsSink S{out, aux, p};
  bssn_rhs_point<GAUGE, CO, true, true>(E, S);
}

template <int GAUGE, bool CO, int ORD>
__global__ void __launch_bounds__(256) rhs_edge_kernel(FieldsIn in, FieldsIn mat, FieldsOut out, AuxOut aux,
                                                       Box box, Shell sh, Coef C, int* flag) {
  int i, j, k;
  if (!edge_index(sh, i, j, k)) return;
  const long p = i + j * box.sy + k * box.sz;
  if (bad_input(in, p)) *flag = 1;
  EdgeEnv<ORD> E(in, mat, C, i, j, k, box.n, box.mlo, box.sy, box.sz);
  RhsSink S{out, aux, p};
  bssn_rhs_point<GAUGE, CO, true, true>(E, S);
}

// ---- RHS fused with the RK4 sub-step ----------------------------------------
template <int GAUGE, int STAGE, bool CO>
AMSS_POINT_KERNEL rk4_interior_kernel(FieldsIn in, FieldsIn u0, FieldsOut acc, FieldsOut out, AuxOut aux, Box box,
                                      Coef C, Rk4Param R, int* flag) {
  int i, j, k;
  if (!interior_index(box, i, j, k)) return;
  const long p = i + j * box.sy + k * box.sz;
  if (bad_input(in, p)) *flag = 1;
  InteriorEnv E{in, in, C, p, box.sy, box.sz};
  Rk4SinkT<STAGE> S{u0, acc, out, aux, p, R.c, R.tinny, {}};
  bssn_rhs_point<GAUGE, CO, false, false>(E, S);
  S.finish();
}

// LDS-staged variant: tiles of a shape in kLdsShape, halo tiles of every
// field group in LDS (double-buffered, filled by direct global->LDS loads).  A
// 1-D grid of tiles in XCD-contiguous order: consecutive tiles, whose halos
// overlap, run behind the same L2.  The tiles cover the box whole: threads of
// a partial tile past it compute on a clamped point and store nothing
// (remainder slabs on the direct kernel took 120-155 us each and sub-step,
// whatever their size: a coarse step of a 64^3 patch and a nested one of 76^3
// with them 10.2 ms, with partial tiles 7.4 ms).  Instantiated in
// bssn_lds_g<G>[_odd].hip; lds_tile_shape (bssn_lds_launch.h) picks the shape.
constexpr int kLdsTX = 8, kLdsTY = 8, kLdsTZ = 4;
constexpr int kLdsShape[3][3] = {{8, 8, 4}, {8, 8, 8}, {32, 4, 4}};
// Tile b of gx x gy x gz: x fastest, then y in strips of `strip` tiles, then
// z, then the strips, so that the tiles an XCD holds at a time (32 of 512
// points) form a block whose halo is small: 128 x 16 x 8 points of 4 x 4 x 2
// wide tiles, 16 x 2 of cubic ones, at 128 points per row.  Sub-step 1 of 128^3
// points in 32x4x4 tiles: 993 us in plain order, 975 / 951 / 972 in strips of
// 2 / 4 / 8.  What bounds the kernel there is memory traffic: 4.3-4.6 GB per
// launch in 0.89-0.92 ms, 4.8 TB/s where a copy reaches 5.7.  The halo is read
// 5.7 times over the state's own bytes, as an XCD's tiles drift apart and its L2
// forgets; holding each 32 tiles together by a counter took 12% off the reads
// and cost 7% of the time, all of them then loading at once.
__device__ __forceinline__ void tile_place(int b, int gx, int gy, int gz, int strip, int& x, int& y, int& z) {
  const int full = gx * strip * gz, s = b / full, r = b - s * full, h = min(strip, gy - s * strip);
  x = r % gx;
  y = s * strip + (r / gx) % h;
  z = r / (gx * h);
}
#ifndef AMSS_LDS_WAVES
#define AMSS_LDS_WAVES 2
#endif
template <int GAUGE, int STAGE, bool CO, int SH, bool ODD>
__global__ void __launch_bounds__(kLdsShape[SH][0] * kLdsShape[SH][1] * kLdsShape[SH][2])
    __attribute__((amdgpu_waves_per_eu(AMSS_LDS_WAVES, AMSS_LDS_WAVES)))
rk4_lds_kernel(FieldsIn in, FieldsIn u0, FieldsOut acc, FieldsOut out, AuxOut aux, Box box,
                                 Coef C, Rk4Param R, int* flag, long nfill) {
  constexpr int TX = kLdsShape[SH][0], TY = kLdsShape[SH][1], TZ = kLdsShape[SH][2];
  using Tl = LdsTile<TX, TY, TZ, ODD>;
  __shared__ __attribute__((aligned(16))) double tiles[kLdsBuffers * Tl::NPAD + lds_stash(TX * TY * TZ, Tl::NPAD)];
  const int gx = (box.hi[0] - box.lo[0] + TX - 1) / TX, gy = (box.hi[1] - box.lo[1] + TY - 1) / TY;
  const int gz = (box.hi[2] - box.lo[2] + TZ - 1) / TZ, ntiles = gx * gy * gz;
  if ((int)blockIdx.x >= ntiles) {
    // the frozen-ghost fill of the nfill points outside [3, n - 3) of the
    // array (nfill is 0 when the caller fills them), in the workgroups after
    // the tiles (they start as the last tiles finish); its points lie
    // outside every tile
    if constexpr (STAGE < 2) {  // rk4_fuses_fill: sub-steps 0 and 1
      const long t = (long)(blockIdx.x - ntiles) * blockDim.x + threadIdx.x;
      if (t < nfill) {
        int i, j, k;
        ghost3_point(t, box.n[0], box.n[1], box.n[2], i, j, k);
        ghost_fill_point(u0, out, i + j * box.sy + k * box.sz, STAGE, R.tinny, flag);
      }
    }
    return;
  }
  int tx, ty, tz;
  Tl::point((int)threadIdx.x, tx, ty, tz);
  int bx, by, bz;
  tile_place(xcd_spread(blockIdx.x, ntiles), gx, gy, gz, TX == 32 ? 4 : gy, bx, by, bz);
  const int i0 = box.lo[0] + bx * TX, j0 = box.lo[1] + by * TY, k0 = box.lo[2] + bz * TZ;
  const int N = box.n[0] * box.n[1] * box.n[2];
  bool live;
  const BufIo io = tile_io(i0 + tx, j0 + ty, k0 + tz, box.hi[0], box.hi[1], box.hi[2], (int)box.sy, (int)box.sz, N, live);
  lds_double* t0 = (lds_double*)tiles;
  using Rk = LdsRk4<STAGE, TX, TY, TZ, FieldsIn, FieldsOut, AuxOut, ODD, (STAGE > 0 ? 2 : 1), SH == 2>;
  Rk X{
      {in, in, C, t0, t0 + (kLdsBuffers / 2) * Tl::NPAD, io, Tl::lds_index(tx, ty, tz, (int)box.sz),
       (int)((i0 - 3) + (j0 - 3) * box.sy + (k0 - 3) * box.sz), (int)box.sy, (int)box.sz, N, (int)threadIdx.x, tz + 3},
      {u0, acc, out, aux, typename Rk::Io{io.vo, io.vs, io.bytes}, R.c, R.tinny, {}},
       t0 + kLdsBuffers * Tl::NPAD + threadIdx.x};
  X.prologue();
  bssn_rhs_point<GAUGE, CO, false, false>(X, X);
  X.finish();
  if (X.bad && live) *flag = 1;
}

// sg: the Sommerfeld faces of the array (none when sg.faces == 0).  The
// sub-step is a template argument, as in the interior kernels (a runtime
// stage costs registers and spills).
#ifndef AMSS_EDGE_WAVES
#define AMSS_EDGE_WAVES 2
#endif
template <int GAUGE, int STAGE, bool CO, int ORD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(AMSS_EDGE_WAVES, AMSS_EDGE_WAVES)))
rk4_edge_kernel(FieldsIn in, FieldsIn u0, FieldsOut acc, FieldsOut out, AuxOut aux, Box box, Shell sh, Coef C,
                Rk4Param R, int* flag, SommerGeom sg) {
  int i, j, k;
  if (!edge_index(sh, i, j, k)) return;
  const long p = i + j * box.sy + k * box.sz;
  if (bad_input(in, p)) *flag = 1;
  // without the residuals, the points of the copy faces need nothing and
  // those of the Sommerfeld faces take sommer_face_kernel
  if (ORD == 0 && !CO && on_faces(sg.copy | sg.faces, box.n, i, j, k)) return;
  EdgeEnv<ORD> E(in, in, C, i, j, k, box.n, box.mlo, box.sy, box.sz);
  SommerRk4Sink<EdgeEnv<ORD>, Rk4SinkT<STAGE>> S{
      {u0, acc, out, aux, p, R.c, R.tinny, {}}, E, sg, sommer_point(sg, box.n, i, j, k)};
  bssn_rhs_point<GAUGE, CO, false, false>(E, S);
  S.finish();
}

// The RK4 sub-step on the Sommerfeld-face points of the outermost layer
// when no residuals are wanted: every field's RHS there is the boundary
// condition's (sommerfeld_rout.f90:376-440, applied to the stage's RHS
// before rungekutta4_rout, bssn_class.C:3106-3117), so the point algebra is
// skipped.  blockIdx.y is the point's work item (UpdateItems): one field
// alone, or before sub-step 3 the 12 fields enforce_ga couples, whose
// boundary RHS are all formed and whose U0 and accumulator values are all
// loaded before the first store.  With test_nan the kernel also applies the
// reference's NaN test to the shell's points (the launcher then runs no
// other kernel on them).
template <int STAGE>
__global__ void __launch_bounds__(256) sommer_face_kernel(FieldsIn in, FieldsIn u0, FieldsOut acc, FieldsOut out,
                                                          AuxOut aux, Box box, Shell sh, Rk4Param R, SommerGeom sg,
                                                          int* flag, bool test_nan) {
  int i, j, k;
  if (!edge_index(sh, i, j, k)) return;
  const long p = i + j * box.sy + k * box.sz;
  const int y = (int)blockIdx.y;
  if (y == 0 && test_nan && bad_input(in, p)) *flag = 1;
  if (on_faces(sg.copy, box.n, i, j, k) || !on_faces(sg.faces, box.n, i, j, k)) return;
  const int q[3] = {i, j, k};
  // the boundary RHS of field v; index -1 is index 0 times the field's
  // parity (the one mirrored layer below a symmetry plane), taken without a
  // branch so that all the reads can be in flight together
  auto rhs = [&](int v) {
    auto rd = [&](int a, int m) {
      int c[3] = {q[0], q[1], q[2]};
      const int t = c[a] + m, neg = t >> 31;
      c[a] = t ^ neg;
      const double x = in.p[v][c[0] + c[1] * box.sy + c[2] * box.sz];
      return (x + 0.0) * (neg ? (double)parity(v, a) : 1.0);
    };
    return sommer_rhs(sg, box.n, q, prop_speed(v), rd);
  };
  Rk4SinkT<STAGE> S{u0, acc, out, aux, p, R.c, R.tinny, {}};
  if (STAGE < 3 && y == 0) {
    double kv[12], uv[12], av[12];
#pragma unroll
    for (int s = 0; s < 12; ++s) kv[s] = rhs(DXX + s);
#pragma unroll
    for (int s = 0; s < 12; ++s) {
      uv[s] = u0.p[DXX + s][p];
      av[s] = STAGE > 0 ? acc.p[DXX + s][p] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < 12; ++s) S.put_loaded(DXX + s, kv[s], uv[s], av[s]);
    S.finish();
  } else {
    const int v = UpdateItems<STAGE>::field(y);
    const double kv = rhs(v), uv = u0.p[v][p], av = STAGE > 0 ? acc.p[v][p] : 0.0;
    S.put_loaded(v, kv, uv, av);
  }
}

inline dim3 interior_grid(const Box& b) {
  return dim3((b.hi[0] - b.lo[0] + kTileX - 1) / kTileX, (b.hi[1] - b.lo[1] + kTileY - 1) / kTileY,
              b.hi[2] - b.lo[2]);
}
inline bool box_empty(const Box& b) { return b.hi[0] <= b.lo[0] || b.hi[1] <= b.lo[1] || b.hi[2] <= b.lo[2]; }
inline unsigned blocks_for(long n, int t) { return (unsigned)((n + t - 1) / t); }

// The plain right-hand side of a whole array in one launch (bssn_rhs_lds.h;
// instantiated in bssn_rhs_inst.hip).
template <int G, bool CO, bool ODD>
void launch_rhs_lds(const FieldsIn& in, const FieldsIn& mat, const FieldsOut& out, const AuxOut& aux, const Box& box,
                    const Coef& C, int* flag, hipStream_t s);

// Whether it may run: no symmetry plane (a variant with the mirror pass gave
// wrong values, for the reason told at EdgeLdsEnv::mirror, and was not kept),
// every axis of 5 points or more (the boundary tiles' windows are laid out
// for those), 32-bit byte offsets, and with an even row
// pitch every state array on 16 bytes (the direct loads' alignment; with an
// odd pitch the layout follows each array's own).
inline bool rhs_lds_ok(const FieldsIn& in, const Box& box) {
  for (int a = 0; a < 3; ++a)
    if (box.n[a] < 5 || box.mlo[a] < 0) return false;
  if ((long)box.n[0] * box.n[1] * box.n[2] >= (1L << 29)) return false;
  for (int v = 0; v < NFIELD; ++v)
    if (((uintptr_t)in.p[v]) % (box.sy % 2 == 0 ? 16 : 8) != 0) return false;
  return true;
}

template <int G>
void launch_rhs_gauge(const FieldsIn& in, const FieldsIn& mat, const FieldsOut& out, const AuxOut& aux,
                      const Box& box, const Coef& C, int co, int* flag, bool edge, hipStream_t s) {
  if (edge && rhs_lds_ok(in, box)) {
    auto* rhs = box.sy % 2 != 0 ? (co == 0 ? launch_rhs_lds<G, true, true> : launch_rhs_lds<G, false, true>)
                                : (co == 0 ? launch_rhs_lds<G, true, false> : launch_rhs_lds<G, false, false>);
    rhs(in, mat, out, aux, box, C, flag, s);
    return;
  }
  if (co == 0) {
    if (!box_empty(box)) rhs_interior_kernel<G, true><<<interior_grid(box), kRhsThreads, 0, s>>>(in, mat, out, aux, box, C, flag);
  } else {
    if (!box_empty(box)) rhs_interior_kernel<G, false><<<interior_grid(box), kRhsThreads, 0, s>>>(in, mat, out, aux, box, C, flag);
  }
  if (!edge) return;
  const EdgeShells es = edge_shells(box);
#define AMSS_REDGE(O)                                                                                       \
  if (es.s[O].size() > 0) {                                                                                 \
    const unsigned gr = blocks_for(es.s[O].size(), 256);                                                    \
    if (co == 0) rhs_edge_kernel<G, true, O><<<gr, 256, 0, s>>>(in, mat, out, aux, box, es.s[O], C, flag);  \
    else rhs_edge_kernel<G, false, O><<<gr, 256, 0, s>>>(in, mat, out, aux, box, es.s[O], C, flag);         \
  }
  AMSS_REDGE(0)
  AMSS_REDGE(1)
  AMSS_REDGE(2)
#undef AMSS_REDGE
}

// The fused sub-step of an interior box on LDS tiles (ODD: an odd row pitch).
template <int G, bool ODD>
void launch_rk4_lds(const FieldsIn& in, const FieldsIn& u0, const FieldsOut& acc, const FieldsOut& out,
                    const AuxOut& aux, const Box& box, const Coef& C, const Rk4Param& R, bool want_res, int* flag,
                    hipStream_t s);

template <int G>
void launch_rk4_gauge(const FieldsIn& in, const FieldsIn& u0, const FieldsOut& acc, const FieldsOut& out,
                      const AuxOut& aux, const Box& box, const Coef& C, const Rk4Param& R, bool want_res, int* flag,
                      bool edge, hipStream_t s, bool interior, const SommerGeom& sg) {
  if (interior && !box_empty(box) && R.variant == 1) {
    if (box.sy % 2 == 0) launch_rk4_lds<G, false>(in, u0, acc, out, aux, box, C, R, want_res, flag, s);
    else launch_rk4_lds<G, true>(in, u0, acc, out, aux, box, C, R, want_res, flag, s);
  } else if (interior && !box_empty(box)) {
    const dim3 gr = interior_grid(box);
    switch (R.stage) {
      case 0:
        if (want_res) rk4_interior_kernel<G, 0, true><<<gr, kRhsThreads, 0, s>>>(in, u0, acc, out, aux, box, C, R, flag);
        else rk4_interior_kernel<G, 0, false><<<gr, kRhsThreads, 0, s>>>(in, u0, acc, out, aux, box, C, R, flag);
        break;
      case 1: rk4_interior_kernel<G, 1, false><<<gr, kRhsThreads, 0, s>>>(in, u0, acc, out, aux, box, C, R, flag); break;
      case 2: rk4_interior_kernel<G, 2, false><<<gr, kRhsThreads, 0, s>>>(in, u0, acc, out, aux, box, C, R, flag); break;
      default: rk4_interior_kernel<G, 3, false><<<gr, kRhsThreads, 0, s>>>(in, u0, acc, out, aux, box, C, R, flag); break;
    }
  }
  if (edge) {
    const EdgeShells es = edge_shells(box);
    // the order-1 and order-2 shells in one LDS launch pair where it may
    // take them (run with edge_order 1; edge_order 2 then has nothing left)
    const EdgeTileSet ts = edge_tile_set(es);
    const bool lds = R.variant == 1 && edge_lds_ok(box, sg, ts, R);
    for (int o = 0; o < 3; ++o) {
      const Shell& sh = es.s[o];
      if (sh.size() <= 0 || (R.edge_order >= 0 && o != R.edge_order)) continue;
      if (lds && o >= 1) {
        if (o == 1 && ts.tiles() > 0) {
          const bool odd = box.sy % 2 != 0, mirror = box.mlo[0] < 0 || box.mlo[1] < 0 || box.mlo[2] < 0;
          auto* rhs = want_res ? edge_lds_launcher<G, true>(odd, mirror) : edge_lds_launcher<G, false>(odd, mirror);
          rhs(in, aux, box, ts, C, R.edge_k, flag, s);
          launch_edge_lds_update(u0, acc, out, aux, box, ts, R.edge_k, R, s);
        }
        continue;
      }
      const unsigned gr = blocks_for(sh.size(), 256);
      // Without the residuals, an outermost layer made of Sommerfeld and
      // copy faces only needs the face kernel.
      const bool faces_only = o == 0 && !want_res && (sg.faces | sg.copy) != 0 &&
                              shell_on_faces(sh, box.n, sg.faces | sg.copy);
      if (!faces_only) {
#define AMSS_EDGE(ST, CO)                                                                                      \
  do {                                                                                                         \
    if (o == 0) rk4_edge_kernel<G, ST, CO, 0><<<gr, 256, 0, s>>>(in, u0, acc, out, aux, box, sh, C, R, flag, sg); \
    else if (o == 1) rk4_edge_kernel<G, ST, CO, 1><<<gr, 256, 0, s>>>(in, u0, acc, out, aux, box, sh, C, R, flag, sg); \
    else rk4_edge_kernel<G, ST, CO, 2><<<gr, 256, 0, s>>>(in, u0, acc, out, aux, box, sh, C, R, flag, sg);       \
  } while (0)
        switch (R.stage) {
          case 0:
            if (want_res) AMSS_EDGE(0, true);
            else AMSS_EDGE(0, false);
            break;
          case 1: AMSS_EDGE(1, false); break;
          case 2: AMSS_EDGE(2, false); break;
          default: AMSS_EDGE(3, false); break;
        }
#undef AMSS_EDGE
      }
      if (o == 0 && !want_res && (faces_only || sg.faces != 0)) {
        const bool nan = faces_only;
#define AMSS_FACE(ST)                                                                                      \
  sommer_face_kernel<ST><<<dim3(gr, UpdateItems<ST>::kCount), 256, 0, s>>>(in, u0, acc, out, aux, box, sh, R, sg, \
                                                                          flag, nan)
        switch (R.stage) {
          case 0: AMSS_FACE(0); break;
          case 1: AMSS_FACE(1); break;
          case 2: AMSS_FACE(2); break;
          default: AMSS_FACE(3); break;
        }
#undef AMSS_FACE
      }
    }
  }
}

}  // namespace amss
