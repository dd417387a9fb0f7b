// bssn_lds.h -- LDS-staged stencil environment for the fused RHS kernels.
//
// A workgroup owns a TX x TY x TZ tile of interior points (one point per
// thread; the threads of a partial tile past the interior compute on clamped
// points and store nothing).  For every field group of the algebra the tile plus a
// 3-point halo of that field, (TX+6)(TY+6)(TZ+6) doubles, sits in LDS; every
// stencil of the group (gradient, Hessian incl. mixed, upwind, KO) reads it
// from there with compile-time offsets.  Two tile buffers alternate: while
// group g computes from one, the halo tile of group g+1 streams into the
// other with gfx950's direct global->LDS loads (global_load_lds_dwordx4:
// each lane moves 16 bytes, a wave fills a contiguous 1 KiB run starting at
// the wave-uniform LDS base), so staging costs no VGPRs.  The centre value of
// the open group's field comes from its tile; the other centre values a pair
// reads (and the RK4 epilogue's U0 and accumulator values of its fields) are
// loaded one pair ahead, so the barrier's full wait settles them and no
// later wait for them stalls on the halo loads in flight.
#pragma once
#include <type_traits>

#include "bssn_env.h"

namespace amss {

// The order in which bssn_rhs_point opens its field groups.
__host__ __device__ constexpr int group_field(int g) {
  constexpr signed char seq[NFIELD] = {BETAX, BETAY, BETAZ, DXX, GXY, GXZ, DYY, GYZ,
                                       DZZ,   GAMX,  GAMY,  GAMZ, CHI, LAP, TRK, DTSFX,
                                       DTSFY, DTSFZ, AXX,   AXY,  AXZ, AYY, AYZ, AZZ};
  return seq[g];
}

// The centre value of another field that the point algebra reads inside a
// group (the shift rhs reads B^i, the metric rhs A_ij), or -1.
__host__ __device__ constexpr int group_extra(int v) {
  return v >= BETAX && v <= BETAX + 2 ? DTSFX + (v - BETAX) : (v >= DXX && v <= DZZ ? AXX + (v - DXX) : -1);
}

// Pointers into LDS (32-bit local addresses; generic pointers would make
// every stencil offset a 64-bit flat address).
typedef __attribute__((address_space(3))) double lds_double;

// Tile row of a thread's row index r (of TY): with 8 rows a 16-lane LDS
// access group can hold rows y and y + 4, whose 14-double pitch puts them
// 112 dwords apart (16 mod 32 banks).
__host__ __device__ constexpr int tile_row(int r, int TY) { return TY == 8 ? ((r & 1) ? 4 + (r >> 1) : (r >> 1)) : r; }

// The LDS layout of one field's halo tile.  The direct loads move 16-byte
// aligned chunks, so an element's LDS index and its index in the array (plus
// the array's own offset from 16 bytes, LdsEnv::odd_base) must have the same
// parity throughout the tile.
//  EVEN row pitch of the arrays: rows of TX + 6 doubles, planes without gaps
//    (rows start at an even x, and so does every chunk).
//  ODD pitch: rows one double longer (elements x = -1 .. TX + 5; -1 is padding
//    whose chunk may hold it and x = 0), planes of an even pitch with room for
//    one more; where the arrays' plane pitch is odd too, odd planes start one
//    double later.  A sub-step of 85^3 points takes 376 us on 8x8x8 tiles and
//    311 on 32x4x4 ones, which lds_tile_shape picks there (the direct kernel,
//    which took odd pitches before, about 650); 8x8x8 tiles filled by 4-byte
//    loads spilled scalar registers (730 us with the residuals).
// LDS banks: a ds_read_b64 serves 16 lanes at a time.  Rows of 16 points or
// more need no care; an 8-point row pairs with one 16 banks away: row y + 4
// (EVEN, tile_row), or the same row of plane z + 1 (ODD: planes of 216
// doubles, a wave of 8 x 4 x 2 points).
template <int TX, int TY, int TZ, bool ODD = false>
struct LdsTile {
  static constexpr int LX = TX + 6, LY = TY + 6, LZ = TZ + 6;
  static constexpr int PY = ODD ? LX + 1 : LX;  // LDS pitches
  static constexpr int PZ = !ODD ? LX * LY : (TX == 8 ? 216 : (PY * LY + 3) / 2 * 2);
  static constexpr int NCH = PZ * LZ / 2;  // 16-byte chunks
  static constexpr int NT = TX * TY * TZ;  // threads
  static constexpr int ROUNDS = (NCH + NT - 1) / NT;
  static constexpr int NPAD = 2 * ROUNDS * NT;  // doubles per buffer: whole rounds, no bounds branches
  static_assert(LX % 2 == 0, "tile rows must hold whole 16-byte chunks");
  static_assert(NT % 64 == 0, "whole waves");
  static_assert(!ODD || (PZ % 2 == 0 && PY * LY + 2 <= PZ && PZ * LZ < NPAD), "room for the shifts");
  static_assert(!ODD || TX >= 16 || (TX == 8 && TY == 8), "odd pitch: 8 x 8 rows or wide ones");

  // the tile point of thread tid
  __device__ __forceinline__ static void point(int tid, int& tx, int& ty, int& tz) {
    if (ODD && TX == 8) {
      tx = tid & 7;
      ty = ((tid >> 4) & 3) + 4 * ((tid >> 6) & 1);
      tz = ((tid >> 3) & 1) + 2 * (tid >> 7);
    } else {
      tx = tid % TX;
      ty = TX <= 8 ? tile_row((tid / TX) % TY, TY) : (tid / TX) % TY;
      tz = tid / (TX * TY);
    }
  }
  // its LDS index (ODD: sz is the arrays' plane pitch)
  __device__ __forceinline__ static int lds_index(int tx, int ty, int tz, int sz) {
    return (tx + 3) + PY * (ty + 3) + PZ * (tz + 3) + (ODD ? (sz & 1 & (tz + 3)) : 0);
  }
};

// Array access of the tile point (i, j, k): live inside the interior [.., hi),
// else clamped into it and storing nothing.
__device__ __forceinline__ BufIo tile_io(int i, int j, int k, int hx, int hy, int hz, int sy, int sz, int n,
                                         bool& live) {
  live = i < hx && j < hy && k < hz;
  const unsigned vo = (unsigned)(min(i, hx - 1) + min(j, hy - 1) * sy + min(k, hz - 1) * sz) * 8u;
  return BufIo{vo, live ? vo : kDropStore, (unsigned)n * 8u};
}

#ifndef AMSS_LDS_FENCE
#define AMSS_LDS_FENCE 1
#endif
// LDS tile buffers per workgroup: two pairs (two field groups per barrier).
constexpr int kLdsBuffers = 4;

// Doubles of the epilogue's stash (LdsRk4) behind a kernel's tile buffers of
// npad doubles each, for workgroups of `points` threads: 6 per thread, or none
// where the workgroups of one CU (2 waves per SIMD: 512 threads) would then
// not fit its 160 KB (the 8x8x4 tiles of odd pitches).
constexpr int lds_stash(int points, int npad) {
  return (512 / points) * (kLdsBuffers * npad + 6 * points) * 8 <= 160 * 1024 ? 6 * points : 0;
}

// When a pair's two halo tiles are issued, one pair ahead: the first at the
// barrier and the second with the second group (1), both with the second group
// (2).  Self::kDmaAt says; 1 by default.
template <class S, class = void>
struct DmaAt {
  static constexpr int v = 1;
};
template <class S>
struct DmaAt<S, std::void_t<decltype(S::kDmaAt)>> {
  static constexpr int v = S::kDmaAt;
};
// Self: a type deriving from this environment and from the RK4 epilogue,
// whose prefetch(v0, v1) the environment calls for each pair (void: none).
template <int TX, int TY, int TZ, class FI = FieldsIn, class Self = void, bool ODD = false>
struct LdsEnv {
  static constexpr bool kFence = AMSS_LDS_FENCE;
  using T = LdsTile<TX, TY, TZ, ODD>;
  static constexpr long SY = T::PY, SZ = T::PZ;

  const FI& F;
  const FI& M;
  const Coef& C;
  lds_double* buf0;   // two pairs of LDS tile buffers (2 x NPAD doubles each)
  lds_double* buf1;
  BufIo at_p;     // this thread's point (clamped into the interior) in the arrays
  int lt;         // LDS index of this thread's point
  int gbase;      // global index of tile element (0,0,0)
  int sy, sz;     // global strides
  int gmax;       // number of points of one field
  int tid;        // thread index in the workgroup
  int plane = 0;  // ODD: the point's plane in the tile, halo included
  // ODD: LDS indices of the point in the open group's tile, and the base of
  // reads an odd number of planes away (the odd planes' shift)
  int ltc = 0, ltz = 0;
  int g = 0;      // next group to open
  bool bad = false;  // a NaN among the centre values of the first 21 fields (bssn_rhs.f90:110-113)
  double top[NFIELD];  // centre values the algebra reads before its first group (in_top)
  int xf[2] = {-1, -1}, nxf[2] = {-1, -1};  // group_extra of the open (next) pair's fields
  double xv[2], nxv[2];                      // ... and their centre values, loaded a pair ahead

  // Stream the halo tile of field v into buffer b by direct global->LDS
  // loads.  The buffer is padded to whole rounds, so chunks past the tile
  // land in the padding and the loop has no bounds branches -- branches here
  // split the point kernel into many blocks and wreck its register
  // allocation.  Addresses outside the array (the front and end corners, and
  // the part of a partial tile past the interior's halo, which no live point
  // reads) are clamped to valid ones.
  __device__ __forceinline__ void issue(int v, lds_double* b) const {
    const auto base = F.ptr(v);
    const int wave = tid >> 6;
    const int ob = odd_base(v);
#pragma unroll
    for (int r = 0; r < T::ROUNDS; ++r) {
      const int c = r * T::NT + tid;
      const int e = 2 * c;
      int gi;
      if constexpr (ODD) {
        const int z = e / T::PZ, t = e - z * T::PZ + 1 - (sz & 1 & z) - ob, y = t / T::PY, x = t - y * T::PY - 1;
        gi = gbase + x + y * sy + z * sz;  // of e's parity: a clamped index keeps it
        gi = min(max(gi, gi & 1), gmax - 2 - ((gi ^ gmax) & 1));
      } else {
        const int x = e % T::LX, y = (e / T::LX) % T::LY, z = e / (T::LX * T::LY);
        gi = gbase + x + y * sy + z * sz;  // < 2^29 points per field
        gi = min(max(gi, 0), gmax - 2);
      }
      __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(base + gi),
                                       (__attribute__((address_space(3))) void*)(b + 2 * (r * T::NT + wave * 64)),
                                       16, 0, 0);
    }
  }
  // ODD: 1 where the tile's first element lies on the second half of a
  // 16-byte chunk of field v; its LDS image then starts at index 1.
  __device__ __forceinline__ int odd_base(int v) const {
    return ODD ? (int)(((uintptr_t)F.ptr(v) >> 3) + (unsigned)gbase) & 1 : 0;
  }
  // Groups are staged two at a time: groups 2q and 2q+1 share pair q & 1,
  // so a tile needs one barrier per two field groups.
  __device__ __forceinline__ lds_double* slot(int grp) const {
    return (((grp >> 1) & 1) ? buf1 : buf0) + (grp & 1) * T::NPAD;
  }
  __device__ __forceinline__ lds_double* cur() const { return slot(g - 1); }  // g already advanced

  // Centre values a pair needs from global memory, loaded one pair ahead
  // (into the n* slots; rotate makes them current at the pair's barrier).
  __device__ __forceinline__ void ahead(int g0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      nxf[h] = group_extra(group_field(g0 + h));
      if (nxf[h] >= 0) nxv[h] = at_p.ld(F.ptr(nxf[h]));
    }
    if constexpr (!std::is_void_v<Self>) static_cast<Self*>(this)->prefetch(group_field(g0), group_field(g0 + 1));
  }
  __device__ __forceinline__ void rotate() {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xf[h] = nxf[h];
      xv[h] = nxv[h];
      nxf[h] = -1;
    }
    if constexpr (!std::is_void_v<Self>) static_cast<Self*>(this)->sink_rotate();
  }

  // the centre values bssn_rhs_point reads before it opens a group
  __device__ __forceinline__ static constexpr bool in_top(int v) {
    return v == CHI || v == TRK || v == LAP || (v >= DXX && v <= AZZ) || (v >= BETAX && v <= BETAX + 2);
  }
  __device__ __forceinline__ void prologue() {
#pragma unroll
    for (int v = 0; v < NFIELD; ++v)
      if (in_top(v)) top[v] = at_p.ld(F.ptr(v));
    ahead(0);
    __builtin_amdgcn_sched_barrier(0);
    issue(group_field(0), slot(0));
    issue(group_field(1), slot(1));
  }
  __device__ __forceinline__ void begin(int v) {
    constexpr int kAt = DmaAt<Self>::v;
    if ((g & 1) == 0) {
      __builtin_amdgcn_s_waitcnt(0);  // this wave's DMA of groups g, g+1 (and everything else) landed
      __syncthreads();                // ... for every wave; and the readers of groups g-2, g-1 are done
      rotate();
      if (g + 2 < NFIELD) ahead(g + 2);
      __builtin_amdgcn_sched_barrier(0);
      if (kAt < 2 && g + 2 < NFIELD) issue(group_field(g + 2), slot(g + 2));
    } else if (g + 1 < NFIELD) {
      // the next pair's halo loads start with the pair's second group
      __builtin_amdgcn_sched_barrier(0);
      if (kAt > 1) issue(group_field(g + 1), slot(g + 1));
      issue(group_field(g + 2), slot(g + 2));
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!std::is_void_v<Self>) static_cast<Self*>(this)->sink_flush();
    ++g;
    if constexpr (ODD) {
      ltc = lt + odd_base(v);
      ltz = ltc + (sz & 1) - 2 * (sz & 1 & plane);
    }
    if (v < 21) {
      const double x = at(v, 0);
      bad |= !(x == x);
    }
  }
  __device__ __forceinline__ void end() const {}

  __device__ __forceinline__ double at(int, long o) const {
    if constexpr (ODD) {
      const long dz = (o + 4 * SZ + SZ / 2) / SZ - 4;  // a constant, as o is
      return cur()[((dz & 1) ? ltz : ltc) + o];
    } else {
      return cur()[lt + o];
    }
  }
  // the centre value of the open group's field is in its halo tile; the
  // pair's extra centre values were loaded at its barrier
  __device__ __forceinline__ double val(int v) const {
    if (g == 0 && in_top(v)) return top[v];
    if (g > 0 && v == group_field(g - 1)) return at(v, 0);
    if (v == xf[0]) return xv[0];
    if (v == xf[1]) return xv[1];
    return at_p.ld(F.ptr(v));
  }
  __device__ __forceinline__ double mat(int m) const { return at_p.ld(M.ptr(m)); }

  __device__ __forceinline__ double d1(int v, long s) const {
    return (at(v, -2 * s) - at(v, 2 * s)) + 8.0 * (at(v, s) - at(v, -s));
  }
  __device__ __forceinline__ void grad(int v, double d[3]) const {
    d[0] = C.d1[0] * d1(v, 1);
    d[1] = C.d1[1] * d1(v, SY);
    d[2] = C.d1[2] * d1(v, SZ);
  }
  __device__ __forceinline__ double row(int v, long o, long s) const {
    return (at(v, o - 2 * s) - at(v, o + 2 * s)) + 8.0 * (at(v, o + s) - at(v, o - s));
  }
  __device__ __forceinline__ double mix(int v, long sa, long sb) const {
    return (row(v, -2 * sb, sa) - row(v, 2 * sb, sa)) + 8.0 * (row(v, sb, sa) - row(v, -sb, sa));
  }
  __device__ __forceinline__ void hess(int v, double d[6]) const {
    const double c = 30.0 * at(v, 0);
    d[0] = C.d2[0] * (16.0 * (at(v, -1) + at(v, 1)) - (at(v, -2) + at(v, 2)) - c);
    d[3] = C.d2[1] * (16.0 * (at(v, -SY) + at(v, SY)) - (at(v, -2 * SY) + at(v, 2 * SY)) - c);
    d[5] = C.d2[2] * (16.0 * (at(v, -SZ) + at(v, SZ)) - (at(v, -2 * SZ) + at(v, 2 * SZ)) - c);
    d[1] = C.dm[0] * mix(v, 1, SY);
    d[2] = C.dm[1] * mix(v, 1, SZ);
    d[4] = C.dm[2] * mix(v, SY, SZ);
  }
  __device__ __forceinline__ double up1(int v, long s, double b, double c) const {
    const double f0 = 10.0 * at(v, 0);
    const double up = (at(v, 3 * s) - 3.0 * at(v, -s)) + (18.0 * at(v, s) - 6.0 * at(v, 2 * s)) - f0;
    const double dn = (at(v, -3 * s) - 3.0 * at(v, s)) + (18.0 * at(v, -s) - 6.0 * at(v, -2 * s)) - f0;
    return c * (fmax(b, 0.0) * up - fmin(b, 0.0) * dn);
  }
  // the two one-sided stencils of every direction, unscaled (adjoint use)
  __device__ __forceinline__ void updn(int v, double up[3], double dn[3]) const {
    const long st[3] = {1, SY, SZ};
    const double f0 = 10.0 * at(v, 0);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const long s = st[a];
      up[a] = (at(v, 3 * s) - 3.0 * at(v, -s)) + (18.0 * at(v, s) - 6.0 * at(v, 2 * s)) - f0;
      dn[a] = (at(v, -3 * s) - 3.0 * at(v, s)) + (18.0 * at(v, -s) - 6.0 * at(v, -2 * s)) - f0;
    }
  }
  __device__ __forceinline__ double adv(int v, double, const double b[3]) const {
    return up1(v, 1, b[0], C.d1[0]) + up1(v, SY, b[1], C.d1[1]) + up1(v, SZ, b[2], C.d1[2]);
  }
  __device__ __forceinline__ double ko1(int v, long s, double c20) const {
    return (at(v, -3 * s) + at(v, 3 * s)) - 6.0 * (at(v, -2 * s) + at(v, 2 * s)) +
           15.0 * (at(v, -s) + at(v, s)) - c20;
  }
  __device__ __forceinline__ double ko(int v) const {
    const double c20 = 20.0 * at(v, 0);
    return C.ko[0] * ko1(v, 1, c20) + C.ko[1] * ko1(v, SY, c20) + C.ko[2] * ko1(v, SZ, c20);
  }
};

// The LDS environment and the RK4 epilogue as one object (passed to the point
// algebra as both), so the environment can hand the epilogue its prefetches.
// The last put's stores wait for the next group boundary, where the
// environment calls sink_flush after its barrier -- a store issued just before
// a barrier would be waited for there (its s_waitcnt(0) waits for every memory
// operation), one issued after it has a group's computation to land: 37
// patches 20.63 -> 20.47 ms, 128^3 +0.9%.  Sub-step 3, one store per field,
// gains nothing.
// DMA: when the halo tiles are issued (DmaAt).  The single-patch kernel's
// correctors issue both late: sub-steps 1-3 of 128^3 points 951 / 921 / 779 ->
// 927 / 899 / 770 us; sub-step 0 with the residuals loses by it (1,066 ->
// 1,151), and so do the tile lists (18.1 -> 18.3 ms).
// Non-temporal traffic (WIDE_NT, wide tiles): what a sub-step writes, and what
// a corrector reads of the old state and the accumulator, is not touched
// again before the next sub-step, and wide tiles are used on boxes of more than
// 262,144 points, whose 24 fields (50 MB) exceed the L2s; marked so, it leaves
// them to the halo tiles.
// The predictor's old state IS the field its halo tiles are filled from, so
// its loads stay plain.  128^3 points, sub-steps 0-3 (residuals in 0):
// 1081 / 932 / 906 / 768 -> 1014 / 916 / 892 / 764 us.  72^3 points on
// 8x8x8 tiles lose 0.7% by it.
// The six metric values that the epilogue keeps to the end wait in the
// workgroup's spare LDS (STASH) instead of in registers, where the compiler
// spilled them to scratch memory: 128^3 sub-steps 1 and 2 932 / 906 -> 893 / 869 us, 72^3
// 215 / 201 -> 206 / 189.
template <int STAGE, int TX, int TY, int TZ, class FI = FieldsIn, class FO = FieldsOut, class AX = AuxOut,
          bool ODD = false, int DMA = 1, bool WIDE_NT = false>
struct LdsRk4 : LdsEnv<TX, TY, TZ, FI, LdsRk4<STAGE, TX, TY, TZ, FI, FO, AX, ODD, DMA, WIDE_NT>, ODD>,
                Rk4SinkT<STAGE, FI, FO, AX, BufIoT<WIDE_NT && (STAGE > 0), WIDE_NT>> {
  using Io = BufIoT<WIDE_NT && (STAGE > 0), WIDE_NT>;
  using Sink = Rk4SinkT<STAGE, FI, FO, AX, Io>;
  static constexpr int kPoints = TX * TY * TZ;
  static constexpr bool kDefer = STAGE < 3;
  static constexpr bool kStash = STAGE < 3 && lds_stash(kPoints, LdsTile<TX, TY, TZ, ODD>::NPAD) > 0;
  static constexpr int kDmaAt = DMA;
  lds_double* stash;  // this thread's first slot, slots kPoints apart (kStash)
  int dv = -1;
  double dacc, dout;
  __device__ __forceinline__ void sink_rotate() { Sink::rotate(); }
  __device__ __forceinline__ void prefetch(int v0, int v1) { Sink::prefetch(v0, v1); }
  __device__ __forceinline__ void sink_flush() {
    if (!kDefer || dv < 0) return;
    if (STAGE < 3) Sink::io.st(Sink::ACC.ptr(dv), dacc);
    if (!(STAGE < 3 && dv >= DXX && dv <= AZZ)) Sink::io.st(Sink::OUT.ptr(dv), dout);
    dv = -1;
  }
  __device__ __forceinline__ void put(int v, double k) {
    if (!kDefer) {
      Sink::put(v, k);
      return;
    }
    double u0v, av, accv, u;
    Sink::u0_acc(v, u0v, av);
    Sink::rk4_values(v, k, u0v, av, accv, u);
    sink_flush();  // an earlier put since the last boundary
    dv = v;
    dacc = accv;
    if (kStash && v >= DXX && v <= DZZ)
      stash[(v - DXX) * kPoints] = u;
    else if (STAGE < 3 && v >= DXX && v <= AZZ)
      Sink::gA[v - DXX] = u;
    else
      dout = u;
  }
  __device__ __forceinline__ void finish() {
    sink_flush();
    if (kStash) {
#pragma unroll
      for (int s = 0; s < 6; ++s) Sink::gA[s] = stash[s * kPoints];
    }
    Sink::finish();
  }
};

}  // namespace amss
