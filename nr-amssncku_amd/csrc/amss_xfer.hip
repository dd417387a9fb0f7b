// amss_xfer.hip -- inter-level transfer between 2:1 cell-centred grids: the
// 6-point, 5th-order prolongation (coarse -> fine) and restriction (fine ->
// coarse) of prolongrestrict_cell.f90 (Cell, ghost_width 3; prolong3
// :1915-2164, restrict3 :2330-2468), on LDS-staged tiles of target cells.
#include "amss_xfer.h"

#include <cmath>

namespace amss {

// Cell numbering of both grids from a common base point (:1958-1990): the
// reference rounds (x - base) / h + 0.4 toward zero, 0.4 being a
// single-precision literal.
static inline int cell_index(double x, double base, double h) {
  return (int)((x - base) / h + (double)0.4f);
}

int xfer_plan(const double* llbc, const double* uubc, const int* extc, const double* llbf, const double* uubf,
              const int* extf, const double* ll, const double* uu, bool prolong, XferPlan& P) {
  double CD[3], FD[3], base[3];
  for (int a = 0; a < 3; ++a) {
    if (extc[a] < 1 || extf[a] < 1) return 2;
    CD[a] = (uubc[a] - llbc[a]) / extc[a];
    FD[a] = (uubf[a] - llbf[a]) / extf[a];
    if (std::fabs(CD[a] - 2 * FD[a]) > 1e-10) return 2;  // not 2:1 (the reference stops)
    // a fine box starting inside a coarse cell shifts the base by half a
    // coarse cell when it starts on an odd fine cell (:1965-1977)
    if (llbc[a] <= llbf[a]) {
      base[a] = llbc[a];
    } else {
      const int j = cell_index(llbc[a], llbf[a], FD[a]);
      base[a] = (j % 2 == 0) ? llbf[a] : llbf[a] - CD[a] / 2;
    }
  }
  for (int a = 0; a < 3; ++a) {
    P.ext_c[a] = extc[a];
    P.ext_f[a] = extf[a];
    P.lbf[a] = cell_index(llbf[a], base[a], FD[a]) + 1;
    P.lbc[a] = cell_index(llbc[a], base[a], CD[a]) + 1;
    const double ht = prolong ? FD[a] : CD[a], hs = prolong ? CD[a] : FD[a];
    const int lt = cell_index(ll[a], base[a], ht) + 1, ut = cell_index(uu[a], base[a], ht);
    const int ls = cell_index(ll[a], base[a], hs) + 1, us = cell_index(uu[a], base[a], hs);
    const int tl = prolong ? P.lbf[a] : P.lbc[a], sl = prolong ? P.lbc[a] : P.lbf[a];
    const int nt = prolong ? extf[a] : extc[a], ns = prolong ? extc[a] : extf[a];
    // target range, 1-based; the reference's sanity test on both ranges
    // (:2001-2021, 2416-2427)
    P.lo[a] = lt - tl + 1;
    P.hi[a] = ut - tl + 1;
    if (P.lo[a] < 1 || ls - sl + 1 < 1 || P.hi[a] > nt || us - sl + 1 > ns - 2) return 1;
  }
  for (int a = 0; a < 3; ++a)
    if (P.hi[a] < P.lo[a]) return 0;  // an empty region: nothing to do
  for (int a = 0; a < 3; ++a) {
    const int ns = prolong ? extc[a] : extf[a];
    // every stencil inside the source and its mirrored halo (prolong:
    // funcc(-2:extc), restrict: funff(-1:extf)); the reference only
    // prints a warning there and reads outside its arrays
    const int c0 = prolong ? (P.lo[a] + P.lbf[a] - 1) / 2 - P.lbc[a] + 1 : 2 * (P.lo[a] + P.lbc[a] - 1) - P.lbf[a];
    const int c1 = prolong ? (P.hi[a] + P.lbf[a] - 1) / 2 - P.lbc[a] + 1 : 2 * (P.hi[a] + P.lbc[a] - 1) - P.lbf[a];
    if (c0 < (prolong ? 0 : 1) || c1 + 3 > ns) return 1;
  }
  return 0;
}

// Both transfers work on tiles of target cells and factorize the 6x6x6
// contraction along z, then y, then x (the reference's summation order).  A
// thread takes a whole column of the source block in z -- all its loads in
// flight together, coalesced along x -- and forms the tile's values along z
// from registers; y and x follow through LDS the same way.  Bound by the
// latency of one such round trip per tile (an 8-16 deep chain of loads, two
// barriers) and by the launch, not by bytes: the earlier kernels staged the
// block in LDS in a loop whose every load waited.  Over 24 fields in turn a
// 134^3 fine array takes 12.9 us (36 before; its 9 bytes a cell 3.8 us at the
// rate of a copy), 61^3 coarse cells 11.4 us (28); the same arrays again and
// again, 11.0 us and (62^3 cells) 8.5.
// blockIdx.y is the field, blockIdx.x a tile of one of the regions.
// Source cells past what the valid target cells read are clamped or skipped;
// cells past the end of the target range are not stored.
constexpr double kProW[6] = {77.0 / 8192.0, -693.0 / 8192.0, 3465.0 / 4096.0,
                             1155.0 / 4096.0, -495.0 / 8192.0, 63.0 / 8192.0};
constexpr double kResW[3] = {3.0 / 256.0, -25.0 / 256.0, 75.0 / 128.0};

namespace {

// A column of the source at 1-based (i, j), cells k0, k0 + 1, ... (at most
// kmax): symmetry_bd's mirror below 1 (q -> 1 - q with the parity of each
// mirrored axis, fmisc.f90:877-901).
template <int N>
__device__ __forceinline__ void load_column(const XferField& F, int n0, int n1, int i, int j, int k0, int kmax,
                                            double (&c)[N]) {
  double s = 1.0;
  if (i < 1) { i = 1 - i; s *= F.S[0]; }
  if (j < 1) { j = 1 - j; s *= F.S[1]; }
  const double* f = F.src + (i - 1) + (long)n0 * (j - 1);
  const long nz = (long)n0 * n1;
#pragma unroll
  for (int q = 0; q < N; ++q) {
    const int k = min(k0 + q, kmax);
    const double v = f[nz * (k < 1 ? -k : k - 1)];
    c[q] = v * (k < 1 ? s * F.S[2] : s);
  }
}

// Fine values d = 0 .. 7 of a line whose first fine cell has an even (odd)
// global index, from coarse values c: cell d reads c[o .. o + 5], o = (ODD + d)
// / 2, with the weights in reverse order on odd cells.
template <bool ODD, int N>
__device__ __forceinline__ void prolong_line(const double (&c)[10], double (&f)[N]) {
#pragma unroll
  for (int d = 0; d < N; ++d) {
    const int g = ODD + d, o = g / 2;
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) s += kProW[(g & 1) ? 5 - q : q] * c[o + q];
    f[d] = s;
  }
}
template <int N>
__device__ __forceinline__ void prolong_line(bool odd, const double (&c)[10], double (&f)[N]) {
  if (odd) prolong_line<true, N>(c, f);
  else prolong_line<false, N>(c, f);
}

// the region of block b, and b's tile in it
__device__ __forceinline__ const XferPlan& xfer_region(const XferBatch& X, int& b) {
  int r = 0;
  while (r + 1 < X.nregion && b >= X.first[r + 1]) ++r;
  b -= X.first[r];
  return X.P[r];
}

}  // namespace

// prolong: fine tile 32 x 8 x 8.  Fine cell p reads coarse cells
// c(p) - 2 .. c(p) + 3, c(p) = (p + lbf - 1) / 2 - lbc + 1; over a tile of F
// cells c advances by at most F / 2, so F / 2 + 6 coarse cells cover it.
constexpr int kPFX = 32, kPFY = 8, kPFZ = 8;
constexpr int kPCX = kPFX / 2 + 6, kPCY = kPFY / 2 + 6;
static_assert(kPFY / 2 + 6 == 10 && kPFZ / 2 + 6 == 10, "prolong_line reads 10 coarse values");

__global__ void __launch_bounds__(256) prolong3_kernel(XferBatch X) {
  __shared__ double T1[kPFZ][kPCY][kPCX];
  __shared__ double T2[kPFZ][kPFY][kPCX];
  int b = blockIdx.x;
  const XferPlan& P = xfer_region(X, b);
  const XferField& F = X.f[blockIdx.y];
  const int T[3] = {kPFX, kPFY, kPFZ};
  int nt[3], p0[3], pe[3], c0[3], nc[3];
  bool odd[3];  // parity of the tile's first fine cell
  for (int a = 0; a < 3; ++a) nt[a] = (P.hi[a] - P.lo[a] + T[a]) / T[a];
  const int tb[3] = {b % nt[0], (b / nt[0]) % nt[1], b / (nt[0] * nt[1])};
  for (int a = 0; a < 3; ++a) {
    p0[a] = P.lo[a] + tb[a] * T[a];
    pe[a] = min(p0[a] + T[a] - 1, P.hi[a]);
    const int g = p0[a] + P.lbf[a] - 1;
    odd[a] = g & 1;
    c0[a] = g / 2 - P.lbc[a] + 1 - 2;  // first coarse cell of the block
    nc[a] = (pe[a] + P.lbf[a] - 1) / 2 - P.lbc[a] + 1 + 3 - c0[a] + 1;  // ... that the valid fine cells read
  }
  const int tid = threadIdx.x;
  if (tid < kPCX * kPCY) {
    const int x = tid % kPCX, y = tid / kPCX;
    if (x < nc[0] && y < nc[1]) {
      double c[10], f[kPFZ];
      load_column(F, P.ext_c[0], P.ext_c[1], c0[0] + x, c0[1] + y, c0[2], c0[2] + nc[2] - 1, c);
      prolong_line(odd[2], c, f);
#pragma unroll
      for (int d = 0; d < kPFZ; ++d) T1[d][y][x] = f[d];
    }
  }
  __syncthreads();
  if (tid < kPCX * kPFZ) {
    const int x = tid % kPCX, z = tid / kPCX;
    double c[10], f[kPFY];
#pragma unroll
    for (int q = 0; q < 10; ++q) c[q] = T1[z][q][x];
    prolong_line(odd[1], c, f);
#pragma unroll
    for (int d = 0; d < kPFY; ++d) T2[z][d][x] = f[d];
  }
  __syncthreads();
  const int fx = tid % kPFX, fy = tid / kPFX, g = (odd[0] ? 1 : 0) + fx, o = g / 2;
  const int i = p0[0] + fx, j = p0[1] + fy;
  if (i > pe[0] || j > pe[1]) return;
  double w[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) w[q] = (g & 1) ? kProW[5 - q] : kProW[q];
  double* out = F.dst + (i - 1) + (long)P.ext_f[0] * (j - 1);
  const long nz = (long)P.ext_f[0] * P.ext_f[1];
#pragma unroll
  for (int fz = 0; fz < kPFZ; ++fz) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 6; ++q) s += w[q] * T2[fz][fy][o + q];
    if (p0[2] + fz <= pe[2]) out[nz * (p0[2] + fz - 1)] = s;
  }
}

// restrict: coarse tile 16 x 4 x 4.  Coarse cell p reads fine cells
// f(p) - 2 .. f(p) + 3, f(p) = 2 (p + lbc - 1) - lbf; over a tile f advances
// by 2 per cell, so a block of 2 C + 4 fine cells per axis covers it.
constexpr int kRCX = 16, kRCY = 4, kRCZ = 4;
constexpr int kRFX = 2 * kRCX + 4, kRFY = 2 * kRCY + 4, kRFZ = 2 * kRCZ + 4;

template <int N>
__device__ __forceinline__ void restrict_line(const double (&f)[2 * N + 4], double (&c)[N]) {
#pragma unroll
  for (int d = 0; d < N; ++d)
    c[d] = kResW[0] * (f[2 * d] + f[2 * d + 5]) + kResW[1] * (f[2 * d + 1] + f[2 * d + 4]) +
           kResW[2] * (f[2 * d + 2] + f[2 * d + 3]);
}

__global__ void __launch_bounds__(256) restrict3_kernel(XferBatch X) {
  __shared__ double T1[kRCZ][kRFY][kRFX];
  __shared__ double T2[kRCZ][kRCY][kRFX];
  int b = blockIdx.x;
  const XferPlan& P = xfer_region(X, b);
  const XferField& F = X.f[blockIdx.y];
  const int T[3] = {kRCX, kRCY, kRCZ};
  int nt[3], p0[3], pe[3], f0[3], nf[3];
  for (int a = 0; a < 3; ++a) nt[a] = (P.hi[a] - P.lo[a] + T[a]) / T[a];
  const int tb[3] = {b % nt[0], (b / nt[0]) % nt[1], b / (nt[0] * nt[1])};
  for (int a = 0; a < 3; ++a) {
    p0[a] = P.lo[a] + tb[a] * T[a];
    pe[a] = min(p0[a] + T[a] - 1, P.hi[a]);
    f0[a] = 2 * (p0[a] + P.lbc[a] - 1) - P.lbf[a] - 2;  // first fine cell of the block
    nf[a] = 2 * (pe[a] - p0[a]) + 6;                    // ... that the valid coarse cells read
  }
  const int tid = threadIdx.x;
#pragma unroll
  for (int e = 0; e < kRFX * kRFY; e += 256) {
    const int x = (e + tid) % kRFX, y = (e + tid) / kRFX;
    if (x < nf[0] && y < nf[1]) {
      double f[kRFZ], c[kRCZ];
      load_column(F, P.ext_f[0], P.ext_f[1], f0[0] + x, f0[1] + y, f0[2], f0[2] + nf[2] - 1, f);
      restrict_line(f, c);
#pragma unroll
      for (int d = 0; d < kRCZ; ++d) T1[d][y][x] = c[d];
    }
  }
  __syncthreads();
  if (tid < kRFX * kRCZ) {
    const int x = tid % kRFX, z = tid / kRFX;
    double f[kRFY], c[kRCY];
#pragma unroll
    for (int q = 0; q < kRFY; ++q) f[q] = T1[z][q][x];
    restrict_line(f, c);
#pragma unroll
    for (int d = 0; d < kRCY; ++d) T2[z][d][x] = c[d];
  }
  __syncthreads();
  const int cx = tid % kRCX, cy = (tid / kRCX) % kRCY, cz = tid / (kRCX * kRCY);
  const double* v = &T2[cz][cy][2 * cx];
  const double r = kResW[0] * (v[0] + v[5]) + kResW[1] * (v[1] + v[4]) + kResW[2] * (v[2] + v[3]);
  const int i = p0[0] + cx, j = p0[1] + cy, k = p0[2] + cz;
  if (i <= pe[0] && j <= pe[1] && k <= pe[2])
    F.dst[(i - 1) + (long)P.ext_c[0] * ((j - 1) + (long)P.ext_c[1] * (k - 1))] = r;
}

static_assert(kRCX * kRCY * kRCZ == 256 && kPFX * kPFY == 256, "one target column or cell per thread");

// The tiles (of size T) of a batch's regions; empty regions give none.
static unsigned batch_tiles(XferBatch& X, const int T[3]) {
  int first = 0;
  for (int r = 0; r < X.nregion; ++r) {
    const XferPlan& P = X.P[r];
    int n = 1;
    for (int a = 0; a < 3; ++a) n *= P.hi[a] >= P.lo[a] ? (P.hi[a] - P.lo[a] + T[a]) / T[a] : 0;
    X.first[r] = first;
    first += n;
  }
  return (unsigned)first;
}

void launch_prolong3(XferBatch X, hipStream_t s) {
  const int T[3] = {kPFX, kPFY, kPFZ};
  const unsigned n = batch_tiles(X, T);
  if (n > 0 && X.nfield > 0) prolong3_kernel<<<dim3(n, X.nfield), 256, 0, s>>>(X);
}

void launch_restrict3(XferBatch X, hipStream_t s) {
  const int T[3] = {kRCX, kRCY, kRCZ};
  const unsigned n = batch_tiles(X, T);
  if (n > 0 && X.nfield > 0) restrict3_kernel<<<dim3(n, X.nfield), 256, 0, s>>>(X);
}

void launch_prolong3(const double* func, double* funf, const XferPlan& P, const double S[3], hipStream_t s) {
  XferBatch X;
  X.add(P);
  X.add(func, funf, S);
  launch_prolong3(X, s);
}

void launch_restrict3(const double* funf, double* func, const XferPlan& P, const double S[3], hipStream_t s) {
  XferBatch X;
  X.add(P);
  X.add(funf, func, S);
  launch_restrict3(X, s);
}

}  // namespace amss
