// Shared definitions of the MI355X CGFDM library (device and host side).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include <cstdint>

namespace cg {

constexpr int H = 3;  // ghost layers on every side of the local domain (reference macro.h:39)

// MacCormack one-sided coefficients (reference macro.h:121-125) and the 3-point
// one-sided stencil one layer under the surface (macro.h:144-146).
constexpr double AF_1 = -0.30874, AF0 = -0.6326, AF1 = 1.2330, AF2 = -0.3334, AF3 = 0.04168;
constexpr double CF1 = -1.16666667, CF2 = 1.33333333, CF3 = -0.16666667;
// Classical RK4 written on (W, t, m) buffers (macro.h:133-142).
constexpr double RK_A2 = 0.5, RK_A3 = 0.5;
constexpr double RK_B1 = 0.16666667, RK_B2 = 0.33333333, RK_B3 = 0.33333333, RK_B4 = 0.16666667;

// Storage type of metric and medium coefficients.
template <class T> struct Store;
template <> struct Store<float> {
  static __device__ __forceinline__ float ld(const float* p) { return *p; }
};
template <> struct Store<double> {
  static __device__ __forceinline__ double ld(const double* p) { return *p; }
};
template <> struct Store<__half> {
  static __device__ __forceinline__ float ld(const __half* p) { return __half2float(*p); }
};
template <> struct Store<__hip_bfloat16> {
  static __device__ __forceinline__ float ld(const __hip_bfloat16* p) { return __bfloat162float(*p); }
};

// 16-bit coefficient storage (fp16 / bf16): the twelve coefficient planes are
// stored in pairs (c = 2q, 2q + 1) as one 32-bit word per cell (code of plane
// 2q in the low half), and each 16-bit value is an affine code over its
// (plane, k) layer: value = mid[c][k] + half[c][k] * code, code in [-1, 1],
// with (mid, half) the centre and half-width of the layer's value range in a
// float table aff[c][k][2]. A layer whose values are all equal is stored
// exactly; otherwise the rounding error is bounded by half * 2^-11 (fp16) or
// half * 2^-8 (bf16) instead of |value| times that.
template <class T> struct Bits16;
template <> struct Bits16<__half> {
  static __device__ __forceinline__ float to_float(unsigned short b) { return __half2float(__ushort_as_half(b)); }
};
template <> struct Bits16<__hip_bfloat16> {
  static __device__ __forceinline__ float to_float(unsigned short b) { return __uint_as_float((unsigned)b << 16); }
};

// Coefficient planes, SoA over the padded grid. Metrics are stored as the
// unit-free products m * DH (i.e. divided by rDH) only when `scaled` is set;
// the default keeps the reference meaning (xi_x ... zt_z in 1/m).
enum { M_XIX = 0, M_XIY, M_XIZ, M_ETX, M_ETY, M_ETZ, M_ZTX, M_ZTY, M_ZTZ, M_MU, M_LAM, M_B, M_NCOEF };

// One PML face slab (reference pml_deriv.cpp:17-37): three RK buffers of 9 SoA
// components over `cnt` cells. a = state at the step start (and the final
// state); x1, x2 = the stage states, each in place of an earlier one (pml_face).
template <class R>
struct FaceBuf {
  R* a;
  R* x1;
  R* x2;
  long long cnt;
};

template <class R>
struct PmlArgs {
  int npml;
  int has_z2;         // bottom-only PML in z when a free surface is present
  const R* alpha[3];  // per axis, padded length
  const R* beta[3];   // inverted beta (1 outside the PML)
  const R* d[3];      // d / beta
  FaceBuf<R> f[6];    // x1, y1, z1, x2, y2, z2
};

// Access at a byte offset from a uniform base pointer: the compiler emits the
// global load/store form with a 64-bit SGPR base and a 32-bit VGPR offset, so
// one offset register serves every plane of every grid array (field, RK,
// coefficient). Every grid plane array spans less than 4 GiB (checked on the
// host before a launch), so byte offsets of cells fit 32 bits.
template <class T>
__device__ __forceinline__ const T* at(const T* base, unsigned boff) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + boff);
}
template <class T>
__device__ __forceinline__ T* at(T* base, unsigned boff) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + boff);
}

// XCD-aware block order of the interior launch. The hardware hands block b to
// XCD b % 8, so block b is the (b / 8)-th block that XCD runs. The (x, y) plane
// is cut into regions of rtx 64-column tiles by rty 4-row tiles (rtx <= 0 or
// larger than the row: whole rows, so that no region is a partial column); regions are
// dealt to the XCDs in turn and each XCD walks its regions one after another,
// plane by plane in k and, within a plane, row of tiles by row of tiles. The
// x, y and z stencil neighbours of a cell are then read by blocks of the same
// XCD a few planes earlier or later and come from that XCD's L2 instead of
// HBM, except across region edges, which the XCDs reach at about the same time.
// The last regions, fewer than eight, are taken as one sequence of blocks of which
// each XCD gets an eighth: dealt whole they leave XCDs idle (333 x 150 x 117 has 19
// regions: 1.64 ms per step dealt whole and 1.41 so; FP64 200 x 180 x 100 2.21 and 2.15;
// the whole range cut into eighths costs the shared edges: 512 x 512 x 256 14.0 and
// 14.8). Returns false for padding blocks.
//
// A last tile column of at most 32 cells, in regions of whole rows, goes in blocks
// of 32 columns by 8 rows: a wave takes two rows of it instead of one with half its
// lanes idle (nx 150: 5 blocks where 6 were; 200: 7 for 8; 333: 11 for 12).
struct CellTile {
  int i, j, k;  // of the thread, from the first cell of the range
};
__device__ __host__ __forceinline__ int region_extent(int r, int n) { return (r <= 0 || r > n) ? n : r; }
// blocks of a region's plane: whole tiles, and those of the narrow last column
__device__ __host__ __forceinline__ void region_blocks(int nx, int ntx, int rtx, int rty, int& wide, int& narrow) {
  const int r = nx % 64;
  const bool has = rtx == ntx && r > 0 && r <= 32;
  wide = (has ? rtx - 1 : rtx) * rty;
  narrow = has ? (rty + 1) / 2 : 0;
}

__device__ __forceinline__ bool interior_tile(int b, int nx, int ny, int nk, int rtx, int rty, CellTile& t) {
  const int ntx = (nx + 63) / 64, nty = (ny + 3) / 4;
  rtx = region_extent(rtx, ntx);  // rtx <= 0: whole rows of tiles
  rty = region_extent(rty, nty);
  const int nrx = (ntx + rtx - 1) / rtx, nry = (nty + rty - 1) / rty;
  int wide, narrow;
  region_blocks(nx, ntx, rtx, rty, wide, narrow);
  const int per_plane = wide + narrow;
  const unsigned per_region = (unsigned)(per_plane * nk);  // the launch has fewer than 2^31 blocks
  const int nreg = nrx * nry;
  const unsigned xcd = (unsigned)b & 7u, seq = (unsigned)b >> 3, whole = (unsigned)(nreg / 8) * per_region;
  int r;
  unsigned within;
  if (seq < whole) {
    r = (int)(seq / per_region * 8u + xcd);
    within = seq % per_region;
  } else {
    const unsigned s = xcd * (((unsigned)(nreg % 8) * per_region + 7u) / 8u) + (seq - whole);
    r = nreg / 8 * 8 + (int)(s / per_region);
    within = s % per_region;
  }
  if (r >= nreg) return false;
  const int kk = (int)within / per_plane, q = (int)within - kk * per_plane;
  const int rx = r % nrx, ry = r / nrx;
  int row;  // in the region
  if (q < wide) {
    const int w = narrow ? rtx - 1 : rtx, ty = q / w;
    t.i = (rx * rtx + q - ty * w) * 64 + (int)(threadIdx.x & 63);
    row = 4 * ty + (int)(threadIdx.x >> 6);
  } else {
    t.i = (ntx - 1) * 64 + (int)(threadIdx.x & 31);
    row = 8 * (q - wide) + (int)(threadIdx.x >> 5);
  }
  t.j = 4 * rty * ry + row;
  t.k = kk;
  return row < 4 * rty && t.i < nx && t.j < ny;
}

// number of blocks of the interior launch for interior_tile()
inline long long interior_blocks(int nx, int ny, int nk, int rtx, int rty) {
  const int ntx = (nx + 63) / 64, nty = (ny + 3) / 4;
  rtx = region_extent(rtx, ntx);
  rty = region_extent(rty, nty);
  const long long nregions = (long long)((ntx + rtx - 1) / rtx) * ((nty + rty - 1) / rty);
  int wide, narrow;
  region_blocks(nx, ntx, rtx, rty, wide, narrow);
  const long long per_region = (long long)(wide + narrow) * nk;
  return 8 * (nregions / 8 * per_region + (nregions % 8 * per_region + 7) / 8);
}

}  // namespace cg
