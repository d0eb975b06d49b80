// Kernel argument blocks and launcher declarations of the CGFDM step.
#pragma once
#include "common.h"

namespace cg {

template <class R>
struct StageArgs {
  int nx, ny, nz;       // interior cells
  int NX, NY;           // padded x/y extents
  long long N;          // padded cells per field
  long long S;          // NX * NY
  unsigned rowb, planeb;  // NX and S in bytes of one grid element (R); N * sizeof(R) < 4 GiB
  int kbeg, kend;       // k range of the interior kernel [kbeg, kend)
  int stage;            // RK4 stage 0..3
  int rtx, rty;         // interior block order: regions of (64 rtx) x (4 rty) columns per XCD
  int kc;               // > 0: z-marching interior kernel with chunks of kc planes
  int zty;              // z-marching tile height: 8 (512 threads) or 4 (256 threads)
  int zreg;             // > 0: register z-marching interior kernel with chunks of zreg planes
  R DT, rDH;
  const float* aff;     // 16-bit coefficient storage: affine table [12][NZ][2] (mid, half); else unused
  int nzp;              // padded z extent (rows of the affine table)
  const R* win;         // stencil input (9 SoA fields)
  const R* wm;          // RK base (state at the start of the step; the last stage's output)
  const R* x1;          // states of stages 1 and 2, read by the last stage
  const R* x2;
  R* wout;              // stage output
  PmlArgs<R> pml;
};

template <class R>
struct SurfArgs {
  const R* jac;         // Jacobian, padded grid
  const R* rdzdx;       // 9 planes [NY][NX]: -DZ^-1 DX on the surface
  const R* rdzdy;       // 9 planes [NY][NX]: -DZ^-1 DY
  float* pgv;           // [ny][nx][2] or nullptr (updated on stage 3)
  R* dis;               // surface displacement, 3 planes [NY][NX]
};

// launcher results: nothing is launched unless LAUNCH_OK; LAUNCH_EMPTY means
// there is nothing to do (an empty k range), the others are caller errors
constexpr int LAUNCH_OK = 0;
constexpr int LAUNCH_EMPTY = 1;       // empty range: no launch needed
constexpr int LAUNCH_BAD_STAGE = 2;   // RK stage outside 0..3
constexpr int LAUNCH_TOO_LARGE = 3;   // grid beyond the launch limits (2^31 - 1 blocks, 65535 in y)

template <class R, class TM>
int launch_interior(StageArgs<R> a, const TM* coef, int fb1, int fb2, int fb3, hipStream_t st);
template <class R, class TM>
int launch_surface(StageArgs<R> a, const TM* coef, SurfArgs<R> s, int fb1, int fb2, int fb3, hipStream_t st);
template <class R, class TM>
int launch_stage(StageArgs<R> a, const TM* coef, SurfArgs<R> s, int fb1, int fb2, int fb3, hipStream_t st);
// Interior and surface blocks of a stage under a free surface where launch_stage takes
// them in one launch (cg_stage), else 0. FP32: up to 1024 blocks, twice what the 256
// CUs hold at two blocks each (the registers of the surface part); the surface
// first and the interior after it otherwise. us per step in two launches and in one:
// 24 x 20 x 16 (80 blocks) 78 and 48, 64 x 60 x 40 (600) 113 and 87, 64 x 64 x 62 (992)
// 128 and 99; above the line still 172 and 158 at 2000 blocks, with the gain falling.
// FP64 would need more registers than there are for two blocks.
template <class R>
inline long long one_launch_blocks(const StageArgs<R>& a) {
  const int nk = a.kend - a.kbeg;
  if (sizeof(R) != 4 || a.kc != 0 || a.zreg != 0 || a.stage < 0 || a.stage > 3 || nk <= 0 || a.nx <= 0 || a.ny <= 0)
    return 0;
  const long long nb = 3LL * ((a.nx + 63) / 64) * ((a.ny + 3) / 4) +
                       interior_blocks(a.nx, a.ny, nk, a.rtx, a.rty < 1 ? 1 : a.rty);
  return nb <= 1024 ? nb : 0;
}
template <class R>
void launch_source(R* W, long long N, int np, const long long* cell, const R* rate, int srcIt, R tw, R DT, hipStream_t st);
template <class R>
void launch_record(const R* W, long long N, int ns, const long long* cell, float* rec, int nt, int it, hipStream_t st);

}  // namespace cg
