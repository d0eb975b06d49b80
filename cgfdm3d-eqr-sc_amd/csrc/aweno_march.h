// Marching form of the ME-AWENO stage for gfx950: the face fluxes stay in
// registers instead of going through a 27-plane array.
//
// A stage is two kernels over the cells below the top three layers:
//   aw_yflux   a wave of 64 x-adjacent columns of one plane marches along y and
//              leaves the eta flux difference in the stage's output buffer;
//   aw_xzstep  a wave of 64 x-adjacent columns of one row marches along z: zeta
//              fluxes from its registers, xi fluxes across its lanes, the TVD-RK3
//              combination; it replaces the eta difference by the stage's result.
// Per cell and stage 24 + 46 plane values move (37 in the first stage's second
// kernel) where the flux array costs 21 + 27 written and 27 + 28 read back.
//
// Marching also shares the reconstruction between faces. Everything a WENO5 face
// value needs is a property of a three-cell window: its second and centred first
// difference A and C, the three smoothness indicators 13 A^2 + 3 {2A + C, C,
// 2A - C}^2, the weights 1 / q^2, and its parabola at the faces -3/2, -1/2, 1/2
// and 3/2 cells from its centre. A window serves the minus side of three faces
// and the plus side of three, each weight twice: 3 + 2 reciprocals per face
// and field instead of 8, about 59 instruction slots instead of 102.
//
// MI355X, 320 x 300 x 200: 2.57 -> 1.61 ms per stage, 77.3 -> 48.3 ms per 10 steps.
// aw_yflux takes 0.43 ms (530 vector instructions per cell, of which 45 are
// reciprocals at a quarter of the rate), aw_xzstep 1.1 ms in the first stage and
// 1.2 in the others (1330 per cell, 90 of them reciprocals, on 54 of 64 lanes):
// both about 80 % bound by instruction issue.
#pragma once
#include "aweno_impl.h"

namespace aw {

// Window of centre w0 with neighbours wl, wr: scaled weights and face values.
// Indicators as in weno5_pair (times 12, eps 12e-6), linear weights (5, 10, 1) / 16.
struct Window {
  float aR, R5, C10, L, L5;  // 1/q^2 of the right, centred and left indicator, times the linear weights used
  float pLL, pL, pR, pRR;    // parabola at -3/2, -1/2, 1/2, 3/2
};
__device__ __forceinline__ Window window(float wl, float w0, float wr) {
  Window s;
  const float A = fmaf(-2.0f, w0, wl + wr), C = wl - wr;
  const float T = fmaf(13.0f * A, A, 12e-6f);
  const float ep = fmaf(2.0f, A, C), em = fmaf(2.0f, A, -C);
  const float qR = fmaf(3.0f * ep, ep, T), qC = fmaf(3.0f * C, C, T), qL = fmaf(3.0f * em, em, T);
  s.aR = __builtin_amdgcn_rcpf(qR * qR);
  const float aC = __builtin_amdgcn_rcpf(qC * qC);
  s.L = __builtin_amdgcn_rcpf(qL * qL);
  s.R5 = 5.0f * s.aR;
  s.C10 = 10.0f * aC;
  s.L5 = 5.0f * s.L;
  const float u1 = fmaf(0.125f, A, w0), u3 = fmaf(1.125f, A, w0);
  s.pL = fmaf(0.25f, C, u1);
  s.pR = fmaf(-0.25f, C, u1);
  s.pLL = fmaf(0.75f, C, u3);
  s.pRR = fmaf(-0.75f, C, u3);
  return s;
}

// Reconstruction of one field along the marching direction. Q is the step's phase,
// n mod 4 up to a constant: every value stays in one register from its first to
// its last use, where a rolled loop would move each of them every step.
// w: values at n - 1, n, n + 1 in slots Q, Q + 1, Q + 2; slot Q + 3 receives n + 2.
// mn / md: numerator and denominator of the minus value of faces n (slot Q) and
// n - 1 (slot Q + 1), which centre n finishes; pn / pd: of the plus value of
// faces n - 2 (slot Q), which centre n finishes, and n - 1 (slot Q + 1).
struct March {
  float w[4], mn[2], md[2], pn[2], pd[2];
  __device__ __forceinline__ void start() {
    // ones in the denominators: values of faces before the first complete one are finite and unused
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      mn[s] = pn[s] = 0.0f;
      md[s] = pd[s] = 1.0f;
    }
  }
  // adds centre n (um: in, the minus value of face n - 2; out, of face n - 1): sum and difference of the two sides of face n - 2
  template <int Q>
  __device__ __forceinline__ void add(float& um, float& us, float& jump) {
    constexpr int e = Q & 1, d = e ^ 1;
    const Window s = window(w[Q], w[(Q + 1) & 3], w[(Q + 2) & 3]);
    const float up = fmaf(s.aR, s.pLL, pn[e]) * __builtin_amdgcn_rcpf(pd[e] + s.aR);
    us = up + um;
    jump = up - um;
    um = fmaf(s.R5, s.pL, mn[d]) * __builtin_amdgcn_rcpf(md[d] + s.R5);
    mn[e] = fmaf(s.C10, s.pR, mn[e]);
    md[e] += s.C10;
    mn[d] = s.L * s.pRR;
    md[d] = s.L;
    pn[d] = fmaf(s.C10, s.pL, pn[d]);
    pd[d] += s.C10;
    pn[e] = s.L5 * s.pR;
    pd[e] = s.L5;
    // a use here keeps the compiler from moving the update to the end of the step,
    // across everything in between, with the window's nine values alive instead
    asm volatile("" ::"v"(mn[0]), "v"(md[0]), "v"(mn[1]), "v"(md[1]), "v"(pn[0]), "v"(pd[0]), "v"(pn[1]), "v"(pd[1]));
  }
};

// Lax-Friedrichs flux of a face from the sum and the difference of both sides'
// values and the six coefficients (cofactor normal, mu, lambda, 1/rho) of the cell
// before it.
__device__ __forceinline__ void lf_flux(const float (&us)[9], const float (&jump)[9], const float (&c)[6], float alpha,
                                        float (&F)[9]) {
  phys_flux<float>(us, c[0], c[1], c[2], c[3], c[4], c[5], F);
#pragma unroll
  for (int v = 0; v < 9; ++v) F[v] = 0.5f * (F[v] - alpha * jump[v]);
}

// Address of the cell at byte offset o in plane c of an array, the plane's base in
// scalar registers. N comes from plane_stride, a
// value that the compiler does not know to be the same in every step: it would
// otherwise keep the addresses of up to 40 planes, more than there are registers,
// or add the plane to the cell's offset in vector registers.
__device__ __forceinline__ long long plane_stride(long long N) {
  asm volatile("" : "+s"(N));
  return N;
}
typedef __attribute__((address_space(1))) float gfloat;
__device__ __forceinline__ gfloat* plane(const float* base, long long N, int c, unsigned o) {
  unsigned long long p = (unsigned long long)(base + c * N);
  asm("" : "+s"(p));
  return (gfloat*)(p + o);
}
__device__ __forceinline__ void ld_face_coef(const float* cjm, long long N, unsigned o, int d, float (&c)[6]) {
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    c[q] = *plane(cjm, N, 3 * d + q, o);
    c[3 + q] = *plane(cjm, N, C_MU + q, o);
  }
}
static_assert(C_LAM == C_MU + 1 && C_B == C_MU + 2, "ld_face_coef reads mu, lambda, 1/rho in a row");

// Values a wave keeps in LDS from step to step, one per lane and field, which
// leaves the registers to the reconstruction (with them the xi/zeta kernel
// spilled, and a spilled load is a load waited for): the differences of the last
// four faces (slots Q, the oldest, to Q + 3), the last face's flux, the finished minus values. A lane
// reads only what it wrote itself, so there is no barrier. d starts undefined: a
// cell's five faces are all added first.
struct Ring {
  float d[4][9][64];
  float F[9][64], um[9][64];
  __device__ __forceinline__ void start(int lane) {
#pragma unroll
    for (int v = 0; v < 9; ++v) F[v][lane] = um[v][lane] = 0.0f;
  }
};
template <int Q>
__device__ __forceinline__ void add_face(Ring& r, int lane, bool complete, float (&F)[9]) {
#pragma unroll
  for (int v = 0; v < 9; ++v) {  // F: flux of face n - 2 in, corrected difference of cell n - 4 out
    const float fv = complete ? F[v] : 0.0f;
    const float D = fv - r.F[v][lane];
    r.F[v][lane] = fv;
    F[v] = fmaf((float)DG, D + r.d[Q][v][lane],
                fmaf((float)DB, r.d[(Q + 3) & 3][v][lane] + r.d[(Q + 1) & 3][v][lane], (float)DA * r.d[(Q + 2) & 3][v][lane]));
    r.d[Q][v][lane] = D;
    asm volatile("" ::"v"(F[v]));  // summed here, not where it is used with the four differences kept until then
  }
}

// Index of a wave of a launch, four to a block: blocks are dealt to the eight XCDs in
// turn, and each XCD takes a contiguous range of waves, so that waves that share
// rows or cache lines of a row run on one XCD.
// The index is the same in all lanes, which readfirstlane tells the compiler: the
// loop's control flow then stays scalar and its loads are not split by branches.
__device__ __forceinline__ int march_wave(unsigned b, unsigned nb8) {
  return __builtin_amdgcn_readfirstlane((int)(((b & 7) * nb8 + (b >> 3)) * 4 + (threadIdx.x >> 6)));
}

// --------------------------------------------------------------------------
// eta: columns (i, k) march along j
// --------------------------------------------------------------------------
struct YWave {
  March m[9];

  // step n at byte offset o; stride between rows a.rowb. A step's loads come first
  // and are used late in the step (row n + 2 in the next): with few waves per
  // SIMD there is little else to hide them.
  template <int Q>
  __device__ __forceinline__ void step(const StageArgs<float>& a, Ring& r, int lane, int n, int ns, int j0, unsigned o) {
    const long long N = plane_stride(a.N);
    float F[9], c[6], us[9], jump[9];
    ld_face_coef(a.cjm, N, n < 2 ? o : o - 2 * a.rowb, 1, c);
    const unsigned on = n < a.NY - 2 ? o + 2 * a.rowb : o;  // row n + 2, if there is one
#pragma unroll
    for (int v = 0; v < 9; ++v) m[v].w[(Q + 3) & 3] = *plane(a.win, N, v, on);
#pragma unroll
    for (int v = 0; v < 9; ++v) m[v].add<Q>(r.um[v][lane], us[v], jump[v]);
    lf_flux(us, jump, c, a.alpha, F);
    add_face<Q>(r, lane, n >= ns + 3 && n < a.NY - 1, F);  // complete and before face NY - 3
    if (n - 4 >= j0) {
#pragma unroll
      for (int v = 0; v < 9; ++v) *plane(a.wout, N, v, o - 4 * a.rowb) = F[v];
    }
  }
};

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
aw_yflux(StageArgs<float> a, int nbx, int nk, int chunk, unsigned nb8) {
  __shared__ Ring ring[4];
  const int w = march_wave(blockIdx.x, nb8);
  const int tx = w % nbx, k = H + w / nbx % nk;
  const int j0 = H + w / nbx / nk * chunk, j1 = min(j0 + chunk, a.NY - H);
  const int lane = threadIdx.x & 63, i = H + tx * 64 + lane;
  if (j0 >= j1 || i >= a.XE - H) return;
  Ring& r = ring[threadIdx.x >> 6];
  const int ns = max(j0 - 4, 1), ne = j1 + 3;  // first centre: face ns + 1 is the first one needed that is not zero
  unsigned o = (unsigned)i * 4u + (unsigned)k * a.planeb + (unsigned)ns * a.rowb;  // row n
  YWave y;
  r.start(lane);
#pragma unroll
  for (int v = 0; v < 9; ++v) {
    y.m[v].start();
#pragma unroll
    for (int s = 0; s < 3; ++s) y.m[v].w[s] = *at(a.win + v * a.N, o + (unsigned)(s - 1) * a.rowb);
  }
  for (int n = ns;; n += 4) {
    y.step<0>(a, r, lane, n, ns, j0, o);
    if (n + 1 > ne) return;
    o += a.rowb;
    y.step<1>(a, r, lane, n + 1, ns, j0, o);
    if (n + 2 > ne) return;
    o += a.rowb;
    y.step<2>(a, r, lane, n + 2, ns, j0, o);
    if (n + 3 > ne) return;
    o += a.rowb;
    y.step<3>(a, r, lane, n + 3, ns, j0, o);
    if (n + 4 > ne) return;
    o += a.rowb;
  }
}

// --------------------------------------------------------------------------
// xi and zeta: columns (i, j) march along k; xi fluxes across the lanes
// --------------------------------------------------------------------------
// value of the lane before / after (0 past the ends of the wave; such lanes' results are not used)
__device__ __forceinline__ float lane_prev(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));  // wave_shr:1
}
__device__ __forceinline__ float lane_next(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));  // wave_shl:1
}

// A wave holds columns ib .. ib + 63, ib = 54 t. A cell's difference needs the
// windows of centres i - 4 .. i + 4, the outermost with a neighbour each, so five
// columns at either end of the wave only feed the others; at the ends of the
// row the faces beyond are zero and up to two more columns are complete.
constexpr int XT = 54;
inline int x_waves(int XE) { return XE <= 64 ? 1 : (XE - 64 + XT - 1) / XT + 1; }

struct XZWave {
  March m[9];
  int lane;
  bool xface, own;

  // step n at byte offset o: the zeta face n - 2, which completes cell n - 4, then
  // that cell's xi fluxes and its update. The cell's own values are loaded before
  // the zeta windows, the rest of what it needs before the xi windows, which hide
  // the loads.
  template <int STAGE, int Q>
  __device__ __forceinline__ void step(const StageArgs<float>& a, Ring& r, int n, int ns, int k0, unsigned o) {
    const long long N = plane_stride(a.N);
    const bool cell = n - 4 >= k0;
    const unsigned oc = cell ? o - 4 * a.planeb : o;  // cell n - 4
    float h[9], wv[9], c[6], us[9], jump[9];
    ld_face_coef(a.cjm, N, n < 2 ? o : o - 2 * a.planeb, 2, c);
#pragma unroll
    for (int v = 0; v < 9; ++v) {
      m[v].w[(Q + 3) & 3] = *plane(a.win, N, v, o + 2 * a.planeb);  // n + 2 <= NZ - 1
      wv[v] = *plane(a.win, N, v, oc);
    }
#pragma unroll
    for (int v = 0; v < 9; ++v) m[v].add<Q>(r.um[v][lane], us[v], jump[v]);
    lf_flux(us, jump, c, a.alpha, h);
    add_face<Q>(r, lane, n >= ns + 3, h);
    if (!cell) return;
    float F[9], mv[9], hy[9];
    ld_face_coef(a.cjm, N, oc, 0, c);
    const float J = *plane(a.cjm, N, C_J, oc);
#pragma unroll
    for (int v = 0; v < 9; ++v) {
      hy[v] = *plane(a.wout, N, v, oc);
      if constexpr (STAGE != 0) mv[v] = __builtin_nontemporal_load(plane(a.wm, N, v, oc));
    }
#pragma unroll
    for (int v = 0; v < 9; ++v) {
      const Window s = window(lane_prev(wv[v]), wv[v], lane_next(wv[v]));
      const float mn = fmaf(s.C10, s.pR, lane_prev(s.L * s.pRR)) + lane_next(s.R5 * s.pL);
      const float md = s.C10 + lane_prev(s.L) + lane_next(s.R5);
      const float pn = fmaf(s.L5, s.pR, lane_next(fmaf(s.C10, s.pL, lane_next(s.aR * s.pLL))));
      const float pd = s.L5 + lane_next(s.C10 + lane_next(s.aR));
      const float um = mn * __builtin_amdgcn_rcpf(md), up = pn * __builtin_amdgcn_rcpf(pd);
      us[v] = up + um;
      jump[v] = up - um;
    }
    lf_flux(us, jump, c, a.alpha, F);
    const float cd = a.DT * a.rDH * (1.0f / J);
#pragma unroll
    for (int v = 0; v < 9; ++v) {
      const float f = xface ? F[v] : 0.0f;
      const float D = f - lane_prev(f), l = lane_prev(D), t = lane_next(D);
      h[v] += hy[v] + fmaf((float)DA, D, fmaf((float)DB, l + t, (float)DG * (lane_prev(l) + lane_next(t))));
    }
    if (own) {
#pragma unroll
      for (int v = 0; v < 9; ++v)
        *plane(a.wout, N, v, oc) = tvd<float>(STAGE, STAGE == 0 ? wv[v] : mv[v], wv[v], -cd * h[v]);
    }
  }
};

template <int STAGE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
aw_xzstep(StageArgs<float> a, int nbx, int chunk, unsigned nb8) {
  __shared__ Ring ring[4];
  const int w = march_wave(blockIdx.x, nb8);
  const int ny = a.NY - 2 * H, kend = a.NZ - H - 3;
  const int tx = w % nbx, j = H + w / nbx % ny;
  const int k0 = H + w / nbx / ny * chunk, k1 = min(k0 + chunk, kend);
  if (k0 >= k1) return;  // whole waves: the lanes of a wave stay together for the lane shifts
  Ring& r = ring[threadIdx.x >> 6];
  XZWave z;
  z.lane = threadIdx.x & 63;
  const int i = tx * XT + z.lane;
  z.xface = i >= 2 && i < a.XE - H;
  z.own = (tx == 0 ? i >= H : z.lane >= 5) && (tx == nbx - 1 ? i < a.XE - H : z.lane <= 58);
  const int ns = max(k0 - 4, 1), ne = k1 + 3;  // k1 + 3 <= NZ - 3: every window lies in the array
  unsigned o = (unsigned)min(i, a.XE - 1) * 4u + (unsigned)j * a.rowb + (unsigned)ns * a.planeb;  // plane n
#pragma unroll
  for (int v = 0; v < 9; ++v) {
    z.m[v].start();
#pragma unroll
    for (int s = 0; s < 3; ++s) z.m[v].w[s] = *at(a.win + v * a.N, o + (unsigned)(s - 1) * a.planeb);
  }
  r.start(z.lane);
  for (int n = ns;; n += 4) {
    z.step<STAGE, 0>(a, r, n, ns, k0, o);
    if (n + 1 > ne) return;
    o += a.planeb;
    z.step<STAGE, 1>(a, r, n + 1, ns, k0, o);
    if (n + 2 > ne) return;
    o += a.planeb;
    z.step<STAGE, 2>(a, r, n + 2, ns, k0, o);
    if (n + 3 > ne) return;
    o += a.planeb;
    z.step<STAGE, 3>(a, r, n + 3, ns, k0, o);
    if (n + 4 > ne) return;
    o += a.planeb;
  }
}

// Cells per wave along the marching direction: `units` waves per chunk of a column
// of `cells`. A wave takes about 12 steps' time more than its cells (8 steps that
// only fill the windows, and the first loads); the 256 CUs hold 1024 waves at one
// per SIMD, and a second one on each costs about two thirds of the first's time.
// Measured in us per stage at 200 x 180 x 100 with chunks of 8, 16, 32 cells: 539,
// 492, 544; at 128 x 120 x 80: 210, 188, 276.
inline int march_cells(long long units, int cells, double* cost_of = nullptr) {
  int best = cells;
  double least = 0.0;
  for (int n = 1; n <= cells; ++n) {
    const int c = (cells + n - 1) / n;
    const long long r = (units * n + 1023) / 1024;
    const double cost = (double)(c + 12) * ((double)(r / 2) + 0.6 * (double)(r % 2));
    if (n > 1 && cost >= least) continue;
    least = cost;
    best = c;
  }
  if (cost_of) *cost_of = least;
  return best;
}

// Whether the marching kernels are the faster ones: us per step from the costs of
// their two launches and the blocks of the top layers, against the blocks of the two
// kernels with the flux array.
// The figures are fitted to both paths on 170 grids of 0.1 to 12 million cells with
// extents from 4 to 2000, most of them near the line. On 68 others the path taken is
// the slower one by more than 6 % once (536 x 77 x 17, 0.487 ms for 0.414), and a mean
// 0.4 % slower than the better one; a line at a number of cells does worse, since
// marching gains with the depth and with the lanes that a row fills. ms per step with
// the array and marching: 59 x 90 x 78 0.320 and 0.397, 400 x 400 x 6 0.655 and 0.786,
// 900 x 800 x 6 2.78 and 3.13, 166 x 80 x 46 0.392 and 0.387, 512 x 500 x 60 6.37 and
// 4.18, 320 x 300 x 200 7.72 and 4.83.
bool march_pays(int nx, int ny, int nz, int rtx, int rty) {
  const int nk = nz - 3;  // at least 1: a grid has four planes
  const long long bx = (nx + 63) / 64;
  double cy, cz;
  march_cells(bx * nk, ny, &cy);
  march_cells((long long)x_waves(nx + 2 * H) * ny, nk, &cz);
  const double march = 33.0 + 10.9 * cy + 11.8 * cz + 0.5 * (double)(bx * ((ny + 3) / 4));
  const double array = 95.0 + 0.0488 * (double)(cg::interior_blocks(nx, ny + 1, nz + 1, rtx, rty) +
                                               cg::interior_blocks(nx, ny + 2 * H, nz + 2 * H, rtx, rty));
  return march < array;
}

inline unsigned march_blocks8(long long waves) { return (unsigned)(((waves + 3) / 4 + 7) / 8); }

void launch_march_y(const StageArgs<float>& a, int nx, int ny, hipStream_t st) {
  const int nk = a.NZ - 2 * H - 3;  // planes below the top three layers
  if (nk <= 0) return;
  const int bx = (nx + 63) / 64, c = march_cells((long long)bx * nk, ny);
  const unsigned b8 = march_blocks8((long long)bx * nk * ((ny + c - 1) / c));
  aw_yflux<<<dim3(8 * b8), dim3(256), 0, st>>>(a, bx, nk, c, b8);
}

void launch_march_xz(const StageArgs<float>& a, int nx, int ny, hipStream_t st) {
  const dim3 block(256);
  aw_update_top<float, true><<<dim3((nx + 63) / 64, (ny + 3) / 4, 6), block, 0, st>>>(a, nx, ny);
  const int nk = a.NZ - 2 * H - 3;
  if (nk <= 0) return;
  const int bx = x_waves(a.XE), c = march_cells((long long)bx * ny, nk);
  const unsigned b8 = march_blocks8((long long)bx * ny * ((nk + c - 1) / c));
  const dim3 g(8 * b8);
  if (a.stage == 0) aw_xzstep<0><<<g, block, 0, st>>>(a, bx, c, b8);
  else if (a.stage == 1) aw_xzstep<1><<<g, block, 0, st>>>(a, bx, c, b8);
  else aw_xzstep<2><<<g, block, 0, st>>>(a, bx, c, b8);
}

}  // namespace aw
