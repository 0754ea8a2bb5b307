// mlau_1d.hip -- 1D ideal-MHD step on gfx950 (FP64).
//
// k_step1d runs one or more whole FP64 steps of 1D/SERIAL/shock/mhd_fd4c_1d.c:60-271 in
// one launch (step1d_body): each block advances a window of cells with its own
// halo, from u0 to u1 or back.  Very long grids, where the repeated halo cells
// cost more than the launches, and the mixed forms take a stage in two launches or one:
//   k_sweep1d   primitives (:121-131, formed per stencil point) + reconstruction
//               + Riemann solver, one wavefront per 63 faces (left face
//               states passed by shuffle)                                :137-207
//   k_update1d  flux difference + SSP-RK combine (:225-255); its last block
//               runs the characteristic open boundary on stage 0 (:209-218,
//               openbc1d_mhd.c:21-175), periodic ghosts are written with their
//               source cells (1D/SERIAL/wave/prdc_1d.c:18-25), and the last
//               stage advances the step's time.
// RK1 with the open boundary updates in place, so there the boundary runs
// first in a launch of its own (k_openbc1d).
// At ODR <= 2 with R_K >= 2 a stage is one launch (k_stage1d: flux and update
// per wavefront) writing a third state u0 -> u1 -> u2 -> u0 (u2: the flux
// arrays, which it does not use); with the open boundary, stage 0 keeps the
// two launches (the boundary rewrites ghosts its stencils read) and stage 1
// copies those fixed ghosts into u2.
// Fields in argument order ro,mx,my,mz,en,by,bz; bx is a constant.
#include "mlau_1d_body.h"

namespace mlau {

template <int ODR, int FLUX, int MIX>
__global__ __launch_bounds__(256) void k_sweep1d(U1d u, W1d w, G1d g)
{
  sweep1d_body<ODR, FLUX, MIX>(u, w, g, blockIdx.x, threadIdx.x);
}

// thread 0 = left edge, thread 1 = right edge
__global__ void k_openbc1d(U1d in, U1d dst0, U1d dst1, G1d g, const StepInfo *info)
{
  openbc1d_body(in, dst0, dst1, g, info->dtdx, threadIdx.x);
}

// obc: the last block runs the open boundary on u0 and u1 (stage 0 of RK2/RK3:
// it reads the stage input u0 and writes only ghosts, the update reads only
// interior cells of u0 and writes u1, so the two are independent).
// adv: block 0 advances the step's time (tim, nstep; the blocks read only dtdx).
template <int ODR, bool PER>
__global__ __launch_bounds__(256) void k_update1d(U1d in, U1d ut, U1d out, W1d w, G1d g, StepInfo *info, double ra,
                                                  double rb, U1d u0, U1d u1, int obc, int adv)
{
  if (obc && blockIdx.x == gridDim.x - 1) {
    openbc1d_body(in, u0, u1, g, info->dtdx, threadIdx.x);
    return;
  }
  const double dtdx = info->dtdx;
  update1d_body<ODR, PER>(in, ut, out, w, g, dtdx, ra, rb, blockIdx.x, threadIdx.x);
  if (adv && blockIdx.x == 0 && threadIdx.x == 0) {
    info->tim += info->dt;
    info->nstep += 1;
  }
}

// K whole steps (step1d_body); block 0 advances the time.
template <int ODR, int FLUX, bool PER>
__global__ __launch_bounds__(PER ? kWin1 : kWin1 + 64) void k_step1d(U1d in, U1d out, G1d g, StepInfo *info, int rk,
                                                                     int K)
{
  __shared__ Lds1d S;
  step1d_body<ODR, FLUX, PER>(in, out, g, info->dtdx, rk, K, blockIdx.x, threadIdx.x, S);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int k = 0; k < K; k++) info->tim += info->dt;
    info->nstep += K;
  }
}

// The state after an odd number of launches: one thread per cell, all seven fields.
__global__ __launch_bounds__(256) void k_copy1d(U1d src, U1d dst, int nx)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nx) return;
#pragma unroll
  for (int n = 0; n < 7; n++) dst.f[n][i] = src.f[n][i];
}

template <int ODR, int FLUX, int MIX, bool PER>
__global__ __launch_bounds__(256) void k_stage1d(U1d in, U1d ut, U1d out, G1d g, StepInfo *info, double ra, double rb,
                                                 int copy_ghosts, int adv)
{
  stage1d_body<ODR, FLUX, MIX, PER>(in, ut, out, g, info->dtdx, ra, rb, blockIdx.x * 4 + (threadIdx.x >> 6),
                                    threadIdx.x & 63, copy_ghosts != 0);
  if (adv && blockIdx.x == 0 && threadIdx.x == 0) {
    info->tim += info->dt;
    info->nstep += 1;
  }
}

__global__ __launch_bounds__(256) void k_cfl1d(U1d u, G1d g, StepInfo *info, double cfl, double vfloor,
                                               double dx, double dy, double dz)
{
  double v = 0.0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < g.nx; i += (int)gridDim.x * 256) {
    const double vt = cfl1d_cell(u, g, i);
    if (vt > v) v = vt;
  }
  v = block_max<256>(v);
  if (threadIdx.x == 0) cfl_finish(info, v, cfl, vfloor, dx, dx, dy, dz);
}

// A cell per thread on short grids, whose check is one cell's chain; few blocks on
// long ones (cfl_blocks).  A step and its check, us, all cells at once and by cfl_blocks: 1000
// cells 19.8 and 20.5, 8192 20.1 and 20.7, 65536 34.0 and 31.6, 200000 69.3 and 58.4, 1000000
// 245 and 203, 4194304 1145 and 980.
static void check1d(Handle *h, const U1d &u, const G1d &g, double cfl, double vfloor)
{
  const unsigned nb = g.nx <= 16384 ? (unsigned)((g.nx + 255) / 256) : cfl_blocks(g.nx);
  MLAU_LAUNCH(h, K_CFL1D, k_cfl1d, dim3(nb), dim3(256), u, g, h->info, cfl, vfloor, h->g.dx, h->g.dy, h->g.dz);
}

static void views1d(Handle *h, U1d &u0, U1d &u1, W1d &w, G1d &g)
{
  for (int n = 0; n < 7; n++) {
    u0.f[n] = h->U0[n];
    u1.f[n] = h->U1[n];
    w.fx[n] = h->fx[n];
  }
  w.vx = h->prim[0]; w.vy = h->prim[1]; w.vz = h->prim[2]; w.pr = h->prim[3];
  g.nx = h->g.nx; g.xoff = h->g.xoff; g.gamma = h->g.gamma; g.bx = h->g.bx;
}

template <int ODR, int FLUX, int MIX>
static void step1d(Handle *h)
{
  U1d u0, u1;
  W1d w;
  G1d g;
  views1d(h, u0, u1, w, g);
  const int R_K = h->s.rk, nx = g.nx;
  const double rkf[3][2] = {{0.0, 1.0}, {0.5 + (R_K - 2) * 0.25, 0.5 - (R_K - 2) * 0.25}, {1. / 3., 2. / 3.}};
  const int tiles = (nx - 5 + 62) / 63;
  const bool open = h->s.bc1d == MLAU_BC1D_OPEN;
  const unsigned ub = (nx - 8 + 255) / 256;
  if constexpr (ODR <= 2) {
    if (R_K >= 2 && !(h->tune & 8)) {  // tune bit 3: separate flux and update launches throughout
      U1d u2;
      for (int n = 0; n < 7; n++) u2.f[n] = h->fx[n];
      const U1d buf[3] = {u0, u1, u2};
      const unsigned sb = (unsigned)(((nx - 8 + 61) / 62 + 3) / 4);  // 4 wavefronts of 62 cells per block
      for (int rk = 0; rk < R_K; rk++) {
        const int sin = (rk == 0) ? 0 : (rk == 1 ? 1 : 2);
        const int sout = (rk == R_K - 1) ? 0 : (rk == 0 ? 1 : 2);
        const int adv = rk == R_K - 1;
        if (rk == 0 && open) {
          MLAU_LAUNCH(h, K_SWEEP1D, (k_sweep1d<ODR, FLUX, MIX>), dim3((tiles + 3) / 4), dim3(256), u0, w, g);
          MLAU_LAUNCH(h, K_UPD1D, (k_update1d<ODR, false>), dim3(ub + 1), dim3(256), u0, u0, u1, w, g, h->info,
                      rkf[0][0], rkf[0][1], u0, u1, 1, 0);
        } else if (open) {
          MLAU_LAUNCH(h, K_STAGE1D, (k_stage1d<ODR, FLUX, MIX, false>), dim3(sb), dim3(256), buf[sin], u0, buf[sout], g,
                      h->info, rkf[rk][0], rkf[rk][1], (int)(sout == 2), adv);
        } else {
          MLAU_LAUNCH(h, K_STAGE1D, (k_stage1d<ODR, FLUX, MIX, true>), dim3(sb), dim3(256), buf[sin], u0, buf[sout], g,
                      h->info, rkf[rk][0], rkf[rk][1], 0, adv);
        }
      }
      return;
    }
  }
  for (int rk = 0; rk < R_K; rk++) {
    const U1d &in = (rk == 0) ? u0 : u1;
    const U1d &out = (rk == R_K - 1) ? u0 : u1;
    MLAU_LAUNCH(h, K_SWEEP1D, (k_sweep1d<ODR, FLUX, MIX>), dim3((tiles + 3) / 4), dim3(256), in, w, g);
    const bool obc_here = rk == 0 && open;
    const int obc = obc_here && R_K > 1;  // RK1 updates in place: boundary first, separately
    if (obc_here && !obc)
      MLAU_LAUNCH(h, K_OPENBC1D, k_openbc1d, dim3(1), dim3(64), in, u0, u1, g, (const StepInfo *)h->info);
    const int adv = rk == R_K - 1;
    if (open)
      MLAU_LAUNCH(h, K_UPD1D, (k_update1d<ODR, false>), dim3(ub + obc), dim3(256), in, u0, out, w, g, h->info,
                  rkf[rk][0], rkf[rk][1], u0, u1, obc, adv);
    else
      MLAU_LAUNCH(h, K_UPD1D, (k_update1d<ODR, true>), dim3(ub), dim3(256), in, u0, out, w, g, h->info, rkf[rk][0],
                  rkf[rk][1], u0, u1, 0, adv);
  }
}

// Whole steps per launch: 1, 2 or 4.  More save launches (about 1.5 us a step each time) but repeat
// more cells at the windows' edges, and a step costs as many rounds of the 256 CUs as its windows
// fill (one window a CU: 11.5 us a round for MUSCL + MLAU, 15.5 for WCNS4 + LHLLD): as many as take no
// further round.  Measured, us a step with a launch or two per stage and with 1, 2, 4 steps per launch, rk 3
// (MUSCL + MLAU open / WCNS4 + LHLLD periodic): 20000 cells 24.7 and 13.8, 13.0, 12.4 / 32.8 and 18.9, 17.2, 16.5;
// 100000 40.2 and 25.1, 23.7, 33.1 / 59.7 and 35.1, 33.3, 47.1; 131072 49.6 and 36.7, 34.2, 33.4 / 70.3 and 51.3, 48.6,
// 62.4; 300000 72.6 and 60.0, 66.9, 75.5 / 106 and 100, 95.9, 124; 393000 91.3 and 82.4, 78.3, 96.4 /
// 129 and 117, 128, 155; 1048576 202 and 215, 217, 255 / 345 and 330, 355, 452.
// 0: separate stage launches.  A periodic grid at ODR 2 takes one launch a stage and is
// better off so from fewer cells on: 262144 60.1 and 62.0, 58.3, 67.4; 300000 61.9 and 62.5, 69.5; 350000 70.4 and
// 74.4, 81.1; and for a single step, whose result is copied back, wherever a step takes more than one round:
// 56000 31.9 and 29.4, 65536 39.3 and 41.9, 200000 62.6 and 71.3.  The mixed forms always: the compiler would
// fuse their multiply-adds otherwise here (rounding differences of 1e-16 with FP64 solvers and of 1e-9 to
// 1e-8 with FP32 or Roe's, between grids on the two sides of a line).
static int steps_per_launch1d(const Handle *h, int nsteps, bool cfl_mode)
{
  const int cells = h->g.nx - 8, rk = h->s.rk;
  if ((h->tune & 8) || h->g.nx > 393216 || h->s.precision != MLAU_FP64) return 0;
  auto rounds = [&](int K) {
    const int own = kWin1 - 2 * (h->s.odr <= 2 ? win1_halo<2>(K, rk) : win1_halo<4>(K, rk));
    return ((cells + own - 1) / own + 255) / 256;
  };
  if (h->s.odr == 2 && rk >= 2 && h->s.bc1d == MLAU_BC1D_PERIODIC &&
      (cells > 280000 || (nsteps == 1 && rounds(1) > 1)))
    return 0;
  if (cfl_mode) return 1;  // the next dt needs the whole grid
  return rounds(4) <= rounds(1) ? 4 : rounds(2) <= rounds(1) ? 2 : 1;
}

// Steps in launches of up to `most` whole steps, from one state to the other and
// back; an odd number of launches ends with a copy into u0.
template <int ODR, int FLUX>
static void steps1d(Handle *h, int nsteps, int most, bool cfl_mode, double cfl, double vfloor)
{
  U1d u0, u1;
  W1d w;
  G1d g;
  views1d(h, u0, u1, w, g);
  const int rk = h->s.rk, nx = g.nx;
  const bool open = h->s.bc1d == MLAU_BC1D_OPEN;
  int m = (nsteps + most - 1) / most;  // launches
  if ((m & 1) && m < nsteps) m++;
  for (int j = 0; j < m; j++) {
    const int K = (int)((long)nsteps * (j + 1) / m - (long)nsteps * j / m);
    const int own = kWin1 - 2 * win1_halo<ODR>(K, rk);
    const dim3 gr((nx - 8 + own - 1) / own);
    const U1d &in = j & 1 ? u1 : u0, &out = j & 1 ? u0 : u1;
    if (open)
      MLAU_LAUNCH(h, K_STEP1D, (k_step1d<ODR, FLUX, false>), gr, dim3(kWin1 + 64), in, out, g, h->info, rk, K);
    else
      MLAU_LAUNCH(h, K_STEP1D, (k_step1d<ODR, FLUX, true>), gr, dim3(kWin1), in, out, g, h->info, rk, K);
    if (cfl_mode) check1d(h, out, g, cfl, vfloor);
  }
  if (m & 1) MLAU_LAUNCH(h, K_STEP1D, k_copy1d, dim3((nx + 255) / 256), dim3(256), u1, u0, nx);
}

typedef void (*Step1Fn)(Handle *);
typedef void (*Steps1Fn)(Handle *, int, int, bool, double, double);
template <int ODR, int MIX>
static Step1Fn pick1f(int flux)
{
  switch (flux) {
  case FLUX_MLAU: return step1d<ODR, FLUX_MLAU, MIX>;
  case FLUX_ROE: return step1d<ODR, FLUX_ROE, MIX>;
  case FLUX_HLLD: return step1d<ODR, FLUX_HLLD, MIX>;
  default: return step1d<ODR, FLUX_LHLLD, MIX>;
  }
}
template <int ODR>
static Step1Fn pick1(int flux, int precision)
{
  switch (precision) {
  case MLAU_MIXED: return pick1f<ODR, MLAU_MIXED>(flux);
  case MLAU_MIXED_RECON: return pick1f<ODR, MLAU_MIXED_RECON>(flux);
  default: return pick1f<ODR, MLAU_FP64>(flux);
  }
}

template <int ODR>
static Steps1Fn pick1s(int flux)
{
  switch (flux) {
  case FLUX_MLAU: return steps1d<ODR, FLUX_MLAU>;
  case FLUX_ROE: return steps1d<ODR, FLUX_ROE>;
  case FLUX_HLLD: return steps1d<ODR, FLUX_HLLD>;
  default: return steps1d<ODR, FLUX_LHLLD>;
  }
}

int run_cfl_1d(Handle *h, double cfl, double vfloor)
{
  U1d u0, u1;
  W1d w;
  G1d g;
  views1d(h, u0, u1, w, g);
  check1d(h, u0, g, cfl, vfloor);
  return (int)hipGetLastError();
}

int run_steps_1d(Handle *h, int nsteps, bool cfl_mode, double cfl, double vfloor)
{
  if (h->g.xoff != 4) return (int)hipErrorInvalidValue;
  if (const int most = steps_per_launch1d(h, nsteps, cfl_mode)) {
    Steps1Fn fs;
    switch (h->s.odr) {
    case 1: fs = pick1s<1>(h->s.flux); break;
    case 2: fs = pick1s<2>(h->s.flux); break;
    case 3: fs = pick1s<3>(h->s.flux); break;
    default: fs = pick1s<4>(h->s.flux); break;
    }
    fs(h, nsteps, most, cfl_mode, cfl, vfloor);
    return (int)hipGetLastError();
  }
  Step1Fn fn;
  switch (h->s.odr) {
  case 1: fn = pick1<1>(h->s.flux, h->s.precision); break;
  case 2: fn = pick1<2>(h->s.flux, h->s.precision); break;
  case 3: fn = pick1<3>(h->s.flux, h->s.precision); break;
  default: fn = pick1<4>(h->s.flux, h->s.precision); break;
  }
  for (int n = 0; n < nsteps; n++) {
    fn(h);  // its last update advances the time
    if (cfl_mode) run_cfl_1d(h, cfl, vfloor);
  }
  return (int)hipGetLastError();
}

}  // namespace mlau
