// mlau_2d.hip -- 2D ideal-MHD + CT step on gfx950 (FP64).
//
// One RK stage (2D/SERIAL/OTvortex/mhd_fd_ct_2d.c:165-639) is five kernels:
//   k_prim2d    face B -> centre (cx,cy) and primitives (vx,vy,vz,pr,m2)   :172-223
//   k_aux2d     CT upwind weight ctx and shock sensors dvx,dvy            :224-271
//   k_sweeps2d  both sweeps, by blocks:
//     x         reconstruction + Riemann solver, one wavefront per 63
//               faces of a row; each lane reconstructs one cell and hands
//               its left face state to the next lane by a wave shuffle    :273-362
//     y         reconstruction + Riemann solver, one lane per column
//               marching up a chunk of rows with the 5-row stencil held in
//               registers (coalesced rows, no reconstruction twice)      :404-493
//   k_ez2d      corner E-field from both sweeps' induction fluxes       :364-402,495-533
//   k_update2d  cell-centre update, CT face-B update, SSP-RK combine    :535-632
// followed by k_bc2d (ghost cells, :636-638); on periodic grids the update
// writes the ghost images itself (k_update2d_per) and no boundary pass follows.  The reference's halo fills of
// the intermediate fields (bc2d on cx,cy,dvx,dvy) are folded into the
// kernels that produce them: a ghost value is computed at its source cell and
// multiplied by the boundary factor.
#include "mlau_2d_fused.h"

namespace mlau {

constexpr int kMarch = 8;  // longest march of the y sweep

// Single-grid kernels: the cell kernels tile their region in flattened
// 256-cell pieces, remapped so that each XCD works on a contiguous band of
// rows (xcd_band).
#define REGION_CELL(W, H, I0, J0)                                                                   \
  int i, j;                                                                                        \
  if (!region_cell((W), (H), (I0), (J0), xcd_band(blockIdx.x, gridDim.x), threadIdx.x, i, j)) return;

template <int ODR>
__global__ __launch_bounds__(256) void k_prim2d(U2 u, W2 w, G2 g, BcFlags bc)
{
  REGION_CELL(g.nx, g.ny, 0, 0)
  prim2d_body<ODR>(u, w, g, bc, i, j);
}

template <int CTW>
__global__ __launch_bounds__(256) void k_aux2d(U2 u, W2 w, G2 g, BcFlags bc)
{
  REGION_CELL(g.nx, g.ny, 0, 0)
  aux2d_body<CTW>(u, w, g, bc, i, j);
}

template <int ODR, int CTW>
__global__ __launch_bounds__(256) void k_primaux2d(U2 u, W2 w, G2 g, BcFlags bc)
{
  REGION_CELL(g.nx, g.ny, 0, 0)
  primaux2d_body<ODR, CTW>(u, w, g, bc, i, j);
}

template <int ODR>
__global__ __launch_bounds__(256) void k_ez2d(W2 w, G2 g)
{
  REGION_CELL(g.nx - 5, g.ny - 5, 3, 3)
  ez2d_body<ODR>(w, g, i, j);
}

template <int ODR, bool FIRST>
__global__ __launch_bounds__(256) void k_update2d(U2 in, U2 ut, U2 out, W2 w, G2 g, StepInfo *info, double ra,
                                                  double rb, int adv)
{
  if (adv) advance_time(info);
  REGION_CELL(g.nx - 2 * g.xoff + 1, g.ny - 2 * g.yoff + 1, g.xoff, g.yoff)
  update2d_body<ODR, FIRST>(in, ut, out, w, g, info->dtdx, info->dtdy, ra, rb, i, j);
}

// periodic grids: interior cells, ghost images written with them (no k_bc2d)
template <int ODR, bool FIRST>
__global__ __launch_bounds__(256) void k_update2d_per(U2 in, U2 ut, U2 out, W2 w, G2 g, StepInfo *info, double ra,
                                                      double rb, int adv)
{
  if (adv) advance_time(info);
  REGION_CELL(g.nx - 2 * g.xoff, g.ny - 2 * g.yoff, g.xoff, g.yoff)
  update2d_body<ODR, FIRST, true>(in, ut, out, w, g, info->dtdx, info->dtdy, ra, rb, i, j);
}

// Both sweeps in one launch: blocks below `ny` are y-sweep blocks (px pieces of a row
// by marches), the others one x-sweep wavefront each (row-flattened).  The sweeps share no output, and both fit two wavefronts to
// a SIMD.  Against two launches on two streams, where a fork and a join
// wait on each other's events, 8 steps, us: 64^2 964 -> 599, 256^2 1278 -> 1041,
// 1024^2 6898 -> 6604, 2048^2 26117 -> 25610; mixed 256^2 1133 -> 826, 1024^2 5587 ->
// 4797 (the x sweep's third wavefront lost nothing); walls 512^2 1991 -> 1825.
// Periodic grids: primitives, shock sensors and CT weights from the state
// itself (mlau_2d_fused.h).
template <int ODR, int FLUX, int MIX, int CTW, bool SPLIT>
__device__ __forceinline__ void sweeps2d_inl_body(const U2 &u, const W2 &w, const G2 &g, int ch, unsigned px,
                                                  unsigned ny)
{
  const unsigned b = blockIdx.x;
  if (b < ny)
    ysweep2d_inl_body<ODR, FLUX, MIX, CTW, SPLIT>(u, w, g, ch, march_mid(ch, b / px, kMarch), b % px, b / px,
                                                  threadIdx.x);
  else
    xsweep2d_inl_body<ODR, FLUX, MIX>(u, w, g, (long)(b - ny), threadIdx.x);
}
template <int ODR, int FLUX, int MIX, int CTW, bool SPLIT>
__global__ __launch_bounds__(64) void k_sweeps2d_inl(U2 u, W2 w, G2 g, int ch, unsigned px, unsigned ny)
{
  sweeps2d_inl_body<ODR, FLUX, MIX, CTW, SPLIT>(u, w, g, ch, px, ny);
}
template <int ODR, int FLUX, int MIX, int CTW, bool SPLIT>
__global__ __launch_bounds__(64) MLAU_TWO_WAVES void k_sweeps2d_inl_two(U2 u, W2 w, G2 g, int ch, unsigned px,
                                                                        unsigned ny)
{
  sweeps2d_inl_body<ODR, FLUX, MIX, CTW, SPLIT>(u, w, g, ch, px, ny);
}
template <int ODR, int FLUX, int MIX, bool SPLIT>
__device__ __forceinline__ void sweeps2d_body(const U2 &u, const W2 &w, const G2 &g, int ch, unsigned px, unsigned ny)
{
  const unsigned b = blockIdx.x;
  if (b < ny)
    ysweep2d_body<ODR, FLUX, MIX, SPLIT>(u, w, g, ch, march_mid(ch, b / px, kMarch), b % px, b / px, threadIdx.x);
  else
    xsweep2d_body<ODR, FLUX, MIX>(u, w, g, (long)(b - ny), threadIdx.x);
}
template <int ODR, int FLUX, int MIX, bool SPLIT>
__global__ __launch_bounds__(64) void k_sweeps2d(U2 u, W2 w, G2 g, int ch, unsigned px, unsigned ny)
{
  sweeps2d_body<ODR, FLUX, MIX, SPLIT>(u, w, g, ch, px, ny);
}
template <int ODR, int FLUX, int MIX, bool SPLIT>
__global__ __launch_bounds__(64) MLAU_TWO_WAVES void k_sweeps2d_two(U2 u, W2 w, G2 g, int ch, unsigned px, unsigned ny)
{
  sweeps2d_body<ODR, FLUX, MIX, SPLIT>(u, w, g, ch, px, ny);
}

// Forms whose joint sweeps take 258 to 272 VGPRs by themselves, and so one wavefront a SIMD.
// Launches of more wavefronts than two for each of the chip's 1024 SIMDs hold them to 256,
// where 0 to 68 bytes are spilled; smaller ones gain nothing by it. us a step: walls, MUSCL + MLAU 64^2
// 65.2 and 67.2, 515^2 237 and 218, 1400^2 1447 and 1239; WCNS4 + LHLLD 256^2 144 and 147, 900^2 739 and 662, 2048^2
// 4015 and 3486; periodic, WCNS4 + MLAU 100^2 73.9 and 75.7, 256^2 141 and 135, 2048^2 4085 and 3299, Roe
// 3963 and 3266. On the others the limit is not needed (WCNS3 + MLAU periodic 2048^2 2897 and 3104).
template <int ODR, int FLUX, int MIX>
constexpr bool two_waves_inl = MIX == MLAU_FP64 && ODR == 4 && (FLUX == FLUX_MLAU || FLUX == FLUX_ROE);
template <int ODR, int FLUX, int MIX>
constexpr bool two_waves = (MIX == MLAU_FP64 && ((FLUX == FLUX_MLAU && ODR >= 2) || (FLUX == FLUX_LHLLD && ODR == 4))) ||
                           (MIX == MLAU_MIXED_RECON && FLUX == FLUX_MLAU && ODR == 4);
constexpr unsigned kTwoWaves = 2048;

// The x sweep by itself, four row-flattened wavefronts to a block.
template <int ODR, int FLUX, int MIX>
__global__ __launch_bounds__(256) void k_xsweep2d_inl(U2 u, W2 w, G2 g)
{
  const long W = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (W >= xsweep_waves(g.ny, g.nx)) return;  // whole wavefront
  xsweep2d_inl_body<ODR, FLUX, MIX>(u, w, g, W, threadIdx.x & 63);
}

// CT weight 1/2 at corners 3..nx-3 x 3..ny-3 (no upwind weighting)
__global__ __launch_bounds__(256) void k_ctx_half2d(W2 w, G2 g)
{
  REGION_CELL(g.nx - 5, g.ny - 5, 3, 3)
  w.ctx[(long)j * g.nx + i] = 0.5;
}

// blockIdx.y = field
__global__ __launch_bounds__(256) void k_bc2d(U2 u, G2 g, BcPack bc)
{
  const BcField b = bc_field(u.f, bc, blockIdx.y);
  bc2d_body(b, g, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

// vmax over the interior, grid-stride with one atomic per block.
__global__ __launch_bounds__(256) void k_cfl2d(U2 u, G2 g, StepInfo *info, double cfl, double vfloor,
                                               double dr, double dx, double dy, double dz)
{
  const long total = (long)(g.nx - 2 * g.xoff) * (g.ny - 2 * g.yoff);
  double v = 0.0;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
    const double vt = cfl2d_cell(u, g, t);
    if (vt > v) v = vt;
  }
  v = block_max<256>(v);
  if (threadIdx.x == 0) cfl_finish(info, v, cfl, vfloor, dr, dx, dy, dz);
}

// ------------------------------------------------------------------ driver
static void make_views(Handle *h, U2 &u0, U2 &u1, W2 &w, G2 &g)
{
  for (int n = 0; n < 8; n++) {
    u0.f[n] = h->U0[n];
    u1.f[n] = h->U1[n];
  }
  w.vx = h->prim[0]; w.vy = h->prim[1]; w.vz = h->prim[2]; w.pr = h->prim[3]; w.m2 = h->prim[4];
  w.cx = h->prim[5]; w.cy = h->prim[6];
  w.ctx = h->aux[0]; w.dvx = h->aux[3]; w.dvy = h->aux[4];
  for (int k = 0; k < 7; k++) {
    w.fx[k] = h->fx[k];
    w.fy[k] = h->fy[k];
  }
  w.fcx = h->fcx[0];
  w.fcy = h->fcy[0];
  w.ez = h->e[2];
  g.nx = h->g.nx; g.ny = h->g.ny; g.xoff = h->g.xoff; g.yoff = h->g.yoff; g.gamma = h->g.gamma;
}

// Marches that may start in the middle of a longest one (march_mid).
template <int MIX>
static bool split_march(int ch)
{
  return MIX != MLAU_FP64 && ch < kMarch;
}

// Faces per lane of the y sweep: march_chunk's choice, or 16, 4 or 8 with tune
// bits 0-1 = 1, 2 or 3.
static int ychunk(const Handle *h, const G2 &g)
{
  static const int fixed[4] = {0, 16, 4, 8};
  const int t = fixed[h->tune & 3];
  return t ? t : march_chunk((g.nx + 63) / 64, g.ny - 5, xsweep_waves(g.ny, g.nx), 0.5, kMarch,
                              h->s.precision != MLAU_FP64);
}

// Launches of both sweeps: `go` takes the kernel id, the grid, whether marches are split,
// their length and the number of y blocks.  Tune bit 6, for profiles of each sweep: one
// after the other, each as its part of the joint launch's blocks, the mixed forms in longest
// marches (same bits, march_mid).
template <int MIX, typename Go>
static void launch_sweeps2d(Handle *h, const G2 &g, int ch, int kx, int ky, Go go)
{
  const bool one_by_one = (h->tune & 64) != 0;
  if (one_by_one && split_march<MIX>(ch)) ch = kMarch;
  const unsigned px = (g.nx + 63) / 64, nyb = px * ((g.ny - 5 + ch - 1) / ch);
  const unsigned xw = (unsigned)xsweep_waves(g.ny, g.nx);
  if (one_by_one) {
    go(kx, dim3(xw), false, ch, px, 0u);
    go(ky, dim3(nyb), false, ch, px, nyb);
  } else {
    go(K_SWEEPS2D, dim3(nyb + xw), split_march<MIX>(ch), ch, px, nyb);
  }
}

template <int ODR, int FLUX, int MIX>
static void sweeps2d(Handle *h, const U2 &in, const W2 &w, const G2 &g)
{
  const int ch = whole_march<FLUX, MIX> ? kMarch : ychunk(h, g);
  launch_sweeps2d<MIX>(h, g, ch, K_XSWEEP2D, K_YSWEEP2D, [&](int k, dim3 gr, bool split, int c, unsigned px, unsigned nyb) {
    if constexpr (MIX != MLAU_FP64 && !whole_march<FLUX, MIX>) {
      if (split) {
        MLAU_LAUNCH(h, k, (k_sweeps2d<ODR, FLUX, MIX, true>), gr, dim3(64), in, w, g, c, px, nyb);
        return;
      }
    }
    if constexpr (two_waves<ODR, FLUX, MIX>) {
      if (gr.x > kTwoWaves) {
        MLAU_LAUNCH(h, k, (k_sweeps2d_two<ODR, FLUX, MIX, false>), gr, dim3(64), in, w, g, c, px, nyb);
        return;
      }
    }
    MLAU_LAUNCH(h, k, (k_sweeps2d<ODR, FLUX, MIX, false>), gr, dim3(64), in, w, g, c, px, nyb);
  });
}

// Primitives and weights in one pass, which forms the neighbours' velocities
// again, or in two: a small grid's pass is its launch and one cell's chain, a
// large one's its bytes.  Walls, 8 steps, us, two passes and one: MUSCL + MLAU 64^2 583
// and 546, 256^2 1002 and 957, 515x391 1505 and 1455, 1024^2 6261 and 6233, 1300^2
// 10152 and 10193; WCNS4 + LHLLD 64^2 631 and 597, 1024^2 7914 and 7875, 1300^2 12509
// and 12554, 2048^2 32554 and 32728; mixed 515x391 1359 and 1320, 1300^2 8574 and
// 8595, 2048^2 22045 and 22191.  Tune bit 2: the other choice.
static bool one_prim_pass(const Handle *h, const G2 &g)
{
  return ((long)g.nx * g.ny < (5L << 18)) != ((h->tune & 4) != 0);
}

template <int ODR, int FLUX, int MIX>
static void stage2d(Handle *h, const U2 &in, const U2 &ut, const U2 &out, const W2 &w, const G2 &g, double ra,
                    double rb, int adv)
{
  const int nx = g.nx, ny = g.ny;
  dim3 b256(256);
  dim3 gcell(region_pieces(nx, ny));
  if (!one_prim_pass(h, g)) {
    MLAU_LAUNCH(h, K_PRIM2D, (k_prim2d<ODR>), gcell, b256, in, w, g, h->bc);
    if (h->s.ctw) MLAU_LAUNCH(h, K_AUX2D, (k_aux2d<1>), gcell, b256, in, w, g, h->bc);
    else MLAU_LAUNCH(h, K_AUX2D, (k_aux2d<0>), gcell, b256, in, w, g, h->bc);
  } else if (h->s.ctw) {
    MLAU_LAUNCH(h, K_PRIMAUX2D, (k_primaux2d<ODR, 1>), gcell, b256, in, w, g, h->bc);
  } else {
    MLAU_LAUNCH(h, K_PRIMAUX2D, (k_primaux2d<ODR, 0>), gcell, b256, in, w, g, h->bc);
  }
  sweeps2d<ODR, FLUX, MIX>(h, in, w, g);
  MLAU_LAUNCH(h, K_EZ2D, (k_ez2d<ODR>), dim3(region_pieces(nx - 5, ny - 5)), b256, w, g);
  if (h->periodic_images && !(h->tune & 16)) {  // tune bit 4: separate boundary pass
    const dim3 gp(region_pieces(nx - 2 * g.xoff, ny - 2 * g.yoff));
    if (ra == 0.0) MLAU_LAUNCH(h, K_UPD2D, (k_update2d_per<ODR, true>), gp, b256, in, ut, out, w, g, h->info, ra, rb, adv);
    else MLAU_LAUNCH(h, K_UPD2D, (k_update2d_per<ODR, false>), gp, b256, in, ut, out, w, g, h->info, ra, rb, adv);
    return;
  }
  const dim3 gu(region_pieces(nx - 2 * g.xoff + 1, ny - 2 * g.yoff + 1));
  if (ra == 0.0)
    MLAU_LAUNCH(h, K_UPD2D, (k_update2d<ODR, true>), gu, b256, in, ut, out, w, g, h->info, ra, rb, adv);
  else
    MLAU_LAUNCH(h, K_UPD2D, (k_update2d<ODR, false>), gu, b256, in, ut, out, w, g, h->info, ra, rb, adv);
  const long nframe = (long)ny * 2 * g.xoff + (long)2 * g.yoff * nx;
  MLAU_LAUNCH(h, K_BC2D, k_bc2d, dim3((unsigned)((nframe + 255) / 256), 8), b256, out, g, bc_pack(h->bc));
}

template <int ODR, int FLUX, int MIX, int CTW>
static void sweeps2d_inl(Handle *h, const U2 &in, const W2 &w, const G2 &g)
{
  if constexpr (MIX != MLAU_FP64 || ODR == 1) {  // x_beside_2d
    const int ch = ychunk(h, g);
    if (!(h->tune & 64) && !split_march<MIX>(ch)) {
      const unsigned px = (g.nx + 63) / 64, nyb = px * ((g.ny - 5 + ch - 1) / ch);
      const unsigned xb = (unsigned)((xsweep_waves(g.ny, g.nx) + 3) / 4);
      if (run_beside(
              h,
              [&] { MLAU_LAUNCH(h, K_XSW2D_INL, (k_xsweep2d_inl<ODR, FLUX, MIX>), dim3(xb), dim3(256), in, w, g); },
              [&] {
                MLAU_LAUNCH(h, K_YSW2D_INL, (k_sweeps2d_inl<ODR, FLUX, MIX, CTW, false>), dim3(nyb), dim3(64), in, w, g,
                            ch, px, nyb);
              }))
        return;
    }
  }
  launch_sweeps2d<MIX>(h, g, ychunk(h, g), K_XSW2D_INL, K_YSW2D_INL,
                       [&](int k, dim3 gr, bool split, int c, unsigned px, unsigned nyb) {
    if constexpr (MIX != MLAU_FP64) {
      if (split) {
        MLAU_LAUNCH(h, k, (k_sweeps2d_inl<ODR, FLUX, MIX, CTW, true>), gr, dim3(64), in, w, g, c, px, nyb);
        return;
      }
    }
    if constexpr (two_waves_inl<ODR, FLUX, MIX>) {
      if (gr.x > kTwoWaves) {
        MLAU_LAUNCH(h, k, (k_sweeps2d_inl_two<ODR, FLUX, MIX, CTW, false>), gr, dim3(64), in, w, g, c, px, nyb);
        return;
      }
    }
    MLAU_LAUNCH(h, k, (k_sweeps2d_inl<ODR, FLUX, MIX, CTW, false>), gr, dim3(64), in, w, g, c, px, nyb);
  });
}

// Periodic grids (with room for the ghost images written by the update): the
// stage without primitive arrays.
template <int ODR, int FLUX, int MIX>
static void stage2d_inl(Handle *h, const U2 &in, const U2 &ut, const U2 &out, const W2 &w, const G2 &g, double ra,
                        double rb, int adv)
{
  if (h->s.ctw) sweeps2d_inl<ODR, FLUX, MIX, 1>(h, in, w, g);
  else sweeps2d_inl<ODR, FLUX, MIX, 0>(h, in, w, g);
  if (!h->s.ctw) {  // constant weight 1/2 (aux2d_body with CTW 0) over the corners the E-field reads
    const dim3 gc(region_pieces(g.nx - 5, g.ny - 5));
    MLAU_LAUNCH(h, K_AUX2D, k_ctx_half2d, gc, dim3(256), w, g);
  }
  MLAU_LAUNCH(h, K_EZ2D, (k_ez2d<ODR>), dim3(region_pieces(g.nx - 5, g.ny - 5)), dim3(256), w, g);
  const dim3 gp(region_pieces(g.nx - 2 * g.xoff, g.ny - 2 * g.yoff));
  if (ra == 0.0) MLAU_LAUNCH(h, K_UPD2D, (k_update2d_per<ODR, true>), gp, dim3(256), in, ut, out, w, g, h->info, ra, rb, adv);
  else MLAU_LAUNCH(h, K_UPD2D, (k_update2d_per<ODR, false>), gp, dim3(256), in, ut, out, w, g, h->info, ra, rb, adv);
}

// The stage without primitive arrays applies to periodic grids whose interior
// spans two ghost widths per axis, unless tune bit 5 asks for the separate
// prim/aux passes (or bit 4 for those with a boundary pass).
static bool inline2d(const Handle *h) { return h->periodic_images && !(h->tune & (16 | 32)); }

template <int ODR, int FLUX, int MIX>
static void step2d(Handle *h)
{
  U2 u0, u1;
  W2 w;
  G2 g;
  make_views(h, u0, u1, w, g);
  const int R_K = h->s.rk;
  const double rkf[3][2] = {{0.0, 1.0}, {0.5 + (R_K - 2) * 0.25, 0.5 - (R_K - 2) * 0.25}, {1. / 3., 2. / 3.}};
  const bool inl = inline2d(h);
  for (int rk = 0; rk < R_K; rk++) {
    const U2 &in = (rk == 0) ? u0 : u1;
    const U2 &out = (rk == R_K - 1) ? u0 : u1;
    const int adv = rk == R_K - 1;
    if (inl) stage2d_inl<ODR, FLUX, MIX>(h, in, u0, out, w, g, rkf[rk][0], rkf[rk][1], adv);
    else stage2d<ODR, FLUX, MIX>(h, in, u0, out, w, g, rkf[rk][0], rkf[rk][1], adv);
  }
}

typedef void (*Step2Fn)(Handle *);
template <int ODR, int MIX>
static Step2Fn pick2f(int flux)
{
  switch (flux) {
  case FLUX_MLAU: return step2d<ODR, FLUX_MLAU, MIX>;
  case FLUX_ROE: return step2d<ODR, FLUX_ROE, MIX>;
  case FLUX_HLLD: return step2d<ODR, FLUX_HLLD, MIX>;
  default: return step2d<ODR, FLUX_LHLLD, MIX>;
  }
}
template <int ODR>
static Step2Fn pick2(int flux, int precision)
{
  switch (precision) {
  case MLAU_MIXED: return pick2f<ODR, MLAU_MIXED>(flux);
  case MLAU_MIXED_RECON: return pick2f<ODR, MLAU_MIXED_RECON>(flux);
  default: return pick2f<ODR, MLAU_FP64>(flux);
  }
}

// Periodic grids whose x sweep, which alone fits three wavefronts a SIMD where the joint launch
// fits two, runs in a launch of its own beside the y sweep: it pays where the sweeps are light beside
// their bytes and the grid is large enough to hide the fork and join. us a step, before the sweeps
// shared a launch, in one launch, beside each other: mixed MUSCL + HLLD 1000^2 393, 408, 403, 1500^2 1005, 1078, 1018,
// 2048^2 1933, 2087, 1956;
// mixed_recon 2048^2 2071, 2257, 2152; mixed WCNS4 + LHLLD 1500^2 1342, 1333, 1360, 1750^2 1814, 1843, 1813, 2048^2 2457, 2568,
// 2485; FP64 ODR 1 + HLLD 1250^2 754, 741, 754, 1500^2 1109, 1140, 1108. mixed_recon + MLAU, whose solver keeps the
// x sweep to two wavefronts, and the other FP64 forms stay in one launch (WCNS4 + MLAU 2048^2 2826, 2756, 2845).
bool x_beside_2d(const Handle *h)
{
  const int odr = h->s.odr, flux = h->s.flux, mix = h->s.precision;
  if (!inline2d(h) || (mix == MLAU_FP64 && odr != 1) || (mix != MLAU_MIXED && flux == FLUX_MLAU)) return false;
  if (mix == MLAU_MIXED && flux == FLUX_HLLD && odr == 2) return h->ncell >= 900000;
  const bool light = odr <= 2 && (flux == FLUX_HLLD || flux == FLUX_LHLLD);
  return h->ncell >= (light ? 2100000 : 3000000);
}

int run_cfl_2d(Handle *h, double cfl, double vfloor)
{
  U2 u0, u1;
  W2 w;
  G2 g;
  make_views(h, u0, u1, w, g);
  const long cells = (long)(g.nx - 2 * g.xoff) * (g.ny - 2 * g.yoff);
  const unsigned nb = cfl_blocks(cells);
  const double dr = (h->g.dx < h->g.dy) ? h->g.dx : h->g.dy;
  MLAU_LAUNCH(h, K_CFL2D, k_cfl2d, dim3(nb), dim3(256), u0, g, h->info, cfl, vfloor, dr, h->g.dx, h->g.dy, h->g.dz);
  return (int)hipGetLastError();
}

int run_steps_2d(Handle *h, int nsteps, bool cfl_mode, double cfl, double vfloor)
{
  Step2Fn fn;
  switch (h->s.odr) {
  case 1: fn = pick2<1>(h->s.flux, h->s.precision); break;
  case 2: fn = pick2<2>(h->s.flux, h->s.precision); break;
  case 3: fn = pick2<3>(h->s.flux, h->s.precision); break;
  default: fn = pick2<4>(h->s.flux, h->s.precision); break;
  }
  for (int n = 0; n < nsteps; n++) {
    fn(h);  // its last update advances the time
    if (cfl_mode) run_cfl_2d(h, cfl, vfloor);
  }
  return (int)hipGetLastError();
}

}  // namespace mlau
