// mlau_ens1d.hip -- batched 1D members of the ensemble engine.
//
// A 1D member keeps the dt of its first step, so the steps of one launch share
// one plan, fill, CFL and dt; a member that ends among them is halted, and the
// bookkeeping between two steps runs in a block of its own of the next first
// sweep (five launches of little work per step took 60 of its 100 us).  A 1D stage is a sweep (primitives formed per stencil point) and an
// update that also runs the open boundary on stage 0 and writes periodic
// ghosts with their source cells, as the single-grid path; at odr <= 2 with
// rk >= 2 the later stages are one launch each (k_ens_stage1d, flux and update
// per wavefront) writing a third state.  Groups of a few open members at odr <= 2
// take whole steps in windows instead (k_ens_win1d).  Following the 1D driver (1D/SERIAL/shock/main.cpp:
// 113-130) the CFL step is taken once from the initial state over all cells
// (|vx| + c_f) and kept; only the last step is clipped at the end time.
// Tiles run the device bodies of mlau_1d_body.h on each member's arrays.
#include <cstring>

#include "mlau_1d_body.h"
#include "mlau_ens.h"

namespace mlau {

struct EnsRec1D {
  U1d u0, u1;
  U1d u2;  // third state of the fused stages (aliases w.fx, which they do not use)
  W1d w;
  G1d g;
  int flux, bc1d;
};

enum { T1_CFL = 0, T1_SWEEP, T1_OBC, T1_UPD, T1_FUSE, T1_WIN, T1_N };

// Kernel variant: 1 = stages after the first fused (odr <= 2, rk >= 2), 2 = also,
// with an open boundary, windows that take several steps per launch while the
// group has few tiles (windows1d).
static int variant1d(const mlau_member &m, int flags)
{
  if ((flags & MLAU_ENS_UNFUSED) || m.scheme.odr > 2 || m.scheme.rk < 2) return 0;
  return m.scheme.bc1d == MLAU_BC1D_OPEN ? 2 : 1;
}

constexpr int kWinSteps = 4;  // most steps of a window launch
// Cells lost at each side of a window over kWinSteps steps: stage 1 leaves the
// window's outer 4 cells stale, each further one the reach of its stencils more.
__host__ __device__ __forceinline__ int win_halo(int rk) { return 4 + (kWinSteps * rk - 1) * kReach<2>; }
__host__ __device__ __forceinline__ int win_own(int rk) { return kWin1 - 2 * win_halo(rk); }

static long long tiles1d(const mlau_grid &g, int kind, int)
{
  const long long nx = g.nx;
  switch (kind) {
  case T1_CFL: return (nx + 255) / 256;
  case T1_SWEEP: return ((nx - 5 + 62) / 63 + 3) / 4;
  case T1_UPD: return (nx - 8 + 255) / 256;
  default: return 0;  // T1_OBC depends on the boundary kind (tiles1d_member)
  }
}

static size_t arrays1d(const mlau_grid &) { return 7 + 7 + 4 + 7; }

static void record1d(void *out, const mlau_member &m, double *base, size_t per)
{
  EnsRec1D r{};
  size_t k = 0;
  auto take = [&]() { return base + (k++) * per; };
  for (int n = 0; n < 7; n++) r.u0.f[n] = take();
  for (int n = 0; n < 7; n++) r.u1.f[n] = take();
  r.w.vx = take(); r.w.vy = take(); r.w.vz = take(); r.w.pr = take();
  for (int n = 0; n < 7; n++) r.w.fx[n] = take();
  for (int n = 0; n < 7; n++) r.u2.f[n] = r.w.fx[n];
  r.g.nx = m.grid.nx; r.g.xoff = m.grid.xoff; r.g.gamma = m.grid.gamma; r.g.bx = m.grid.bx;
  r.flux = m.scheme.flux;
  r.bc1d = m.scheme.bc1d;
  memcpy(out, &r, sizeof r);
}

static void state1d(const void *rec, double **u0, int *nf, size_t *cells)
{
  const EnsRec1D *r = (const EnsRec1D *)rec;
  for (int n = 0; n < 7; n++) u0[n] = r->u0.f[n];
  *nf = 7;
  *cells = (size_t)r->g.nx;
}

// Tile counts that depend on the member's boundary kind.
static long long tiles1d_member(const mlau_member &m, int kind, int tune, int variant)
{
  if (kind == T1_WIN) return variant == 2 ? (m.grid.nx - 8 + win_own(m.scheme.rk) - 1) / win_own(m.scheme.rk) : 0;
  if (kind == T1_OBC) return m.scheme.bc1d == MLAU_BC1D_OPEN ? 1 : 0;
  if (kind == T1_FUSE) return variant ? ((m.grid.nx - 8 + 61) / 62 + 3) / 4 : 0;  // 4 wavefronts of 62 cells
  return tiles1d(m.grid, kind, tune);
}

// A member's clock over several steps of its fixed dt (ens_dt_slot and
// ens_advance_slot step by step), the same in every tile of the member.
struct WinClock {
  double dt = 0.0, tim, dtc, tend, dx;
  long long nstep, max_steps;
  bool last = false, ended;
  __device__ __forceinline__ explicit WinClock(const EnsState &S)
      : tim(S.tim), dtc(S.dtc), tend(S.tend), dx(S.dx), nstep(S.nstep), max_steps(S.max_steps), ended(S.halt != 0)
  {
  }
  __device__ __forceinline__ bool next()  // one more step, with its dt; false once the member has ended
  {
    if (ended) return false;
    dt = dtc;
    if (tim + dt >= tend) {
      dt = tend - tim;
      last = true;
    }
    tim = last ? tend : tim + dt;
    nstep += 1;
    ended = last || (max_steps > 0 && nstep >= max_steps);
    return true;
  }
};

// ------------------------------------------------------------------ kernels
#define ENS_LOOP(KIND)                                                           \
  for (PRange r_ = pers_range(count[KIND]); r_.t < r_.end; r_.t += r_.stride) { \
    const int2 e_ = tiles[r_.t];                                                 \
    const EnsRec1D &R = rec[e_.x];                                               \
    const unsigned l_ = (unsigned)e_.y;

// CFL speed over all cells, first step of each member only.
__global__ __launch_bounds__(256) void k_ens_cfl1d(const EnsRec1D *__restrict__ rec, EnsState *st,
                                                   const int2 *__restrict__ tiles, const int *__restrict__ count)
{
  __shared__ double red[4];
  ENS_LOOP(T1_CFL)
    if (st[e_.x].nstep > 0) continue;  // uniform per tile
    const int i = l_ * 256 + threadIdx.x;
    const double v = (i < R.g.nx) ? cfl1d_cell_checked(R.u0, R.g, i) : 0.0;
    ens_vmax_block(v, &st[e_.x].vmax_bits, red);
  }
}

// instantiated per Riemann solver (a group holds one solver)
template <int ODR, int FLUX, int MIX>
__global__ __launch_bounds__(256) void k_ens_sweep1d(const EnsRec1D *__restrict__ rec,
                                                     const int2 *__restrict__ tiles, const int *__restrict__ count,
                                                     int sin, EnsPlan p, int next)
{
  ENS_LOOP(T1_SWEEP)
    sweep1d_body<ODR, FLUX, MIX>(sin ? R.u1 : R.u0, R.w, R.g, l_, threadIdx.x);
  }
  // The first sweep of a step reads no dt: its last block, which has no tiles,
  // ends the members' previous step and forms this one's dt meanwhile.
  if (next && blockIdx.x == gridDim.x - 1)
    for (int s = threadIdx.x; s < kEnsSlots; s += blockDim.x)
      if (p.act[s] && ens_advance_slot(p, s)) ens_dt_slot(p, s);
}

// stage 0 only: the stage input is u0; ghosts go to u0 and u1
__global__ __launch_bounds__(64) void k_ens_openbc1d(const EnsRec1D *__restrict__ rec, const EnsState *st,
                                                     const int2 *__restrict__ tiles, const int *__restrict__ count)
{
  ENS_LOOP(T1_OBC)
    if (st[e_.x].halt) continue;  // failed at this step's CFL check, or ended
    (void)l_;
    openbc1d_body(R.u0, R.u0, R.u1, R.g, st[e_.x].dtdx, threadIdx.x);
  }
}

// obc (stage 0 of RK2/RK3): the open-boundary tiles run in the same launch
// (the boundary reads u0 and writes ghosts only; the update reads interior
// cells of u0 and writes u1).
template <int ODR>
__global__ __launch_bounds__(256) void k_ens_update1d(const EnsRec1D *__restrict__ rec, const EnsState *st,
                                                      const int2 *__restrict__ tiles, const int2 *__restrict__ otiles,
                                                      const int *__restrict__ count, int sin, int sout, double ra,
                                                      double rb, int obc)
{
  ENS_LOOP(T1_UPD)
    if (st[e_.x].halt) continue;  // failed at this step's CFL check, or ended
    const U1d in = sin ? R.u1 : R.u0, out = sout ? R.u1 : R.u0;
    if (R.bc1d == MLAU_BC1D_PERIODIC)
      update1d_body<ODR, true>(in, R.u0, out, R.w, R.g, st[e_.x].dtdx, ra, rb, l_, threadIdx.x);
    else
      update1d_body<ODR, false>(in, R.u0, out, R.w, R.g, st[e_.x].dtdx, ra, rb, l_, threadIdx.x);
  }
  if (!obc) return;
  tiles = otiles;
  ENS_LOOP(T1_OBC)
    if (st[e_.x].halt) continue;  // failed at this step's CFL check, or ended
    (void)l_;
    openbc1d_body(R.u0, R.u0, R.u1, R.g, st[e_.x].dtdx, threadIdx.x);
  }
}
// stages after the first: tile = 4 wavefronts of stage1d_body (62 cells each);
// sin/sout: 0 = u0, 1 = u1, 2 = u2
__device__ __forceinline__ U1d ubuf1(const EnsRec1D &R, int s) { return s == 0 ? R.u0 : (s == 1 ? R.u1 : R.u2); }

template <int ODR, int FLUX, int MIX>
__global__ __launch_bounds__(256) void k_ens_stage1d(const EnsRec1D *__restrict__ rec, const EnsState *st,
                                                     const int2 *__restrict__ tiles, const int *__restrict__ count,
                                                     int sin, int sout, double ra, double rb)
{
  ENS_LOOP(T1_FUSE)
    if (st[e_.x].halt) continue;  // failed at this step's CFL check, or ended
    const U1d in = ubuf1(R, sin), out = ubuf1(R, sout);
    const double dtdx = st[e_.x].dtdx;
    const unsigned wave = l_ * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (R.bc1d == MLAU_BC1D_PERIODIC)
      stage1d_body<ODR, FLUX, MIX, true>(in, R.u0, out, R.g, dtdx, ra, rb, wave, lane, false);
    else  // the open boundary's ghosts, fixed over the step, go into u2 with it
      stage1d_body<ODR, FLUX, MIX, false>(in, R.u0, out, R.g, dtdx, ra, rb, wave, lane, sout == 2);
  }
}

// ------------------------------------------------------------------ windows
// Up to kWinSteps whole steps of members with an open boundary at odr <= 2 and
// rk >= 2: a tile advances kWin1 consecutive cells of the member, held in LDS,
// by the bodies that the stage launches run on whole grids (a window is a small
// grid whose outer cells lose their meaning by the stencils' reach per stage, so
// that win_own cells are left), and writes those from u0 to u1 or back.  The bodies
// get the grid's constants anew at each call: the mixed forms fuse
// multiply-adds within a basic block, and products of constants hoisted out of
// the loop over steps would be rounded otherwise than in the stage launches.
// What bounds a step of few members is the chain of three stages' cells and, as
// four launches, the gaps between them: 5000 cells, MLAU, odr 2, rk 3 took 31.9
// us a step in mixed precision (36.2 in FP64) for 1 to 16 members, now 12.7 (17.4).
// Four steps a launch: two take 14.2 us, and six or eight, of which fewer cells
// are left (146 and 110), 12.4, but 1.2 and 1.5 times as long on 24 members.
struct LdsWin1d {
  double u[3][7][kWin1];  // u0, u1 and u2 (with stage 0's fluxes in its place)
};
__device__ __forceinline__ G1d win_grid(int W, double gamma, double bx)
{
  G1d g;
  g.nx = W;
  g.xoff = 4;
  g.gamma = gamma;
  g.bx = bx;
  asm volatile("" : "+s"(g.bx), "+s"(g.gamma));
  return g;
}

// One step of a window of W cells; e0, e1: its ends are the grid's.  320 threads.
template <int ODR, int FLUX, int MIX>
__device__ __forceinline__ void win1d_step(LdsWin1d &S, int W, double gamma, double bx, double dtdx, int rk, bool e0,
                                           bool e1, unsigned tid)
{
  U1d u0, u1, u2;
  W1d w{};
#pragma unroll
  for (int n = 0; n < 7; n++) {
    u0.f[n] = S.u[0][n];
    u1.f[n] = S.u[1][n];
    u2.f[n] = S.u[2][n];
    w.fx[n] = S.u[2][n];
  }
  const unsigned lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double vals[7];
  if (wave < 4) {
    sweep1d_body<ODR, FLUX, MIX>(u0, w, win_grid(W, gamma, bx), 0, tid);
  } else if (e0 || e1) {  // the ends' new ghosts: even lanes left, odd lanes right
    const int side = lane & 1, si = side ? W - 5 : 4, so = side ? W - 4 : 3;
    double q[7][2];
    prim1d_pair(u0, si, so, gamma, bx, q);
    G1d g;
    g.nx = W;
    g.xoff = 4;
    g.gamma = gamma;
    g.bx = bx;
    openbc1d_cell<false>(q, g, dtdx, side, vals);
  }
  __syncthreads();
  if (wave < 4) {
    update1d_body<ODR, false>(u0, u0, u1, w, win_grid(W, gamma, bx), dtdx, 0.0, 1.0, 0, tid);
  } else if (lane < 8) {  // outer cells: new ghosts, or what the window's edge holds
    const int side = lane & 1, c = (side ? W - 4 : 0) + (lane >> 1);
    const bool end = side ? e1 : e0;
#pragma unroll
    for (int n = 0; n < 7; n++) {
      const double v = end ? vals[n] : u0.f[n][c];
      u0.f[n][c] = v;
      u1.f[n][c] = v;
    }
  }
  __syncthreads();
  const double rkf[3][2] = {{0.0, 1.0}, {0.5 + (rk - 2) * 0.25, 0.5 - (rk - 2) * 0.25}, {1. / 3., 2. / 3.}};
  for (int s = 1; s < rk; s++) {  // u1 -> u2 -> u0 or u1 -> u0
    if (wave < 4)
      stage1d_body<ODR, FLUX, MIX, false>(s == 1 ? u1 : u2, u0, s == rk - 1 ? u0 : u2, win_grid(W, gamma, bx), dtdx,
                                          s == 1 ? rkf[1][0] : rkf[2][0], s == 1 ? rkf[1][1] : rkf[2][1], wave, lane,
                                          s != rk - 1);
    __syncthreads();
  }
}

template <int ODR, int FLUX, int MIX>
__global__ __launch_bounds__(kWin1 + 64) void k_ens_win1d(const EnsRec1D *__restrict__ rec,
                                                          const EnsState *__restrict__ st,
                                                          const int2 *__restrict__ tiles,
                                                          const int *__restrict__ count, int sin, int done, int K,
                                                          int rk)
{
  __shared__ LdsWin1d S;
  ENS_LOOP(T1_WIN)
    const int nx = R.g.nx, W = nx < kWin1 ? nx : kWin1, own = win_own(rk);
    const int first = 4 + (int)l_ * own, last = first + own < nx - 4 ? first + own : nx - 4;
    int c0 = first - win_halo(rk);
    c0 = c0 > nx - W ? nx - W : c0;
    c0 = c0 < 0 ? 0 : c0;
    const bool e0 = c0 == 0, e1 = c0 + W == nx;
    const U1d in = sin ? R.u1 : R.u0, out = sin ? R.u0 : R.u1;
    const int t = (int)threadIdx.x;
    if (t < W)
#pragma unroll
      for (int n = 0; n < 7; n++) S.u[0][n][t] = in.f[n][c0 + t];
    const double gamma = R.g.gamma, bx = R.g.bx;
    WinClock ck(st[e_.x]);
    for (int k = 0; k < done; k++) ck.next();  // the steps of the launches before this one
    __syncthreads();
    for (int k = 0; k < K && ck.next(); k++)
      win1d_step<ODR, FLUX, MIX>(S, W, gamma, bx, ck.dt / ck.dx, rk, e0, e1, threadIdx.x);
    const int c = c0 + t;
    if (t < W && ((c >= first && c < last) || (c < 4 && first == 4) || (c >= nx - 4 && last == nx - 4)))
#pragma unroll
      for (int n = 0; n < 7; n++) out.f[n][c] = S.u[0][n][t];
    __syncthreads();
  }
}

// The members' clocks after the n steps that the windows took.
__global__ __launch_bounds__(256) void k_ens_win_clock(EnsPlan p, int n)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= kEnsSlots || !p.act[s] || p.stat[s] != MLAU_MEMBER_RUNNING) return;
  EnsState &S = p.st[s];
  WinClock ck(S);
  for (int k = 0; k < n && ck.next(); k++) {
    S.dt = ck.dt;
    S.dtdx = ck.dt / S.dx;
    S.dtdy = ck.dt / S.dy;
    S.dtdz = ck.dt / S.dz;
  }
  S.tim = ck.tim;
  S.nstep = ck.nstep;
  if (ck.ended) {
    p.stat[s] = ck.last ? MLAU_MEMBER_DONE : MLAU_MEMBER_CAPPED;
    S.last = ck.last;
    S.halt = 1;
  }
  S.vmax_bits = (unsigned long long)__double_as_longlong(S.vfloor);
}
#undef ENS_LOOP

// ------------------------------------------------------------------- driver
static unsigned pers_blocks1(const Ensemble *e)
{
  const int m = (e->tune >> 4) & 15;
  return (unsigned)((m ? m : 2) * ens_cus(e));
}

template <int ODR, int MIX>
static void sweep1d(Ensemble *e, int flux, unsigned pb, const EnsRec1D *rec, const EnsPlan &p, int sin, int next)
{
  pb += next;  // one block more than the whole sets of kXcds that share the tiles (pers_range)
  const int2 *t = (const int2 *)p.tiles[T1_SWEEP];
  const int *cnt = p.count;
  const dim3 b(256);
  switch (flux) {
  case FLUX_MLAU: ENS_LAUNCH(e, E_XSWEEP, (k_ens_sweep1d<ODR, FLUX_MLAU, MIX>), dim3(pb), b, rec, t, cnt, sin, p, next);
    break;
  case FLUX_ROE: ENS_LAUNCH(e, E_XSWEEP, (k_ens_sweep1d<ODR, FLUX_ROE, MIX>), dim3(pb), b, rec, t, cnt, sin, p, next);
    break;
  case FLUX_HLLD: ENS_LAUNCH(e, E_XSWEEP, (k_ens_sweep1d<ODR, FLUX_HLLD, MIX>), dim3(pb), b, rec, t, cnt, sin, p, next);
    break;
  default: ENS_LAUNCH(e, E_XSWEEP, (k_ens_sweep1d<ODR, FLUX_LHLLD, MIX>), dim3(pb), b, rec, t, cnt, sin, p, next);
    break;
  }
}

template <int ODR, int MIX>
static void stage1d(Ensemble *e, int flux, unsigned pb, const EnsRec1D *rec, const EnsPlan &p, int sin, int sout,
                    double ra, double rb)
{
  const int2 *t = (const int2 *)p.tiles[T1_FUSE];
  const int *cnt = p.count;
  const EnsState *st = p.st;
  const dim3 b(256);
  const dim3 g(pb);
  switch (flux) {
  case FLUX_MLAU:
    ENS_LAUNCH(e, E_STAGE, (k_ens_stage1d<ODR, FLUX_MLAU, MIX>), g, b, rec, st, t, cnt, sin, sout, ra, rb);
    break;
  case FLUX_ROE:
    ENS_LAUNCH(e, E_STAGE, (k_ens_stage1d<ODR, FLUX_ROE, MIX>), g, b, rec, st, t, cnt, sin, sout, ra, rb);
    break;
  case FLUX_HLLD:
    ENS_LAUNCH(e, E_STAGE, (k_ens_stage1d<ODR, FLUX_HLLD, MIX>), g, b, rec, st, t, cnt, sin, sout, ra, rb);
    break;
  default:
    ENS_LAUNCH(e, E_STAGE, (k_ens_stage1d<ODR, FLUX_LHLLD, MIX>), g, b, rec, st, t, cnt, sin, sout, ra, rb);
    break;
  }
}

template <int ODR, int MIX>
static int step1d_group(Ensemble *e, EnsGroup *G, bool first, bool last)
{
  const EnsPlan &p = G->p;
  const EnsRec1D *rec = (const EnsRec1D *)G->rec;
  const unsigned pb = pers_blocks1(e);
  const dim3 b256(256), b64(64), slots(kEnsSlots / 256);
  const int *cnt = p.count;
  if (first) {
    ENS_LAUNCH(e, E_PLAN, k_ens_plan, dim3(1), dim3(kPlanThreads), p, (int)T1_N);
    ENS_LAUNCH(e, E_FILL, k_ens_fill, dim3(kEnsSlots), b256, p, (int)T1_N);
    ENS_LAUNCH(e, E_CFL, k_ens_cfl1d, dim3(pb), b256, rec, p.st, (const int2 *)p.tiles[T1_CFL], cnt);
    ENS_LAUNCH(e, E_DT, k_ens_dt, slots, b256, p);
  }
  const int R_K = G->rk;
  const double rkf[3][2] = {{0.0, 1.0}, {0.5 + (R_K - 2) * 0.25, 0.5 - (R_K - 2) * 0.25}, {1. / 3., 2. / 3.}};
  for (int rk = 0; rk < R_K; rk++) {
    if constexpr (ODR <= 2) {
      if (G->variant && rk > 0) {  // u1 -> u2 -> u0 (rk 3) or u1 -> u0 (rk 2)
        stage1d<ODR, MIX>(e, G->flux, pb, rec, p, rk == 1 ? 1 : 2, rk == R_K - 1 ? 0 : 2, rkf[rk][0], rkf[rk][1]);
        continue;
      }
    }
    const int sin = (rk == 0) ? 0 : 1;
    const int sout = (rk == R_K - 1) ? 0 : 1;
    sweep1d<ODR, MIX>(e, G->flux, pb, rec, p, sin, rk == 0 && !first);
    const int obc = rk == 0 && R_K > 1;  // RK1 updates in place: boundary first, separately
    if (rk == 0 && !obc)
      ENS_LAUNCH(e, E_BC, k_ens_openbc1d, dim3(e->cus), b64, rec, (const EnsState *)p.st,
                 (const int2 *)p.tiles[T1_OBC], cnt);
    ENS_LAUNCH(e, E_UPD, (k_ens_update1d<ODR>), dim3(pb), b256, rec, (const EnsState *)p.st,
               (const int2 *)p.tiles[T1_UPD], (const int2 *)p.tiles[T1_OBC], cnt, sin, sout, rkf[rk][0], rkf[rk][1],
               obc);
  }
  if (last) ENS_LAUNCH(e, E_ADVANCE, k_ens_advance, slots, b256, p);
  return (int)hipGetLastError();
}

typedef int (*EnsStepFn)(Ensemble *, EnsGroup *, bool, bool);

template <int ODR>
static EnsStepFn pick1_odr(int precision)
{
  switch (precision) {
  case MLAU_MIXED: return step1d_group<ODR, MLAU_MIXED>;
  case MLAU_MIXED_RECON: return step1d_group<ODR, MLAU_MIXED_RECON>;
  default: return step1d_group<ODR, MLAU_FP64>;
  }
}

template <int ODR, int MIX>
static int win1d_group(Ensemble *e, EnsGroup *G, int n)
{
  const EnsPlan &p = G->p;
  const EnsRec1D *rec = (const EnsRec1D *)G->rec;
  const EnsState *st = p.st;
  const unsigned pb = pers_blocks1(e);
  const dim3 b256(256), slots(kEnsSlots / 256), g(pb), b(kWin1 + 64);
  const int *cnt = p.count;
  ENS_LAUNCH(e, E_PLAN, k_ens_plan, dim3(1), dim3(kPlanThreads), p, (int)T1_N);
  ENS_LAUNCH(e, E_FILL, k_ens_fill, dim3(kEnsSlots), b256, p, (int)T1_N);
  ENS_LAUNCH(e, E_CFL, k_ens_cfl1d, dim3(pb), b256, rec, p.st, (const int2 *)p.tiles[T1_CFL], cnt);
  ENS_LAUNCH(e, E_DT, k_ens_dt, slots, b256, p);
  const int2 *t = (const int2 *)p.tiles[T1_WIN];
  const int m = (n + 2 * kWinSteps - 1) / (2 * kWinSteps) * 2;  // an even number of launches ends in u0
  for (int j = 0; j < m; j++) {
    const int done = (int)((long)n * j / m), K = (int)((long)n * (j + 1) / m) - done, sin = j & 1;
    switch (G->flux) {
    case FLUX_MLAU:
      ENS_LAUNCH(e, E_STAGE, (k_ens_win1d<ODR, FLUX_MLAU, MIX>), g, b, rec, st, t, cnt, sin, done, K, G->rk);
      break;
    case FLUX_ROE:
      ENS_LAUNCH(e, E_STAGE, (k_ens_win1d<ODR, FLUX_ROE, MIX>), g, b, rec, st, t, cnt, sin, done, K, G->rk);
      break;
    case FLUX_HLLD:
      ENS_LAUNCH(e, E_STAGE, (k_ens_win1d<ODR, FLUX_HLLD, MIX>), g, b, rec, st, t, cnt, sin, done, K, G->rk);
      break;
    default:
      ENS_LAUNCH(e, E_STAGE, (k_ens_win1d<ODR, FLUX_LHLLD, MIX>), g, b, rec, st, t, cnt, sin, done, K, G->rk);
      break;
    }
  }
  ENS_LAUNCH(e, E_ADVANCE, k_ens_win_clock, slots, b256, p, n);
  return (int)hipGetLastError();
}

template <int ODR>
static int win1d_odr(Ensemble *e, EnsGroup *G, int n)
{
  switch (G->precision) {
  case MLAU_MIXED: return win1d_group<ODR, MLAU_MIXED>(e, G, n);
  case MLAU_MIXED_RECON: return win1d_group<ODR, MLAU_MIXED_RECON>(e, G, n);
  default: return win1d_group<ODR, MLAU_FP64>(e, G, n);
  }
}

// Windows while they fill the CUs at most three times (one block of 320 threads
// per CU by its registers): a window forms 256 cells for the 182 it gives, so
// a full chip is left to the stages.  Members of 5000 cells, 28 windows each, in
// FP64 as stages and as windows, us a step: 16 members 42.1 and 30.5, 24 44.0 and
// 41.0, 32 54.1 and 55.9, 128 156 and 189.  One step by itself takes two launches of windows
// too, so only while they fill the CUs once: us a call, 256 windows 91 and 86, 352 91 and 104, 700
// 102 and 120 (two steps 136 and 100, 137 and 129, 160 and 158).  Members that ended are
// taken to be of the mean size.  Both give the same bits, so a group may change over at any launch.
static bool windows1d(const Ensemble *e, const EnsGroup *G, int steps)
{
  if (G->variant != 2) return false;
  long long n = 0;
  for (int id : G->slot_id) n += id >= 0;
  return G->need[T1_WIN] * G->nrun <= (steps == 1 ? 1ll : 3ll) * ens_cus(e) * n;
}

// The plan, fill, CFL and dt passes once per 32 steps of windows: 14.7 us a step
// with 8 of them, 12.8 with 32, 12.7 with 64.
static int graph_steps1d(const Ensemble *e, const EnsGroup *G)
{
  return windows1d(e, G, 4 * e->gsteps) ? 4 * e->gsteps : e->gsteps;
}

static int launch_many1d(Ensemble *e, EnsGroup *G, int n)
{
  if (!windows1d(e, G, n)) return -1;
  const int most = graph_steps1d(e, G);
  for (; n > 0; n -= most) {
    const int k = n < most ? n : most;
    const int rc = G->odr == 1 ? win1d_odr<1>(e, G, k) : win1d_odr<2>(e, G, k);
    if (rc) return rc;
  }
  return 0;
}

static int launch1d(Ensemble *e, EnsGroup *G, bool first, bool last)
{
  EnsStepFn fn;
  switch (G->odr) {
  case 1: fn = pick1_odr<1>(G->precision); break;
  case 2: fn = pick1_odr<2>(G->precision); break;
  case 3: fn = pick1_odr<3>(G->precision); break;
  default: fn = pick1_odr<4>(G->precision); break;
  }
  return fn(e, G, first, last);
}

static const EnsDim kDim1d = {sizeof(EnsRec1D), T1_N, tiles1d_member, arrays1d, record1d, launch1d, state1d,
                              variant1d, launch_many1d, graph_steps1d};
const EnsDim *ens_dim1d() { return &kDim1d; }

}  // namespace mlau
