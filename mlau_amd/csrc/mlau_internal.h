// mlau_internal.h -- handle layout and launch helpers shared by the HIP
// translation units of libmlau_hip.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "mlau_common.h"

namespace mlau {

// Kernel identifiers for the per-kernel timing table.
enum KernelId {
  K_PRIM2D = 0, K_AUX2D, K_XSWEEP2D, K_YSWEEP2D, K_EZ2D, K_UPD2D, K_BC2D, K_CFL2D,
  K_SWEEP1D, K_OPENBC1D, K_UPD1D, K_CFL1D,
  K_PRIM3D, K_AUX3D, K_XSWEEP3D, K_YSWEEP3D, K_ZSWEEP3D, K_EDGE3D, K_UPD3D, K_BC3D, K_CFL3D,
  K_FINALIZE, K_PRIMAUX2D, K_STAGE1D, K_XSW2D_INL, K_YSW2D_INL, K_STEP1D, K_SWEEPS2D, K_SWEEPS3D, K_COUNT
};
extern const char *kKernelNames[K_COUNT];

struct Timing {
  bool enabled = false;
  std::vector<hipEvent_t> pool;       // free events
  struct Rec { int k; hipEvent_t a, b; };
  std::vector<Rec> pending;
  double total_ms[K_COUNT] = {};
  long long count[K_COUNT] = {};
};

// Boundary flags per field (field order), plus stagger flags.
struct BcFlags {
  int dnx[8], dny[8], dnz[8];
  int stx[8], sty[8], stz[8];
};

// Array and flags of one field.
struct BcField {
  double *f;
  int dnx, dny, dnz, stx, sty, stz;
};
// The flags of all fields as kernel arguments: two bits per field (dn + 1).
struct BcPack {
  unsigned x, y, z;
};
inline BcPack bc_pack(const BcFlags &bc)
{
  BcPack p{0, 0, 0};
  for (int n = 0; n < 8; n++) {
    p.x |= (unsigned)(bc.dnx[n] + 1) << (2 * n);
    p.y |= (unsigned)(bc.dny[n] + 1) << (2 * n);
    p.z |= (unsigned)(bc.dnz[n] + 1) << (2 * n);
  }
  return p;
}
// Field fld (the same in all threads of a block) out of kernel arguments.  A
// run-time index into arrays of arguments makes every thread copy them to LDS or
// scratch first (the 515x391 frame took 17 us instead of 6); the pointers pass
// through an empty asm so that their selects stay selects of scalar registers.
__device__ __forceinline__ BcField bc_field(double *const (&f)[8], BcPack p, int fld)
{
  double *at = nullptr;
#pragma unroll
  for (int n = 0; n < 8; n++) {
    double *a = f[n];
    asm("" : "+s"(a));
    at = fld == n ? a : at;
  }
  return BcField{at, (int)(p.x >> (2 * fld) & 3u) - 1, (int)(p.y >> (2 * fld) & 3u) - 1,
                 (int)(p.z >> (2 * fld) & 3u) - 1, fld == 5, fld == 6, fld == 7};
}

struct Handle {
  mlau_grid g;
  mlau_scheme s;
  BcFlags bc;
  int nf;                  // 7 (1D) or 8
  long long ncell;         // nx*ny*nz including ghosts
  hipStream_t stream = nullptr;
  // second stream, where the x sweep runs beside the others (large grids of some forms, else null)
  hipStream_t side = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  int device = 0;
  double *base = nullptr;  // one device allocation carved into the arrays below
  size_t base_bytes = 0;
  double *U0[8] = {};      // state (step start / result)
  double *U1[8] = {};      // stage state
  // scratch (meaning depends on dim; see the per-dim step files)
  double *prim[8] = {};    // vx,vy,vz,pr,m2,cx,cy,cz
  double *aux[6] = {};     // ct0,ct1,ct2,dvx,dvy,dvz
  double *fx[8] = {}, *fy[8] = {}, *fz[8] = {};
  double *fcx[2] = {}, *fcy[2] = {}, *fcz[2] = {};
  double *e[3] = {};       // ex,ey,ez (2D: ez only)
  double *lr = nullptr;    // 1D face states
  StepInfo *info = nullptr;  // device
  int tune = 0;              // launch-shape variant (autotuner choice), see the per-dim drivers
  bool periodic_images = false;  // 2D periodic: the update writes the ghost images (no boundary pass)
  Timing timing;
  // HIP graph of kGraphSteps steps (replayed by mlau_step / mlau_step_cfl)
  hipGraphExec_t gexec = nullptr;
  bool graph_off = false;    // MLAU_NO_GRAPH set at creation
  bool g_cfl_mode = false;
  double g_cfl = 0.0, g_vfloor = 0.0;
};

// error reporting (message kept per host thread for mlau_last_error)
int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *where);

// launch bookkeeping
void timing_begin(Handle *h, int k, hipEvent_t *a);
void timing_end(Handle *h, int k, hipEvent_t a);

#define MLAU_LAUNCH(h, kid, kernel, grid, block, ...)                                 \
  do {                                                                                \
    hipEvent_t _ev = nullptr;                                                         \
    if ((h)->timing.enabled) timing_begin((h), (kid), &_ev);                          \
    hipLaunchKernelGGL(kernel, grid, block, 0, (h)->stream, __VA_ARGS__);             \
    if ((h)->timing.enabled) timing_end((h), (kid), _ev);                             \
  } while (0)

// `beside` on the handle's side stream, between a fork from and a join into its own,
// and `here` on its own meanwhile; false (nothing launched) where there is no side stream.
template <typename A, typename B>
bool run_beside(Handle *h, A here, B beside)
{
  const hipStream_t own = h->stream;
  if (!h->side || hipEventRecord(h->ev_fork, own) != hipSuccess ||
      hipStreamWaitEvent(h->side, h->ev_fork, 0) != hipSuccess)
    return false;
  here();
  h->stream = h->side;
  beside();
  h->stream = own;
  if (hipEventRecord(h->ev_join, h->side) != hipSuccess || hipStreamWaitEvent(own, h->ev_join, 0) != hipSuccess)
    hipStreamSynchronize(h->side);
  return true;
}

// Whether a handle gets a side stream for its sweeps.
bool x_beside_2d(const Handle *h);
bool x_beside_3d(const Handle *h);

// per-dimension drivers (return hipError_t as int)
int run_steps_1d(Handle *h, int nsteps, bool cfl_mode, double cfl, double vfloor);
int run_steps_2d(Handle *h, int nsteps, bool cfl_mode, double cfl, double vfloor);
int run_steps_3d(Handle *h, int nsteps, bool cfl_mode, double cfl, double vfloor);
int run_cfl_1d(Handle *h, double cfl, double vfloor);
int run_cfl_2d(Handle *h, double cfl, double vfloor);
int run_cfl_3d(Handle *h, double cfl, double vfloor);

__global__ void k_set_dt(StepInfo *info, double dt, double dx, double dy, double dz);

// Argument checks of mlau_create (grid and scheme).
int mlau_validate(const mlau_grid *g, const mlau_scheme *s);

}  // namespace mlau
