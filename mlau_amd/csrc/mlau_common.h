// mlau_common.h -- host/device shared declarations of the HIP path.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/mlau.h"
#include "mlau_dev.h"

// Register budget of the marching sweeps: at most 256 VGPRs + AGPRs per lane,
// so two waves share each SIMD (one wave alone leaves the SIMD idle while it
// waits on the next row's loads).
#define MLAU_TWO_WAVES __attribute__((amdgpu_waves_per_eu(2)))

namespace mlau {

// Per-step scalars kept on the device so a step loop never waits on the host:
// dt and the ratios the reference forms once per call (dtdx=dt/dx, ...).
struct StepInfo {
  double dt, dtdx, dtdy, dtdz;
  double vmax;                    // last CFL speed (reference cflcheck vmax)
  unsigned long long vmax_bits;   // reduction accumulator (non-negative doubles order like their bits); 0 between checks
  double tim;                     // accumulated time (driver's tim+=dt)
  long long nstep;                // steps taken
  unsigned blocks_done;           // blocks of the running check that have added their maximum; 0 between checks
};

// Ghost-cell source of one axis under the reference's boundary rules
// (2D/SERIAL/OTvortex/boundary.c:18-74, 3D/MPI/OTvortex/boundary.c:91-309):
// periodic (dn==0) copies the image across the domain; Neumann/Dirichlet
// (dn=+1/-1) mirrors about the boundary (stagger st shifts the mirror and
// leaves one more face on the right to the solver) and multiplies by dn.
// Returns the source index; multiplies *sg by the factor.  Interior indices map
// to themselves.
__host__ __device__ __forceinline__ int bc_src(int i, int n, int off, int st, int dn, double *sg)
{
  if (dn == 0) {
    if (i < off) return n - 2 * off + i;
    if (i >= n - off) return i - (n - 2 * off);
    return i;
  }
  if (i < off) {
    *sg *= (double)dn;
    return 2 * off - 1 + st - i;
  }
  if (i >= n - (off - st)) {
    *sg *= (double)dn;
    return n - 2 * off + st + (n - 1 - i);
  }
  return i;
}

constexpr int kWave = 64;
constexpr unsigned kXcds = 8;  // MI355X: 8 accelerator dies, each with its own L2

// Workgroups are handed to the XCDs round-robin (block b -> XCD b % 8).  For
// stencils that reuse neighbouring rows, remap the linear block index so each
// XCD walks one contiguous band of the grid and finds its neighbours in its own
// L2.  A bijection on [0, nb).
__device__ __forceinline__ unsigned xcd_band(unsigned b, unsigned nb)
{
  const unsigned x = b % kXcds, k = b / kXcds;
  const unsigned q = nb / kXcds, r = nb % kXcds;
  return x * q + (x < r ? x : r) + k;
}

__device__ __forceinline__ double shfl_up1(double v)
{
  return __shfl_up(v, 1, kWave);
}

// Block-wide max of a non-negative speed (NaN never wins: comparisons with >
// as in the reference's "if (vtmp > vmax) vmax=vtmp"), in thread 0.
template <int BLOCK>
__device__ __forceinline__ double block_max(double v)
{
  __shared__ double red[BLOCK / 64];
  for (int o = 32; o > 0; o >>= 1) {
    const double t = __shfl_xor(v, o, 64);
    if (t > v) v = t;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int k = 1; k < BLOCK / 64; k++)
      if (red[k] > v) v = red[k];
  return v;
}

// End of a signal-speed check, called by one thread per block with the block's
// maximum, added as a bit pattern (non-negative doubles order like theirs).
// The count waits for the value that the maximum's atomic returns, so the last
// block to arrive sees every maximum; a fence in its place writes back each
// XCD's L2 per block (2048^2: +100 us a check, 128^3: +500).  That block turns the maximum (at least vfloor)
// into the next dt and the ratios the reference forms from it, and leaves the
// accumulator and the counter as it found them, so a check is one launch.  The
// reset before it and the dt after it as launches of their own, with the time
// advance (now in the last update), took 15 us of a 64^2 step's 83.
__device__ __forceinline__ void cfl_finish(StepInfo *info, double v, double cfl, double vfloor, double dr, double dx,
                                           double dy, double dz)
{
  unsigned one = 1u;
  if (v > 0.0) {
    unsigned long long was = atomicMax(&info->vmax_bits, (unsigned long long)__double_as_longlong(v));
    asm volatile("" : "+v"(was));
    one += (unsigned)(was == ~0ull);  // never: no sum or product of doubles has these bits
  }
  if (atomicAdd(&info->blocks_done, one) != gridDim.x - 1) return;
  unsigned long long bits = atomicExch(&info->vmax_bits, 0ull);
  const unsigned long long least = (unsigned long long)__double_as_longlong(vfloor);
  if (least > bits) bits = least;
  atomicExch(&info->blocks_done, 0u);
  const double vmax = __longlong_as_double((long long)bits);
  info->vmax = vmax;
  if (isfinite(vmax)) {
    const double dt = cfl * dr / vmax;
    info->dt = dt;
    info->dtdx = dt / dx;
    info->dtdy = dt / dy;
    info->dtdz = dt / dz;
  }
}

// Blocks of a signal-speed check over `cells` cells.  Each adds its maximum and
// its count to the same two words, about 18 ns apart, so few are better until the
// reads need more in flight: 200k cells take 19 us with 787 blocks, 13.8 with
// 512, 8.5-9 with 128-256; 4.2M cells 68 us with 256, 55 with 512, 58 with 1024.
inline unsigned cfl_blocks(long cells)
{
  const long most = cells < (1L << 20) ? 256 : 512, want = (cells + 511) / 512;
  return (unsigned)(want < most ? want : most);
}

// Advance of the step's time by block 0 of a step's last update (the other
// blocks read only the dt ratios).
__device__ __forceinline__ void advance_time(StepInfo *info)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    info->tim += info->dt;
    info->nstep += 1;
  }
}

// Wavefronts of the row-flattened x sweeps: cells 2..nx-3 of `rows` rows at a
// stride of 63 cells per 64-lane wavefront.
__host__ __device__ __forceinline__ long xsweep_waves(long rows, int nx) { return (rows * (nx - 4) - 1 + 62) / 63; }

// Faces per lane of a marching sweep (y in 2D, y and z in 3D).  A lane that
// marches ch faces reconstructs ch+1 cells one after the other: a long march
// wastes fewer reconstructions (1 in ch+1), a short one makes more wavefronts.
// Times in units of one cell's issue time on a SIMD (6.1 us at WCNS4 + LHLLD):
// the chip's 1024 SIMDs issue `pieces` columns of wavefronts marching the
// faces plus the `others` wavefronts of the sweeps that run beside this one;
// a wavefront with a SIMD to itself needs kLone of them per cell (7.5-9 us);
// and at the end a SIMD idles for `tail` of a march on average, less in 3D where the two other
// sweeps fill the gap.  Measured over 2D 64..2048 squared and 3D 24..128 cubed
// (8 steps, us), fixed chunk 8 (2D) and 16 (3D) -> this choice:
// 64^2 2268 -> 1045 (1 face), 256^2 2320 -> 1356 (1), 512^2 2774 -> 2497 (2), 768^2 4646 -> 4413 (4),
// 2048^2 27159 (8), 32^3 6211 -> 3713 (1), 64^3 6905 -> 5729 (4), 128^3 29220 -> 29190 (8);
// never more than 2 % above the best of 1, 2, 4, 8, 16.  `most` is 8 in 2D (16
// gained nothing there at any size) and 16 in 3D.
inline int march_chunk(long pieces, int faces, long others, double tail, int most, bool mixed)
{
  const double kSimds = 1024, kLone = 1.5;
  int best = 1;
  double least = 0.0;
  for (int ch = 1; ch <= most; ch *= 2) {
    const double cells = ch + (mixed && ch < most ? 1.6 : 1.0);  // a whole cell and a longer loop: march_mid
    const double issue = ((double)(pieces * ((faces + ch - 1) / ch)) * cells + (double)others) / kSimds;
    const double lone = kLone * (ch + 1);
    const double t = issue + tail * lone > lone ? issue + tail * lone : lone;
    if (ch == 1 || t < least) {
      least = t;
      best = ch;
    }
  }
  return best;
}

// Whether a march that starts at face 3 + ch*c begins in the middle of a march
// of `most` faces.  The left state of the cell below a march's first face
// comes from a copy of the reconstruction that makes nothing else, in which the
// compiler fuses other multiply-adds of the FP32 form than in the march's own
// copy: the mixed forms therefore take that copy at the cells where the longest
// march takes it and the march's own elsewhere, so that their results do not
// depend on the march length.  FP64 fuses nothing and always takes the short
// copy; so do longest marches, whose kernels are compiled without the choice
// (with it the 128^3 mixed sweeps took 1 % longer).
// The FP32 LHLLD solver and the contracted FP64 Roe solver themselves fuse otherwise in
// the kernels with the choice of the sweeps that read primitive arrays, so
// these keep to longest marches.
template <int FLUX, int MIX>
constexpr bool whole_march =
    (MIX == MLAU_MIXED && FLUX == FLUX_LHLLD) || (MIX == MLAU_MIXED_RECON && FLUX == FLUX_ROE);
__device__ __forceinline__ bool march_mid(int ch, unsigned c, int most) { return (ch * c) % most != 0; }

}  // namespace mlau
