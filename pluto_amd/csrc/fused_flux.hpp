// Flux kernels of the fused stage (k_flux_xy_rows, k_flux_xy,
// k_flux_xy_items, k_flux_z) and their launcher template, shared by
// fused_kernels.hip (the FP64 instantiations, compiled without FMA
// contraction: bit-exact with the reference), fused_f32.hip (the FP32-flux
// instantiations, compiled with contraction) and fused_fast.hip (the
// tolerance-mode FP64 instantiations).
// Fused flux kernels of the stage (the fast path used by pgpu_run and
// AdvanceStep).  Same arithmetic as the modular kernels in stage_kernels.hip
// (and thus as the reference), organised to move fewer bytes:
//
//   k_flux_xy_rows    (the default x/y kernel) a workgroup holds whole box
//                     rows, or a window of the rows of all planes one after
//                     another, and marches up a y segment: each cell
//                     reconstructed once per direction, x neighbours through
//                     LDS, y carried in registers (see the kernel).
//   k_flux_xy<STAGE>  one z-plane tile per workgroup.  The primitive state of
//                     the tile plus its stencil halo is staged in LDS once;
//                     each thread solves one x and one y interface (PLM +
//                     HLLD) from LDS, fluxes go to LDS, and each cell adds
//                     -dt/dx (F_{i+1/2}-F_{i-1/2}) and the y counterpart to
//                     its conservative state in registers.  Writes U, the
//                     UCT_HLL face speeds of its own
//                     faces/cells, and C_dt's x+y part.
//   k_flux_z<STAGE>   one thread per (i,j) column marching up a z segment:
//                     each cell's z PLM and each z interface is computed
//                     once, the previous interface's flux is carried in
//                     registers; adds the z flux difference to U, finishes
//                     C_dt ((0 + cx) + cy) + cz (update_stage.c:229-235) and
//                     its maximum.
//
// The flux differences are added in x, y, z order as in update_stage.c:134-242.

#pragma once
#include <hip/hip_runtime.h>
#include "mhd_device.hpp"
#include "stage_cells.hpp"
#include "stage_kernels.hpp"
#include "fused_kernels.hpp"

namespace pgpu {

namespace {

// face speed / velocity slope of the EMF stencil at cell c: FP64 values as
// double, FP32 values as float in the first half of the buffer (exact, and
// half the bytes for the EMF kernel to read back)
template <class R>
__device__ __forceinline__ void face_store(double* a, long c, R v)
{
  if constexpr (sizeof(R) == 4) reinterpret_cast<float*>(a)[c] = v;
  else a[c] = v;
}

// what the flux kernels store per face for the EMF: the UCT_HLL face speeds
// (the EMF kernel reconstructs the velocity slopes; not storing them took
// the x/y rows from 1255 to 1150 us and the z march from 653 to 600 at
// 256^3), or the face EMFs from the normal fluxes of B
// and the mass flux (ARITHMETIC, UCT0, UCT_CONTACT)
constexpr int FACE_UCT_HLL = 0;
constexpr int FACE_BFLUX = 1;

// periodic index for -n <= q < 2n
__device__ __forceinline__ int wrap(int q, int n)
{
  q = q < 0 ? q + n : q;
  return q >= n ? q - n : q;
}

// periodic index for any q (tiles may be wider than the box)
__device__ __forceinline__ int wrap_any(int q, int n)
{
  q %= n;
  return q < 0 ? q + n : q;
}

__device__ __forceinline__ void block_max(double v, unsigned long long* dst, double* red)
{
  const int lane = threadIdx.x + threadIdx.y * blockDim.x;
  const int wave = lane / warpSize;
  const int nwave = (blockDim.x * blockDim.y + warpSize - 1) / warpSize;
  for (int off = warpSize / 2; off > 0; off >>= 1) {
    double o = __shfl_xor(v, off, warpSize);
    v = o > v ? o : v;
  }
  if ((lane % warpSize) == 0) red[wave] = v;
  __syncthreads();
  if (lane == 0) {
    double m = red[0];
    for (int w = 1; w < nwave; w++) m = red[w] > m ? red[w] : m;
    atomicMax(dst, (unsigned long long)__double_as_longlong(m));
  }
}

// PLM of one cell from its neighbours: right-face (vp) and left-face (vm)
// states of all variables.
template <typename R>
__device__ __forceinline__ void plm_cell(const R* vm1, const R* v0, const R* vp1, R* vp, R* vm)
{
#pragma unroll
  for (int q = 0; q < NV; q++) {
    const R s = mc_slope(vm1[q], v0[q], vp1[q]);
    vp[q] = v0[q] + s * R(0.5);
    vm[q] = v0[q] - s * R(0.5);
  }
}

}  // namespace

// ---------------------------------------------------------------------
// x and y sweeps of one z-plane tile
// ---------------------------------------------------------------------

// A TXx8 workgroup produces the (TX-1)x7 cells (i0..i0+TX-2, j0..j0+6) of an
// overlapping tile: thread (tx, ty) solves the x interface on the left of
// cell (i0+tx, j0+ty) and the y interface below cell (i0+tx, j0+ty), so
// every thread does exactly one x and one y interface (two full passes).
// The staged state spans x in [i0-2, i0+TX] and y in [j0-2, j0+8].  TX is
// 32 for FP64 (LDS-limited: three workgroups per CU) and 64 for FP32.
// V: 0 for the builds of fused_kernels.hip and fused_f32.hip, 1 for the
// tolerance-mode FP64 build of fused_fast.hip (distinct kernel symbols)
template <int STAGE, typename R, int TX, int S, int E, int V = 0>
__global__ void __launch_bounds__(64 * XY_TY)
k_flux_xy(Geo g, StageIn in, Cons U, FaceData fd, double* cdt_xy, DevScalars* sc)
{
  constexpr int TY = XY_TY;
  constexpr int OX = TX - 1, OY = TY - 1;     // output cells of the workgroup
  constexpr int LX = TX + 3, LY = TY + 3;     // staged region
  constexpr int NT = TX * TY;
  __shared__ R sv[NV][LY][LX];
  __shared__ R fx[6][TY][TX];                 // rho, mx, my, mz, E, p at x_{i0+tx-1/2}
  __shared__ R cmx[TY][TX];
  __shared__ R fy[6][TY][TX];                 // same at y_{j0+ty-1/2}
  __shared__ R cmy[TY][TX];
  __shared__ double red[NT / 64 + 1];

  const int tx = threadIdx.x, ty = threadIdx.y;
  const int tid = tx + ty * TX;
  const dim3 tb = xcd_tile();
  const int i0 = tb.x * OX, j0 = tb.y * OY, k = tb.z;
  const long plane = (long)k * g.ny * g.nx;
  sc = scal(sc, g, k);

  // stage the primitive state (periodic wrap)
  for (int q = tid; q < LX * LY; q += NT) {
    const int lx = q % LX, ly = q / LX;
    const int gi = wrap_any(i0 + lx - 2, g.nx), gj = wrap_any(j0 + ly - 2, g.ny);
    const long c = plane + (long)gj * g.nx + gi;
#pragma unroll
    for (int v = 0; v < NV; v++) sv[v][ly][lx] = R(in.V[v][c]);
  }
  __syncthreads();

  const double dt = sc->dt;
  const R gam = R(g.gamma), gm1 = R(g.gmm1);
  double mach = 0.0;
  const int ci = i0 + tx, cj = j0 + ty;                 // unwrapped cell of this thread
  const bool row_in = cj < g.ny, col_in = ci < g.nx;

  // x interface between cells (ci-1, cj) and (ci, cj): cells ci-2 .. ci+1 at LDS x = tx .. tx+3
  {
    R a[4][NV], vL[NV], vR[NV], vm0[NV], vpn[NV], vmn[NV];
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int v = 0; v < NV; v++) a[s][v] = sv[v][ty + 2][tx + s];
    plm_cell(a[0], a[1], a[2], vL, vm0);
    plm_cell(a[1], a[2], a[3], vpn, vmn);
#pragma unroll
    for (int v = 0; v < NV; v++) vR[v] = vmn[v];
    const int oi = wrap_any(ci - 1, g.nx), oj = wrap_any(cj, g.ny);   // owner cell of the face
    const long cf = plane + (long)oj * g.nx + oi;
    const R bface = R(in.b[0][cf]);
    vL[BX1] = bface;
    vR[BX1] = bface;
    RiemannOut<R> r;
    riemann<S, 0, E == FACE_BFLUX>(vL, vR, gam, gm1, r, g.dims == 2);
    fx[0][ty][tx] = r.f[RHO];
    fx[1][ty][tx] = r.f[VX1];
    fx[2][ty][tx] = r.f[VX2];
    fx[3][ty][tx] = r.f[VX3];
    fx[4][ty][tx] = r.f[ENG];
    fx[5][ty][tx] = r.press;
    cmx[ty][tx] = r.cmax;
    // the face belongs to cell ci-1, an output cell of this tile when tx >= 1
    if (tx >= 1 && ty < OY && row_in && ci - 1 < g.nx) {
      if constexpr (E == FACE_BFLUX) {
        fd.SL[0][cf] = -r.f[BX2];   // ezi, eyi (ct_emf.c:131-133)
        fd.SR[0][cf] = r.f[BX3];
        fd.mf[0][cf] = r.f[RHO];
      } else {
        face_store(fd.SL[0], cf, max_ge(R(0), -r.SL));
        face_store(fd.SR[0], cf, max_ge(R(0), r.SR));
      }
    }
    const double rm = double(r.mach);
    if (in_sweep(g, 0, ci - 1, cj, k)) mach = rm > mach ? rm : mach;
  }
  // y interface between cells (ci, cj-1) and (ci, cj): rows cj-2 .. cj+1 at LDS y = ty .. ty+3
  {
    R a[4][NV], vL[NV], vR[NV], vm0[NV], vpn[NV], vmn[NV];
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int v = 0; v < NV; v++) a[s][v] = sv[v][ty + s][tx + 2];
    plm_cell(a[0], a[1], a[2], vL, vm0);
    plm_cell(a[1], a[2], a[3], vpn, vmn);
#pragma unroll
    for (int v = 0; v < NV; v++) vR[v] = vmn[v];
    const int oi = wrap_any(ci, g.nx), oj = wrap_any(cj - 1, g.ny);   // owner cell of the face
    const long cf = plane + (long)oj * g.nx + oi;
    const R bface = R(in.b[1][cf]);
    vL[BX2] = bface;
    vR[BX2] = bface;
    RiemannOut<R> r;
    riemann<S, 1, E == FACE_BFLUX>(vL, vR, gam, gm1, r, g.dims == 2);
    fy[0][ty][tx] = r.f[RHO];
    fy[1][ty][tx] = r.f[VX1];
    fy[2][ty][tx] = r.f[VX2];
    fy[3][ty][tx] = r.f[VX3];
    fy[4][ty][tx] = r.f[ENG];
    fy[5][ty][tx] = r.press;
    cmy[ty][tx] = r.cmax;
    // the face belongs to cell cj-1, an output cell of this tile when ty >= 1
    if (ty >= 1 && tx < OX && col_in && cj - 1 < g.ny) {
      if constexpr (E == FACE_BFLUX) {
        fd.SL[1][cf] = r.f[BX1];    // ezj, exj (ct_emf.c:153-155)
        fd.SR[1][cf] = -r.f[BX3];
        fd.mf[1][cf] = r.f[RHO];
      } else {
        face_store(fd.SL[1], cf, max_ge(R(0), -r.SL));
        face_store(fd.SR[1], cf, max_ge(R(0), r.SR));
      }
    }
    const double rm = double(r.mach);
    if (in_sweep(g, 1, ci, cj - 1, k)) mach = rm > mach ? rm : mach;
  }
  __syncthreads();

  // output cells: base state plus x then y flux differences
  if (tx < OX && ty < OY && col_in && row_in) {
    const long c = plane + (long)cj * g.nx + ci;
    double u[5];
    if (STAGE == 1) {
      double v[NV];
      if constexpr (sizeof(R) == sizeof(double)) {
#pragma unroll
        for (int q = 0; q < NV; q++) v[q] = sv[q][ty + 2][tx + 2];
      } else {
#pragma unroll
        for (int q = 0; q < NV; q++) v[q] = in.V[q][c];   // U0 from the FP64 state
      }
      u[0] = v[RHO];
      u[1] = v[RHO] * v[VX1];
      u[2] = v[RHO] * v[VX2];
      u[3] = v[RHO] * v[VX3];
      u[4] = total_energy(v, g.gmm1);
    } else {
#pragma unroll
      for (int q = 0; q < 5; q++) u[q] = U.u[q][c];
    }
    const double dtdx = dt / g.dx[0], dtdy = dt / g.dx[1];
    double r[5];
#pragma unroll
    for (int q = 0; q < 5; q++) r[q] = -dtdx * (double(fx[q][ty][tx + 1]) - double(fx[q][ty][tx]));
    r[1] -= dtdx * (double(fx[5][ty][tx + 1]) - double(fx[5][ty][tx]));
#pragma unroll
    for (int q = 0; q < 5; q++) u[q] += r[q];
#pragma unroll
    for (int q = 0; q < 5; q++) r[q] = -dtdy * (double(fy[q][ty + 1][tx]) - double(fy[q][ty][tx]));
    r[2] -= dtdy * (double(fy[5][ty + 1][tx]) - double(fy[5][ty][tx]));
#pragma unroll
    for (int q = 0; q < 5; q++) u[q] += r[q];
#pragma unroll
    for (int q = 0; q < 5; q++) U.u[q][c] = u[q];
    if (STAGE == 1) {
      double cdt = 0.0;
      cdt += 0.5 * (double(cmx[ty][tx]) + double(cmx[ty][tx + 1])) * g.inv_dx[0];
      cdt += 0.5 * (double(cmy[ty][tx]) + double(cmy[ty + 1][tx])) * g.inv_dx[1];
      cdt_xy[c] = cdt;
    }
  }
  block_max(mach, &sc->mach_max, red);
}

// Non-overlapping variant (the FP32-flux path): a 32x8 tile plus a two-cell
// halo; the (TX+1)*TY x and TX*(TY+1) y interfaces of the tile are spread
// over the workgroup (three passes).  With FP32 state the workgroup is not
// LDS-limited and this layout measured faster than the overlapping one.
template <int STAGE, typename R, int S>
__global__ void __launch_bounds__(XY_TX * XY_TY)
k_flux_xy_items(Geo g, StageIn in, Cons U, FaceData fd, double* cdt_xy, DevScalars* sc)
{
  constexpr int TX = XY_TX, TY = XY_TY;
  constexpr int LX = TX + 4, LY = TY + 4;     // staged region with 2-cell halo
  constexpr int NXI = (TX + 1) * TY;          // x interfaces of the tile (one halo)
  constexpr int NYI = TX * (TY + 1);          // y interfaces
  constexpr int NT = TX * TY;
  __shared__ R sv[NV][LY][LX];
  __shared__ R fx[6][TY][TX + 1];             // rho, mx, my, mz, E, p
  __shared__ R cmx[TY][TX + 1];
  __shared__ R fy[6][TY + 1][TX];
  __shared__ R cmy[TY + 1][TX];
  __shared__ double red[NT / 64 + 1];

  const int tid = threadIdx.x + threadIdx.y * TX;
  const int i0 = blockIdx.x * TX, j0 = blockIdx.y * TY, k = blockIdx.z;
  const long plane = (long)k * g.ny * g.nx;
  sc = scal(sc, g, k);

  // stage the primitive state of the tile plus halo (periodic wrap); the
  // second stage's input was stored as float by the first stage
  for (int q = tid; q < LX * LY; q += NT) {
    const int lx = q % LX, ly = q / LX;
    const int gi = wrap_any(i0 + lx - 2, g.nx), gj = wrap_any(j0 + ly - 2, g.ny);
    const long c = plane + (long)gj * g.nx + gi;
#pragma unroll
    for (int v = 0; v < NV; v++)
      sv[v][ly][lx] = (STAGE == 2 && sizeof(R) == 4) ? R(reinterpret_cast<const float*>(in.V[v])[c])
                                                     : R(in.V[v][c]);
  }
  __syncthreads();

  const double dt = sc->dt;
  const R gam = R(g.gamma), gm1 = R(g.gmm1);
  double mach = 0.0;

  // interfaces: x items first, then y items; items that no cell of the
  // box needs (tiles wider than the box) are skipped
  for (int item = tid; item < NXI + NYI; item += NT) {
    RiemannOut<R> r;
    R vL[NV], vR[NV];
    R a[4][NV];
    int li, lj, own, gi, gj;
    if (item < NXI) {
      const int row = item / (TX + 1), col = item % (TX + 1);
      if (j0 + row >= g.ny || i0 + col - 1 >= g.nx) continue;
      // interface between tile cells col-1 and col of row `row`
      li = col + 1;   // LDS x of the left cell
      lj = row + 2;
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int v = 0; v < NV; v++) a[s][v] = sv[v][lj][li - 1 + s];
      gi = i0 + col - 1;
      gj = j0 + row;
      own = (col >= 1) && (gi < g.nx) && (gj < g.ny);
      R vm0[NV], vpn[NV], vmn[NV];
      plm_cell(a[0], a[1], a[2], vL, vm0);
      plm_cell(a[1], a[2], a[3], vpn, vmn);
#pragma unroll
      for (int v = 0; v < NV; v++) vR[v] = vmn[v];
      const long cf = plane + (long)wrap(gj, g.ny) * g.nx + wrap(gi, g.nx);
      const R bface = R(in.b[0][cf]);
      vL[BX1] = bface;
      vR[BX1] = bface;
      riemann<S, 0, false>(vL, vR, gam, gm1, r, g.dims == 2);
      fx[0][row][col] = r.f[RHO];
      fx[1][row][col] = r.f[VX1];
      fx[2][row][col] = r.f[VX2];
      fx[3][row][col] = r.f[VX3];
      fx[4][row][col] = r.f[ENG];
      fx[5][row][col] = r.press;
      cmx[row][col] = r.cmax;
      if (own) {
        const long c = plane + (long)gj * g.nx + gi;
        face_store(fd.SL[0], c, max_ge(R(0), -r.SL));
        face_store(fd.SR[0], c, max_ge(R(0), r.SR));
      }
    } else {
      const int it = item - NXI;
      const int row = it / TX, col = it % TX;   // row 0 is the halo interface j0-1/2
      if (i0 + col >= g.nx || j0 + row - 1 >= g.ny) continue;
      li = col + 2;
      lj = row + 1;
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int v = 0; v < NV; v++) a[s][v] = sv[v][lj - 1 + s][li];
      gi = i0 + col;
      gj = j0 + row - 1;
      own = (row >= 1) && (gi < g.nx) && (gj < g.ny);
      R vm0[NV], vpn[NV], vmn[NV];
      plm_cell(a[0], a[1], a[2], vL, vm0);
      plm_cell(a[1], a[2], a[3], vpn, vmn);
#pragma unroll
      for (int v = 0; v < NV; v++) vR[v] = vmn[v];
      const long cf = plane + (long)wrap(gj, g.ny) * g.nx + wrap(gi, g.nx);
      const R bface = R(in.b[1][cf]);
      vL[BX2] = bface;
      vR[BX2] = bface;
      riemann<S, 1, false>(vL, vR, gam, gm1, r, g.dims == 2);
      fy[0][row][col] = r.f[RHO];
      fy[1][row][col] = r.f[VX1];
      fy[2][row][col] = r.f[VX2];
      fy[3][row][col] = r.f[VX3];
      fy[4][row][col] = r.f[ENG];
      fy[5][row][col] = r.press;
      cmy[row][col] = r.cmax;
      if (own) {
        const long c = plane + (long)gj * g.nx + gi;
        face_store(fd.SL[1], c, max_ge(R(0), -r.SL));
        face_store(fd.SR[1], c, max_ge(R(0), r.SR));
      }
    }
    const double rm = double(r.mach);
    mach = rm > mach ? rm : mach;
  }
  __syncthreads();

  // per cell: base state plus x then y flux differences
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int i = i0 + tx, j = j0 + ty;
  if (i < g.nx && j < g.ny) {
    const long c = plane + (long)j * g.nx + i;
    double u[5];
    if (STAGE == 1) {
      double v[NV];
      if constexpr (sizeof(R) == sizeof(double)) {
#pragma unroll
        for (int q = 0; q < NV; q++) v[q] = sv[q][ty + 2][tx + 2];
      } else {
#pragma unroll
        for (int q = 0; q < NV; q++) v[q] = in.V[q][c];   // U0 from the FP64 state
      }
      u[0] = v[RHO];
      u[1] = v[RHO] * v[VX1];
      u[2] = v[RHO] * v[VX2];
      u[3] = v[RHO] * v[VX3];
      u[4] = total_energy(v, g.gmm1);
    } else {
#pragma unroll
      for (int q = 0; q < 5; q++) u[q] = U.u[q][c];
    }
    const double dtdx = dt / g.dx[0], dtdy = dt / g.dx[1];
    double r[5];
#pragma unroll
    for (int q = 0; q < 5; q++) r[q] = -dtdx * (double(fx[q][ty][tx + 1]) - double(fx[q][ty][tx]));
    r[1] -= dtdx * (double(fx[5][ty][tx + 1]) - double(fx[5][ty][tx]));
#pragma unroll
    for (int q = 0; q < 5; q++) u[q] += r[q];
#pragma unroll
    for (int q = 0; q < 5; q++) r[q] = -dtdy * (double(fy[q][ty + 1][tx]) - double(fy[q][ty][tx]));
    r[2] -= dtdy * (double(fy[5][ty + 1][tx]) - double(fy[5][ty][tx]));
#pragma unroll
    for (int q = 0; q < 5; q++) u[q] += r[q];
#pragma unroll
    for (int q = 0; q < 5; q++) U.u[q][c] = u[q];
    if (STAGE == 1) {
      double cdt = 0.0;
      cdt += 0.5 * (double(cmx[ty][tx]) + double(cmx[ty][tx + 1])) * g.inv_dx[0];
      cdt += 0.5 * (double(cmy[ty][tx]) + double(cmy[ty + 1][tx])) * g.inv_dx[1];
      cdt_xy[c] = cdt;
    }
  }
  block_max(mach, &sc->mach_max, red);
}

// ---------------------------------------------------------------------
// x and y sweeps, one workgroup per row marching up a y segment
// ---------------------------------------------------------------------

// The variables a cell exchanges with its x neighbours: all but B_x (the x
// interfaces take the staggered face value instead of the reconstruction).
constexpr int XROW_NV = NV - 1;
__device__ __forceinline__ constexpr int xrow_var(int q) { return q < BX1 ? q : q + 1; }

// A workgroup takes up to MAXT cells along x and marches up the rows
// j0 .. j0+seg-1 of their planes.  How its threads sit on the box (RowMap)
// is a launch parameter:
//   rows > 0   thread t = cell t % nx of plane blockIdx.y * rows + t / nx:
//              whole rows of `rows` planes, each periodic within itself
//   rows = 0   the rows of all planes, each with the images of its last two
//              cells before it and of its first two after it (nx + 4 threads),
//              one after another; workgroup w takes the window of blockDim.x
//              threads that starts at w * (blockDim.x - 4).  The window's
//              two outer threads at either end and the images only feed their
//              neighbours: any row length, about 1 - 4/256 - 4/nx of the lanes
//              busy
// Rows of the primitive state go through a ring of three LDS row buffers,
// filled by direct global-to-LDS copies (global_load_lds_dword, no registers
// on the way, any alignment) one row ahead, every wave its own 64 cells.
// For row j each thread
//   - reconstructs its own cell in x (PLM from the ring, periodic
//     neighbours), solves the x interface i-1/2 with its left neighbour's
//     right-face state from LDS, and takes the flux at i+1/2 from its right
//     neighbour through LDS;
//   - reconstructs cell (i, j+1) in y from rows j, j+1, j+2 of the ring and
//     solves the y interface j+1/2; the flux at j-1/2 and the right-face
//     state of cell (i, j) are carried from the previous row;
//   - adds the x then the y flux difference to U and writes the face data
//     of its faces and C_dt's x+y part.
// Every cell is reconstructed once per direction and every interface solved
// once (plus, per segment, the y interface j0-1/2 and two y
// reconstructions), where the tile kernel reconstructs each cell twice per
// direction and solves its halo interfaces again.  Two workgroup barriers
// per row.  The arithmetic per interface and per cell is the tile kernel's,
// so the results are identical.
// LDS (dynamic): 3 * NV * blockDim.x ring values and (NV + 7) * blockDim.x
// values of R.

// thread t of workgroup w: its cell (ic, k), whether it owns that cell's
// results, and the threads of its x neighbours
struct RowCell {
  int ic, k, tl, tr;
  bool act;
};

__device__ __forceinline__ RowCell row_cell(const Geo& g, int rows, int w, int t, int nt)
{
  RowCell c;
  if (rows > 0) {
    int r = t / g.nx;
    c.act = r < rows && w * rows + r < g.nz;
    r = min(r, rows - 1);
    c.ic = t - r * g.nx;
    c.k = min(w * rows + r, g.nz - 1);
    c.tl = c.ic == 0 ? t + g.nx - 1 : t - 1;
    c.tr = c.ic == g.nx - 1 ? t - (g.nx - 1) : t + 1;
    if (c.ic >= g.nx) {   // past the last row
      c.ic = g.nx - 1;
      c.tl = c.tr = t;
    }
  } else {
    const int f = w * (nt - 4) + t, len = g.nx + 4;
    c.k = f / len;
    const int q = f - c.k * len - 2;   // -2, -1: images of the last cells, nx, nx + 1: of the first
    c.act = t > 1 && t < nt - 2 && q >= 0 && q < g.nx && c.k < g.nz;
    c.ic = q < 0 ? q + g.nx : (q >= g.nx ? q - g.nx : q);
    c.k = min(c.k, g.nz - 1);
    c.tl = max(t - 1, 0);
    c.tr = min(t + 1, nt - 1);
  }
  return c;
}

template <int STAGE, typename R, int S, int E, int V, int MAXT>
__global__ void __launch_bounds__(MAXT, 2)
k_flux_xy_rows(Geo g, StageIn in, Cons U, FaceData fd, double* cdt_xy, int seg, int rows,
               DevScalars* sc)
{
  // rows of the state as they are stored: FP64, or float for the FP32-flux
  // path's second stage; a lane copies 4 bytes, CPC lanes a cell
  using RT = std::conditional_t<(STAGE == 2 && sizeof(R) == 4), float, double>;
  constexpr int CPC = int(sizeof(RT)) / 4, CCH = 64 / CPC;   // cells per copy
  extern __shared__ __align__(16) unsigned char xrow_lds[];
  __shared__ double red[MAXT / 64 + 1];
  const int nt = blockDim.x;
  RT* ring = reinterpret_cast<RT*>(xrow_lds);          // [3][NV][nt] rows of the state
  R* xp = reinterpret_cast<R*>(ring + 3 * NV * nt);   // [NV][nt] right-face states, B_x: the face value
  R* xf = xp + NV * nt;                               // [7][nt] flux at i-1/2: rho mx my mz E p cmax

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const dim3 tb = xcd_tile();
  const int j0 = tb.x * seg;
  const int j1 = min(j0 + seg, g.ny);
  const RowCell rc = row_cell(g, rows, tb.y, t, nt);
  const bool act = rc.act;
  const int ic = rc.ic, k = rc.k, tl = rc.tl, tr = rc.tr;
  sc = scal(sc, g, (int)tb.y * rows);   // (a stack: the workgroup's rows are of one patch)
  // 32-bit byte offsets of FP64 fields (the launcher keeps this kernel to
  // boxes under 4 GiB per field): the loop's addresses stay one VGPR each
  const unsigned row8 = (unsigned)g.nx * 8u;
  const unsigned plane8 = row8 * (unsigned)g.ny;
  const unsigned col8 = (unsigned)k * plane8 + (unsigned)ic * 8u;    // cell (ic, 0, k)
  const unsigned coll8 = col8 - (ic == 0 ? 0u - (row8 - 8u) : 8u);   // its left neighbour
  const double dt = sc->dt;
  const double dtdx = dt / g.dx[0], dtdy = dt / g.dx[1];
  const R gam = R(g.gamma), gm1 = R(g.gmm1);
  double mach = 0.0;

  auto off8 = [&](int jj) { return col8 + (unsigned)jj * row8; };
  auto load = [&](int jj, R* v) {
    const unsigned o = off8(wrap_any(jj, g.ny));
#pragma unroll
    for (int q = 0; q < NV; q++)
      v[q] = sizeof(RT) == 4 ? R(at_byte(reinterpret_cast<const float*>(in.V[q]), o >> 1))
                             : R(at_byte(in.V[q], o));
  };
  // face data: FP64, or float in the first half of the buffer
  auto fstore = [&](double* a, unsigned o, R v) {
    if constexpr (sizeof(R) == 4) at_byte(reinterpret_cast<float*>(a), o >> 1) = v;
    else at_byte(a, o) = v;
  };
  // copy row jj of every variable into ring slot sl: each wave the cells of
  // its own threads, CCH of them per copy
  unsigned soff[CPC];
#pragma unroll
  for (int c = 0; c < CPC; c++) {
    const RowCell s = row_cell(g, rows, tb.y, wave * 64 + c * CCH + lane / CPC, nt);
    soff[c] = ((unsigned)s.k * plane8 + (unsigned)s.ic * 8u) / (8u / sizeof(RT)) +
              (unsigned)(lane % CPC) * 4u;
  }
  auto stage_row = [&](int jj, int sl) {
    const unsigned o = (unsigned)wrap_any(jj, g.ny) * (row8 / (8u / (unsigned)sizeof(RT)));
#pragma unroll
    for (int q = 0; q < NV; q++)
#pragma unroll
      for (int c = 0; c < CPC; c++)
        __builtin_amdgcn_global_load_lds(
            (const void*)(reinterpret_cast<const char*>(in.V[q]) + (o + soff[c])),
            (__attribute__((address_space(3))) void*)(ring + (sl * NV + q) * nt + wave * 64 + c * CCH),
            4, 0, 0);
  };
  // wait for every vector memory access of this thread (the ring copies
  // among them) before a barrier that publishes the copies
  auto wait_vm = [] { __builtin_amdgcn_s_waitcnt(0x0070); };   // vmcnt(0) lgkmcnt(0)
  auto rv = [&](int sl, int q, int ii) -> R { return R(ring[(sl * NV + q) * nt + ii]); };
  stage_row(j0, 0);
  stage_row(j0 + 1, 1);
  // the y right-face state of cell (i, j0) and the y flux at j0-1/2
  R vpy[NV], fyb[6], cmyb;
  {
    R a[NV], b[NV], w0[NV], w1[NV], vpb[NV], vmb[NV], vm0[NV];
    load(j0 - 2, a);
    load(j0 - 1, b);
    load(j0, w0);
    load(j0 + 1, w1);
    plm_cell(a, b, w0, vpb, vmb);      // cell (i, j0-1)
    plm_cell(b, w0, w1, vpy, vm0);     // cell (i, j0)
    R vL[NV], vR[NV];
#pragma unroll
    for (int q = 0; q < NV; q++) {
      vL[q] = vpb[q];
      vR[q] = vm0[q];
    }
    const R bface = R(at_byte(in.b[1], off8(wrap_any(j0 - 1, g.ny))));
    vL[BX2] = bface;
    vR[BX2] = bface;
    RiemannOut<R> r;
    riemann<S, 1, E == FACE_BFLUX>(vL, vR, gam, gm1, r, g.dims == 2);
    fyb[0] = r.f[RHO]; fyb[1] = r.f[VX1]; fyb[2] = r.f[VX2];
    fyb[3] = r.f[VX3]; fyb[4] = r.f[ENG]; fyb[5] = r.press;
    cmyb = r.cmax;
    if (act && in_sweep(g, 1, ic, j0 - 1, k)) mach = double(r.mach);
  }
  wait_vm();
  __syncthreads();

  // FP64: the face values of a row are loaded during the row before, ahead
  // of its stores (vector memory completes in order: loaded after them, they
  // would wait for them), and are in place by that row's last barrier
  // (1.33 -> 1.30 ms at 256^3; the FP32 kernel measured slower so and loads
  // them at the top of the row)
  constexpr bool kPrefetch = sizeof(R) == sizeof(double);
  R bfx_n = R(0), bfy_n = R(0);
  if (kPrefetch) {
    bfx_n = R(at_byte(in.b[0], coll8 + (unsigned)j0 * row8));
    bfy_n = R(at_byte(in.b[1], off8(j0)));
  }
  int s0 = 0, s1 = 1, s2 = 2;   // ring slots of rows j, j+1, j+2
  for (int j = j0; j < j1; j++) {
    const unsigned c = off8(j);
    const unsigned cf = coll8 + (unsigned)j * row8;   // owner cell of the x face i-1/2
    const R bfx = kPrefetch ? bfx_n : R(at_byte(in.b[0], cf));
    const R bfy = kPrefetch ? bfy_n : R(at_byte(in.b[1], c));

    // x reconstruction of cell (i, j)
    R vmx[NV];
    {
      R w0[NV], a[NV], b[NV], vpx[NV];
#pragma unroll
      for (int q = 0; q < NV; q++) w0[q] = rv(s0, q, t);
#pragma unroll
      for (int q = 0; q < XROW_NV; q++) {
        a[xrow_var(q)] = rv(s0, xrow_var(q), tl);
        b[xrow_var(q)] = rv(s0, xrow_var(q), tr);
      }
      a[BX1] = w0[BX1];   // not used: the x interfaces take the face value
      b[BX1] = w0[BX1];
      plm_cell(a, w0, b, vpx, vmx);
      // (every thread writes its slot: the face value's load then stays
      // at the top of the row instead of sinking into a branch)
#pragma unroll
      for (int q = 0; q < NV; q++) xp[q * nt + t] = q == BX1 ? bfx : vpx[q];
    }
    __syncthreads();
    // row j+2 into the slot of row j-1 (last read before the barrier)
    if (j + 1 < j1) {
      stage_row(j + 2, s2);
      if (kPrefetch) {
        bfx_n = R(at_byte(in.b[0], coll8 + (unsigned)(j + 1) * row8));
        bfy_n = R(at_byte(in.b[1], off8(j + 1)));
      }
    }

    // x interface i-1/2
    R xsl, xsr, xe[3];
    {
      R vL[NV], vR[NV];
#pragma unroll
      for (int q = 0; q < NV; q++) vL[q] = xp[q * nt + tl];
#pragma unroll
      for (int q = 0; q < NV; q++) vR[q] = vmx[q];
      const R bface = xp[BX1 * nt + t];
      vL[BX1] = bface;
      vR[BX1] = bface;
      RiemannOut<R> r;
      riemann<S, 0, E == FACE_BFLUX>(vL, vR, gam, gm1, r, g.dims == 2);
      const R fxl[6] = {r.f[RHO], r.f[VX1], r.f[VX2], r.f[VX3], r.f[ENG], r.press};
      if constexpr (E == FACE_BFLUX) {
        xe[0] = -r.f[BX2];   // ezi, eyi (ct_emf.c:131-133)
        xe[1] = r.f[BX3];
        xe[2] = r.f[RHO];
      } else {
        xsl = max_ge(R(0), -r.SL);
        xsr = max_ge(R(0), r.SR);
      }
#pragma unroll
      for (int q = 0; q < 6; q++) xf[q * nt + t] = fxl[q];
      xf[6 * nt + t] = r.cmax;
      if (act) {
        const double rm = double(r.mach);
        if (in_sweep(g, 0, ic - 1, j, k)) mach = rm > mach ? rm : mach;
      }
    }
    wait_vm();
    __syncthreads();   // the copy of row j+2 is in place
    double U0[5];
    if (STAGE == 2) {
#pragma unroll
      for (int q = 0; q < 5; q++) U0[q] = at_byte(U.u[q], c);
    }
    if (act) {
      if constexpr (E == FACE_BFLUX) {
        at_byte(fd.SL[0], cf) = xe[0];
        at_byte(fd.SR[0], cf) = xe[1];
        at_byte(fd.mf[0], cf) = xe[2];
      } else {
        fstore(fd.SL[0], cf, xsl);
        fstore(fd.SR[0], cf, xsr);
      }
    }
    // y reconstruction of cell (i, j+1) and the y interface j+1/2
    R vpn[NV], vmn[NV];
    {
      R a[NV], b[NV], w2[NV];
#pragma unroll
      for (int q = 0; q < NV; q++) {
        a[q] = rv(s0, q, t);
        b[q] = rv(s1, q, t);
      }
      if (j + 1 < j1) {
#pragma unroll
        for (int q = 0; q < NV; q++) w2[q] = rv(s2, q, t);
      } else {
        load(j + 2, w2);   // the segment's last row: row j+2 is not staged
      }
      plm_cell(a, b, w2, vpn, vmn);
    }
    {
      R vL[NV], vR[NV];
#pragma unroll
      for (int q = 0; q < NV; q++) {
        vL[q] = vpy[q];
        vR[q] = vmn[q];
      }
      vL[BX2] = bfy;
      vR[BX2] = bfy;
      RiemannOut<R> r;
      riemann<S, 1, E == FACE_BFLUX>(vL, vR, gam, gm1, r, g.dims == 2);
      const R fcur[6] = {r.f[RHO], r.f[VX1], r.f[VX2], r.f[VX3], r.f[ENG], r.press};
      if (act) {
        if constexpr (E == FACE_BFLUX) {
          at_byte(fd.SL[1], c) = r.f[BX1];    // ezj, exj (ct_emf.c:153-155)
          at_byte(fd.SR[1], c) = -r.f[BX3];
          at_byte(fd.mf[1], c) = r.f[RHO];
        } else {
          fstore(fd.SL[1], c, max_ge(R(0), -r.SL));
          fstore(fd.SR[1], c, max_ge(R(0), r.SR));
        }
        const double rm = double(r.mach);
        if (in_sweep(g, 1, ic, j, k)) mach = rm > mach ? rm : mach;
        // the x fluxes and signal speeds of both faces, still in LDS: held in
        // registers through the y solve they and U0 spilled (256^3, us a
        // launch: Roe 2012 -> 1390, HLLD with magnetic face fluxes 1385 ->
        // 1225; HLLD alone fitted before too, 1186 either way)
        double rx[5], cdt = 0.0;
#pragma unroll
        for (int q = 0; q < 5; q++) rx[q] = -dtdx * (double(xf[q * nt + tr]) - double(xf[q * nt + t]));
        rx[1] -= dtdx * (double(xf[5 * nt + tr]) - double(xf[5 * nt + t]));
        if (STAGE == 1) cdt += 0.5 * (double(xf[6 * nt + t]) + double(xf[6 * nt + tr])) * g.inv_dx[0];
        double ry[5];
#pragma unroll
        for (int q = 0; q < 5; q++) ry[q] = -dtdy * (double(fcur[q]) - double(fyb[q]));
        ry[2] -= dtdy * (double(fcur[5]) - double(fyb[5]));
        double u[5];
        if (STAGE == 2) {
#pragma unroll
          for (int q = 0; q < 5; q++) u[q] = U0[q];
        } else {
          // U0 from the FP64 state of row j, still in the ring (formed before
          // the solves it held ten registers through both of them)
          double v[NV];
#pragma unroll
          for (int q = 0; q < NV; q++) v[q] = double(ring[(s0 * NV + q) * nt + t]);
          u[0] = v[RHO];
          u[1] = v[RHO] * v[VX1];
          u[2] = v[RHO] * v[VX2];
          u[3] = v[RHO] * v[VX3];
          u[4] = total_energy(v, g.gmm1);
        }
#pragma unroll
        for (int q = 0; q < 5; q++) u[q] += rx[q];
#pragma unroll
        for (int q = 0; q < 5; q++) u[q] += ry[q];
#pragma unroll
        for (int q = 0; q < 5; q++) at_byte(U.u[q], c) = u[q];
        if (STAGE == 1) {
          cdt += 0.5 * (double(cmyb) + double(r.cmax)) * g.inv_dx[1];
          at_byte(cdt_xy, c) = cdt;
        }
      }
#pragma unroll
      for (int q = 0; q < 6; q++) fyb[q] = fcur[q];
      cmyb = r.cmax;
    }
#pragma unroll
    for (int q = 0; q < NV; q++) vpy[q] = vpn[q];
    const int st = s0;
    s0 = s1;
    s1 = s2;
    s2 = st;
  }
  block_max(mach, &sc->mach_max, red);
}

// ---------------------------------------------------------------------
// z sweep, one thread per column marching over a z segment
// ---------------------------------------------------------------------

// A workgroup takes 256 consecutive columns of the plane, whatever the row
// length, so only the plane's last workgroup has idle lanes (rows cut into
// 64-wide tiles left 31% of the lanes of a 133-cell row idle: 133^3 171 ->
// 121 us a launch, 131 x 93 x 77 81 -> 53).  At 256^3 the march moves its
// 171 B per cell at 4.8 TB/s, the rate of a large copy; small boxes are
// bound by the solves one after another along a segment (march_len).

template <int STAGE, typename R, int S, int E, int V = 0>
__global__ void __launch_bounds__(Z_COLS)
k_flux_z(Geo g, StageIn in, Cons U, FaceData fd, const double* cdt_xy, int seg, DevScalars* sc)
{
  __shared__ double red[Z_COLS / 64 + 1];
  const unsigned col = blockIdx.x * (unsigned)Z_COLS + threadIdx.x;   // cell of the plane
  // (its indices: only the reductions of a ghosted box ask for them)
  const int j = g.ghost ? (int)(col / (unsigned)g.nx) : 0;
  const int i = g.ghost ? (int)(col - (unsigned)j * (unsigned)g.nx) : 0;
  const ZSeg zs = zseg(g, blockIdx.y, seg);   // (a patch of a stack: z periodic within it)
  const int k0 = zs.k0, k1 = zs.k1;
  sc = scal(sc, g, k0);
  double mach = 0.0, cdt_max = 0.0;
  if (col < (unsigned)g.nx * (unsigned)g.ny) {
    // 32-bit byte offsets (the launcher keeps the z march to fields under
    // 4 GiB): the column's addresses stay one VGPR each
    const unsigned col8 = col * 8u;
    const unsigned pl8 = (unsigned)g.nx * (unsigned)g.ny * 8u;
    const double dt = sc->dt;
    const double dtdz = dt / g.dx[2];
    const R gam = R(g.gamma), gm1 = R(g.gmm1);
    auto load = [&](int kk, R* v) {
      const unsigned o = (unsigned)zwrap(g, zs.kb, kk) * pl8 + col8;
#pragma unroll
      for (int q = 0; q < NV; q++)   // the FP32 path's second stage reads its input as float
        v[q] = (STAGE == 2 && sizeof(R) == 4) ? R(at_byte(reinterpret_cast<const float*>(in.V[q]), o >> 1))
                                              : R(at_byte(in.V[q], o));
    };
    auto fstore = [&](double* a, unsigned o, R v) {
      if constexpr (sizeof(R) == 4) at_byte(reinterpret_cast<float*>(a), o >> 1) = v;
      else at_byte(a, o) = v;
    };
    // vb = v(k), vc = v(k+1); vp_k: right-face state of cell k
    R vb[NV], vc[NV], vp_k[NV];
    R fprev[6], cmprev;
    {
      R va[NV], vm_k[NV], vp_n[NV], vm_n[NV];
      load(k0 - 2, va);
      load(k0 - 1, vb);
      load(k0, vc);
      plm_cell(va, vb, vc, vp_k, vm_k);      // cell k0-1
#pragma unroll
      for (int q = 0; q < NV; q++) va[q] = vb[q];
#pragma unroll
      for (int q = 0; q < NV; q++) vb[q] = vc[q];
      load(k0 + 1, vc);
      plm_cell(va, vb, vc, vp_n, vm_n);      // cell k0
      R vL[NV], vR[NV];
#pragma unroll
      for (int q = 0; q < NV; q++) {
        vL[q] = vp_k[q];
        vR[q] = vm_n[q];
      }
      const R bface = R(at_byte(in.b[2], (unsigned)zwrap(g, zs.kb, k0 - 1) * pl8 + col8));
      vL[BX3] = bface;
      vR[BX3] = bface;
      RiemannOut<R> r;
      riemann<S, 2, false>(vL, vR, gam, gm1, r);
      if (in_sweep(g, 2, i, j, k0 - 1)) mach = double(r.mach);
      fprev[0] = r.f[RHO]; fprev[1] = r.f[VX1]; fprev[2] = r.f[VX2];
      fprev[3] = r.f[VX3]; fprev[4] = r.f[ENG]; fprev[5] = r.press;
      cmprev = r.cmax;
#pragma unroll
      for (int q = 0; q < NV; q++) vp_k[q] = vp_n[q];   // cell k0
    }
    // march: vb = v(k), vc = v(k+1)
    for (int k = k0; k < k1; k++) {
      const unsigned c = (unsigned)k * pl8 + col8;
      R vn[NV], vp_n[NV], vm_n[NV];
      load(k + 2, vn);
      const R bface = R(at_byte(in.b[2], c));
      // U and C_dt(x+y) of cell k read here, ahead of this plane's stores
      // (which may alias them as far as the compiler knows): their latency
      // then passes under the solve
      double u[5], cdt = 0.0;
#pragma unroll
      for (int q = 0; q < 5; q++) u[q] = at_byte(U.u[q], c);
      if (STAGE == 1) cdt = at_byte(cdt_xy, c);
      plm_cell(vb, vc, vn, vp_n, vm_n);     // cell k+1
      R vL[NV], vR[NV];
#pragma unroll
      for (int q = 0; q < NV; q++) {
        vL[q] = vp_k[q];
        vR[q] = vm_n[q];
      }
      vL[BX3] = bface;
      vR[BX3] = bface;
      RiemannOut<R> r;
      riemann<S, 2, E == FACE_BFLUX>(vL, vR, gam, gm1, r);
      const double rm = double(r.mach);
      if (in_sweep(g, 2, i, j, k)) mach = rm > mach ? rm : mach;
      const R fcur[6] = {r.f[RHO], r.f[VX1], r.f[VX2], r.f[VX3], r.f[ENG], r.press};
      double rr[5];
#pragma unroll
      for (int q = 0; q < 5; q++) rr[q] = -dtdz * (double(fcur[q]) - double(fprev[q]));
      rr[3] -= dtdz * (double(fcur[5]) - double(fprev[5]));
#pragma unroll
      for (int q = 0; q < 5; q++) u[q] += rr[q];
#pragma unroll
      for (int q = 0; q < 5; q++) at_byte(U.u[q], c) = u[q];
      if constexpr (E == FACE_BFLUX) {
        at_byte(fd.SL[2], c) = -r.f[BX1];    // eyk, exk (ct_emf.c:175-176)
        at_byte(fd.SR[2], c) = r.f[BX2];
        at_byte(fd.mf[2], c) = r.f[RHO];
      } else {
        fstore(fd.SL[2], c, max_ge(R(0), -r.SL));
        fstore(fd.SR[2], c, max_ge(R(0), r.SR));
      }
      if (STAGE == 1) {
        cdt += 0.5 * (double(cmprev) + double(r.cmax)) * g.inv_dx[2];
        if (in_dom(g, i, j, k)) cdt_max = cdt > cdt_max ? cdt : cdt_max;
      }
#pragma unroll
      for (int q = 0; q < 6; q++) fprev[q] = fcur[q];
      cmprev = r.cmax;
#pragma unroll
      for (int q = 0; q < NV; q++) {
        vp_k[q] = vp_n[q];
        vb[q] = vc[q];
        vc[q] = vn[q];
      }
    }
  }
  block_max(mach, &sc->mach_max, red);
  if (STAGE == 1) {
    __syncthreads();
    block_max(cdt_max, &sc->invdt_max, red);
  }
}

// 2D problems: C_dt's maximum directly from the x+y part.
// (a template so that each translation unit that launches it has its own)
template <int = 0>
__global__ void k_cdt_max2d(Geo g, const double* cdt_xy, DevScalars* sc)
{
  __shared__ double red[4];
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  double v = c < g.n ? cdt_xy[c] : 0.0;
  block_max(v, &sc->invdt_max, red);
}

template <typename R, int S, int E = FACE_UCT_HLL, int V = 0>
static void launch_flux_fused_t(const Geo& g, int stage, const StageIn& in, const Cons& U,
                                const FaceData& fd, double* cdt_xy, DevScalars* sc,
                                hipStream_t s, KernelTimer* kt)
{
  if (kt) kt->begin(KT_FLUX_XY, s);
  bool rows = false;
  {
    const RowLaunch rl = row_launch(g, (int)sizeof(R));
    rows = rl.nt > 0;
    if (rows) {
      const dim3 grid((g.ny + rl.seg - 1) / rl.seg, rl.wgs), block(rl.nt);
      // ring rows: FP64, except the FP32-flux path's float second-stage input
      const size_t rt = (stage == 2 && sizeof(R) == 4) ? 4 : 8;
      const size_t lds = 3 * NV * rl.nt * rt + (NV + 7) * rl.nt * sizeof(R);
      if (stage == 1)
        hipLaunchKernelGGL((k_flux_xy_rows<1, R, S, E, V, 256>), grid, block, lds, s, g, in, U, fd, cdt_xy, rl.seg, rl.rows, sc);
      else
        hipLaunchKernelGGL((k_flux_xy_rows<2, R, S, E, V, 256>), grid, block, lds, s, g, in, U, fd, cdt_xy, rl.seg, rl.rows, sc);
    }
  }
  if (rows) {
  } else if constexpr (sizeof(R) == sizeof(double)) {
    constexpr int TX = 32;
    const dim3 bxy(TX, XY_TY), gxy((g.nx + TX - 2) / (TX - 1), (g.ny + XY_TY - 2) / (XY_TY - 1), g.nz);
    if (stage == 1) hipLaunchKernelGGL((k_flux_xy<1, R, TX, S, E, V>), gxy, bxy, 0, s, g, in, U, fd, cdt_xy, sc);
    else hipLaunchKernelGGL((k_flux_xy<2, R, TX, S, E, V>), gxy, bxy, 0, s, g, in, U, fd, cdt_xy, sc);
  } else {
    static_assert(E == FACE_UCT_HLL, "the FP32 x/y kernel stores UCT_HLL face data only");
    const dim3 bxy(XY_TX, XY_TY), gxy((g.nx + XY_TX - 1) / XY_TX, (g.ny + XY_TY - 1) / XY_TY, g.nz);
    if (stage == 1) hipLaunchKernelGGL((k_flux_xy_items<1, R, S>), gxy, bxy, 0, s, g, in, U, fd, cdt_xy, sc);
    else hipLaunchKernelGGL((k_flux_xy_items<2, R, S>), gxy, bxy, 0, s, g, in, U, fd, cdt_xy, sc);
  }
  if (kt) kt->end(KT_FLUX_XY, s);
  if (g.dims == 3) {
    const unsigned cols = (unsigned)g.nx * (unsigned)g.ny, wgs = (cols + Z_COLS - 1) / Z_COLS;
    // (the FP32 z march is memory-bound and best on short segments: 256^3
    // 518 us at 8 planes, 534 at 32)
    const int seg = march_len(sizeof(R) == 4 ? 8 : 32, patch_depth(g), [&](int len) {
      return (long)wgs * (Z_COLS / 64) * zblocks(g, len);
    });
    const dim3 bz(Z_COLS), gz(wgs, zblocks(g, seg));
    if (kt) kt->begin(KT_FLUX_Z, s);
    if (stage == 1)
      hipLaunchKernelGGL((k_flux_z<1, R, S, E, V>), gz, bz, 0, s, g, in, U, fd, cdt_xy, seg, sc);
    else
      hipLaunchKernelGGL((k_flux_z<2, R, S, E, V>), gz, bz, 0, s, g, in, U, fd, cdt_xy, seg, sc);
    if (kt) kt->end(KT_FLUX_Z, s);
  } else if (stage == 1) {
    hipLaunchKernelGGL(k_cdt_max2d<>, dim3((unsigned)((g.n + 255) / 256)), dim3(256), 0, s, g,
                       cdt_xy, sc);
  }
}

}  // namespace pgpu
