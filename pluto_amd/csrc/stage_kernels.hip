// Stage kernels of the unsplit RK2 MHD step (FP64 path), gfx950.
//
// One RK2 step (Time_Stepping/rk_step.c:27-254) is two stages, each:
//   sweep<x>, sweep<y>, sweep<z>   PLM + HLLD at every interface along a
//                                  direction (update_stage.c:155-242): flux,
//                                  pressure, UCT_HLL face data, velocity
//                                  slopes, Mach estimate
//   update<S>                      U += -dt/dx (F_{i+1/2} - F_{i-1/2}) and the
//                                  separate pressure-gradient term, in x, y, z
//                                  order (rhs.c:193-201); stage 1 also C_dt
//                                  and its maximum (update_stage.c:229-235,
//                                  308-313)
//   emf                            UCT_HLL edge EMFs (ct_emf_average.c:179-352)
//                                  with MC-limited staggered slopes
//                                  (ct_stag_slopes.c:51-106)
//   ct<S>                          Stokes update of the faces (ct_update.c:29-220);
//                                  stage 2 blends with the step-start faces
//                                  (rk_step.c:172-174)
//   c2p<S>                         face average of B (ct_field_average.c:64-66),
//                                  stage-2 blend of U (rk_step.c:168-170),
//                                  ConsToPrim with floors (mappers.c:88-254)
// followed by step_end, which forms invDt_hyp and the next dt on the device
// (NextTimeStep, main.c:459-532) so a run of steps never waits on the host.
//
// Layout: periodic box, no ghost zones, structure of arrays.  Cell
// c = (k*ny + j)*nx + i.  Face arrays hold the face at i+1/2 (x), j+1/2 (y)
// and k+1/2 (z) of cell c; edge arrays hold ez at (i+1/2, j+1/2, k), ex at
// (i, j+1/2, k+1/2), ey at (i+1/2, j, k+1/2).  Periodic neighbours are
// index wraps; the reference's periodic ghost zones hold exactly these
// values, so results agree bit for bit.

#include <hip/hip_runtime.h>
#include "mhd_device.hpp"
#include "stage_kernels.hpp"
#include "stage_cells.hpp"

namespace pgpu {

__device__ __forceinline__ unsigned long long as_bits(double x)
{
  return (unsigned long long)__double_as_longlong(x);
}

// Block-wide max of a non-negative double, one atomic per block.
__device__ __forceinline__ void block_max_to(double v, unsigned long long* dst)
{
  __shared__ double red[16];
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
    atomicMax(dst, as_bits(m));
  }
}

// ---------------------------------------------------------------------
// sweep: PLM + HLLD at interface (q+1/2) of every cell along direction D
// ---------------------------------------------------------------------

template <int D, int S>
__global__ void __launch_bounds__(256) k_sweep(Geo g, StageIn in, SweepOut out, DevScalars* sc)
{
  Cell p;
  double mach = 0.0;
  if (cell_of(g, p)) {
    mach = sweep_cell<D, S>(g, p, in, out);
    if (!in_sweep(g, D, p.i, p.j, p.k)) mach = 0.0;
  }
  block_max_to(mach, &sc->mach_max);
}

// ---------------------------------------------------------------------
// update: conservative accumulation in direction order, C_dt (stage 1)
// ---------------------------------------------------------------------

// FROM_V / CDT as update_cell; CDT also reduces the C_dt maximum.
template <bool FROM_V, bool CDT>
__global__ void __launch_bounds__(256) k_update(Geo g, StageIn in, Sweeps sw, Cons U, DevScalars* sc)
{
  Cell p;
  double cdt = 0.0;
  if (cell_of(g, p)) {
    cdt = update_cell<FROM_V, CDT>(g, p, in, sw, U, sc->dt);
    if (!in_dom(g, p.i, p.j, p.k)) cdt = 0.0;
  }
  if (CDT) block_max_to(cdt, &sc->invdt_max);
}

// ---------------------------------------------------------------------
// emf: UCT_HLL edge EMFs
// ---------------------------------------------------------------------

template <class FT>
__global__ void __launch_bounds__(256) k_emf(Geo g, StageIn in, Sweeps sw, EdgeOut e)
{
  Cell p;
  if (!cell_of(g, p)) return;
  emf_cell<FT>(g, p, in, sw, e);
}

// ARITHMETIC / UCT0 / UCT_CONTACT edge EMFs from the face EMFs (per cell)
template <int MODE>
__global__ void __launch_bounds__(256) k_emf_faces(Geo g, StageIn in, Sweeps sw, EdgeOut e)
{
  Cell p;
  if (!cell_of(g, p)) return;
  emf_faces_cell<MODE>(g, p, in, sw, e);
}

// UCT0 and UCT_CONTACT in 3D, marching up z: a workgroup takes 256 consecutive columns of
// the plane and kz planes.  What Ex and Ey of plane k read from plane k+1 (the
// cell EMFs of three columns, four face values) is computed once, kept in
// registers and is plane k's own part at the next step, so a cell reads about
// 47 values (UCT_CONTACT) where the per-cell form reads over a hundred and
// forms every cell EMF up to eight times.  Same expressions in the same
// order.  UCT_CONTACT 256^3 1184 -> 644 us a launch, 128^3 137 -> 91, 131 x 93
// x 77 75 -> 38; UCT0 607 -> 544, 83 -> 77, 38 -> 33.  (ARITHMETIC, which reads
// no cell EMF, is bound by its 12 values in either form: 228 us per cell, 237
// marching.)
template <int MODE>
__global__ void __launch_bounds__(256) k_emf_faces_z(Geo g, StageIn in, Sweeps sw, EdgeOut e, int kz)
{
  const unsigned col = blockIdx.x * 256u + threadIdx.x;
  const unsigned nxy = (unsigned)g.nx * (unsigned)g.ny;
  if (col >= nxy) return;
  const int j = (int)(col / (unsigned)g.nx), i = (int)(col - (unsigned)j * (unsigned)g.nx);
  // byte offsets in a plane: the cell, and those one further along x, y, both
  const unsigned jp = (unsigned)wrap2(j, 1, g.ny) * (unsigned)g.nx, ip = (unsigned)wrap2(i, 1, g.nx);
  const unsigned o00 = col * 8u, o10 = ((unsigned)j * (unsigned)g.nx + ip) * 8u, o01 = (jp + (unsigned)i) * 8u,
                 o11 = (jp + ip) * 8u;
  const int k0 = blockIdx.y * kz, k1 = min(k0 + kz, g.nz);
  // component A of the cell EMF at byte offset o of the arrays
  auto E = [&](int A, unsigned o) -> double {
    if (A == 0) return at_byte(in.V[VX3], o) * at_byte(in.V[BX2], o) - at_byte(in.V[VX2], o) * at_byte(in.V[BX3], o);
    if (A == 1) return at_byte(in.V[VX1], o) * at_byte(in.V[BX3], o) - at_byte(in.V[VX3], o) * at_byte(in.V[BX1], o);
    return at_byte(in.V[VX2], o) * at_byte(in.V[BX1], o) - at_byte(in.V[VX1], o) * at_byte(in.V[BX2], o);
  };
  // upwind sign of the mass flux at the d-face at byte offset o (ct_emf.c:136-141)
  auto S = [&](int d, unsigned o) -> int {
    const double f = at_byte(sw.d[d].dv[0], o);
    return f > 1.e-6 ? 1 : (f < -1.e-6 ? -1 : 0);
  };
  // what plane k + 1 gives to the edges of plane k
  struct Roll {
    double ex00, ex01, ey00, ey10;   // cell EMFs
    double eyi, exj;                 // face EMFs of the x and y faces
    int sx = 0, sy = 0;              // mass flux signs there
  };
  auto roll = [&](unsigned pk) {
    Roll r;
    r.ex00 = E(0, pk + o00);
    r.ex01 = E(0, pk + o01);
    r.ey00 = E(1, pk + o00);
    r.ey10 = E(1, pk + o10);
    r.eyi = at_byte(sw.d[0].SR, pk + o00);
    r.exj = at_byte(sw.d[1].SR, pk + o00);
    if constexpr (MODE == EMF_UCT_CONTACT) {
      r.sx = S(0, pk + o00);
      r.sy = S(1, pk + o00);
    }
    return r;
  };
  Roll c = roll((unsigned)k0 * nxy * 8u);
  for (int k = k0; k < k1; k++) {
    const unsigned pk = (unsigned)k * nxy * 8u;
    const Roll n = roll((unsigned)wrap2(k, 1, g.nz) * nxy * 8u);
    const double ezi00 = at_byte(sw.d[0].SL, pk + o00), ezi01 = at_byte(sw.d[0].SL, pk + o01);
    const double ezj00 = at_byte(sw.d[1].SL, pk + o00), ezj10 = at_byte(sw.d[1].SL, pk + o10);
    const double eyk00 = at_byte(sw.d[2].SL, pk + o00), eyk10 = at_byte(sw.d[2].SL, pk + o10);
    const double exk00 = at_byte(sw.d[2].SR, pk + o00), exk01 = at_byte(sw.d[2].SR, pk + o01);
    double ez, ex, ey;
    if constexpr (MODE == EMF_UCT0) {
      // ct_emf.c:261-283: each face EMF doubled minus the mean of its two cells'
      auto U0 = [](double f, double a, double b) { return f * 2.0 - 0.5 * (a + b); };
      const double z00 = E(2, pk + o00), z10 = E(2, pk + o10), z01 = E(2, pk + o01), z11 = E(2, pk + o11);
      ez = 0.25 * (U0(ezi00, z00, z10) + U0(ezi01, z01, z11) + U0(ezj00, z00, z01) + U0(ezj10, z10, z11));
      ex = 0.25 * (U0(exk00, c.ex00, n.ex00) + U0(exk01, c.ex01, n.ex01) + U0(c.exj, c.ex00, c.ex01) +
                   U0(n.exj, n.ex00, n.ex01));
      ey = 0.25 * (U0(c.eyi, c.ey00, c.ey10) + U0(n.eyi, n.ey00, n.ey10) + U0(eyk00, c.ey00, n.ey00) +
                   U0(eyk10, c.ey10, n.ey10));
    } else {
      ez = ezi00 + ezi01 + ezj00 + ezj10;
      ex = exk00 + exk01 + c.exj + n.exj;
      ey = c.eyi + n.eyi + eyk00 + eyk10;
      // the term of the upwind side, or the mean of both (s == 0)
      auto up = [](int s, double a, double b) { return s == 0 ? 0.5 * (a + b) : (s > 0 ? a : b); };
      const double z00 = E(2, pk + o00), z10 = E(2, pk + o10), z01 = E(2, pk + o01), z11 = E(2, pk + o11);
      const int sz = S(2, pk + o00);
      ez += up(c.sx, ezj00 - z00, ezj10 - z10);
      ez += up(c.sy, ezi00 - z00, ezi01 - z01);
      ez -= up(S(1, pk + o10), z10 - ezi00, z11 - ezi01);
      ez -= up(S(0, pk + o01), z01 - ezj00, z11 - ezj10);
      ez *= 0.25;
      ex += up(c.sy, exk00 - c.ex00, exk01 - c.ex01);
      ex += up(sz, c.exj - c.ex00, n.exj - n.ex00);
      ex -= up(S(2, pk + o01), c.ex01 - c.exj, n.ex01 - n.exj);
      ex -= up(n.sy, n.ex00 - exk00, n.ex01 - exk01);
      ex *= 0.25;
      ey += up(c.sx, eyk00 - c.ey00, eyk10 - c.ey10);
      ey += up(sz, c.eyi - c.ey00, n.eyi - n.ey00);
      ey -= up(S(2, pk + o10), c.ey10 - c.eyi, n.ey10 - n.eyi);
      ey -= up(n.sx, n.ey00 - eyk00, n.ey10 - eyk10);
      ey *= 0.25;
    }
    at_byte(e.ez, pk + o00) = ez;
    at_byte(e.ex, pk + o00) = ex;
    at_byte(e.ey, pk + o00) = ey;
    c = n;
  }
}

template <int MODE>
static void launch_emf_faces(const Geo& g, const StageIn& in, const Sweeps& sw, const EdgeOut& e,
                             hipStream_t s)
{
  if (g.dims == 3 && (unsigned long long)g.n * 8ull < (1ull << 32)) {   // 32-bit byte offsets
    // 16 planes a segment (each segment reads one plane twice), fewer where
    // that would leave less than eight workgroups a CU
    const unsigned wgs = (unsigned)(((long)g.nx * g.ny + 255) / 256);
    int kz = 16;
    while (kz > 1 && (long)wgs * ((g.nz + kz - 1) / kz) < 2048) kz /= 2;
    hipLaunchKernelGGL(k_emf_faces_z<MODE>, dim3(wgs, (g.nz + kz - 1) / kz), dim3(256), 0, s, g, in, sw, e, kz);
  } else {
    hipLaunchKernelGGL(k_emf_faces<MODE>, dim3((g.nx + 63) / 64, (g.ny + 3) / 4, g.nz), dim3(64, 4), 0, s, g, in,
                       sw, e);
  }
}

// z-marching EMF (3D): a workgroup covers a bx x by patch of a plane and
// marches kz planes.  The stencil reads 100 values per cell; 26 of them
// (field, i-offset, j-offset) are read on both planes k and k+1, and the
// field columns bx(i, j), by(i, j) on planes k-1 .. k+2, so a thread loads
// those once, on the leading plane, and keeps them in registers for the
// following planes: 67 loads per cell.  Every field is addressed by a 32-bit
// byte offset (in-plane part fixed per thread, plane part uniform), which
// keeps the loop's address registers to a handful.  Requires 8 n < 2^32.

// (field, i-offset, j-offset) read on planes k and k+1 by emf_edges
#define PGPU_EMF_ROLL(X)                                                                       \
  X(F_XSR, 0, 0) X(F_XSL, 0, 0) X(F_YSR, 0, 0) X(F_YSL, 0, 0)                                  \
  X(F_VX, 0, 0) X(F_VX, 1, 0) X(F_VY, 0, 0) X(F_VY, 0, 1) X(F_VZ, 0, 0) X(F_VZ, 0, 1)          \
  X(F_VZ, 1, 0)                                                                                \
  X(F_XDV0, 0, 0) X(F_XDV0, 1, 0) X(F_YDV1, 0, 0) X(F_YDV1, 0, 1) X(F_YDV2, 0, 0)              \
  X(F_YDV2, 0, 1) X(F_ZDV1, 0, 0) X(F_ZDV1, 0, 1) X(F_ZDV2, 0, 0) X(F_ZDV2, 0, 1)              \
  X(F_ZDV2, 1, 0) X(F_ZDV0, 0, 0) X(F_ZDV0, 1, 0) X(F_XDV2, 0, 0) X(F_XDV2, 1, 0)

constexpr int emf_roll_slot(int a, int i, int j)
{
  int s = 0;
#define X(A_, I_, J_)                        \
  if (a == A_ && i == I_ && j == J_) return s; \
  ++s;
  PGPU_EMF_ROLL(X)
#undef X
  return -1;
}

#define X(A_, I_, J_) +1
constexpr int kEmfRoll = 0 PGPU_EMF_ROLL(X);
#undef X

template <class FT>
struct EmfZLoader {
  const EmfFields& f;
  unsigned col[4], row[4], pk[4];   // byte offsets of the offsets -1 .. 2 along i, j, k
  double cur[kEmfRoll];             // rolled values on plane k
  double nxt[kEmfRoll];             // ... on plane k+1
  double wbx[4], wby[4];            // bx(i, j), by(i, j) on planes k-1 .. k+2

  template <int A, int I, int J, int K>
  __device__ __forceinline__ double load() const
  {
    const unsigned o = col[I + 1] + row[J + 1] + pk[K + 1];
    if constexpr (emf_f32<FT>(A))
      return double(at_byte(reinterpret_cast<const float*>(f.a[A]), o >> 1));
    else
      return at_byte(f.a[A], o);
  }

  template <int A, int I, int J, int K>
  __device__ __forceinline__ double get() const
  {
    constexpr int s = emf_roll_slot(A, I, J);
    if constexpr (A == F_BX && I == 0 && J == 0) return wbx[K + 1];
    else if constexpr (A == F_BY && I == 0 && J == 0) return wby[K + 1];
    else if constexpr (s >= 0 && K == 0) return cur[s];
    else if constexpr (s >= 0 && K == 1) return nxt[s];
    else return load<A, I, J, K>();
  }
};

// 2 waves per SIMD, the three edges scheduled one after the other (202 VGPRs,
// no spills): left alone the scheduler issues every load of an iteration at
// once and needs more than 256 VGPRs.  FT: storage type of the face speeds
// and velocity slopes.
template <class FT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_emf_z(Geo g, StageIn in, Sweeps sw, EdgeOut e, int kz)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= g.nx || j >= g.ny) return;
  const EmfFields f = emf_fields(in, sw);
  EmfZLoader<FT> ld{f};
  const unsigned rowb = (unsigned)g.nx * 8u;
  const unsigned planeb = rowb * (unsigned)g.ny;
#pragma unroll
  for (int o = -1; o <= 2; o++) {
    ld.col[o + 1] = (unsigned)wrap2(i, o, g.nx) * 8u;
    ld.row[o + 1] = (unsigned)wrap2(j, o, g.ny) * rowb;
  }
  const int k0 = blockIdx.z * kz;
  const int k1 = min(k0 + kz, g.nz);
  auto planes = [&](int k) {
#pragma unroll
    for (int o = -1; o <= 2; o++) ld.pk[o + 1] = (unsigned)wrap2(k, o, g.nz) * planeb;
  };
  // leading values for the first plane
  planes(k0);
#define X(A_, I_, J_) ld.cur[emf_roll_slot(A_, I_, J_)] = ld.template load<A_, I_, J_, 0>();
  PGPU_EMF_ROLL(X)
#undef X
  ld.wbx[0] = ld.template load<F_BX, 0, 0, -1>();
  ld.wbx[1] = ld.template load<F_BX, 0, 0, 0>();
  ld.wbx[2] = ld.template load<F_BX, 0, 0, 1>();
  ld.wby[0] = ld.template load<F_BY, 0, 0, -1>();
  ld.wby[1] = ld.template load<F_BY, 0, 0, 0>();
  ld.wby[2] = ld.template load<F_BY, 0, 0, 1>();
  for (int k = k0; k < k1; k++) {
    planes(k);
#define X(A_, I_, J_) ld.nxt[emf_roll_slot(A_, I_, J_)] = ld.template load<A_, I_, J_, 1>();
    PGPU_EMF_ROLL(X)
#undef X
    ld.wbx[3] = ld.template load<F_BX, 0, 0, 2>();
    ld.wby[3] = ld.template load<F_BY, 0, 0, 2>();
    double ez, ex, ey;
    emf_edges<true>(ld, true, ez, ex, ey);
    const unsigned o = ld.col[1] + ld.row[1] + ld.pk[1];
    at_byte(e.ez, o) = ez;
    at_byte(e.ex, o) = ex;
    at_byte(e.ey, o) = ey;
#pragma unroll
    for (int q = 0; q < kEmfRoll; q++) ld.cur[q] = ld.nxt[q];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      ld.wbx[q] = ld.wbx[q + 1];
      ld.wby[q] = ld.wby[q + 1];
    }
  }
}

// ---------------------------------------------------------------------
// ct: Stokes update of the faces owned by each cell
// ---------------------------------------------------------------------

template <int STAGE>
__global__ void __launch_bounds__(256) k_ct(Geo g, EdgeOut e, FaceIn bin, FaceIn b0, FaceOut bout,
                                            DevScalars* sc)
{
  Cell p;
  if (!cell_of(g, p)) return;
  ct_cell<STAGE>(g, p, e, bin, b0, bout, sc->dt);
}

// ---------------------------------------------------------------------
// c2p: face average, stage-2 blend, ConsToPrim
// ---------------------------------------------------------------------

template <int STAGE>
__global__ void __launch_bounds__(256) k_c2p(Geo g, Cons U, FaceIn b, StageIn vn,
                                             Prims Vout, unsigned char* flag,
                                             DevScalars* sc)
{
  Cell p;
  if (!cell_of(g, p)) return;
  bool nan = false;
  const unsigned char f = c2p_cell<STAGE>(g, p, U, b, vn, Vout, &nan);
  if (f) {
    flag[p.c] |= f;
    atomicAdd(&sc->fail_cells, 1u);
  }
  if (nan) atomicAdd(STAGE == 1 ? &sc->nan_cells : &sc->nan_next, 1u);
}

// Start of a step: clear the flags; the NaN cells of the previous step's
// output become stage-input NaNs now that a stage takes them as input.
__global__ void k_zero_flags(Geo g, unsigned char* flag, DevScalars* sc)
{
  if (sc && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0 &&
      threadIdx.y == 0) {
    sc->nan_cells += sc->nan_next;
    sc->nan_next = 0;
  }
  Cell p;
  if (!cell_of(g, p)) return;
  flag[p.c] = 0;
}

__global__ void k_step_end(DevScalars* sc, int dims, double cfl, double cfl_max_var, int fixed_dt)
{
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  close_step(sc, dims, cfl, cfl_max_var, fixed_dt);
}

// ---------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------

static inline dim3 grid_of(const Geo& g) { return dim3((g.nx + 63) / 64, (g.ny + 3) / 4, g.nz); }
static const dim3 kBlock(64, 4, 1);

#define PGPU_TIMED(id, ...)              \
  do {                                   \
    if (kt) kt->begin(id, s);            \
    hipLaunchKernelGGL(__VA_ARGS__);     \
    if (kt) kt->end(id, s);              \
  } while (0)

int launch_sweeps(const Geo& g, const StageIn& in, const Sweeps& sw, DevScalars* sc,
                  hipStream_t s, KernelTimer* kt)
{
  const dim3 gr = grid_of(g);
  if (g.solver == SOLVER_HLL) {
    PGPU_TIMED(KT_SWEEP_X, (k_sweep<0, SOLVER_HLL>), gr, kBlock, 0, s, g, in, sw.d[0], sc);
    PGPU_TIMED(KT_SWEEP_Y, (k_sweep<1, SOLVER_HLL>), gr, kBlock, 0, s, g, in, sw.d[1], sc);
    if (g.dims == 3) PGPU_TIMED(KT_SWEEP_Z, (k_sweep<2, SOLVER_HLL>), gr, kBlock, 0, s, g, in, sw.d[2], sc);
  } else if (g.solver == SOLVER_HLLC) {
    PGPU_TIMED(KT_SWEEP_X, (k_sweep<0, SOLVER_HLLC>), gr, kBlock, 0, s, g, in, sw.d[0], sc);
    PGPU_TIMED(KT_SWEEP_Y, (k_sweep<1, SOLVER_HLLC>), gr, kBlock, 0, s, g, in, sw.d[1], sc);
    if (g.dims == 3) PGPU_TIMED(KT_SWEEP_Z, (k_sweep<2, SOLVER_HLLC>), gr, kBlock, 0, s, g, in, sw.d[2], sc);
  } else if (g.solver == SOLVER_TVDLF) {
    PGPU_TIMED(KT_SWEEP_X, (k_sweep<0, SOLVER_TVDLF>), gr, kBlock, 0, s, g, in, sw.d[0], sc);
    PGPU_TIMED(KT_SWEEP_Y, (k_sweep<1, SOLVER_TVDLF>), gr, kBlock, 0, s, g, in, sw.d[1], sc);
    if (g.dims == 3) PGPU_TIMED(KT_SWEEP_Z, (k_sweep<2, SOLVER_TVDLF>), gr, kBlock, 0, s, g, in, sw.d[2], sc);
  } else if (g.solver == SOLVER_ROE) {
    PGPU_TIMED(KT_SWEEP_X, (k_sweep<0, SOLVER_ROE>), gr, kBlock, 0, s, g, in, sw.d[0], sc);
    PGPU_TIMED(KT_SWEEP_Y, (k_sweep<1, SOLVER_ROE>), gr, kBlock, 0, s, g, in, sw.d[1], sc);
    if (g.dims == 3) PGPU_TIMED(KT_SWEEP_Z, (k_sweep<2, SOLVER_ROE>), gr, kBlock, 0, s, g, in, sw.d[2], sc);
  } else {
    PGPU_TIMED(KT_SWEEP_X, (k_sweep<0, SOLVER_HLLD>), gr, kBlock, 0, s, g, in, sw.d[0], sc);
    PGPU_TIMED(KT_SWEEP_Y, (k_sweep<1, SOLVER_HLLD>), gr, kBlock, 0, s, g, in, sw.d[1], sc);
    if (g.dims == 3) PGPU_TIMED(KT_SWEEP_Z, (k_sweep<2, SOLVER_HLLD>), gr, kBlock, 0, s, g, in, sw.d[2], sc);
  }
  return (int)hipGetLastError();
}

int launch_update(const Geo& g, bool from_v, bool cdt, const StageIn& in, const Sweeps& sw,
                  const Cons& U, DevScalars* sc, hipStream_t s, KernelTimer* kt)
{
  const dim3 gr = grid_of(g);
  if (from_v && cdt) PGPU_TIMED(KT_UPDATE, (k_update<true, true>), gr, kBlock, 0, s, g, in, sw, U, sc);
  else if (from_v) PGPU_TIMED(KT_UPDATE, (k_update<true, false>), gr, kBlock, 0, s, g, in, sw, U, sc);
  else if (cdt) PGPU_TIMED(KT_UPDATE, (k_update<false, true>), gr, kBlock, 0, s, g, in, sw, U, sc);
  else PGPU_TIMED(KT_UPDATE, (k_update<false, false>), gr, kBlock, 0, s, g, in, sw, U, sc);
  return (int)hipGetLastError();
}

// Tiling of k_emf_z (process-wide; pgpu_set_emf_tiling).
static int g_emf_bx = 64, g_emf_by = 4, g_emf_kz = 16;
// UCT_HLL EMF kernel of FP64 3D boxes (process-wide; pgpu_set_emf_kernel):
// 0 register-rolling k_emf_z, 1 LDS-staged k_emf_zs with 64 x 4 tiles, 2 with
// 32 x 4, 3 with 32 x 8
static int g_emf_kernel = 3, g_emf_lds_kz = 16;

int set_emf_kernel(int kind, int kz)
{
  if (kind < 0 || kind > 3 || kz < 0) return -1;
  g_emf_kernel = kind;
  g_emf_lds_kz = kz > 0 ? kz : 16;
  return 0;
}

int set_emf_tiling(int bx, int by, int kz)
{
  if (bx == 0 && by == 0 && kz == 0) {
    g_emf_bx = 64;
    g_emf_by = 4;
    g_emf_kz = 16;
    return 0;
  }
  if (bx < 1 || by < 1 || kz < 1 || bx * by > 256 || (bx * by) % 64 != 0) return -1;
  g_emf_bx = bx;
  g_emf_by = by;
  g_emf_kz = kz;
  return 0;
}

void get_emf_tiling(int* bx, int* by, int* kz)
{
  *bx = g_emf_bx;
  *by = g_emf_by;
  *kz = g_emf_kz;
}

// Whether the register kernels beat the LDS one where the sweeps have stored the
// velocity slopes (modular pipeline): on small boxes, but for narrow ones that
// an LDS tile holds whole.  us a launch, register and LDS: 33^3 11.5 and 14.1,
// 64^3 18.4 and 22.1, 300 x 3 x 300 22.9 and 49.4, 256^2 6.8 and 8.1, 3 x 3 x
// 2000 29.5 and 43.2; 100^3 84.7 and 75.3, 7 x 7 x 500 23.1 and 14.6, 3 x 300
// x 300 292.8 and 155.5, 1000^2 34.1 and 26.7.
static bool emf_by_registers(const Geo& g)
{
  return g.n <= 300000 && (g.nx >= 16 || g.nx * g.ny < 16);
}

// f32_faces: face speeds and velocity slopes stored as float (FP32 flux);
// f32_state: the velocities of the stage input too (FP32 flux, stage 2);
// slopes: the velocity slopes are in sw already
static bool enqueue_emf(const Geo& g, const StageIn& in, const Sweeps& sw, const EdgeOut& e,
                        hipStream_t s, KernelTimer* kt, bool f32_faces = false,
                        bool f32_state = false, bool slopes = false)
{
  if (g.pz > 0 && g.emf_avg != EMF_UCT_HLL) return false;
  if (g.emf_avg == EMF_ARITHMETIC) {
    PGPU_TIMED(KT_EMF, k_emf_faces<EMF_ARITHMETIC>, grid_of(g), kBlock, 0, s, g, in, sw, e);
  } else if (g.emf_avg == EMF_UCT0) {
    if (kt) kt->begin(KT_EMF, s);
    launch_emf_faces<EMF_UCT0>(g, in, sw, e, s);
    if (kt) kt->end(KT_EMF, s);
  } else if (g.emf_avg == EMF_UCT_CONTACT) {
    if (kt) kt->begin(KT_EMF, s);
    launch_emf_faces<EMF_UCT_CONTACT>(g, in, sw, e, s);
    if (kt) kt->end(KT_EMF, s);
  } else if ((g_emf_kernel || g.pz > 0 || g.dims != 3) && !(slopes && emf_by_registers(g)) &&
             launch_emf_lds(g, in, sw, e, s, g_emf_kernel ? g_emf_kernel : 3, g_emf_lds_kz, kt,
                            f32_state ? 2 : (f32_faces ? 1 : 0))) {
    // LDS-staged z-march (the only EMF kernel for a stack of patches)
  } else if (g.pz > 0 ||
             (!slopes && launch_vel_slopes(g, in, sw, s, f32_state ? 2 : (f32_faces ? 1 : 0)) != 0)) {
    return false;
  } else if (g.dims == 3 && (unsigned long long)g.n * 8ull < (1ull << 32)) {
    const dim3 b(g_emf_bx, g_emf_by, 1);
    const long xy = (long)((g.nx + b.x - 1) / b.x) * ((g.ny + b.y - 1) / b.y);
    // fewer planes per workgroup on small boxes: keep >= 2048 workgroups
    // (8 per CU) in flight where the box has them
    int kz = g_emf_kz;
    while (kz > 1 && xy * ((g.nz + kz - 1) / kz) < 2048) kz /= 2;
    const dim3 gr((g.nx + b.x - 1) / b.x, (g.ny + b.y - 1) / b.y, (g.nz + kz - 1) / kz);
    if (f32_state) PGPU_TIMED(KT_EMF, k_emf_z<F32State>, gr, b, 0, s, g, in, sw, e, kz);
    else if (f32_faces) PGPU_TIMED(KT_EMF, k_emf_z<float>, gr, b, 0, s, g, in, sw, e, kz);
    else PGPU_TIMED(KT_EMF, k_emf_z<double>, gr, b, 0, s, g, in, sw, e, kz);
  } else {
    if (f32_state) PGPU_TIMED(KT_EMF, k_emf<F32State>, grid_of(g), kBlock, 0, s, g, in, sw, e);
    else if (f32_faces) PGPU_TIMED(KT_EMF, k_emf<float>, grid_of(g), kBlock, 0, s, g, in, sw, e);
    else PGPU_TIMED(KT_EMF, k_emf<double>, grid_of(g), kBlock, 0, s, g, in, sw, e);
  }
  return true;
}

int launch_emf(const Geo& g, const StageIn& in, const Sweeps& sw, const EdgeOut& e, hipStream_t s,
               KernelTimer* kt, bool f32_faces, bool f32_state)
{
  if (!enqueue_emf(g, in, sw, e, s, kt, f32_faces, f32_state)) return (int)hipErrorInvalidValue;
  return (int)hipGetLastError();
}

int launch_emf_ct(const Geo& g, bool blend, const StageIn& in, const Sweeps& sw, const EdgeOut& e,
                  const FaceIn& bin, const FaceIn& b0, const FaceOut& bout, DevScalars* sc,
                  hipStream_t s, KernelTimer* kt)
{
  // the modular sweeps store the UCT_HLL face data only
  if (g.emf_avg != EMF_UCT_HLL) return (int)hipErrorInvalidValue;
  const dim3 gr = grid_of(g);
  enqueue_emf(g, in, sw, e, s, kt, false, false, true);
  if (!blend) PGPU_TIMED(KT_CT, k_ct<1>, gr, kBlock, 0, s, g, e, bin, b0, bout, sc);
  else PGPU_TIMED(KT_CT, k_ct<2>, gr, kBlock, 0, s, g, e, bin, b0, bout, sc);
  return (int)hipGetLastError();
}

int launch_ct(const Geo& g, bool blend, const EdgeOut& e, const FaceIn& bin, const FaceIn& b0,
              const FaceOut& bout, DevScalars* sc, hipStream_t s)
{
  const dim3 gr = grid_of(g);
  if (!blend) hipLaunchKernelGGL(k_ct<1>, gr, kBlock, 0, s, g, e, bin, b0, bout, sc);
  else hipLaunchKernelGGL(k_ct<2>, gr, kBlock, 0, s, g, e, bin, b0, bout, sc);
  return (int)hipGetLastError();
}

int launch_c2p(const Geo& g, int stage, const Cons& U, const FaceIn& b, const StageIn& vn,
               const Prims& Vout, unsigned char* flag, DevScalars* sc, hipStream_t s,
               KernelTimer* kt)
{
  const dim3 gr = grid_of(g);
  if (stage == 1) PGPU_TIMED(KT_C2P, k_c2p<1>, gr, kBlock, 0, s, g, U, b, vn, Vout, flag, sc);
  else PGPU_TIMED(KT_C2P, k_c2p<2>, gr, kBlock, 0, s, g, U, b, vn, Vout, flag, sc);
  return (int)hipGetLastError();
}

int launch_stage(const Geo& g, int stage, const StageIn& in, const Sweeps& sw, const Cons& U,
                 const EdgeOut& e, const FaceIn& bin, const FaceIn& b0, const FaceOut& bout,
                 const StageIn& vn, const Prims& Vout, unsigned char* flag, DevScalars* sc,
                 hipStream_t s, KernelTimer* kt)
{
  int rc = launch_sweeps(g, in, sw, sc, s, kt);
  if (!rc) rc = launch_update(g, stage == 1, stage == 1, in, sw, U, sc, s, kt);
  if (!rc) rc = launch_emf_ct(g, stage == 2, in, sw, e, bin, b0, bout, sc, s, kt);
  FaceIn bnew;
  for (int d = 0; d < 3; d++) bnew.b[d] = bout.b[d];
  if (!rc) rc = launch_c2p(g, stage, U, bnew, vn, Vout, flag, sc, s, kt);
  return rc;
}
#undef PGPU_TIMED

int launch_zero_flags(const Geo& g, unsigned char* flag, hipStream_t s, DevScalars* sc)
{
  hipLaunchKernelGGL(k_zero_flags, grid_of(g), kBlock, 0, s, g, flag, sc);
  return (int)hipGetLastError();
}

int launch_step_end(DevScalars* sc, int dims, double cfl, double cfl_max_var, int fixed_dt,
                    hipStream_t s)
{
  hipLaunchKernelGGL(k_step_end, dim3(1), dim3(64), 0, s, sc, dims, cfl, cfl_max_var, fixed_dt);
  return (int)hipGetLastError();
}

}  // namespace pgpu
