// Discrete adjoint of one RK2 step of the unsplit MHD stage (FP64, 3D,
// fixed dt), the reverse of the forward step in stage_kernels.hip:
//
//   stage 1   U*   = U0 + L(V, b),     b*  = b  - dt curl E(V, b),
//             V1   = ConsToPrim(U*, avg b*)
//   stage 2   U**  = U* + L(V1, b*),   b** = b* - dt curl E(V1, b*)
//   blend     U'   = (U0 + U**)/2,     b'  = (b + b**)/2,
//             V'   = ConsToPrim(U', avg b')          (rk_step.c:140-176)
//
// with U0 = PrimToCons(V), L the flux differences of update_stage.c /
// rhs.c (x, y, z; PLM-MC + HLLD), E the UCT_HLL edge EMF
// (ct_emf_average.c:179-352) and avg the face average of B
// (ct_field_average.c:64-66).  The adjoint step recomputes the forward
// step from the domain's state (the fused kernels), then runs the stages
// backwards.  Stencil adjoints that land on neighbouring cells are not
// scattered with atomics: the EMF's are written as per-edge partials and
// gathered per cell, the interfaces' are summed per cell in LDS (x rows) or
// in a per-thread ring while marching along y and z, so the adjoint is
// deterministic.  Floors are assumed inactive (smooth
// flows).

#include <hip/hip_runtime.h>

#include "domain.hpp"
#include "fused_kernels.hpp"
#include "mhd_adjoint.hpp"
#include "mhd_device.hpp"
#include "stage_cells.hpp"
#include "stage_kernels.hpp"

namespace pgpu {

namespace {

struct AdjCell {
  int i, j, k;
  long c;
};

__device__ __forceinline__ bool adj_cell(const Geo& g, AdjCell& p)
{
  p.i = blockIdx.x * blockDim.x + threadIdx.x;
  p.j = blockIdx.y * blockDim.y + threadIdx.y;
  p.k = blockIdx.z;
  if (p.i >= g.nx || p.j >= g.ny) return false;
  p.c = ((long)p.k * g.ny + p.j) * g.nx + p.i;
  return true;
}

// periodic neighbour at offset o (|o| <= 2) along axis A
template <int A>
__device__ __forceinline__ long nbr(const Geo& g, const AdjCell& p, int o)
{
  const int q = (A == 0 ? p.i : A == 1 ? p.j : p.k);
  const int nq = (A == 0 ? g.nx : A == 1 ? g.ny : g.nz);
  const long s = (A == 0 ? 1L : A == 1 ? (long)g.nx : (long)g.nx * g.ny);
  int qq = q + o;
  if (qq < 0) qq += nq;
  else if (qq >= nq) qq -= nq;
  return p.c + (long)(qq - q) * s;
}

__device__ __forceinline__ long nbr(const Geo& g, const AdjCell& p, int a, int o)
{
  return a == 0 ? nbr<0>(g, p, o) : a == 1 ? nbr<1>(g, p, o) : nbr<2>(g, p, o);
}

const dim3 kAdjBlock(64, 4);

dim3 adj_grid(const Geo& g)
{
  return dim3((g.nx + 63) / 64, (g.ny + 3) / 4, g.nz);
}

}  // namespace

// Adjoint work arrays (device), allocated on the first adjoint call.
struct AdjArrays {
  double* lamV[8];      // adjoint of the stage input primitives (cell B included)
  double* lamU[5];      // adjoint of the conservative accumulator
  double* lamU0[5];     // adjoint of U0 = PrimToCons(V^n) from the blend
  double* lamB[3];      // adjoint of the faces of the current stage
  double* lamB0[3];     // adjoint of b^n from the blend
  double* lamE[3];      // ex, ey, ez
  double* lamS[3][2];   // [direction][0: max(0,-SL), 1: max(0,SR)]
  double* lamDV[3][3];  // [direction][velocity component]
  double* lamBc[3];     // adjoint of the cell-centred field (temporary)
  double* VN[8];        // forward V^{n+1}
  double* bN[3];        // forward b^{n+1}
  double* ep[3][12];    // per-edge partials of the EMF adjoint, per edge family
  double* sw1[3][5];    // stage-1 sweep outputs kept for its reverse: SR, SL, dv[3]
};

// ---------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------

// Output side: V' = ConsToPrim(U', avg b'); lam_prim -> lamU (= lamU0 =
// half of the U' adjoint) and lamBc.
__global__ void __launch_bounds__(256)
k_adj_out(Geo g, AdjArrays A, const double* lam_prim)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
  double v[NV], lv[NV];
#pragma unroll
  for (int q = 0; q < NV; q++) {
    v[q] = A.VN[q][p.c];
    lv[q] = lam_prim[(long)q * g.n + p.c];
  }
  double au[5] = {0, 0, 0, 0, 0}, ab[3] = {lv[BX1], lv[BX2], lv[BX3]};
  cons2prim_vjp(v, lv, au, ab, g.gmm1);
#pragma unroll
  for (int q = 0; q < 5; q++) {
    A.lamU[q][p.c] = 0.5 * au[q];
    A.lamU0[q][p.c] = 0.5 * au[q];
  }
#pragma unroll
  for (int a = 0; a < 3; a++) A.lamBc[a][p.c] = ab[a];
#pragma unroll
  for (int q = 0; q < NV; q++) A.lamV[q][p.c] = 0.0;   // scatter target of stage 2
}

// lam_face + avg^T lamBc, halved into the stage-2 faces and the b^n part.
__global__ void __launch_bounds__(256)
k_adj_out_faces(Geo g, AdjArrays A, const double* lam_face)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const long cp = nbr(g, p, a, 1);
    const double lb = lam_face[(long)a * g.n + p.c] + 0.5 * (A.lamBc[a][p.c] + A.lamBc[a][cp]);
    A.lamB[a][p.c] = 0.5 * lb;
    A.lamB0[a][p.c] = 0.5 * lb;
  }
}

// CT transpose: lamE from the face adjoint (ct_update.c:87-196 reversed).
__global__ void __launch_bounds__(256)
k_adj_ct(Geo g, AdjArrays A, const DevScalars* sc)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
  const double dt = sc->dt;
  const double dtx = dt / g.dx[0], dty = dt / g.dx[1], dtz = dt / g.dx[2];
  const long c = p.c;
  const long cip = nbr<0>(g, p, 1), cjp = nbr<1>(g, p, 1), ckp = nbr<2>(g, p, 1);
  const double *lbx = A.lamB[0], *lby = A.lamB[1], *lbz = A.lamB[2];
  A.lamE[2][c] = -dty * (lbx[c] - lbx[cjp]) + dtx * (lby[c] - lby[cip]);
  A.lamE[1][c] = dtz * (lbx[c] - lbx[ckp]) - dtx * (lbz[c] - lbz[cip]);
  A.lamE[0][c] = -dtz * (lby[c] - lby[ckp]) + dty * (lbz[c] - lbz[cjp]);
}

// ---------------------------------------------------------------------
// EMF adjoint in two passes without atomics, for the UCT_HLL edge families
// with axes (P, Q): Ez = <0,1>, Ex = <1,2>, Ey = <2,0> (the stencils of
// k_emf).  Pass 1 (per edge, for each family F) stores 12 partials:
//   0-3   speed adjoints SP.SR, SP.SL, SQ.SR, SQ.SL, each going to the cell
//         the edge's max() selected (c or c+Q for SP, c or c+P for SQ); the
//         gather redoes the comparison
//   4-7   adjoints of the corner EMFs of SW (c), SE (c+P), NE (c+P+Q),
//         NW (c+Q)
//   8-11  adjoints of the limited faces S, N, W, E
// Pass 2 (per cell) gathers what the neighbouring edges sent to the cell: it
// forms the face states and the limiters' branches of the few cells that it
// needs from the fields, and multiplies there what pass 1 otherwise had to
// multiply out and store (24 partials an edge).  Both passes are bound by
// memory, 480 and 580 B a cell instead of 770 and 840: at 128^3 577 -> 318 and
// 441 -> 369 us a launch.
// ---------------------------------------------------------------------

// byte offsets of a cell and, periodic, of its neighbours up to two away (32
// bits: the adjoint's arrays of a box with fields of 4 GiB would not fit the
// device); one VGPR an address where 64-bit ones took two and a multiply
struct AdjOffs {
  unsigned c;
  unsigned d[3][5];   // [axis][offset + 2], to add to c
};

__device__ __forceinline__ AdjOffs adj_offs(const Geo& g, const AdjCell& p)
{
  AdjOffs o;
  o.c = (unsigned)p.c * 8u;
  const unsigned st[3] = {8u, 8u * (unsigned)g.nx, 8u * (unsigned)g.nx * (unsigned)g.ny};
  const int q[3] = {p.i, p.j, p.k}, n[3] = {g.nx, g.ny, g.nz};
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int m = -2; m <= 2; m++) {
      const int w = wrap2(q[a], m, n[a]) - q[a];
      o.d[a][m + 2] = m == 0 ? 0u : (unsigned)w * st[a];
    }
  return o;
}

template <int P, int Q>
__device__ __forceinline__ void emf_edge_partials(const AdjOffs& of, const StageIn& in,
                                                  const Sweeps& sw, const AdjArrays& A)
{
  constexpr int E = 3 - P - Q;
  constexpr int F = (P == 0 ? 0 : P == 1 ? 1 : 2);
  const unsigned c = of.c;
  double o[12];
#pragma unroll
  for (int q = 0; q < 12; q++) o[q] = 0.0;
  const double le = at_byte(A.lamE[E], c);
  if (le != 0.0) {
    const unsigned cP = c + of.d[P][3], cQ = c + of.d[Q][3];
    const unsigned cPQ = cP + of.d[Q][3];
    const SweepOut &SP = sw.d[P], &SQ = sw.d[Q];
    const double* vP = in.V[VX1 + P];
    const double* vQ = in.V[VX1 + Q];
    const double* bP = in.b[P];
    const double* bQ = in.b[Q];
    const bool sxp = at_byte(SP.SR, c) >= at_byte(SP.SR, cQ), sxm = at_byte(SP.SL, c) >= at_byte(SP.SL, cQ);
    const bool syp = at_byte(SQ.SR, c) >= at_byte(SQ.SR, cP), sym = at_byte(SQ.SL, c) >= at_byte(SQ.SL, cP);
    double x[12];
    x[0] = sxp ? at_byte(SP.SR, c) : at_byte(SP.SR, cQ);
    x[1] = sxm ? at_byte(SP.SL, c) : at_byte(SP.SL, cQ);
    x[2] = syp ? at_byte(SQ.SR, c) : at_byte(SQ.SR, cP);
    x[3] = sym ? at_byte(SQ.SL, c) : at_byte(SQ.SL, cP);
    const unsigned cQm = c + of.d[Q][1], cPm = c + of.d[P][1];
    const unsigned cQQ = c + of.d[Q][4], cPP = c + of.d[P][4];
    const double dpS = at_byte(bP, cQ) - at_byte(bP, c), dmS = at_byte(bP, c) - at_byte(bP, cQm);
    const double dpN = at_byte(bP, cQQ) - at_byte(bP, cQ), dmN = at_byte(bP, cQ) - at_byte(bP, c);
    const double dpW = at_byte(bQ, cP) - at_byte(bQ, c), dmW = at_byte(bQ, c) - at_byte(bQ, cPm);
    const double dpE = at_byte(bQ, cPP) - at_byte(bQ, cP), dmE = at_byte(bQ, cP) - at_byte(bQ, c);
    const double bS = at_byte(bP, c) + 0.5 * mc_lim2(dpS, dmS);
    const double bW = at_byte(bQ, c) + 0.5 * mc_lim2(dpW, dmW);
    const double bN = at_byte(bP, cQ) - 0.5 * mc_lim2(dpN, dmN);
    const double bE = at_byte(bQ, cP) - 0.5 * mc_lim2(dpE, dmE);
    const double qSW = at_byte(vQ, c) + 0.5 * (at_byte(SP.dv[Q], c) + at_byte(SQ.dv[Q], c));
    const double pSW = at_byte(vP, c) + 0.5 * (at_byte(SP.dv[P], c) + at_byte(SQ.dv[P], c));
    const double qSE = at_byte(vQ, cP) - 0.5 * (at_byte(SP.dv[Q], cP) - at_byte(SQ.dv[Q], cP));
    const double pSE = at_byte(vP, cP) - 0.5 * (at_byte(SP.dv[P], cP) - at_byte(SQ.dv[P], cP));
    const double qNE = at_byte(vQ, cPQ) - 0.5 * (at_byte(SP.dv[Q], cPQ) + at_byte(SQ.dv[Q], cPQ));
    const double pNE = at_byte(vP, cPQ) - 0.5 * (at_byte(SP.dv[P], cPQ) + at_byte(SQ.dv[P], cPQ));
    const double qNW = at_byte(vQ, cQ) + 0.5 * (at_byte(SP.dv[Q], cQ) - at_byte(SQ.dv[Q], cQ));
    const double pNW = at_byte(vP, cQ) + 0.5 * (at_byte(SP.dv[P], cQ) - at_byte(SQ.dv[P], cQ));
    x[4] = qSW * bS - pSW * bW;
    x[5] = qSE * bS - pSE * bE;
    x[6] = qNE * bN - pNE * bE;
    x[7] = qNW * bN - pNW * bW;
    x[8] = bS;
    x[9] = bN;
    x[10] = bW;
    x[11] = bE;
    double ax[12] = {0};
    uct_hll_vjp(x, le, ax);
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = ax[q];
    o[8] = ax[8] + ax[4] * qSW + ax[5] * qSE;
    o[9] = ax[9] + ax[6] * qNE + ax[7] * qNW;
    o[10] = ax[10] - ax[4] * pSW - ax[7] * pNW;
    o[11] = ax[11] - ax[5] * pSE - ax[6] * pNE;
  }
#pragma unroll
  for (int q = 0; q < 12; q++) at_byte(A.ep[F][q], c) = o[q];
}

__global__ void __launch_bounds__(256)
k_adj_emf_partials(Geo g, StageIn in, Sweeps sw, AdjArrays A)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
  const AdjOffs of = adj_offs(g, p);
  emf_edge_partials<0, 1>(of, in, sw, A);   // Ez
  emf_edge_partials<1, 2>(of, in, sw, A);   // Ex
  emf_edge_partials<2, 0>(of, in, sw, A);   // Ey
}

// branch of the MC limiter of the cell between a and b (a, v, b in order): the
// slope, and its derivatives by the differences b - v and v - a
struct LimBranch {
  double s, kp, km;
};

__device__ __forceinline__ LimBranch lim_branch(double a, double v, double b)
{
  const double dp = b - v, dm = v - a;
  const double dc = 0.5 * (dp + dm);
  const bool none = dp * dm < 0.0, small = fabs(dp) < fabs(dm);
  const double sc = 2.0 * (small ? dp : dm);
  const bool mid = fabs(dc) < fabs(sc);
  return {none ? 0.0 : mid ? dc : sc, none ? 0.0 : mid ? 0.5 : small ? 2.0 : 0.0,
          none ? 0.0 : mid ? 0.5 : small ? 0.0 : 2.0};
}

template <int P, int Q>
__device__ __forceinline__ void emf_gather_family(const AdjOffs& of, const AdjArrays& A,
                                                  const StageIn& in,
                                                  const Sweeps& sw,
                                                  double (&sS)[3][2],
                                                  double (&sdv)[3][3], double (&sv)[3],
                                                  double (&sb)[3])
{
  constexpr int F = (P == 0 ? 0 : P == 1 ? 1 : 2);
  auto off = [&](int dp, int dq) { return of.c + of.d[P][dp + 2] + of.d[Q][dq + 2]; };
  const unsigned c = of.c;
  const double* const* e = A.ep[F];
  const unsigned cQ = off(0, 1), cQm = off(0, -1), cQmm = off(0, -2), cQQ = off(0, 2);
  const unsigned cP = off(1, 0), cPm = off(-1, 0), cPmm = off(-2, 0), cPP = off(2, 0);
  const unsigned cPQm = off(-1, -1);
  // speeds: the max() of edge c picked cell c, that of edge c-Q (c-P)
  // picked its upper cell c (the comparisons of emf_edge_partials)
  {
    const SweepOut &SP = sw.d[P], &SQ = sw.d[Q];
    // (all loaded, then chosen: loads under a condition cost a branch and
    // 64-bit addresses each, 256 VGPRs instead of 96)
    auto to_c = [&](const double* sp, const double* part, unsigned lo, unsigned hi) {
      const double own = at_byte(sp, c), up = at_byte(sp, hi), dn = at_byte(sp, lo);
      const double pc = at_byte(part, c), pl = at_byte(part, lo);
      return (own >= up ? pc : 0.0) + (dn >= own ? 0.0 : pl);
    };
    sS[P][1] += to_c(SP.SR, e[0], cQm, cQ);
    sS[P][0] += to_c(SP.SL, e[1], cQm, cQ);
    sS[Q][1] += to_c(SQ.SR, e[2], cPm, cP);
    sS[Q][0] += to_c(SQ.SL, e[3], cPm, cP);
  }
  // limiters along Q of the P faces c-Q, c, c+Q and c-P, along P of the Q
  // faces c-P, c, c+P and c-Q
  const double *bP = in.b[P], *bQ = in.b[Q];
  const double p0 = at_byte(bP, c), pm = at_byte(bP, cQm), pp = at_byte(bP, cQ), pl = at_byte(bP, cPm);
  const double q0 = at_byte(bQ, c), qm = at_byte(bQ, cPm), qp = at_byte(bQ, cP), ql = at_byte(bQ, cQm);
  const LimBranch Pm = lim_branch(at_byte(bP, cQmm), pm, p0), P0 = lim_branch(pm, p0, pp), Pp = lim_branch(p0, pp, at_byte(bP, cQQ));
  const LimBranch Qm = lim_branch(at_byte(bQ, cPmm), qm, q0), Q0 = lim_branch(qm, q0, qp), Qp = lim_branch(q0, qp, at_byte(bQ, cPP));
  const double sPl = mc_lim2(at_byte(bP, off(-1, 1)) - pl, pl - at_byte(bP, cPQm));
  const double sQl = mc_lim2(at_byte(bQ, off(1, -1)) - ql, ql - at_byte(bQ, cPQm));
  // corners: c is SW of edge c, SE of c-P, NE of c-P-Q, NW of c-Q
  const double wSW = at_byte(e[4], c), wSE = at_byte(e[5], cPm), wNE = at_byte(e[6], cPQm), wNW = at_byte(e[7], cQm);
  const double aSW = wSW * (p0 + 0.5 * P0.s), pSWv = -wSW * (q0 + 0.5 * Q0.s);
  const double aSE = wSE * (pl + 0.5 * sPl), pSEv = -wSE * (q0 - 0.5 * Q0.s);
  const double aNE = wNE * (pl - 0.5 * sPl), pNEv = -wNE * (ql - 0.5 * sQl);
  const double aNW = wNW * (p0 - 0.5 * P0.s), pNWv = -wNW * (ql + 0.5 * sQl);
  sv[Q] += aSW + aSE + aNE + aNW;
  sv[P] += pSWv + pSEv + pNEv + pNWv;
  sdv[P][Q] += 0.5 * aSW - 0.5 * aSE - 0.5 * aNE + 0.5 * aNW;
  sdv[Q][Q] += 0.5 * aSW + 0.5 * aSE - 0.5 * aNE - 0.5 * aNW;
  sdv[P][P] += 0.5 * pSWv - 0.5 * pSEv - 0.5 * pNEv + 0.5 * pNWv;
  sdv[Q][P] += 0.5 * pSWv + 0.5 * pSEv - 0.5 * pNEv - 0.5 * pNWv;
  // faces: face c is limited as S of edge c and N of c-Q, and is a neighbour
  // in the limiters of c-Q (S of edge c-Q, N of c-2Q) and c+Q (S of c+Q, N of
  // c); the same along P for W and E
  auto faces = [&](const double* lo, const double* hi, unsigned m2, unsigned m1, unsigned p1, const LimBranch& Lm,
                   const LimBranch& L0, const LimBranch& Lp) {
    const double l0 = 0.5 * at_byte(lo, c), h0 = -0.5 * at_byte(hi, m1);
    return (at_byte(lo, c) - L0.kp * l0 + L0.km * l0) + Lm.kp * (0.5 * at_byte(lo, m1)) - Lp.km * (0.5 * at_byte(lo, p1)) +
           (at_byte(hi, m1) - L0.kp * h0 + L0.km * h0) + Lm.kp * (-0.5 * at_byte(hi, m2)) - Lp.km * (-0.5 * at_byte(hi, c));
  };
  sb[P] += faces(e[8], e[9], cQmm, cQm, cQ, Pm, P0, Pp);
  sb[Q] += faces(e[10], e[11], cPmm, cPm, cP, Qm, Q0, Qp);
}

__global__ void __launch_bounds__(256) k_adj_emf_gather(Geo g, StageIn in, Sweeps sw,
                                                        AdjArrays A)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
  const AdjOffs of = adj_offs(g, p);
  double sS[3][2] = {{0, 0}, {0, 0}, {0, 0}};
  double sdv[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  double sv[3] = {0, 0, 0}, sb[3] = {0, 0, 0};
  emf_gather_family<0, 1>(of, A, in, sw, sS, sdv, sv, sb);
  asm volatile("" ::: "memory");   // one family's loads at a time
  emf_gather_family<1, 2>(of, A, in, sw, sS, sdv, sv, sb);
  asm volatile("" ::: "memory");   // one family's loads at a time
  emf_gather_family<2, 0>(of, A, in, sw, sS, sdv, sv, sb);
  const long c = p.c;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    A.lamS[d][0][c] = sS[d][0];
    A.lamS[d][1][c] = sS[d][1];
#pragma unroll
    for (int k = 0; k < 3; k++) A.lamDV[d][k][c] = sdv[d][k];
    A.lamV[VX1 + d][c] += sv[d];
    A.lamB[d][c] += sb[d];
  }
}

// What the adjoint of the interface q+1/2 along D reads besides the primitives
// of the cells q-1 .. q+2: the adjoints of U of q and q+1, and of cell q the
// face value, the adjoints of its face speeds and velocity slopes.
struct Iface {
  double u0[5], u1[5], b, lS[2], ldv[3];
};

// Adjoint of the interface q+1/2 along D: U += -dt/dx (F_{q+1/2} -
// F_{q-1/2}) and the pressure term, the UCT_HLL face speeds and the velocity
// slopes of cell q, through HLLD and the MC-limited PLM.  cell(k, v) is
// variable v of the cell q + k, in LDS: it is read again for the limiters, so
// that its 32 values are not held through the solver.  part[4 s + k]
// receives what variable slot s (BN skipped) of the cell at offset k - 1 from
// q along D gets; returns the adjoint of the face value.
template <int D, typename Cell>
__device__ __forceinline__ double adj_interface(const Geo& g, const Cell& cell, const Iface& f,
                                                double dtdx, double part[28])
{
  constexpr int BN = BX1 + Dir<D>::n;
  double vL[NV], vR[NV];
#pragma unroll
  for (int q = 0; q < NV; q++) {
    const double v0 = cell(0, q), vp = cell(1, q);
    vL[q] = v0 + mc_slope(cell(-1, q), v0, vp) * 0.5;
    vR[q] = vp - mc_slope(v0, vp, cell(2, q)) * 0.5;
  }
  vL[BN] = f.b;
  vR[BN] = f.b;

  HlldSeed s;
#pragma unroll
  for (int q = 0; q < NV; q++) s.f[q] = 0.0;
  s.f[RHO] = dtdx * (f.u1[0] - f.u0[0]);
  s.f[VX1] = dtdx * (f.u1[1] - f.u0[1]);
  s.f[VX2] = dtdx * (f.u1[2] - f.u0[2]);
  s.f[VX3] = dtdx * (f.u1[3] - f.u0[3]);
  s.f[ENG] = dtdx * (f.u1[4] - f.u0[4]);
  s.press = dtdx * (f.u1[1 + D] - f.u0[1 + D]);
  // stored speeds max(0, -SL), max(0, SR): derivative on the active side
  double slmin, slmax, srmin, srmax;
  fast_speeds<D>(vL, g.gamma, slmin, slmax);
  fast_speeds<D>(vR, g.gamma, srmin, srmax);
  const double SL = min_le(slmin, srmin), SR = max_ge(slmax, srmax);
  s.SL = (0.0 >= -SL) ? 0.0 : -f.lS[0];
  s.SR = (0.0 >= SR) ? 0.0 : f.lS[1];

  double aL[NV] = {0}, aR[NV] = {0};
  hlld_vjp<D>(vL, vR, g.gamma, g.gmm1, s, aL, aR);

  asm volatile("" ::: "memory");   // the cells are read again from here on
#pragma unroll
  for (int q = 0; q < NV; q++) {
    if (q == BN) continue;
    const double vm = cell(-1, q), v0 = cell(0, q), vp = cell(1, q), vq = cell(2, q);
    double a_s0 = 0.5 * aL[q];
    if (q >= VX1 && q <= VX3) a_s0 += f.ldv[q - VX1];
    const double a_s1 = -0.5 * aR[q];
    double am = 0.0, a0 = aL[q], ap = aR[q], aq = 0.0;
    mc_slope_vjp(vm, v0, vp, a_s0, am, a0, ap);
    mc_slope_vjp(v0, vp, vq, a_s1, a0, ap, aq);
    const int sl = 4 * (q < BN ? q : q - 1);
    part[sl + 0] = am;
    part[sl + 1] = a0;
    part[sl + 2] = ap;
    part[sl + 3] = aq;
  }
  return aL[BN] + aR[BN];
}

// The interface adjoints keep about 400 registers a lane, one wave per SIMD, so
// no other wave hides a load: with each interface's 45 values loaded where they
// are used they waited for memory 54% of the time.  Both kernels below
// therefore load what the next interface needs before they solve the present
// one, take what two interfaces share from registers or LDS, and read the
// sums that they add to with the same loads.  128^3: x rows 448 -> 260 us a
// launch, marches 454 -> 255.  (Two waves per SIMD would leave 256 registers a
// lane: 212 spilled, 741 and 1126 us.)

// The x interfaces of box rows r0 .. r0 + len - 1 of the ny nz rows, one row
// after another (thread i = cell i, nx <= 256): the row's primitives and U
// adjoints go through LDS, each thread solves the interface i+1/2, the 28
// partials go through LDS, and cell i sums what the interfaces i+3/2, i+1/2,
// i-1/2, i-3/2 sent it into lamV (periodic along the row).
__global__ void __launch_bounds__(256) k_adj_flux_x_rows(Geo g, StageIn in, AdjArrays A,
                                                         const DevScalars* sc, int len)
{
  extern __shared__ double sm[];   // [28][blockDim.x] partials, [13][blockDim.x] cells
  const int nt = blockDim.x, t = threadIdx.x;
  double* cell = sm + 28 * nt;
  const bool act = t < g.nx;
  const int i = act ? t : g.nx - 1;   // (idle lanes load the last cell)
  const int r0 = blockIdx.x * len, r1 = min(r0 + len, g.ny * g.nz);
  const int p1 = i + 1 < g.nx ? i + 1 : i + 1 - g.nx;
  const int p2 = i + 2 < g.nx ? i + 2 : i + 2 - g.nx;
  const int m1 = i >= 1 ? i - 1 : i - 1 + g.nx;
  const int m2 = i >= 2 ? i - 2 : i - 2 + g.nx;
  const double dtdx = sc->dt / g.dx[0];
  struct Row {
    double v[NV], u[5], b, lS[2], ldv[3], lb, lv[7];
  };
  auto load = [&](int r) {
    const unsigned c = ((unsigned)r * (unsigned)g.nx + (unsigned)i) * 8u;
    Row w;
#pragma unroll
    for (int q = 0; q < NV; q++) w.v[q] = at_byte(in.V[q], c);
#pragma unroll
    for (int q = 0; q < 5; q++) w.u[q] = at_byte(A.lamU[q], c);
    w.b = at_byte(in.b[0], c);
    w.lS[0] = at_byte(A.lamS[0][0], c);
    w.lS[1] = at_byte(A.lamS[0][1], c);
#pragma unroll
    for (int q = 0; q < 3; q++) w.ldv[q] = at_byte(A.lamDV[0][q], c);
    w.lb = at_byte(A.lamB[0], c);
#pragma unroll
    for (int s = 0; s < 7; s++) w.lv[s] = at_byte(A.lamV[s < BX1 ? s : s + 1], c);
    return w;
  };
  Row w = load(r0);
  for (int r = r0; r < r1; r++) {
    const unsigned c = ((unsigned)r * (unsigned)g.nx + (unsigned)i) * 8u;
    if (act) {
#pragma unroll
      for (int q = 0; q < NV; q++) cell[q * nt + i] = w.v[q];
#pragma unroll
      for (int q = 0; q < 5; q++) cell[(NV + q) * nt + i] = w.u[q];
    }
    const Row cur = w;
    w = load(min(r + 1, r1 - 1));
    __syncthreads();
    if (act) {
      Iface f;
#pragma unroll
      for (int q = 0; q < 5; q++) {
        f.u0[q] = cur.u[q];
        f.u1[q] = cell[(NV + q) * nt + p1];
      }
      f.b = cur.b;
      f.lS[0] = cur.lS[0];
      f.lS[1] = cur.lS[1];
#pragma unroll
      for (int q = 0; q < 3; q++) f.ldv[q] = cur.ldv[q];
      double part[28];
      const double ab = adj_interface<0>(
          g, [&](int k, int q) { return cell[q * nt + (k < 0 ? m1 : k == 0 ? i : k == 1 ? p1 : p2)]; }, f,
          dtdx, part);
      at_byte(A.lamB[0], c) = cur.lb + ab;
#pragma unroll
      for (int m = 0; m < 28; m++) sm[m * nt + i] = part[m];
    }
    __syncthreads();
    if (act) {
#pragma unroll
      for (int s = 0; s < 7; s++)
        at_byte(A.lamV[s < BX1 ? s : s + 1], c) =
            cur.lv[s] + (sm[4 * s * nt + p1] + sm[(4 * s + 1) * nt + i] + sm[(4 * s + 2) * nt + m1] +
                         sm[(4 * s + 3) * nt + m2]);
    }
  }
}

// The interfaces along D of one line segment per thread: lanes run along
// the first transverse axis (x for D = 1, 2; y for D = 0), blockIdx.y picks
// the line in the other one, blockIdx.z the segment [q0, q0 + len) of
// cells along D.  The thread solves the interfaces q+1/2 for q = q0-2 ..
// q0+len in order (the three beyond the segment, q0-2, q0-1 and q0+len, are
// solved again by the neighbouring segments), adds each one's partials into a ring of four
// cells kept in LDS, and after interface q adds the now complete cell q-1
// to lamV.  Only the interfaces q0..q0+len-1 add their face adjoint.
template <int D>
__global__ void __launch_bounds__(256) k_adj_flux_march(Geo g, StageIn in, AdjArrays A,
                                                        const DevScalars* sc, int len)
{
  constexpr int BN = BX1 + Dir<D>::n;
  __shared__ double ring[28][256];   // [4 * slot + cell (mod 4)][thread]
  __shared__ double vcell[4 * NV][256];   // the cells q-1 .. q+2: [NV * (cell mod 4) + variable][thread]
  const int t = threadIdx.y * blockDim.x + threadIdx.x;
  const int nD = D == 0 ? g.nx : D == 1 ? g.ny : g.nz;
  const int l0 = blockIdx.x * blockDim.x + threadIdx.x;           // first transverse axis
  const int l1 = blockIdx.y * blockDim.y + threadIdx.y;           // second one
  const int n0 = D == 0 ? g.ny : g.nx, n1 = D == 2 ? g.ny : g.nz;
  if (l0 >= n0 || l1 >= n1) return;
  const int q0 = blockIdx.z * len;
  const int q1 = min(q0 + len, nD);
#pragma unroll
  for (int m = 0; m < 28; m++) ring[m][t] = 0.0;
  const double dtdx = sc->dt / g.dx[D];
  // byte offset of the line's cell q, periodic
  const unsigned sD = 8u * (D == 0 ? 1u : D == 1 ? (unsigned)g.nx : (unsigned)g.nx * (unsigned)g.ny);
  const unsigned base = 8u * (D == 0   ? ((unsigned)l1 * (unsigned)g.ny + (unsigned)l0) * (unsigned)g.nx
                              : D == 1 ? (unsigned)l1 * (unsigned)g.ny * (unsigned)g.nx + (unsigned)l0
                                       : (unsigned)l1 * (unsigned)g.nx + (unsigned)l0);
  auto off = [&](int q) { return base + (unsigned)(q < 0 ? q + nD : q >= nD ? q - nD : q) * sD; };
  // what an interface does not share with the one before it: cell q+2, the U
  // adjoint of q+1, what it reads of cell q, and the sums of cell q-1
  struct Ahead {
    double vq[NV], u1[5], b, lS[2], ldv[3], lb, lv[7];
  };
  auto load = [&](int q) {
    const unsigned c = off(q), c1 = off(q + 1), c2 = off(q + 2), cm = off(q - 1);
    Ahead w;
#pragma unroll
    for (int v = 0; v < NV; v++) w.vq[v] = at_byte(in.V[v], c2);
#pragma unroll
    for (int v = 0; v < 5; v++) w.u1[v] = at_byte(A.lamU[v], c1);
    w.b = at_byte(in.b[D], c);
    w.lS[0] = at_byte(A.lamS[D][0], c);
    w.lS[1] = at_byte(A.lamS[D][1], c);
#pragma unroll
    for (int v = 0; v < 3; v++) w.ldv[v] = at_byte(A.lamDV[D][v], c);
    w.lb = at_byte(A.lamB[D], c);
#pragma unroll
    for (int s = 0; s < 7; s++) w.lv[s] = at_byte(A.lamV[s < BN ? s : s + 1], cm);
    return w;
  };
  Iface f;
  Ahead w = load(q0 - 2);
  {
    const unsigned cm = off(q0 - 3), c = off(q0 - 2), c1 = off(q0 - 1);
#pragma unroll
    for (int v = 0; v < NV; v++) {
      vcell[NV * ((q0 - 3) & 3) + v][t] = at_byte(in.V[v], cm);
      vcell[NV * ((q0 - 2) & 3) + v][t] = at_byte(in.V[v], c);
      vcell[NV * ((q0 - 1) & 3) + v][t] = at_byte(in.V[v], c1);
    }
#pragma unroll
    for (int v = 0; v < 5; v++) f.u0[v] = at_byte(A.lamU[v], c);
  }
  for (int q = q0 - 2; q <= q1; q++) {
    const Ahead cur = w;
    w = load(min(q + 1, q1));
#pragma unroll
    for (int v = 0; v < NV; v++) vcell[NV * ((q + 2) & 3) + v][t] = cur.vq[v];
#pragma unroll
    for (int v = 0; v < 5; v++) f.u1[v] = cur.u1[v];
    f.b = cur.b;
    f.lS[0] = cur.lS[0];
    f.lS[1] = cur.lS[1];
#pragma unroll
    for (int v = 0; v < 3; v++) f.ldv[v] = cur.ldv[v];
    double part[28];
    const double ab = adj_interface<D>(
        g, [&](int k, int v) { return vcell[NV * ((q + k) & 3) + v][t]; }, f, dtdx, part);
    if (q >= q0 && q < q1) at_byte(A.lamB[D], off(q)) = cur.lb + ab;
    // targets q-1 .. q+2 (k = 0..3) sit in ring slots (q - 1 + k) mod 4
#pragma unroll
    for (int s = 0; s < 7; s++)
#pragma unroll
      for (int k = 0; k < 4; k++) ring[4 * s + ((q - 1 + k) & 3)][t] += part[4 * s + k];
    // cell q-1 is complete: its last interface was q+1/2
    const int done = (q - 1) & 3;
    if (q - 1 >= q0) {
      const unsigned cc = off(q - 1);
#pragma unroll
      for (int s = 0; s < 7; s++) at_byte(A.lamV[s < BN ? s : s + 1], cc) = cur.lv[s] + ring[4 * s + done][t];
    }
#pragma unroll
    for (int s = 0; s < 7; s++) ring[4 * s + done][t] = 0.0;
#pragma unroll
    for (int v = 0; v < 5; v++) f.u0[v] = f.u1[v];
  }
}

// Between the stages: V1 = ConsToPrim(U*, avg b*).  lamU += (dV1/dU*)^T lamV,
// lamBc = field part; lamV is cleared for the stage-1 pass.
__global__ void __launch_bounds__(256)
k_adj_mid(Geo g, AdjArrays A, StageIn in)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
  double v[NV], lv[NV];
#pragma unroll
  for (int q = 0; q < NV; q++) {
    v[q] = in.V[q][p.c];
    lv[q] = A.lamV[q][p.c];
    A.lamV[q][p.c] = 0.0;
  }
  double au[5] = {0, 0, 0, 0, 0}, ab[3] = {lv[BX1], lv[BX2], lv[BX3]};
  cons2prim_vjp(v, lv, au, ab, g.gmm1);
#pragma unroll
  for (int q = 0; q < 5; q++) A.lamU[q][p.c] += au[q];
#pragma unroll
  for (int a = 0; a < 3; a++) A.lamBc[a][p.c] = ab[a];
}

// lamB += avg^T lamBc
__global__ void __launch_bounds__(256) k_adj_avgT(Geo g, AdjArrays A)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const long cp = nbr(g, p, a, 1);
    A.lamB[a][p.c] += 0.5 * (A.lamBc[a][p.c] + A.lamBc[a][cp]);
  }
}

// Input side: U0 = PrimToCons(V^n) takes lamU (stage 1) + lamU0 (blend);
// writes the primitive adjoint (field components folded into lamBc).
__global__ void __launch_bounds__(256)
k_adj_in(Geo g, AdjArrays A, StageIn in, double* lam_prim)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
  double v[NV], lv[NV], au[NV] = {0};
#pragma unroll
  for (int q = 0; q < NV; q++) {
    v[q] = in.V[q][p.c];
    lv[q] = A.lamV[q][p.c];
  }
  au[RHO] = A.lamU[0][p.c] + A.lamU0[0][p.c];
  au[VX1] = A.lamU[1][p.c] + A.lamU0[1][p.c];
  au[VX2] = A.lamU[2][p.c] + A.lamU0[2][p.c];
  au[VX3] = A.lamU[3][p.c] + A.lamU0[3][p.c];
  au[ENG] = A.lamU[4][p.c] + A.lamU0[4][p.c];
  prim2cons_vjp(v, au, lv, g.gmm1);
#pragma unroll
  for (int a = 0; a < 3; a++) {
    A.lamBc[a][p.c] = lv[BX1 + a];
    lv[BX1 + a] = 0.0;
  }
#pragma unroll
  for (int q = 0; q < NV; q++) lam_prim[(long)q * g.n + p.c] = lv[q];
}

__global__ void __launch_bounds__(256)
k_adj_faces_final(Geo g, AdjArrays A, double* lam_face)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const long cp = nbr(g, p, a, 1);
    lam_face[(long)a * g.n + p.c] =
        A.lamB[a][p.c] + 0.5 * (A.lamBc[a][p.c] + A.lamBc[a][cp]) + A.lamB0[a][p.c];
  }
}

// Cell-centred field as the face average (after a device-side state copy).
__global__ void __launch_bounds__(256) k_cell_field(Geo g, Prims V, FaceIn b)
{
  AdjCell p;
  if (!adj_cell(g, p)) return;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (a == 2 && g.dims != 3) {
      V.v[BX3][p.c] = 0.0;
      continue;
    }
    const long cm = nbr(g, p, a, -1);
    V.v[BX1 + a][p.c] = 0.5 * (b.b[a][p.c] + b.b[a][cm]);
  }
}

// Segment length of the interface march along D: the longest of 64, 32, 16
// that still gives one workgroup per CU (the march runs one wave per SIMD,
// one workgroup per CU at a time); each segment solves the three interfaces
// beyond its cells again.
static int adj_march_len(const Geo& g, int D)
{
  const int nD = D == 0 ? g.nx : D == 1 ? g.ny : g.nz;
  const long lines = D == 0 ? (long)((g.ny + 63) / 64) * ((g.nz + 3) / 4)
                            : (long)((g.nx + 63) / 64) * (((D == 1 ? g.nz : g.ny) + 3) / 4);
  int len = 64;
  while (len > 16 && lines * ((nD + len - 1) / len) < 256) len /= 2;
  return len;
}

// Rows a workgroup of the x interfaces takes one after another (only the first
// one's loads are waited for): 16, fewer where that would leave less than two
// workgroups for each place (four waves a CU)
static int adj_rows_len(int rows, int nt)
{
  const int places = 256 * (256 / nt);
  int len = 16;
  while (len > 1 && (rows + len - 1) / len < 2 * places) len /= 2;
  return len;
}

// One stage in reverse: CT transpose, EMF adjoint, flux adjoints.
static void adj_stage(const Geo& g, const StageIn& in, const Sweeps& sw, const AdjArrays& A,
                      const DevScalars* sc, hipStream_t s)
{
  const dim3 gr = adj_grid(g);
  hipLaunchKernelGGL(k_adj_ct, gr, kAdjBlock, 0, s, g, A, sc);
  hipLaunchKernelGGL(k_adj_emf_partials, gr, kAdjBlock, 0, s, g, in, sw, A);
  hipLaunchKernelGGL(k_adj_emf_gather, gr, kAdjBlock, 0, s, g, in, sw, A);
  // x: whole rows through LDS where they fit a workgroup, else marching
  if (g.nx <= 256) {
    const int nt = (g.nx + 63) / 64 * 64;
    const int rows = g.ny * g.nz, len = adj_rows_len(rows, nt);
    hipLaunchKernelGGL(k_adj_flux_x_rows, dim3((rows + len - 1) / len), dim3(nt),
                       41 * nt * sizeof(double), s, g, in, A, sc, len);
  } else {
    const int len = adj_march_len(g, 0);
    hipLaunchKernelGGL(k_adj_flux_march<0>, dim3((g.ny + 63) / 64, (g.nz + 3) / 4, (g.nx + len - 1) / len),
                       kAdjBlock, 0, s, g, in, A, sc, len);
  }
  const int ly = adj_march_len(g, 1), lz = adj_march_len(g, 2);
  hipLaunchKernelGGL(k_adj_flux_march<1>, dim3((g.nx + 63) / 64, (g.nz + 3) / 4, (g.ny + ly - 1) / ly),
                     kAdjBlock, 0, s, g, in, A, sc, ly);
  hipLaunchKernelGGL(k_adj_flux_march<2>, dim3((g.nx + 63) / 64, (g.ny + 3) / 4, (g.nz + lz - 1) / lz),
                     kAdjBlock, 0, s, g, in, A, sc, lz);
}

}  // namespace pgpu

using namespace pgpu;

struct pgpu_adjoint_state {
  AdjArrays a;
  void* block = nullptr;
  size_t bytes = 0;
};

static int adj_alloc(pgpu_domain* d)
{
  if (d->adj) return PGPU_OK;
  const size_t per = (size_t)d->g.n * sizeof(double);
  const int narr = 8 + 5 + 5 + 3 + 3 + 3 + 6 + 9 + 3 + 8 + 3 + 36 + 15;
  pgpu_adjoint_state* st = new pgpu_adjoint_state;
  st->bytes = per * narr;
  if (hipMalloc(&st->block, st->bytes) != hipSuccess) {
    const size_t b = st->bytes;
    delete st;
    return fail(PGPU_ENOMEM, "hipMalloc of %zu bytes for the adjoint failed", b);
  }
  char* cur = (char*)st->block;
  auto take = [&]() {
    double* p = (double*)cur;
    cur += per;
    return p;
  };
  AdjArrays& A = st->a;
  for (int q = 0; q < 8; q++) A.lamV[q] = take();
  for (int q = 0; q < 5; q++) A.lamU[q] = take();
  for (int q = 0; q < 5; q++) A.lamU0[q] = take();
  for (int a = 0; a < 3; a++) A.lamB[a] = take();
  for (int a = 0; a < 3; a++) A.lamB0[a] = take();
  for (int a = 0; a < 3; a++) A.lamE[a] = take();
  for (int dd = 0; dd < 3; dd++)
    for (int k = 0; k < 2; k++) A.lamS[dd][k] = take();
  for (int dd = 0; dd < 3; dd++)
    for (int k = 0; k < 3; k++) A.lamDV[dd][k] = take();
  for (int a = 0; a < 3; a++) A.lamBc[a] = take();
  for (int q = 0; q < 8; q++) A.VN[q] = take();
  for (int a = 0; a < 3; a++) A.bN[a] = take();
  for (int f = 0; f < 3; f++)
    for (int q = 0; q < 12; q++) A.ep[f][q] = take();
  for (int dd = 0; dd < 3; dd++)
    for (int q = 0; q < 5; q++) A.sw1[dd][q] = take();
  d->adj = st;
  return PGPU_OK;
}

void pgpu_adjoint_free(pgpu_domain* d)
{
  if (!d || !d->adj) return;
  (void)hipFree(d->adj->block);
  delete d->adj;
  d->adj = nullptr;
}

extern "C" int pgpu_set_state_device(pgpu_domain* d, const double* prim8, const double* face3)
{
  if (!d || !prim8 || !face3) return fail(PGPU_EINVAL, "NULL argument");
  if (d->g.ghost) return fail(PGPU_EINVAL, "a bounded box takes its state through pgpu_set_state");
  const Geo& g = d->g;
  const size_t nb = (size_t)g.n * sizeof(double);
  for (int q = 0; q < 8; q++)
    if (hipMemcpyAsync(d->V[q], prim8 + (size_t)q * g.n, nb, hipMemcpyDeviceToDevice,
                       d->stream) != hipSuccess)
      return fail(PGPU_EDEVICE, "device state copy failed");
  for (int a = 0; a < 3; a++)
    if (hipMemcpyAsync(d->bA[a], face3 + (size_t)a * g.n, nb, hipMemcpyDeviceToDevice,
                       d->stream) != hipSuccess)
      return fail(PGPU_EDEVICE, "device state copy failed");
  Prims V;
  FaceIn b;
  for (int q = 0; q < 8; q++) V.v[q] = d->V[q];
  for (int a = 0; a < 3; a++) b.b[a] = d->bA[a];
  hipLaunchKernelGGL(k_cell_field, adj_grid(g), kAdjBlock, 0, d->stream, g, V, b);
  if (hipGetLastError() != hipSuccess) return fail(PGPU_EDEVICE, "cell field kernel failed");
  return PGPU_OK;
}

extern "C" int pgpu_get_state_device(pgpu_domain* d, double* prim8, double* face3)
{
  if (!d || !prim8 || !face3) return fail(PGPU_EINVAL, "NULL argument");
  if (d->g.ghost) return fail(PGPU_EINVAL, "a bounded box returns its state through pgpu_get_state");
  const Geo& g = d->g;
  const size_t nb = (size_t)g.n * sizeof(double);
  for (int q = 0; q < 8; q++)
    if (hipMemcpyAsync(prim8 + (size_t)q * g.n, d->V[q], nb, hipMemcpyDeviceToDevice,
                       d->stream) != hipSuccess)
      return fail(PGPU_EDEVICE, "device state copy failed");
  for (int a = 0; a < 3; a++)
    if (hipMemcpyAsync(face3 + (size_t)a * g.n, d->bA[a], nb, hipMemcpyDeviceToDevice,
                       d->stream) != hipSuccess)
      return fail(PGPU_EDEVICE, "device state copy failed");
  return PGPU_OK;
}

// What the reverse of one step reads from its forward: the step's input
// (V^n, b^n), the stage-1 output (V1, b*), the face speeds and velocity
// slopes of both stages, and the output V^{n+1}.  Held in the domain's and
// the adjoint's own arrays (pgpu_adjoint_step) or in a caller's tape of
// PGPU_ADJOINT_TAPE_ARRAYS arrays of n doubles, in this order.
struct StepTape {
  double* V[8];
  double* b[3];
  double* V1[8];
  double* b1[3];
  double* sw[2][3][5];   // [stage][direction][SR, SL, dv0, dv1, dv2]
  double* VN[8];
};

static StepTape tape_view(double* base, long n)
{
  StepTape T;
  double* cur = base;
  auto take = [&]() {
    double* p = cur;
    cur += n;
    return p;
  };
  for (int q = 0; q < 8; q++) T.V[q] = take();
  for (int a = 0; a < 3; a++) T.b[a] = take();
  for (int q = 0; q < 8; q++) T.V1[q] = take();
  for (int a = 0; a < 3; a++) T.b1[a] = take();
  for (int st = 0; st < 2; st++)
    for (int dd = 0; dd < 3; dd++)
      for (int q = 0; q < 5; q++) T.sw[st][dd][q] = take();
  for (int q = 0; q < 8; q++) T.VN[q] = take();
  return T;
}

static Sweeps tape_sweeps(const pgpu_domain* d, const StepTape& T, int st)
{
  Sweeps sw = d->sw;   // flux arrays of the modular sweeps: unused here
  for (int dd = 0; dd < 3; dd++) {
    sw.d[dd].SR = T.sw[st][dd][0];
    sw.d[dd].SL = T.sw[st][dd][1];
    for (int c = 0; c < 3; c++) sw.d[dd].dv[c] = T.sw[st][dd][2 + c];
  }
  return sw;
}

static int adj_checks(const pgpu_domain* d)
{
  const Geo& g = d->g;
  if (g.dims != 3) return fail(PGPU_EINVAL, "the adjoint step needs DIMENSIONS 3");
  if (g.solver != SOLVER_HLLD) return fail(PGPU_EINVAL, "the adjoint step is the HLLD solver's");
  if (g.emf_avg != EMF_UCT_HLL) return fail(PGPU_EINVAL, "the adjoint step uses the UCT_HLL EMF average");
  if (g.ghost) return fail(PGPU_EINVAL, "the adjoint step is for periodic boxes");
  if (!d->fixed_dt) return fail(PGPU_EINVAL, "the adjoint step needs a fixed dt (pgpu_set_dt)");
  if (g.nx < 3 || g.ny < 3 || g.nz < 3)
    return fail(PGPU_EINVAL, "the adjoint step needs at least 3 cells per direction");
  return PGPU_OK;
}

// The forward step from T.V, T.b (the fused FP64 kernels, bit-identical to
// the step pgpu_run takes): stage 1 into (T.V1, T.b1), stage 2 into
// (T.VN, outB), face data into T.sw.  U, the edges, C_dt and the flags are
// the domain's scratch.
static int adj_forward(pgpu_domain* d, const StepTape& T, double* const outB[3])
{
  const Geo& g = d->g;
  hipStream_t s = d->stream;
  StageIn in1, in2, vn;
  for (int q = 0; q < 8; q++) {
    in1.V[q] = T.V[q];
    in2.V[q] = T.V1[q];
    vn.V[q] = T.V[q];
  }
  for (int a = 0; a < 3; a++) {
    in1.b[a] = T.b[a];
    in2.b[a] = T.b1[a];
    vn.b[a] = T.b[a];
  }
  Cons U;
  for (int q = 0; q < 5; q++) U.u[q] = d->U[q];
  Prims V1, VN;
  for (int q = 0; q < 8; q++) {
    V1.v[q] = T.V1[q];
    VN.v[q] = T.VN[q];
  }
  FaceIn fA, fB;
  FaceOut oB, oN;
  for (int a = 0; a < 3; a++) {
    fA.b[a] = T.b[a];
    fB.b[a] = T.b1[a];
    oB.b[a] = T.b1[a];
    oN.b[a] = outB[a];
  }
  const Sweeps sw1 = tape_sweeps(d, T, 0), sw2 = tape_sweeps(d, T, 1);
  FaceData fd1, fd2;
  for (int dd = 0; dd < 3; dd++) {
    fd1.SR[dd] = sw1.d[dd].SR;
    fd1.SL[dd] = sw1.d[dd].SL;
    fd2.SR[dd] = sw2.d[dd].SR;
    fd2.SL[dd] = sw2.d[dd].SL;
    fd1.mf[dd] = sw1.d[dd].dv[0];
    fd2.mf[dd] = sw2.d[dd].dv[0];
  }
  int rc = launch_flux_fused(g, 1, false, in1, U, fd1, d->cdt, d->sc, s, nullptr);
  if (!rc) rc = launch_vel_slopes(g, in1, sw1, s);
  if (!rc) rc = launch_emf(g, in1, sw1, d->e, s, nullptr);
  if (!rc) rc = launch_ct_c2p(g, 1, d->e, fA, fA, oB, U, vn, V1, d->flag, d->sc, s, nullptr);
  if (!rc) rc = launch_flux_fused(g, 2, false, in2, U, fd2, d->cdt, d->sc, s, nullptr);
  if (!rc) rc = launch_vel_slopes(g, in2, sw2, s);
  if (!rc) rc = launch_emf(g, in2, sw2, d->e, s, nullptr);
  if (!rc) rc = launch_ct_c2p(g, 2, d->e, fB, fA, oN, U, vn, VN, d->flag, d->sc, s, nullptr);
  if (rc) return fail(PGPU_EDEVICE, "forward recomputation failed: %s", hipGetErrorString((hipError_t)rc));
  return PGPU_OK;
}

// The reverse of the step T holds: output side, stage 2, stage 1, input side.
static int adj_reverse(pgpu_domain* d, const StepTape& T, double* lam_prim, double* lam_face)
{
  const Geo& g = d->g;
  hipStream_t s = d->stream;
  AdjArrays A = d->adj->a;
  for (int q = 0; q < 8; q++) A.VN[q] = T.VN[q];
  StageIn in1, in2;
  for (int q = 0; q < 8; q++) {
    in1.V[q] = T.V[q];
    in2.V[q] = T.V1[q];
  }
  for (int a = 0; a < 3; a++) {
    in1.b[a] = T.b[a];
    in2.b[a] = T.b1[a];
  }
  const Sweeps sw1 = tape_sweeps(d, T, 0), sw2 = tape_sweeps(d, T, 1);
  const dim3 gr = adj_grid(g);
  // output side and blend
  hipLaunchKernelGGL(k_adj_out, gr, kAdjBlock, 0, s, g, A, (const double*)lam_prim);
  hipLaunchKernelGGL(k_adj_out_faces, gr, kAdjBlock, 0, s, g, A, (const double*)lam_face);
  // stage 2
  adj_stage(g, in2, sw2, A, d->sc, s);
  hipLaunchKernelGGL(k_adj_mid, gr, kAdjBlock, 0, s, g, A, in2);
  hipLaunchKernelGGL(k_adj_avgT, gr, kAdjBlock, 0, s, g, A);
  // stage 1
  adj_stage(g, in1, sw1, A, d->sc, s);
  hipLaunchKernelGGL(k_adj_in, gr, kAdjBlock, 0, s, g, A, in1, lam_prim);
  hipLaunchKernelGGL(k_adj_faces_final, gr, kAdjBlock, 0, s, g, A, lam_face);
  if (hipGetLastError() != hipSuccess) return fail(PGPU_EDEVICE, "adjoint kernel launch failed");
  return PGPU_OK;
}

extern "C" int pgpu_adjoint_step(pgpu_domain* d, double* lam_prim, double* lam_face)
{
  if (!d || !lam_prim || !lam_face) return fail(PGPU_EINVAL, "NULL argument");
  int rc = adj_checks(d);
  if (!rc) rc = adj_alloc(d);
  if (rc) return rc;
  AdjArrays& A = d->adj->a;
  // the recomputation in the domain's arrays: stage 1 into (V1, bB), the
  // stage-1 face data into the adjoint's own arrays (its reverse needs them
  // after stage 2 has overwritten the domain's), the output into (VN, bN)
  StepTape T;
  for (int q = 0; q < 8; q++) {
    T.V[q] = d->V[q];
    T.V1[q] = d->V1[q];
    T.VN[q] = A.VN[q];
  }
  for (int a = 0; a < 3; a++) {
    T.b[a] = d->bA[a];
    T.b1[a] = d->bB[a];
  }
  for (int dd = 0; dd < 3; dd++) {
    for (int q = 0; q < 5; q++) T.sw[0][dd][q] = A.sw1[dd][q];
    T.sw[1][dd][0] = d->sw.d[dd].SR;
    T.sw[1][dd][1] = d->sw.d[dd].SL;
    for (int c = 0; c < 3; c++) T.sw[1][dd][2 + c] = d->sw.d[dd].dv[c];
  }
  rc = adj_forward(d, T, A.bN);
  if (!rc) rc = adj_reverse(d, T, lam_prim, lam_face);
  return rc;
}

extern "C" int pgpu_adjoint_record(pgpu_domain* d, double* tape)
{
  if (!d || !tape) return fail(PGPU_EINVAL, "NULL argument");
  int rc = adj_checks(d);
  if (rc) return rc;
  const long n = d->g.n;
  const size_t nb = (size_t)n * sizeof(double);
  const StepTape T = tape_view(tape, n);
  hipStream_t s = d->stream;
  for (int q = 0; q < 8; q++)
    if (hipMemcpyAsync(T.V[q], d->V[q], nb, hipMemcpyDeviceToDevice, s) != hipSuccess)
      return fail(PGPU_EDEVICE, "tape copy failed");
  for (int a = 0; a < 3; a++)
    if (hipMemcpyAsync(T.b[a], d->bA[a], nb, hipMemcpyDeviceToDevice, s) != hipSuccess)
      return fail(PGPU_EDEVICE, "tape copy failed");
  // the step reads its input from the tape, so the output faces can go
  // straight to the domain; the output primitives are copied there after
  rc = adj_forward(d, T, d->bA);
  if (rc) return rc;
  for (int q = 0; q < 8; q++)
    if (hipMemcpyAsync(d->V[q], T.VN[q], nb, hipMemcpyDeviceToDevice, s) != hipSuccess)
      return fail(PGPU_EDEVICE, "state copy failed");
  return PGPU_OK;
}

extern "C" int pgpu_adjoint_step_taped(pgpu_domain* d, const double* tape, double* lam_prim,
                                       double* lam_face)
{
  if (!d || !tape || !lam_prim || !lam_face) return fail(PGPU_EINVAL, "NULL argument");
  int rc = adj_checks(d);
  if (!rc) rc = adj_alloc(d);
  if (rc) return rc;
  return adj_reverse(d, tape_view(const_cast<double*>(tape), d->g.n), lam_prim, lam_face);
}

// ---------------------------------------------------------------------
// point-level tangent and adjoint of HLLD (for checking the adjoint)
// ---------------------------------------------------------------------

namespace pgpu {
namespace {

constexpr int kHlldOut = 8;   // rho, mx, my, mz, E fluxes, press, SL, SR

template <int D>
__global__ void k_hlld_tangent(int n, double gamma, const double* vL, const double* vR,
                               const double* tL, const double* tR, double* out, double* dout)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  Dual L[NV], R[NV];
#pragma unroll
  for (int q = 0; q < NV; q++) {
    L[q] = Dual(vL[(long)r * NV + q], tL[(long)r * NV + q]);
    R[q] = Dual(vR[(long)r * NV + q], tR[(long)r * NV + q]);
  }
  RiemannOut<Dual> o;
  hlld<D, false>(L, R, Dual(gamma), Dual(gamma - 1.0), o);
  const Dual res[kHlldOut] = {o.f[RHO], o.f[VX1], o.f[VX2], o.f[VX3], o.f[ENG], o.press, o.SL, o.SR};
#pragma unroll
  for (int q = 0; q < kHlldOut; q++) {
    out[(long)r * kHlldOut + q] = res[q].v;
    dout[(long)r * kHlldOut + q] = res[q].d;
  }
}

template <int D>
__global__ void k_hlld_adjoint(int n, double gamma, const double* vL, const double* vR,
                               const double* lam, double* aL, double* aR)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  double L[NV], R[NV], a_L[NV] = {0}, a_R[NV] = {0};
#pragma unroll
  for (int q = 0; q < NV; q++) {
    L[q] = vL[(long)r * NV + q];
    R[q] = vR[(long)r * NV + q];
  }
  HlldSeed s;
  const double* l = lam + (long)r * kHlldOut;
#pragma unroll
  for (int q = 0; q < NV; q++) s.f[q] = 0.0;
  s.f[RHO] = l[0];
  s.f[VX1] = l[1];
  s.f[VX2] = l[2];
  s.f[VX3] = l[3];
  s.f[ENG] = l[4];
  s.press = l[5];
  s.SL = l[6];
  s.SR = l[7];
  hlld_vjp<D>(L, R, gamma, gamma - 1.0, s, a_L, a_R);
#pragma unroll
  for (int q = 0; q < NV; q++) {
    aL[(long)r * NV + q] = a_L[q];
    aR[(long)r * NV + q] = a_R[q];
  }
}

// copies host rows to a temporary device block and back
struct RowScratch {
  void* p = nullptr;
  ~RowScratch() { if (p) (void)hipFree(p); }
};

}  // namespace
}  // namespace pgpu

extern "C" int pgpu_hlld_tangent_rows(int dir, int n, double gamma, const double* vL,
                                      const double* vR, const double* tL, const double* tR,
                                      double* out, double* dout)
{
  if (dir < 0 || dir > 2 || n < 0) return fail(PGPU_EINVAL, "bad direction or count");
  if (n == 0) return PGPU_OK;
  if (!vL || !vR || !tL || !tR || !out || !dout) return fail(PGPU_EINVAL, "NULL argument");
  const size_t in_b = (size_t)n * NV * sizeof(double), out_b = (size_t)n * kHlldOut * sizeof(double);
  RowScratch m;
  if (hipMalloc(&m.p, 4 * in_b + 2 * out_b) != hipSuccess) return fail(PGPU_ENOMEM, "hipMalloc failed");
  double* base = (double*)m.p;
  double *dL = base, *dR = dL + (size_t)n * NV, *dtL = dR + (size_t)n * NV, *dtR = dtL + (size_t)n * NV;
  double *dout_v = dtR + (size_t)n * NV, *dout_d = dout_v + (size_t)n * kHlldOut;
  if (hipMemcpy(dL, vL, in_b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dR, vR, in_b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dtL, tL, in_b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dtR, tR, in_b, hipMemcpyHostToDevice) != hipSuccess)
    return fail(PGPU_EDEVICE, "row upload failed");
  const dim3 b(64), gr((n + 63) / 64);
  if (dir == 0) hipLaunchKernelGGL(k_hlld_tangent<0>, gr, b, 0, 0, n, gamma, dL, dR, dtL, dtR, dout_v, dout_d);
  if (dir == 1) hipLaunchKernelGGL(k_hlld_tangent<1>, gr, b, 0, 0, n, gamma, dL, dR, dtL, dtR, dout_v, dout_d);
  if (dir == 2) hipLaunchKernelGGL(k_hlld_tangent<2>, gr, b, 0, 0, n, gamma, dL, dR, dtL, dtR, dout_v, dout_d);
  if (hipGetLastError() != hipSuccess ||
      hipMemcpy(out, dout_v, out_b, hipMemcpyDeviceToHost) != hipSuccess ||
      hipMemcpy(dout, dout_d, out_b, hipMemcpyDeviceToHost) != hipSuccess)
    return fail(PGPU_EDEVICE, "tangent kernel failed");
  return PGPU_OK;
}

extern "C" int pgpu_hlld_adjoint_rows(int dir, int n, double gamma, const double* vL,
                                      const double* vR, const double* lam, double* aL,
                                      double* aR)
{
  if (dir < 0 || dir > 2 || n < 0) return fail(PGPU_EINVAL, "bad direction or count");
  if (n == 0) return PGPU_OK;
  if (!vL || !vR || !lam || !aL || !aR) return fail(PGPU_EINVAL, "NULL argument");
  const size_t in_b = (size_t)n * NV * sizeof(double), l_b = (size_t)n * kHlldOut * sizeof(double);
  RowScratch m;
  if (hipMalloc(&m.p, 4 * in_b + l_b) != hipSuccess) return fail(PGPU_ENOMEM, "hipMalloc failed");
  double* base = (double*)m.p;
  double *dL = base, *dR = dL + (size_t)n * NV, *daL = dR + (size_t)n * NV, *daR = daL + (size_t)n * NV;
  double* dlam = daR + (size_t)n * NV;
  if (hipMemcpy(dL, vL, in_b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dR, vR, in_b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dlam, lam, l_b, hipMemcpyHostToDevice) != hipSuccess)
    return fail(PGPU_EDEVICE, "row upload failed");
  const dim3 b(64), gr((n + 63) / 64);
  if (dir == 0) hipLaunchKernelGGL(k_hlld_adjoint<0>, gr, b, 0, 0, n, gamma, dL, dR, dlam, daL, daR);
  if (dir == 1) hipLaunchKernelGGL(k_hlld_adjoint<1>, gr, b, 0, 0, n, gamma, dL, dR, dlam, daL, daR);
  if (dir == 2) hipLaunchKernelGGL(k_hlld_adjoint<2>, gr, b, 0, 0, n, gamma, dL, dR, dlam, daL, daR);
  if (hipGetLastError() != hipSuccess ||
      hipMemcpy(aL, daL, in_b, hipMemcpyDeviceToHost) != hipSuccess ||
      hipMemcpy(aR, daR, in_b, hipMemcpyDeviceToHost) != hipSuccess)
    return fail(PGPU_EDEVICE, "adjoint kernel failed");
  return PGPU_OK;
}
