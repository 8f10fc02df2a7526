// UCT_HLL edge EMFs (ct_emf_average.c:179-352 with the MC_LIM2 face slopes
// of ct_stag_slopes.c:51-106 and the PLM velocity slopes of
// CT_StoreVelSlopes), z-marching with each plane staged in LDS by direct
// global-to-LDS loads.
//
// A TX x TY workgroup owns a column tile and marches planes k0 .. k1-1.  At
// every plane the tile of the 12 EMF fields, with the in-plane halo the
// stencil reads, is copied from HBM straight into LDS with global_load_lds (no
// registers on the way), so each element of a plane is fetched once per
// workgroup, and the cells read their neighbours from LDS:
//
//   face speeds (6)   rows j0 .. j0+TY,     columns i0 .. i0+TX (+1: LB 16)
//   velocities (3), b_x, b_y, b_z
//                     rows j0-1 .. j0+TY+1, columns i0-1 .. i0+TX+1 (i0-2: LB 16)
//
// (one footprint for the second group, though b_x and b_y need a little
// less: every footprint costs registers for its lane offsets.)
//
// The velocity slopes are reconstructed here, once per cell, with the sweeps'
// own expressions on the sweeps' own operands, so they are the values the
// sweeps had, and shared through LDS; stored by the flux kernels and read
// back they were 72 B written and 72 B read per cell of kernels bound by
// memory.  The stencil's z offsets are split: Ex and Ey at plane k read
// planes k and k+1, so each is computed in two parts, the plane-k part while
// plane k is staged (kept in registers) and the plane-(k+1) part when plane
// k+1 is; b_x, b_y and the velocities at the cell itself on the planes below
// and above (their z slopes) are rolled in registers.  Every quantity is the expression of emf_edges with the same operands in the same
// order, so the FP64 results are the register kernel's bits (the FP32-flux
// path's float face data are widened exactly).

#include <hip/hip_runtime.h>

#include <type_traits>

#include "mhd_device.hpp"
#include "stage_cells.hpp"
#include "stage_kernels.hpp"

namespace pgpu {

namespace {

__device__ __forceinline__ int wrap_mod(int q, int n)
{
  const int r = q % n;
  return r < 0 ? r + n : r;
}

// LDS layout in bytes of a TX x TY tile: face speeds (FT float: float), the
// velocities (float for F32State), the velocity slopes (as the speeds), b_x,
// b_y, b_z.  D3: three dimensions (2D: Ez only, from the x and y faces of its
// one plane).
template <int TX, int TY, class FT, bool D3, int LB>
struct EmfTile {
  static constexpr int ND = D3 ? 3 : 2, NS = 2 * ND, NC = ND;   // directions, speeds, components
  static constexpr int SE = emf_f32<FT>(F_XSR) ? 4 : 8, VE = emf_f32<FT>(F_VX) ? 4 : 8;
  static constexpr int PAD = LB == 16 ? 2 : 1;   // columns before the tile
  static constexpr int SW = TX + PAD, SN = (TY + 1) * SW;
  static constexpr int VW = TX + 2 * PAD + (LB == 16 ? 0 : 1), VN = (TY + 3) * VW;
  static constexpr int up(int b) { return (b + 15) / 16 * 16; }
  static constexpr int SB = up(SN * SE), VB = up(VN * VE);   // bytes of one field
  static constexpr int V0 = NS * SB, PB = V0 + NC * VB;   // one buffer of speeds and velocities
  static constexpr int D0 = (D3 ? 2 : 1) * PB, X0 = D0 + ND * NC * SB;
  static constexpr int BB = up(VN * 8), BYTES = X0 + ND * BB;
  static constexpr int NW = TX * TY / 64;   // waves
  static constexpr int VL = LB == 16 ? VN : VN - 1;   // elements copied (the last corner is not read)
  // 64-lane copies of a footprint of n elements, and a wave's share
  static constexpr int chunks(int n, int es) { return (n * es / LB + 63) / 64; }
  static constexpr int share(int n, int es) { return (chunks(n, es) + NW - 1) / NW; }
  static constexpr int SC = share(SN, SE), VC = share(VL, VE), BC = share(VL, 8);
};

constexpr unsigned kNoLane = 0xffffffffu;

// byte offset in a plane of the LB bytes that lane `lane` copies in chunk c
// of a footprint of n elements of es bytes, rows of w elements from (ia, ja);
// kNoLane past its end
template <int LB>
__device__ __forceinline__ unsigned lane_offset(const Geo& g, int c, int lane, int n, int es, int w,
                                                int ia, int ja)
{
  const int d = (c * 64 + lane) * LB, el = d / es;
  if (el >= n) return kNoLane;
  const int r = el / w, q = el - r * w;
  const int i = wrap_mod(ia + q, g.nx), j = wrap_mod(ja + r, g.ny);
  return ((unsigned)j * (unsigned)g.nx + (unsigned)i) * (unsigned)es + (unsigned)(d % es);
}

}  // namespace

// Two buffers of speeds and velocities: plane p+1's are on the way while
// plane p's edges are computed, and plane p's faces while its slopes are, so
// a plane costs two barriers and no memory latency of its own.  Bound by the
// instructions of the edges and slopes (about 790 VALU and 80 LDS per cell)
// between those barriers.  256^3, per launch: 32 x 8 tiles at two waves per
// SIMD 0.68 ms (0.83 with the slopes read from memory; one buffer 0.74; slopes
// reconstructed at every use 1.05; three waves per SIMD, which spill, 0.83;
// 16 x 16 tiles 0.82; 4-byte copies on an even row length 3% slower).  WPE
// waves per SIMD caps the VGPRs.  LB: bytes a lane copies at a time, 16 on
// even row lengths (column pairs; FP64 fields), else 4.  FT: storage of the face speeds (double, float) and of the
// stage-2 input (F32State), as for k_emf_z.
template <int TX, int TY, int WPE, class FT, bool D3, int LB>
__global__ void __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(WPE)))
k_emf_zs(Geo g, StageIn in, Sweeps sw, EdgeOut e, int kz)
{
  using T = EmfTile<TX, TY, FT, D3, LB>;
  using SF = std::conditional_t<T::SE == 4, float, double>;   // speeds, slopes: the sweeps' type
  using VF = std::conditional_t<T::VE == 4, float, double>;
  __shared__ __attribute__((aligned(16))) char s[T::BYTES];

  const int tx = threadIdx.x, ty = threadIdx.y, tid = tx + TX * ty;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // shortened segments (boxes that 16 planes a workgroup would not fill): tiles
  // numbered so that each XCD runs one contiguous range of them and finds the
  // halos in its L2.  us a launch, plain and so: 64^3 26.3 and 23.2, 96^3 71.3
  // and 62, 128^3 117 and 108, 160^3 211 and 196, 192^3 322 and 307.  Not where
  // all workgroups run at once (32^3: the divisions cost more), nor with whole
  // segments (256^3 683 and 703, 384 x 288 x 320 1511 and 1530)
  const unsigned wgs = gridDim.x * gridDim.y * gridDim.z;
  const dim3 tb = D3 && kz < 16 && wgs > 512u ? xcd_tile() : dim3(blockIdx.x, blockIdx.y, blockIdx.z);
  const int i0 = tb.x * TX, j0 = tb.y * TY;
  const int i = i0 + tx, j = j0 + ty;
  const bool active = i < g.nx && j < g.ny;
  const EmfFields f = emf_fields(in, sw);
  const unsigned nxy = (unsigned)g.nx * (unsigned)g.ny;
  const ZSeg zs = zseg(g, tb.z, kz);   // (a patch of a stack: z periodic within it)

  // in-plane byte offsets of this lane in the chunks its wave copies
  // (chunk c of every footprint goes to wave c % NW)
  unsigned oS[T::SC], oB[T::BC], oV[T::VC];
#pragma unroll
  for (int c = 0; c < T::SC; c++) oS[c] = lane_offset<LB>(g, c * T::NW + wave, lane, T::SN, T::SE, T::SW, i0, j0);
#pragma unroll
  for (int c = 0; c < T::BC; c++)
    oB[c] = lane_offset<LB>(g, c * T::NW + wave, lane, T::VL, 8, T::VW, i0 - T::PAD, j0 - 1);
#pragma unroll
  for (int c = 0; c < T::VC; c++)
    oV[c] = T::VE == 8 ? oB[c] : lane_offset<LB>(g, c * T::NW + wave, lane, T::VL, T::VE, T::VW, i0 - T::PAD, j0 - 1);

  // chunk c (of this wave) of a field whose plane starts pb bytes in, to dst
  auto chunk = [&](const void* a, unsigned off, unsigned pb, int dst, int c) {
    const void* src = (const void*)(reinterpret_cast<const char*>(a) + (pb + off));
    auto lds = (__attribute__((address_space(3))) void*)(s + dst + (c * T::NW + wave) * (64 * LB));
    if (off == kNoLane) return;
    if constexpr (LB == 16) __builtin_amdgcn_global_load_lds(src, lds, 16, 0, 0);
    else __builtin_amdgcn_global_load_lds(src, lds, 4, 0, 0);
  };
  // velocities and face speeds of plane k into buffer buf, its faces
  auto stage_vs = [&](int k, int buf) {
    const unsigned pl = (unsigned)zwrap(g, zs.kb, k) * nxy;
#pragma unroll
    for (int q = 0; q < T::NC; q++)
#pragma unroll
      for (int c = 0; c < T::VC; c++)
        chunk(f.a[F_VX + q], oV[c], pl * (unsigned)T::VE, buf * T::PB + T::V0 + q * T::VB, c);
#pragma unroll
    for (int q = 0; q < T::NS; q++)
#pragma unroll
      for (int c = 0; c < T::SC; c++)
        chunk(f.a[F_XSR + q], oS[c], pl * (unsigned)T::SE, buf * T::PB + q * T::SB, c);
  };
  auto stage_b = [&](int k) {
    const unsigned pl = (unsigned)zwrap(g, zs.kb, k) * nxy;
#pragma unroll
    for (int q = 0; q < T::ND; q++)
#pragma unroll
      for (int c = 0; c < T::BC; c++) chunk(f.a[F_BX + q], oB[c], pl * 8u, T::X0 + q * T::BB, c);
  };
  // this thread's copies done, then every wave's
  auto landed = [] {
    __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    __syncthreads();
  };

  // LDS lookups of this thread's cell (I, J: in-plane offsets)
  const SF* sp0 = reinterpret_cast<const SF*>(s) + ty * T::SW + tx;
  const VF* vp0 = reinterpret_cast<const VF*>(s + T::V0) + (ty + 1) * T::VW + tx + T::PAD;
  SF* dp = reinterpret_cast<SF*>(s + T::D0) + ty * T::SW + tx;
  const double* bp = reinterpret_cast<const double*>(s + T::X0) + (ty + 1) * T::VW + tx + T::PAD;
  constexpr int SS = T::SB / T::SE, VS = T::VB / T::VE;   // elements of one field
#define S(A_, I_, J_) double(sp[(A_ - F_XSR) * SS + (J_) * T::SW + (I_)])
#define V(C_, I_, J_) double(vp[(C_) * VS + (J_) * T::VW + (I_)])
#define DV(D_, C_, I_, J_) double(dp[((D_) * T::NC + (C_)) * SS + (J_) * T::SW + (I_)])
#define BX(J_) bp[(J_) * T::VW]
#define BY(I_) bp[T::BB / 8 + (I_)]
#define BZ(I_, J_) bp[2 * (T::BB / 8) + (J_) * T::VW + (I_)]
  // velocity slope of a cell (v_+ - v_- of its PLM states)
  auto slope = [](VF m, VF c, VF p) -> SF {
    const SF sl = mc_slope(SF(m), SF(c), SF(p));
    const SF a = SF(c) + sl * SF(0.5), b = SF(c) - sl * SF(0.5);
    return a - b;
  };

  // The slopes of the (TX + 1) x (TY + 1) cells go through LDS: every thread
  // takes its own cell, and thread t < NC * (TX + TY + 1) component
  // t / (TX + TY + 1) of one cell of the tile's upper row and column (hx, hy).
  // Their neighbours in the plane come from LDS, those above and below from
  // registers (own cell: vdn, vup; the other: hdn, hup).
  constexpr int HN = TX + TY + 1;
  auto vel = [&](const double* a, unsigned c, int k) -> VF {
    return at_byte(reinterpret_cast<const VF*>(a), ((unsigned)zwrap(g, zs.kb, k) * nxy + c) * (unsigned)T::VE);
  };
  const bool halo = tid < T::NC * HN;
  const int hq = halo ? tid / HN : 0, hc = tid % HN;
  const int hx = hc <= TX ? hc : TX, hy = hc <= TX ? TY : hc - TX - 1;
  const VF* hv0 = reinterpret_cast<const VF*>(s + T::V0) + hq * VS + (hy + 1) * T::VW + hx + T::PAD;
  SF* hd = reinterpret_cast<SF*>(s + T::D0) + hq * SS + hy * T::SW + hx;
  const unsigned hcell = (unsigned)wrap_mod(j0 + hy, g.ny) * (unsigned)g.nx + (unsigned)wrap_mod(i0 + hx, g.nx);
  // (pinned as values: a choice among the struct's members would put the
  // struct in scratch memory)
  const double *va0 = f.a[F_VX], *va1 = f.a[F_VY], *va2 = f.a[F_VZ];
  asm volatile("" : "+s"(va0), "+s"(va1), "+s"(va2));
  const double* ha = hq == 0 ? va0 : (hq == 1 ? va1 : va2);
  // (cells past the box's edge in its last tiles: their periodic images)
  const unsigned cell = (unsigned)(j < g.ny ? j : wrap_mod(j, g.ny)) * (unsigned)g.nx +
                        (unsigned)(i < g.nx ? i : wrap_mod(i, g.nx));
  auto col = [&](const double* a, int k) -> double {
    return at_byte(a, ((unsigned)zwrap(g, zs.kb, k) * nxy + cell) * 8u);
  };
  auto put = [&](double* a, int k, double v) {
    if (active) at_byte(a, ((unsigned)k * nxy + cell) * 8u) = v;
  };
  const int k0 = zs.k0, k1 = zs.k1;
  // b_x, b_y at the cell on planes p-1 and p+1 (plane p: LDS)
  double bx_m = 0, bx_p = 0, by_m = 0, by_p = 0;
  VF vdn[3] = {0, 0, 0}, vup[3] = {0, 0, 0}, hdn = 0, hup = 0;
  if constexpr (D3) {
    bx_m = col(f.a[F_BX], k0 - 1), bx_p = col(f.a[F_BX], k0 + 1);
    by_m = col(f.a[F_BY], k0 - 1), by_p = col(f.a[F_BY], k0 + 1);
#pragma unroll
    for (int q = 0; q < 3; q++) {
      vdn[q] = vel(f.a[F_VX + q], cell, k0 - 1);
      vup[q] = vel(f.a[F_VX + q], cell, k0 + 1);
    }
    hdn = vel(ha, hcell, k0 - 1);
    hup = vel(ha, hcell, k0 + 1);
  }
  // the plane-k parts of Ex(k), Ey(k)
  double x_ysr0 = 0, x_ysl0 = 0, x_ayp = 0, x_aym = 0, x_bS = 0, x_bW = 0, x_bE = 0, x_eSW = 0,
         x_eSE = 0;
  double y_axp = 0, y_axm = 0, y_xsr0 = 0, y_xsl0 = 0, y_bS = 0, y_bN = 0, y_bW = 0, y_eSW = 0,
         y_eNW = 0;

  stage_vs(k0, 0);
  stage_b(k0);
  int buf = 0;
  for (int p = k0; p <= k1; p++) {
    landed();   // plane p's velocities and speeds (and every wave is done with plane p-1)
    if (p > k0) stage_b(p);
    const SF* sp = reinterpret_cast<const SF*>(reinterpret_cast<const char*>(sp0) + buf * T::PB);
    const VF* vp = reinterpret_cast<const VF*>(reinterpret_cast<const char*>(vp0) + buf * T::PB);
    // velocity slopes of plane p, while its faces are on the way
#pragma unroll
    for (int q = 0; q < T::NC; q++) {
      const VF* c = vp + q * VS;
      const VF v = c[0];
      dp[(0 * T::NC + q) * SS] = slope(c[-1], v, c[1]);
      dp[(1 * T::NC + q) * SS] = slope(c[-T::VW], v, c[T::VW]);
      if constexpr (D3) {
        dp[(2 * T::NC + q) * SS] = slope(vdn[q], v, vup[q]);
        vdn[q] = v;
      }
    }
    if (halo) {
      const VF* c = reinterpret_cast<const VF*>(reinterpret_cast<const char*>(hv0) + buf * T::PB);
      const VF v = c[0];
      hd[0 * T::NC * SS] = slope(c[-1], v, c[1]);
      hd[1 * T::NC * SS] = slope(c[-T::VW], v, c[T::VW]);
      if constexpr (D3) {
        hd[2 * T::NC * SS] = slope(hdn, v, hup);
        hdn = v;
      }
    }
    landed();   // the slopes, and plane p's faces
    double bx_n = 0, by_n = 0;
    if constexpr (D3) {
      // plane p+1 (and the cell's values on p+2): on the way under the edges
      if (p < k1) {
        stage_vs(p + 1, buf ^ 1);
        bx_n = col(f.a[F_BX], p + 2), by_n = col(f.a[F_BY], p + 2);
#pragma unroll
        for (int q = 0; q < 3; q++) vup[q] = vel(f.a[F_VX + q], cell, p + 2);
        hup = vel(ha, hcell, p + 2);
      }
    }
    if constexpr (D3) {
      // Ex(p-1): the plane-p part (offset K = 1 of emf_edges); Ex(p): the
      // plane-p part (K = 0)
      {
        const double by_0 = BY(0), sBY = mc_lim2(by_p - by_0, by_0 - by_m);   // z slope at plane p
        if (p > k0) {
          const double a_xp = max_ge(x_ysr0, S(F_YSR, 0, 0));
          const double a_xm = max_ge(x_ysl0, S(F_YSL, 0, 0));
          const double bN = by_0 - 0.5 * sBY;
          const double eNE = (V(2, 0, 1) - 0.5 * (DV(1, 2, 0, 1) + DV(2, 2, 0, 1))) * bN
                           - (V(1, 0, 1) - 0.5 * (DV(1, 1, 0, 1) + DV(2, 1, 0, 1))) * x_bE;
          const double eNW = (V(2, 0, 0) + 0.5 * (DV(1, 2, 0, 0) - DV(2, 2, 0, 0))) * bN
                           - (V(1, 0, 0) + 0.5 * (DV(1, 1, 0, 0) - DV(2, 1, 0, 0))) * x_bW;
          put(e.ex, p - 1, uct_hll(a_xp, a_xm, x_ayp, x_aym, x_eSW, x_eSE, eNE, eNW, x_bS, bN, x_bW, x_bE));
        }
        x_ysr0 = S(F_YSR, 0, 0);
        x_ysl0 = S(F_YSL, 0, 0);
        x_ayp = max_ge(S(F_ZSR, 0, 0), S(F_ZSR, 0, 1));
        x_aym = max_ge(S(F_ZSL, 0, 0), S(F_ZSL, 0, 1));
        x_bS = by_0 + 0.5 * sBY;
        x_bW = BZ(0, 0) + 0.5 * mc_lim2(BZ(0, 1) - BZ(0, 0), BZ(0, 0) - BZ(0, -1));
        x_bE = BZ(0, 1) - 0.5 * mc_lim2(BZ(0, 2) - BZ(0, 1), BZ(0, 1) - BZ(0, 0));
        x_eSW = (V(2, 0, 0) + 0.5 * (DV(1, 2, 0, 0) + DV(2, 2, 0, 0))) * x_bS
              - (V(1, 0, 0) + 0.5 * (DV(1, 1, 0, 0) + DV(2, 1, 0, 0))) * x_bW;
        x_eSE = (V(2, 0, 1) - 0.5 * (DV(1, 2, 0, 1) - DV(2, 2, 0, 1))) * x_bS
              - (V(1, 0, 1) - 0.5 * (DV(1, 1, 0, 1) - DV(2, 1, 0, 1))) * x_bE;
      }
      __builtin_amdgcn_sched_barrier(0);
      // Ey(p-1) and Ey(p) the same way
      {
        const double bx_0 = BX(0), sBX = mc_lim2(bx_p - bx_0, bx_0 - bx_m);
        if (p > k0) {
          const double a_yp = max_ge(y_xsr0, S(F_XSR, 0, 0));
          const double a_ym = max_ge(y_xsl0, S(F_XSL, 0, 0));
          const double bE = bx_0 - 0.5 * sBX;
          const double eSE = (V(0, 0, 0) - 0.5 * (DV(2, 0, 0, 0) - DV(0, 0, 0, 0))) * y_bS
                           - (V(2, 0, 0) - 0.5 * (DV(2, 2, 0, 0) - DV(0, 2, 0, 0))) * bE;
          const double eNE = (V(0, 1, 0) - 0.5 * (DV(2, 0, 1, 0) + DV(0, 0, 1, 0))) * y_bN
                           - (V(2, 1, 0) - 0.5 * (DV(2, 2, 1, 0) + DV(0, 2, 1, 0))) * bE;
          put(e.ey, p - 1, uct_hll(y_axp, y_axm, a_yp, a_ym, y_eSW, eSE, eNE, y_eNW, y_bS, y_bN, y_bW, bE));
        }
        y_axp = max_ge(S(F_ZSR, 0, 0), S(F_ZSR, 1, 0));
        y_axm = max_ge(S(F_ZSL, 0, 0), S(F_ZSL, 1, 0));
        y_xsr0 = S(F_XSR, 0, 0);
        y_xsl0 = S(F_XSL, 0, 0);
        y_bS = BZ(0, 0) + 0.5 * mc_lim2(BZ(1, 0) - BZ(0, 0), BZ(0, 0) - BZ(-1, 0));
        y_bW = bx_0 + 0.5 * sBX;
        y_bN = BZ(1, 0) - 0.5 * mc_lim2(BZ(2, 0) - BZ(1, 0), BZ(1, 0) - BZ(0, 0));
        y_eSW = (V(0, 0, 0) + 0.5 * (DV(2, 0, 0, 0) + DV(0, 0, 0, 0))) * y_bS
              - (V(2, 0, 0) + 0.5 * (DV(2, 2, 0, 0) + DV(0, 2, 0, 0))) * y_bW;
        y_eNW = (V(0, 1, 0) + 0.5 * (DV(2, 0, 1, 0) - DV(0, 0, 1, 0))) * y_bN
              - (V(2, 1, 0) + 0.5 * (DV(2, 2, 1, 0) - DV(0, 2, 1, 0))) * y_bW;
      }
      if (p == k1) break;
      __builtin_amdgcn_sched_barrier(0);
    }
    // Ez(p)
    {
      const double a_xp = max_ge(S(F_XSR, 0, 0), S(F_XSR, 0, 1));
      const double a_xm = max_ge(S(F_XSL, 0, 0), S(F_XSL, 0, 1));
      const double a_yp = max_ge(S(F_YSR, 0, 0), S(F_YSR, 1, 0));
      const double a_ym = max_ge(S(F_YSL, 0, 0), S(F_YSL, 1, 0));
      const double bS = BX(0) + 0.5 * mc_lim2(BX(1) - BX(0), BX(0) - BX(-1));
      const double bW = BY(0) + 0.5 * mc_lim2(BY(1) - BY(0), BY(0) - BY(-1));
      const double bN = BX(1) - 0.5 * mc_lim2(BX(2) - BX(1), BX(1) - BX(0));
      const double bE = BY(1) - 0.5 * mc_lim2(BY(2) - BY(1), BY(1) - BY(0));
      const double eSW = (V(1, 0, 0) + 0.5 * (DV(0, 1, 0, 0) + DV(1, 1, 0, 0))) * bS
                       - (V(0, 0, 0) + 0.5 * (DV(0, 0, 0, 0) + DV(1, 0, 0, 0))) * bW;
      const double eSE = (V(1, 1, 0) - 0.5 * (DV(0, 1, 1, 0) - DV(1, 1, 1, 0))) * bS
                       - (V(0, 1, 0) - 0.5 * (DV(0, 0, 1, 0) - DV(1, 0, 1, 0))) * bE;
      const double eNE = (V(1, 1, 1) - 0.5 * (DV(0, 1, 1, 1) + DV(1, 1, 1, 1))) * bN
                       - (V(0, 1, 1) - 0.5 * (DV(0, 0, 1, 1) + DV(1, 0, 1, 1))) * bE;
      const double eNW = (V(1, 0, 1) + 0.5 * (DV(0, 1, 0, 1) - DV(1, 1, 0, 1))) * bN
                       - (V(0, 0, 1) + 0.5 * (DV(0, 0, 0, 1) - DV(1, 0, 0, 1))) * bW;
      put(e.ez, p, uct_hll(a_xp, a_xm, a_yp, a_ym, eSW, eSE, eNE, eNW, bS, bN, bW, bE));
    }
    if constexpr (!D3) break;
    __builtin_amdgcn_sched_barrier(0);
    bx_m = BX(0);
    by_m = BY(0);
    bx_p = bx_n;
    by_p = by_n;
    buf ^= 1;
  }
#undef S
#undef V
#undef DV
#undef BX
#undef BY
#undef BZ
}

template <int TX, int TY, int WPE, class FT, bool D3, int LB>
static void launch_tile(const Geo& g, const StageIn& in, const Sweeps& sw, const EdgeOut& e,
                        hipStream_t s, int kz)
{
  const long xy = (long)((g.nx + TX - 1) / TX) * ((g.ny + TY - 1) / TY);
  // fewer planes per workgroup on small boxes: keep >= 2048 workgroups
  while (kz > 1 && xy * zblocks(g, kz) < 2048) kz /= 2;
  const dim3 b(TX, TY, 1), gr((g.nx + TX - 1) / TX, (g.ny + TY - 1) / TY, zblocks(g, kz));
  hipLaunchKernelGGL((k_emf_zs<TX, TY, WPE, FT, D3, LB>), gr, b, 0, s, g, in, sw, e, kz);
}

// The LDS kernel for fields under 4 GiB (32-bit byte offsets); ft: face data
// double (0), float (1) or float with an FP32 stage input (2).  False: the
// caller takes another kernel.
bool launch_emf_lds(const Geo& g, const StageIn& in, const Sweeps& sw, const EdgeOut& e,
                    hipStream_t s, int shape, int kz, KernelTimer* kt, int ft)
{
  if ((unsigned long long)g.n * 8ull >= (1ull << 32)) return false;
  if (kt) kt->begin(KT_EMF, s);
  if (g.dims != 3) {
    if (ft == 1) launch_tile<32, 8, 3, float, false, 4>(g, in, sw, e, s, 1);
    else if (ft == 2) launch_tile<32, 8, 3, F32State, false, 4>(g, in, sw, e, s, 1);
    else launch_tile<32, 8, 3, double, false, 4>(g, in, sw, e, s, 1);
  } else if (ft == 1) {
    launch_tile<32, 8, 3, float, true, 4>(g, in, sw, e, s, kz);
  } else if (ft == 2) {
    launch_tile<32, 8, 3, F32State, true, 4>(g, in, sw, e, s, kz);
  } else if (shape == 1) {
    launch_tile<64, 4, 2, double, true, 4>(g, in, sw, e, s, kz);
  } else if (shape == 2) {
    launch_tile<32, 4, 3, double, true, 4>(g, in, sw, e, s, kz);
  } else if (g.nx % 2 == 0) {
    launch_tile<32, 8, 2, double, true, 16>(g, in, sw, e, s, kz);
  } else {
    launch_tile<32, 8, 2, double, true, 4>(g, in, sw, e, s, kz);
  }
  if (kt) kt->end(KT_EMF, s);
  return true;
}

// ---------------------------------------------------------------------
// the velocity slopes as arrays
// ---------------------------------------------------------------------

// The PLM velocity slopes of every cell into sw's dv arrays, for the kernels
// that read them (the register EMF kernels, the adjoint's tape, the branch
// signature): the values the sweeps reconstruct, in FT's storage.
template <class FT>
__global__ void __launch_bounds__(256) k_vel_slopes(Geo g, StageIn in, Sweeps sw)
{
  using RS = std::conditional_t<emf_f32<FT>(F_XDV0), float, double>;
  Cell p;
  if (!cell_of(g, p)) return;
  const EmfFields f = emf_fields(in, sw);
  const int nd = g.dims == 3 ? 3 : 2;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    if (d >= nd) break;
    const long m = d == 0 ? nb<0>(g, p, -1) : d == 1 ? nb<1>(g, p, -1) : nb<2>(g, p, -1);
    const long n = d == 0 ? nb<0>(g, p, 1) : d == 1 ? nb<1>(g, p, 1) : nb<2>(g, p, 1);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      auto at = [&](long o) -> RS {
        if constexpr (emf_f32<FT>(F_VX)) return RS(reinterpret_cast<const float*>(f.a[F_VX + c])[o]);
        else return RS(f.a[F_VX + c][o]);
      };
      const RS v = at(p.c), sl = mc_slope(at(m), v, at(n));
      const RS a = v + sl * RS(0.5), b = v - sl * RS(0.5);
      if constexpr (emf_f32<FT>(F_XDV0)) reinterpret_cast<float*>(sw.d[d].dv[c])[p.c] = a - b;
      else sw.d[d].dv[c][p.c] = a - b;
    }
  }
}

int launch_vel_slopes(const Geo& g, const StageIn& in, const Sweeps& sw, hipStream_t s, int ft)
{
  const dim3 gr((g.nx + 63) / 64, (g.ny + 3) / 4, g.nz), b(64, 4);
  if (ft == 1) hipLaunchKernelGGL(k_vel_slopes<float>, gr, b, 0, s, g, in, sw);
  else if (ft == 2) hipLaunchKernelGGL(k_vel_slopes<F32State>, gr, b, 0, s, g, in, sw);
  else hipLaunchKernelGGL(k_vel_slopes<double>, gr, b, 0, s, g, in, sw);
  return (int)hipGetLastError();
}

}  // namespace pgpu
