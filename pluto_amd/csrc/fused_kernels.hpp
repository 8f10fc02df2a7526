// Fused stage kernels (fused_kernels.hip): tile shapes and launchers.
#pragma once
#include <hip/hip_runtime.h>
#include "stage_kernels.hpp"

namespace pgpu {

constexpr int XY_TX = 32, XY_TY = 8;   // k_flux_xy workgroup (one z-plane); FP64 tiles overlap
constexpr int Z_COLS = 256;            // k_flux_z columns per workgroup, consecutive in the plane

// Cells of a march's segment (a power of two up to `most`, no longer than the
// line needs) for kernels that solve Riemann problems one after another
// along it at two waves per SIMD; waves(len): waves of the launch.  A wave
// does len + 2 interfaces' work (one solved again and two reconstructions
// at the segment's start), the 1024 SIMDs take up to 2048 waves at a time,
// and a round with two waves per SIMD takes 1.5 times one with a single
// wave (measured).  The estimate orders the measured times right: z march
// of 64^3 seg 4: 26 us (8: 32, 16: 50), 96^3 8: 51 (16: 57, 4: 58), 128^3 16: 93
// (8: 100, 32: 113), 133^3 8: 121 (16: 132, 4: 133), 384 x 288 x 320 32: 1414
// (16: 1448, 64: 1465), 32^3 1: 13 (8: 30).
template <class W>
inline int march_len(int most, int line, W waves)
{
  int best = 1;
  double cost = 0.0;
  for (int len = 1; len <= most && (len == 1 || len < 2 * line); len *= 2) {
    const long w = waves(len), rest = w % 2048;
    const double rounds = 1.5 * (double)(w / 2048) + (rest > 1024 ? 1.5 : (rest > 0 ? 1.0 : 0.0));
    const double c = rounds * (len + 2);
    if (len == 1 || c <= cost) {
      best = len;
      cost = c;
    }
  }
  return best;
}

// Per-face UCT_HLL speeds written by the flux kernels for the EMF kernel; for
// the other EMF averages the face EMFs and the mass flux mf (same arrays as
// SweepOut's: SL, SR, dv[0]).
struct FaceData {
  double* SL[3];
  double* SR[3];
  double* mf[3];
};

// fp32_flux: PLM and HLLD in FP32 (states rounded from FP64 on load); the
// flux differences and U are FP64; the face speeds are
// stored as float in the first half of fd's buffers (launch_emf with
// f32_faces reads them).
int launch_flux_fused(const Geo& g, int stage, bool fp32_flux, const StageIn& in, const Cons& U,
                      const FaceData& fd, double* cdt_xy, DevScalars* sc, hipStream_t s,
                      KernelTimer* kt);
// the tolerance-mode FP64 launches (fused_fast.hip: FMA contraction, Newton
// division and square root; HLLD, UCT_HLL)
int launch_flux_fused_fast(const Geo& g, int stage, const StageIn& in, const Cons& U,
                           const FaceData& fd, double* cdt_xy, DevScalars* sc, hipStream_t s,
                           KernelTimer* kt);
// x/y flux kernel of the fused stage (process-wide; FP64 results identical,
// FP32-flux ones to FP32 rounding: the two kernels contract differently):
// 0 the overlapping z-plane tiles (k_flux_xy, k_flux_xy_items), 1 rows
// marching up y segments of seg rows (k_flux_xy_rows; 0: by the box's size,
// and the FP64 tiles on boxes so small that they take less time)
int set_flux_xy_kernel(int kind, int seg);
int flux_xy_kind();
int flux_xy_seg();

// Launch shape of the row kernel: nt threads, wgs workgroups across the
// planes (nt = 0: this box takes the tiles), rows per workgroup (0: windows)
// and rows of a y segment, the combination with the least estimated time.
// In units of a row of two-waves-per-SIMD work (9.6 us): a workgroup takes
// len + 1.3 of them (an interface and two reconstructions more at a
// segment's start), 512 workgroups of three or four waves (three: 0.8 of
// the time) run at once, half as many in 0.65 of the time; whole rows go in
// rounds, the windows' workgroups drift apart and end ragged (f + 0.4).
// The units were measured when both kernels still wrote the velocity slopes;
// the choice needs their ratios only.  Present times in us, the choice and
// another: 256^3 32 rows 1153 (16: 1174), 128^3 as two rows a workgroup, 16
// rows, 161 (8: 167, 32: 189), 64^3 2 rows 34 (1: 39, tiles 49), 16 x 256^2 8
// rows 85 (16: 96, tiles 110), 133^3 windows 209 (8 rows, the best, 199; 32:
// 288, tiles 253), 261 x 256^2 16 rows 1217 (8: 1286, tiles 1648), 96^3 98 (4
// rows, the best, 91; tiles 113); of the sizes near the tiles' line, 48^3 24.6
// (tiles 25.0), a 512^2 plane 34.5 by tiles (1 to 4 rows: 43 to 50), 32^3 16.7 (tiles 19.5).
struct RowLaunch {
  int nt = 0, wgs = 0, rows = 0, seg = 0;
};

inline RowLaunch row_launch(const Geo& g, int real_bytes)
{
  RowLaunch best;
  if (flux_xy_kind() != 1 || g.n * 8 >= (1l << 32)) return best;
  double cost = 0.0;
  auto offer = [&](int nt, long wgs, int rows) {
    const int lens = flux_xy_seg() > 0 ? flux_xy_seg() : 32;
    for (int len = flux_xy_seg() > 0 ? lens : 1; len <= lens && (len <= g.ny || lens == len); len++) {
      const double f = (double)(wgs * ((g.ny + len - 1) / len)) * (nt <= 128 ? nt / 256.0 : 1.0) / 512.0;
      const double all = rows > 0 ? (f <= 4.0 ? (double)(long)(f + 0.9999) : f)
                                  : (f <= 0.75 ? 1.0 : f + 0.4);
      const double c = (f <= 0.5 ? 0.65 : all) * (len + 1.3) * (nt == 192 ? 0.8 : (nt < 192 ? 1.1 : 1.0));
      if (best.nt && c > cost) continue;
      best.nt = nt;
      best.wgs = (int)wgs;
      best.rows = rows;
      best.seg = len;
      cost = c;
    }
  };
  const int deep = patch_depth(g);
  // (a workgroup's rows belong to one patch of a stack, which has no windows;
  // the grid's y, the planes', holds 65535 workgroups: long rows of many planes
  // take the tiles)
  if (g.pz <= 0)
    for (int nt = 64; nt <= 256; nt += 64) {
      const long wgs = ((long)g.nz * (g.nx + 4) - 4 + nt - 5) / (nt - 4);
      if (wgs <= 65535) offer(nt, wgs, 0);
    }
  for (int r = 1; r * g.nx <= 256 && r <= deep; r++)
    if (g.pz <= 0 || deep % r == 0) offer((r * g.nx + 63) / 64 * 64, ((long)g.nz + r - 1) / r, r);
  if (real_bytes == 8 && g.pz <= 0 && flux_xy_seg() <= 0) {
    // the tiles: 768 workgroups at once, 17 us a round (48^3: 26 us, rows 30;
    // a 512^2 plane 37, rows 48; 64^3: 51, rows 36)
    const double f = (double)((g.nx + 30) / 31) * ((g.ny + 6) / 7) * g.nz / 768.0;
    const double us = f <= 1.0 ? 12.0 + 14.0 * f : 3.0 + 17.0 * (f <= 4.0 ? (double)(long)(f + 0.9999) : f + 0.3);
    if (us < 5.0 + 9.6 * cost) best.nt = 0;
  }
  if (real_bytes == 4 && g.pz <= 0 && flux_xy_seg() <= 0 && best.nt == 64) {
    // FP32 rows too short and in too few planes for more than one wave a
    // workgroup: tiles where there are many such rows and few tiles.  us, tiles
    // and rows: planes of 3 x 2000 14.8 and 24.0, 16 x 800 12.3 and 20.2, 60 x 5000
    // 32.7 and 35.0, 9 x 1200 x 3 16.7 and 20.4; 3 x 1500 x 15 44.7 and 23.2,
    // 3 x 500 16.0 and 15.0, 64^2 13.4 and 11.2
    const double us = 12.0 + 0.013 * (double)((g.nx + 31) / 32) * ((g.ny + 7) / 8) * g.nz;
    if ((long)best.wgs * g.ny > 700 && us < 5.0 + 7.0 * cost) best.nt = 0;
  }
  return best;
}
// the FP32-flux launches (fused_f32.hip, compiled with FMA contraction)
int launch_flux_fused_f32(const Geo& g, int stage, const StageIn& in, const Cons& U,
                          const FaceData& fd, double* cdt_xy, DevScalars* sc, hipStream_t s,
                          KernelTimer* kt);

// CT face update fused with the face average and ConsToPrim.  Stage 2
// blends with the step-start faces b0 and writes the new faces to bout,
// which must not alias bin or b0.
// Stage 1 sets the cells' flags, stage 2 adds to them; ends.on: the step's
// ends are taken here too (StepEnds).
// f32_out (stage 1 of the FP32-flux path): Vout, the next stage's input,
// is stored as float in the first half of each buffer; the stage-2 flux and
// EMF kernels of that path read it so.
int launch_ct_c2p(const Geo& g, int stage, const EdgeOut& e, const FaceIn& bin, const FaceIn& b0,
                  const FaceOut& bout, const Cons& U, const StageIn& vn, const Prims& Vout,
                  unsigned char* flag, DevScalars* sc, hipStream_t s, KernelTimer* kt,
                  bool f32_out = false, const StepEnds& ends = StepEnds());

}  // namespace pgpu
