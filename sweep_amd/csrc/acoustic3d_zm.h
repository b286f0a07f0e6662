// z-marching kernels of the 3-D acoustic path (see acoustic3d_zm.hip).
#pragma once

#include "acoustic3d.h"

namespace swp {
namespace a3d {

// Smallest launch (shots x runtime-grid cells) that runs on the z-marching
// kernels by default; smaller ones run one thread per cell.  From here to
// kBigCells3 shot-cells the choice goes by order and shape (march_fwd and
// march_adj in acoustic3d.hip).
constexpr int64_t kZmMinCells3 = int64_t(4) << 20;
// From here up the forward step adds the last axes' second derivatives to the
// CPML sum in one rounding each; below, every term is rounded first, as in the
// per-cell kernels, so that a record there does not depend on the family.  The
// times are equal.  It is so for the records' bits: when the border to the
// per-cell kernels moved down from this size, the records below kept theirs at
// every order, and those from here up at orders 4, 6 and 8 (order 2's moved, by
// 7e-7 of the record after 400 steps).  Consequently one shot's record may differ by rounding between
// launches of few and of many shots.  SWP_KERNELS=zmarch_big runs this form at
// any size.
constexpr int64_t kBigCells3 = int64_t(32) << 20;
// Smallest reconstruction box (shots x cells) on its z-marching kernel: the
// box holds far fewer cells than the grid, and its kernel walks whole z
// segments (1.4M cells 47 us against 16 us per-cell; from 2M to 8M the step
// times are within 2%).
constexpr int64_t kZmMinRecon3 = int64_t(4) << 20;

// The cells that the z-march's tiles cover, masked lanes included, over those
// that the per-cell kernels' 64 x 4 blocks cover.  It is near 1 where each x
// range fills its 64-column tiles, and 1.33 to 1.6 where the middle range of a
// narrow grid takes a tile more for a few columns.
double zm_lane_ratio(const Geo &g);

// Orders 2..8, and a z segment of tz planes plus its 2M + 1 halo and prefetch
// planes addressable with 32-bit byte offsets (tz is clamped to fit).
bool zm_supported(const Geo &g, int &tz);
// The slabs of the computed box around the lean interior [lo + M + 1,
// hi - M - 1) per axis (the whole box when that interior is empty); returns
// how many of out[0..5] it filled.
int shell_boxes(const Geo &g, Box out[6]);
// Interior z-march launch, plus the z-march shell when `shell` is set.
void launch_fwd_zm(const Ctx &x, const StepFields &f, float *u_this, float *strip, bool shell);
void launch_adj_zm(const Ctx &x, const AdjFields &f, const float *img, float *grad, bool shell);
void launch_recon_zm(const Ctx &x, const float *vp, const float *u_prev, const float *u_now, float *u_next,
                     const float *adj, float *grad, int x0, int x1, int y0, int y1, int z0, int z1);

}  // namespace a3d
}  // namespace swp
