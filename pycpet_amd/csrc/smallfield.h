// Field and potential of few point-charge pairs, in one launch (smallfield.hip).
#pragma once

#include "cpet_internal.h"

namespace cpet {

// Grids: the interpolating path (fargrid.h) takes 35 to 70 us from there on,
// whatever the grid: 31^3 x 2,000 (6e7 pairs) 51 us here, 47 there, 21^3 x 8,000
// (7e7) 81 and 37, 21^3 x 2,000 (1.9e7) 24 and 35, 11^3 x 30,000 (4e7) 70 and 68.
// Scattered points have only the direct kernel beside this one, which is at its
// worst with few points: 3,000 points x 30,000 charges (9e7 pairs) 101 us here,
// 112 there; 3,000 x 60,000 (1.8e8) 195 and 527.
constexpr double kSmallMaxPairs = 5e7;
constexpr long long kSmallFewPoints = 4096;

// Whether M points (of a grid, or scattered) and N charges take this path
// (default precision, float32 results).
bool small_field_ok(bool grid, long long M, int N);

// Whether the small grids of a batch, of so many pairs together and at most so many
// charges each, take this path.  It does 1.1e12 pairs/s, the direct batch kernel
// 2.5e12 once it has enough workgroups, but a wave of that one goes through all
// charges of its frame: 90 ns a charge at least.  256 frames of 10^3 points, here and
// direct, us: E of 1,000 charges 238, 150, of 64 of them 65, 119; phi 171, 164 and 49, 127;
// 21^3 x 2,000, E, 8 frames 142, 201, 64 frames 973, 516.
bool small_batch_ok(double pairs, int most_charges, bool phi);

// Float32 E and / or phi (null: not wanted; both only softened) of charges
// x (N,3), q (N) at the points of a grid (ax, ay, az) or at pts (M,3), all on
// the device, queued on the context's stream.
int small_field_launch(cpet_ctx* ctx, int ny, int nz, const float* ax, const float* ay,
                       const float* az, long long M, const float* pts, int N, const float* x,
                       const float* q, float* e, float* phi, bool soft);

// The same for grids of a batch: one workgroup per blk entry (frame, block of P
// points of it), P as small_field_points gives it for the points of all of them.
struct SmallBatch {
  const int32_t* blk;
  const int32_t* geo;      // (F, 4): nx, ny, nz, -
  const int32_t* ax_off;   // (F) offset of the frame's axes
  const int64_t* out_off;  // (F) its first output point
  const int32_t* chg_off;  // (F+1) offsets of the packed charges
  const float* axes;
  const float4* ch;
};

int small_field_points(const cpet_ctx* ctx, long long M);
int small_batch_launch(cpet_ctx* ctx, int P, int blocks, const SmallBatch& t, float* e, float* phi,
                       bool soft);

}  // namespace cpet
