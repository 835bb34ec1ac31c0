// Grid field with the far charges interpolated (fargrid.hip).
#pragma once

#include <memory>
#include <vector>

#include "cpet_internal.h"

namespace cpet {

// One grid of a call: axis i is n[i] values from ax0[i] on, its charges are
// [ch0, ch0 + npad) of the packed array, its points go from out0 on.
struct FarGrid {
  int n[3];
  long long ax0[3];
  int npad;
  long long ch0;
  long long out0;
};

// Axes shorter than the 12 nodes by more than a third would sum at more nodes
// than points.  The launches and node sums cost 35 to 70 us, which the one-launch
// path takes at 5e7 point-charge pairs (smallfield.h has both sides).  In a batch
// the launches are shared, and the direct kernel has no charge split: a 21^3 x
// 40k frame alone keeps it busy for 1.5 ms.
constexpr int kFarMinAxis = 8;
constexpr double kFarMinPairs = 5e7;
constexpr double kFarMinPairsBatch = 2e7;
// Smaller frames of a batch that has more pairs in such frames than the one-launch
// path takes at a time (kSmallMaxPairs).  A frame costs its 1,728 nodes instead of its
// points, and the weights of its axes whatever its charges: 256 frames, E, kernels
// alone, direct -> here: 21^3 x 2,000 2,054 -> 866 us, 21^3 x 250 257 -> 175, 15^3 x
// 1,000 442 -> 410, 15^3 x 250 129 -> 149, 13^3 x 1,000 296 -> 404; 31^3 x 60 216 -> 455.
constexpr long long kFarMinPointsMany = 3000;
constexpr int kFarMinChargesMany = 192;

// Whether an nx x ny x nz grid of npad (padded) charges takes the
// interpolating path, from min_pairs (points x charges) on.
bool far_grid_ok(int nx, int ny, int nz, int npad, double min_pairs);

// The launches of some grids.  Null where their scratch cannot be had (memory has
// run out, or the stream is being captured and they have not run on this context
// before): the direct kernel takes them then.
struct FarPlan;
std::shared_ptr<const FarPlan> far_grid_plan(cpet_ctx* ctx, const std::vector<FarGrid>& grids,
                                             bool want_e, bool want_phi);

// Float32 E and / or phi (as planned) of the grids, queued on the context's
// stream.  ax: the device arrays that hold the grids' x, y and z axes.
int far_grid_run(cpet_ctx* ctx, const FarPlan& plan, const float* const (&ax)[3], const float4* ch,
                 bool soft, void* e, void* phi);

}  // namespace cpet
