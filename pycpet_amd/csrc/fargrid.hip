// Field and potential on a box grid with the far charges interpolated.
//
// The direct sum over a grid costs (points x charges) pair terms, but a box
// grid samples the smooth field of a charge a few box widths away far more
// densely than that field varies.  Here the grid is cut into cells, halved
// per axis level by level; a charge far from a cell contributes to the cell's
// 12 x 12 x 12 Chebyshev nodes instead of its points, at the coarsest level
// whose cell it is far from, and the node sums are interpolated down to the
// points (tensor-product Lagrange).  Charges far from no cell of a point's
// path are summed directly at the point.  All sums, nodes and interpolation
// are FP64 (the pair terms as in the "mixed" precision: FP64 displacement and
// r^2, FP32 rsq seed, FP64 correction), so nothing needs the FP32 error check
// and recompute of the direct grid kernel; points where E nearly cancels are
// summed again without interpolation, in far_eval (see kCancel).
//
// Far means that along every axis the nearest singularity of the charge's
// field, seen from any point of the cell, lies outside the Bernstein ellipse
// of parameter kRho = 7: the kP nodes then miss one charge's term by at most
// 1e-9 of itself (E; 1e-10 for phi) at the threshold, and by much less beyond
// it, against the 6e-8 rounding of one FP32 pair term.  On the frames below
// the results are the FP64 sums rounded to float32, also where E or phi is
// 1e-3 of its RMS (measured: within 6e-11 RMS there).  kRho = 6 was 10-15 %
// faster and up to 1e-10 RMS off at those points, kRho = 8 10-13 % slower and
// no nearer.
//
// Stages, each one launch for all frames of a call:
//   far_classify  which charges are far from, or near, which cells: one
//                 64-bit mask per (cell, 64 charges); and, in its last
//                 workgroups, cell extents, Lagrange weights of every axis
//                 value and the node transfer matrices
//   far_nodes     node sums of every cell, split over its far charges
//   far_reduce    the splits' partial sums in a fixed order
//   far_eval      nodes -> points, plus the near charges, and the store
// Every list and sum has a fixed order: results are reproducible bit for bit.

#include <algorithm>
#include <type_traits>
#include <vector>

#include "cpet_internal.h"
#include "fargrid.h"
#include "pairterm.h"

namespace cpet {
namespace {

constexpr int kP = 12;                 // nodes per axis
constexpr int kNodes = kP * kP * kP;
constexpr int kLeafMax = 27;           // points per axis of a leaf, at most
constexpr int kMaxHalvings = 4;        // per axis: grids of up to 432 points
constexpr int kMaxLevels = kMaxHalvings + 1;
constexpr int kMaxAxis = kLeafMax << kMaxHalvings;
constexpr int kMaxSegs = 2048;         // 64-charge segments: up to 131,072 charges
constexpr int kTableBlocks = 2;        // classification workgroups per axis's tables
constexpr int kClassWaves = 8;         // waves that share a segment's cells
constexpr int kClassThreads = 64 * kClassWaves;
constexpr int kThirds = 3;             // node workgroups per (cell, split)
constexpr int kNodeLanes = 192;        // 48 node lines x 4 threads of 3 nodes
constexpr int kNodeGroups = 4;         // that split a workgroup's charges
constexpr int kNodeThreads = kNodeLanes * kNodeGroups;
constexpr int kBatch = kNodeThreads;   // far charges staged per round
constexpr int kRedThreads = 256;
constexpr int kEvalThreads = 256;
constexpr int kPlanes = 2;             // x planes per eval workgroup
constexpr int kNearLds = kEvalThreads; // near charges staged at once

constexpr int kGeoPerAxis = (2 << kMaxHalvings) - 1;  // intervals of all levels

// Bernstein parameter kRho: sigma = (rho + 1 / rho) / 2; a charge at offset d
// from the cell's centre (per axis) and gap g from its faces is outside the
// ellipse of axis i when d_i^2 / sigma^2 + (|g|^2 - g_i^2) / (sigma^2 - 1)
// >= a_i^2.
constexpr float kRho = 7.0f;
constexpr float kSigma = (kRho + 1.0f / kRho) / 2.0f;
constexpr float kInvS2 = 1.0f / (kSigma * kSigma);
constexpr float kInvS21 = 1.0f / (kSigma * kSigma - 1.0f);
constexpr float kMinGap2 = 1e-4f;   // 0.01 A: far charges never reach the r^2 floor
constexpr float kMaxCoord = 1e6f;   // beyond (or not finite): summed directly
// A point whose E is below this share of S = sum |q| / gap^2 over the charges
// interpolated for its leaf (gap: from the cell at whose nodes) is summed directly: what
// the interpolation misses, some 1e-12 S where charges are placed so that their
// misses add up (a shell of equal charges, mirrored ones), would be more than E's
// rounding there (2-norm error of a shell's E 1.4e-7, with this 2.5e-8).  Hardly a
// point of other frames: 1 in 1e8 at random.  S costs the classification 0.2 us (12k
// x 61 x 47 x 38) to 1.1 us (30k x 101^3), the test 0.2 us of far_eval.
constexpr double kCancel = 2e-5;

// cos((2k + 1) pi / 24) and (-1)^k sin((2k + 1) pi / 24): the Chebyshev nodes
// of the first kind and their barycentric weights.
__constant__ const double kNodeX[kP] = {
    0.9914448613738104,  0.9238795325112867,  0.7933533402912352,  0.6087614290087207,
    0.3826834323650898,  0.13052619222005157, -0.13052619222005157, -0.3826834323650898,
    -0.6087614290087207, -0.7933533402912352, -0.9238795325112867, -0.9914448613738104};
__constant__ const double kNodeW[kP] = {
    0.13052619222005157, -0.3826834323650898, 0.6087614290087207, -0.7933533402912352,
    0.9238795325112867,  -0.9914448613738104, 0.9914448613738104, -0.9238795325112867,
    0.7933533402912352,  -0.6087614290087207, 0.3826834323650898, -0.13052619222005157};

__host__ __device__ inline int part_begin(int n, int level, int t) { return (n * t) >> level; }

// One frame of a call.  Offsets are in elements of the buffers in FarArgs.
struct FarFrame {
  int n[3];            // grid points per axis
  int l[3];            // halvings per axis
  int levels;          // max(l) + 1
  int nseg;            // 64-charge segments
  int cells;           // of all levels
  int splits[kMaxLevels];
  int xblocks;         // eval workgroups per leaf
  int class_blk0, node_blk0, red_blk0, eval_blk0;
  long long ch0;       // first charge
  long long part0;     // partial node sums
  long long val0;      // node sums of every cell, level by level
  long long geo0;      // 3 x kGeoPerAxis x (centre, half width)
  long long lag0[3];   // per axis: level x axis value x kP weights
  long long tr0[3];    // per axis: leaf part x ancestor level x kP x kP
  long long mask0;     // (cells + leaves) x nseg: far masks, then the leaves' near masks
  long long mag0;      // cells x nseg: sum |q| / gap^2 of a segment's charges far from the cell
  long long near0;     // per leaf: number of near charges, S, then their numbers (64 nseg)
  int leaf0;           // the launch's first leaf (see Group::range)
  long long out0;      // first output point
  long long ax0[3];    // first value of each axis
};

struct FarArgs {
  int F;
  const float* ax[3];
  const FarFrame* frames;  // (F) when F > 1
  FarFrame one;            // F == 1
  const float4* ch;
  double* part;
  double* val;
  double* geo;
  double* lag;
  unsigned long long* mask;
  float* mag;
  int* near;
  void* e;
  void* phi;
};

// A frame as kernels read it: in constant memory (the kernel's arguments or
// the uploaded table, neither of which a kernel writes), by scalar loads.
typedef const __attribute__((address_space(4))) FarFrame Frame;

template <class Fr>
__host__ __device__ inline int axis_level(const Fr& f, int axis, int level) {
  return level < f.l[axis] ? level : f.l[axis];
}

template <class Fr>
__host__ __device__ inline int cells_at(const Fr& f, int level) {
  return 1 << (axis_level(f, 0, level) + axis_level(f, 1, level) + axis_level(f, 2, level));
}

// Parts (tx, ty, tz) of cell number c at a level (z fastest).
__device__ __forceinline__ void cell_parts(Frame& f, int level, int c, int (&t)[3]) {
  const int ly = axis_level(f, 1, level), lz = axis_level(f, 2, level);
  t[2] = c & ((1 << lz) - 1);
  t[1] = (c >> lz) & ((1 << ly) - 1);
  t[0] = c >> (lz + ly);
}

// Number of the cell at `level` that holds the cell (t) of a deeper level.
__device__ __forceinline__ int ancestor(Frame& f, int level, int deep, const int (&t)[3]) {
  int c = 0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int al = axis_level(f, i, level);
    c = (c << al) | (t[i] >> (axis_level(f, i, deep) - al));
  }
  return c;
}

// The frame that block b belongs to.  A is the kernels' only argument.
__device__ __forceinline__ Frame& frame_of_block(int FarFrame::*first, int b) {
  typedef const __attribute__((address_space(4))) FarArgs Args;
  Args* a = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
  if (a->F == 1) return a->one;
  Frame* frames = (Frame*)(unsigned long long)a->frames;
  int lo = 0, hi = a->F - 1;  // the last frame whose first block is <= b
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (frames[mid].*first <= b)
      lo = mid;
    else
      hi = mid - 1;
  }
  return frames[lo];
}

// Lagrange weights of the kP nodes at t (barycentric, exact at a node); 0 in
// an interval that no charge is far from, where t is not a number.
__device__ __forceinline__ void lagrange(double t, double* __restrict__ w) {
  double v[kP], s = 0.0;
  int at = -1;
#pragma unroll
  for (int k = 0; k < kP; ++k) {
    const double d = t - kNodeX[k];
    if (d == 0.0) at = k;
    v[k] = kNodeW[k] / d;
    s += v[k];
  }
  const double r = isfinite(t) ? 1.0 / s : 0.0;
#pragma unroll
  for (int k = 0; k < kP; ++k)
    w[k] = at >= 0 ? (k == at ? 1.0 : 0.0) : r != 0.0 ? v[k] * r : 0.0;
}

// ---- extents and weights --------------------------------------------------

// Centre and half width of every interval (level by level) of the axes that x
// (per axis, in LDS; null: left out) holds, into m and a (3 x kGeoPerAxis, LDS).
// An interval that holds a value that is not finite is infinitely wide (its
// centre not a number): no charge is far from it.  Called by a whole workgroup; the
// same result wherever it is computed.  The values are read once, by a lane per leaf
// interval of any axis, and the coarser intervals join their halves.
__device__ __forceinline__ void axis_extents(const float* const (&x)[3], Frame& f, double* m,
                                             double* a) {
  const int l = max(f.l[0], max(f.l[1], f.l[2]));
  for (int e = threadIdx.x; e < 3 << l; e += kClassThreads) {
    const int axis = e >> l, t = e & ((1 << l) - 1);
    if (!x[axis] || t >> f.l[axis]) continue;
    const int n = f.n[axis], k = f.l[axis], i1 = part_begin(n, k, t + 1);
    const float* v = x[axis];
    float lo = INFINITY, hi = -INFINITY, sum = 0.f;
#pragma unroll 4
    for (int i = part_begin(n, k, t); i < i1; ++i) {
      lo = fminf(lo, v[i]);
      hi = fmaxf(hi, v[i]);
      sum += 0.f * v[i];  // not a number for a value that is not finite
    }
    const int at = axis * kGeoPerAxis + (1 << k) - 1 + t;
    m[at] = sum == 0.f ? (double)lo : (double)NAN;
    a[at] = (double)hi;
  }
  __syncthreads();
  for (int k = l - 1; k >= 0; --k) {
    for (int e = threadIdx.x; e < 3 << k; e += kClassThreads) {
      const int axis = e >> k, t = e & ((1 << k) - 1);
      if (!x[axis] || k >= f.l[axis]) continue;
      const int at = axis * kGeoPerAxis + (1 << k) - 1 + t;
      const int half = axis * kGeoPerAxis + (2 << k) - 1 + 2 * t;  // of two
      const double lo0 = m[half], lo1 = m[half + 1];
      m[at] = lo0 != lo0 || lo1 != lo1 ? (double)NAN : fmin(lo0, lo1);
      a[at] = fmax(a[half], a[half + 1]);
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < 3 * kGeoPerAxis; e += kClassThreads) {
    const int axis = e / kGeoPerAxis;
    if (!x[axis] || e - axis * kGeoPerAxis >= (2 << f.l[axis]) - 1) continue;
    const double lo = m[e], hi = a[e];
    const bool fine = lo == lo;
    m[e] = fine ? 0.5 * (lo + hi) : (double)NAN;
    a[e] = fine ? fmax(0.5 * (hi - lo), 1e-12) : (double)INFINITY;
  }
  __syncthreads();
}

// One axis: extents to memory, the weights of its values at every level and
// the ancestors' weights at the leaf intervals' nodes.
// Shared by kTableBlocks workgroups: a row is 12 FP64 divisions.
__device__ void axis_tables(const FarArgs& A, Frame& f, int axis, int share, const float* x,
                            const double* m, const double* a) {
  const int n = f.n[axis], l = f.l[axis];
  const int first = share * kClassThreads + threadIdx.x, stride = kClassThreads * kTableBlocks;
  double* geo = A.geo + f.geo0 + (long long)axis * kGeoPerAxis * 2;
  for (int e = first; e < (2 << l) - 1; e += stride) {
    geo[2 * e] = m[e];
    geo[2 * e + 1] = a[e];
  }
  for (int r = first; r < (l + 1) * n; r += stride) {
    const int k = r / n, i = r - k * n;
    int t = (int)(((long long)i << k) / n);  // the part that holds value i, or one off
    while (t > 0 && i < part_begin(n, k, t)) --t;
    while (i >= part_begin(n, k, t + 1)) ++t;
    const int e = (1 << k) - 1 + t;
    lagrange(((double)x[i] - m[e]) / a[e], A.lag + f.lag0[axis] + (long long)r * kP);
  }
  const int rows = (1 << l) * l * kP;
  for (int r = first; r < rows; r += stride) {
    const int j = r % kP, k = (r / kP) % l, t = r / (kP * l);
    const int e = (1 << l) - 1 + t, anc = (1 << k) - 1 + (t >> (l - k));
    const double X = fma(a[e], kNodeX[j], m[e]);
    lagrange((X - m[anc]) / a[anc], A.lag + f.tr0[axis] + (long long)r * kP);
  }
}

// Sum of v over the wave, in lane 63.
__device__ __forceinline__ float wave_sum63(float v) {
  auto add = [&](auto ctrl, auto rows) __attribute__((always_inline)) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value,
                                                    decltype(rows)::value, 0xf, false));
  };
  using std::integral_constant;
  add(integral_constant<int, 0x111>(), integral_constant<int, 0xf>());  // row_shr:1, 2, 4, 8
  add(integral_constant<int, 0x112>(), integral_constant<int, 0xf>());
  add(integral_constant<int, 0x114>(), integral_constant<int, 0xf>());
  add(integral_constant<int, 0x118>(), integral_constant<int, 0xf>());
  add(integral_constant<int, 0x142>(), integral_constant<int, 0xa>());  // row_bcast:15, 31
  add(integral_constant<int, 0x143>(), integral_constant<int, 0xc>());
  return v;
}

// Whether a charge is far from the cell with centre m and half widths a; gap2: its
// squared distance from the cell.
__device__ __forceinline__ bool far_from(const float4& c, const float (&m)[3], const float (&a)[3],
                                         float& gap2) {
  const float x[3] = {c.x, c.y, c.z};
  float d2[3], g2[3];
  bool ok = fabsf(c.w) < 1e30f;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float d = fabsf(x[i] - m[i]);
    const float gap = fmaxf(d - a[i], 0.0f);
    ok = ok && d < kMaxCoord && a[i] < kMaxCoord;
    d2[i] = d * d;
    g2[i] = gap * gap;
  }
  gap2 = g2[0] + g2[1] + g2[2];
  ok = ok && gap2 >= kMinGap2;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    ok = ok && fmaf(d2[i], kInvS2, (g2[(i + 1) % 3] + g2[(i + 2) % 3]) * kInvS21) >= a[i] * a[i];
  return ok;
}

// One workgroup per 64 charges, its waves sharing the cells of a level (a cell is a
// chain of some 1,000 cycles; one wave for all 73 cells of a 101^3 grid took 36
// us, eight take 11): the far mask of every cell (far from it, near all
// its ancestors) and the near mask of every leaf, so that each charge is in
// exactly one mask of every leaf's path.  A cell whose parent is near none
// of the wave's charges is skipped.  Padding is in no mask.  The frame's last
// workgroups make the tables, kTableBlocks those of one axis.
template <bool E>
__global__ __launch_bounds__(kClassThreads) void far_classify_kernel(FarArgs A) {
  extern __shared__ char dyn[];
  Frame& f = frame_of_block(&FarFrame::class_blk0, blockIdx.x);
  const int b = blockIdx.x - f.class_blk0;
  float* sx = (float*)dyn;  // the axes
  const int values = f.n[0] + f.n[1] + f.n[2];
  double* sm = (double*)(dyn + ((values * 4 + 15) & ~15));  // 3 x kGeoPerAxis
  double* sa = sm + 3 * kGeoPerAxis;
  unsigned long long* far = (unsigned long long*)(sa + 3 * kGeoPerAxis);  // cells
  unsigned long long* near = far + f.cells;                               // cells
  float* mag = (float*)(near + f.cells);                                  // cells
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int only = b < f.nseg ? -1 : (b - f.nseg) / kTableBlocks;  // table workgroups: their axis
  float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
  if (only < 0) c = A.ch[f.ch0 + (long long)b * 64 + lane];
  const float* axes[3];
  float* to = sx;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float* __restrict__ x = A.ax[i] + f.ax0[i];
    const bool used = only < 0 || i == only;
    if (used)
      for (int k = threadIdx.x; k < f.n[i]; k += kClassThreads) to[k] = x[k];
    axes[i] = used ? to : nullptr;
    to += f.n[i];
  }
  __syncthreads();
  axis_extents(axes, f, sm, sa);
  if (only >= 0) {
    axis_tables(A, f, only, (b - f.nseg) % kTableBlocks,
                only == 0 ? axes[0] : only == 1 ? axes[1] : axes[2], sm + only * kGeoPerAxis,
                sa + only * kGeoPerAxis);
    return;
  }
  const bool real = !(c.x == kPadCoord && c.y == kPadCoord && c.z == kPadCoord && c.w == 0.f);
  const unsigned long long all = __ballot(real);
  int cell0 = 0, parent0 = 0;
  for (int level = 0; level < f.levels; ++level) {
    const int cells = cells_at(f, level);
    for (int k = wave; k < cells; k += kClassWaves) {
      int t[3];
      cell_parts(f, level, k, t);
      const unsigned long long pm =
          level ? near[parent0 + ancestor(f, level - 1, level, t)] : all;
      unsigned long long mf = 0ull;
      [[maybe_unused]] float s = 0.f;
      if (pm) {
        float m[3], a[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const int e = i * kGeoPerAxis + (1 << axis_level(f, i, level)) - 1 + t[i];
          m[i] = (float)sm[e];
          a[i] = (float)sa[e];
        }
        float gap2;
        const bool mine = far_from(c, m, a, gap2) && ((pm >> lane) & 1);
        mf = __ballot(mine);
        if constexpr (E) s = wave_sum63(mine ? fabsf(c.w) * __builtin_amdgcn_rcpf(gap2) : 0.f);
      }
      if (lane == 63) {
        far[cell0 + k] = mf;
        near[cell0 + k] = pm & ~mf;
        if constexpr (E) mag[cell0 + k] = s;
      }
    }
    __syncthreads();
    parent0 = cell0;
    cell0 += cells;
  }
  const int leaves = cell0 - parent0;
  unsigned long long* out = A.mask + f.mask0 + b;
  for (int k = threadIdx.x; k < f.cells; k += kClassThreads) {
    out[(long long)k * f.nseg] = far[k];
    if constexpr (E) A.mag[f.mag0 + (long long)k * f.nseg + b] = mag[k];
  }
  for (int k = threadIdx.x; k < leaves; k += kClassThreads)
    out[(long long)(f.cells + k) * f.nseg] = near[parent0 + k];
}

constexpr int kNearHead = 2;  // number of near charges, S

__host__ __device__ inline long long near_stride(int nseg) { return kNearHead + 64LL * nseg; }

// ---- charges of a mask list ------------------------------------------------

// Exclusive prefix counts of the list's nseg masks into off (nseg + 1, LDS);
// returns the total.  Called by the whole workgroup of T threads; tmp (T).
template <int T>
__device__ __forceinline__ int list_prefix(const unsigned long long* __restrict__ mask, int nseg,
                                           int* off, int* tmp) {
  const int per = (nseg + T - 1) / T;
  const int s0 = min((int)threadIdx.x * per, nseg), s1 = min(s0 + per, nseg);
  int n = 0;
  for (int s = s0; s < s1; ++s) n += __popcll(mask[s]);
  int run = n;  // inclusive scan inside the wave, then over the waves
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(run, d);
    if ((int)(threadIdx.x & 63) >= d) run += v;
  }
  if ((threadIdx.x & 63) == 63) tmp[threadIdx.x >> 6] = run;
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) {
    if (w < (int)(threadIdx.x >> 6)) before += tmp[w];
    total += tmp[w];
  }
  int o = before + run - n;
  for (int s = s0; s < s1; ++s) {
    off[s] = o;
    o += __popcll(mask[s]);
  }
  if (threadIdx.x == 0) off[nseg] = total;
  __syncthreads();
  return total;
}

// Number of the list's r-th charge.
__device__ __forceinline__ int list_charge(const unsigned long long* __restrict__ mask, int nseg,
                                           const int* off, int r) {
  int lo = 0, hi = nseg - 1;  // the last segment with off <= r
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= r)
      lo = mid;
    else
      hi = mid - 1;
  }
  unsigned long long m = mask[lo];
  int k = r - off[lo], bit = 0;
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) {  // the k-th set bit
    const int n = __popcll(m & ((1ull << w) - 1ull));
    if (k >= n) {
      k -= n;
      bit += w;
      m >>= w;
    }
  }
  return lo * 64 + bit;
}

// ---- node sums ---------------------------------------------------------------

// q / r^3 (and q / r) from the FP32 seed of 1 / r and an FP64 correction:
// with y the seed and e = 1 - r^2 y^2 (|e| ~ 2e-7), 1/r = y (1 + e/2) and
// 1/r^3 = y^3 (1 + 3e/2) up to e^2 ~ 5e-14.
template <bool E, bool PHI>
__device__ __forceinline__ void far_pair(double r2, double q, double& s, double& v) {
  const double y = (double)__builtin_amdgcn_rsqf((float)r2);
  const double y2 = y * y;
  const double e = fma(-r2, y2, 1.0);
  const double qy = q * y;
  if constexpr (PHI) v = fma(qy, fma(0.5, e, 1.0), v);
  if constexpr (E) s = (qy * y2) * fma(1.5, e, 1.0);
}

// Node workgroups of one frame come level by level, (cell, split, third of the
// nodes) each; one workgroup per leaf follows, which lists its near charges.
template <bool E, bool PHI>
__global__ __launch_bounds__(kNodeThreads, 6) void far_nodes_kernel(FarArgs A) {
  constexpr int C = (E ? 3 : 0) + (PHI ? 1 : 0);
  constexpr int kAcc = 3 * C;
  Frame& f = frame_of_block(&FarFrame::node_blk0, blockIdx.x);
  __shared__ double4 list[kBatch];  // also the groups' sums: 3 x kAcc x kNodeLanes doubles
  __shared__ int off[kMaxSegs + 1], tmp[kNodeThreads / 64];
  static_assert(sizeof(list) >= sizeof(double) * kNodeLanes * kAcc, "one group's sums");
  const int tid = threadIdx.x;
  int b = blockIdx.x - f.node_blk0;
  int level = 0, cell0 = 0;
  long long part = f.part0;
  for (; level < f.levels; ++level) {
    const int cells = cells_at(f, level);
    const int nb = cells * f.splits[level];
    if (b < nb * kThirds) break;
    b -= nb * kThirds;
    part += (long long)nb * C * kNodes;
    cell0 += cells;
  }
  if (level == f.levels) {  // the launch's b-th near list
    const unsigned long long* __restrict__ mask =
        A.mask + f.mask0 + (long long)(f.cells + f.leaf0 + b) * f.nseg;
    const int total = list_prefix<kNodeThreads>(mask, f.nseg, off, tmp);
    int* out = A.near + f.near0 + (long long)b * near_stride(f.nseg);
    for (int r = tid; r < total; r += kNodeThreads)
      out[kNearHead + r] = list_charge(mask, f.nseg, off, r);
    if (tid == 0) out[0] = total;
    if (E && tid >= kNodeThreads - 64) {  // S: the cells of the leaf's path, in a fixed order
      int t[3];
      cell_parts(f, f.levels - 1, f.leaf0 + b, t);
      double s = 0.0;
      for (int k = 0, first = 0; k < f.levels; first += cells_at(f, k++)) {
        const float* __restrict__ mag =
            A.mag + f.mag0 + (long long)(first + ancestor(f, k, f.levels - 1, t)) * f.nseg;
        for (int i = tid & 63; i < f.nseg; i += 64) s += (double)mag[i];
      }
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d);
      if ((tid & 63) == 0) out[1] = __float_as_int((float)s);
    }
    return;
  }
  const int third = b % kThirds, slot = b / kThirds;
  const int splits = f.splits[level];
  const int cell = slot / splits, split = slot % splits;
  part += (long long)slot * C * kNodes;
  int t[3];
  cell_parts(f, level, cell, t);
  const double* __restrict__ geo = A.geo + f.geo0;
  int en[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) en[i] = i * kGeoPerAxis + (1 << axis_level(f, i, level)) - 1 + t[i];

  // this thread's three nodes, one (x, y) line, and its share of the charges
  const int nl = tid % kNodeLanes, group = tid / kNodeLanes;
  const int line = third * (kP * kP / kThirds) + nl / 4, z0 = (nl & 3) * 3;
  const double px = fma(geo[2 * en[0] + 1], kNodeX[line / kP], geo[2 * en[0]]);
  const double py = fma(geo[2 * en[1] + 1], kNodeX[line % kP], geo[2 * en[1]]);
  double pz[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) pz[k] = fma(geo[2 * en[2] + 1], kNodeX[z0 + k], geo[2 * en[2]]);
  double acc[3][C];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int c = 0; c < C; ++c) acc[k][c] = 0.0;

  const unsigned long long* __restrict__ mask = A.mask + f.mask0 + (long long)(cell0 + cell) * f.nseg;
  const float4* __restrict__ ch = A.ch + f.ch0;
  const int total = list_prefix<kNodeThreads>(mask, f.nseg, off, tmp);
  const int r0 = (int)((long long)total * split / splits);
  const int r1 = (int)((long long)total * (split + 1) / splits);
  for (int base = r0; base < r1; base += kBatch) {
    const int n = min(kBatch, r1 - base);
    if (tid < n) {
      const float4 c = ch[list_charge(mask, f.nseg, off, base + tid)];
      list[tid] = make_double4(c.x, c.y, c.z, c.w);
    }
    __syncthreads();
#pragma unroll 2
    for (int i = group; i < n; i += kNodeGroups) {
      const double4 s = list[i];
      const double dx = px - s.x, dy = py - s.y;
      const double dxy2 = fma(dy, dy, dx * dx);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double dz = pz[k] - s.z;
        double w = 0.0;
        far_pair<E, PHI>(fma(dz, dz, dxy2), s.w, w, acc[k][C - 1]);
        if constexpr (E) {
          acc[k][0] = fma(w, dx, acc[k][0]);
          acc[k][1] = fma(w, dy, acc[k][1]);
          acc[k][2] = fma(w, dz, acc[k][2]);
        }
      }
    }
    __syncthreads();
  }
  // the groups' sums, added in order to group 0's
  double* sums = (double*)list;
  for (int g = 1; g < kNodeGroups; ++g) {
    if (group == g) {
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int c = 0; c < C; ++c) sums[(k * C + c) * kNodeLanes + nl] = acc[k][c];
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[k][c] += sums[(k * C + c) * kNodeLanes + nl];
    }
    __syncthreads();
  }
  if (group) return;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int c = 0; c < C; ++c)
      A.part[part + (long long)c * kNodes + line * kP + z0 + k] = acc[k][c];
}

// ---- the splits' sums --------------------------------------------------------

// Threads per value of a level: the more splits, the more.
__host__ __device__ inline int red_groups(int splits) {
  return splits >= 24 ? 8 : splits >= 4 ? 4 : 1;
}

// Workgroups of a level: none where there is one split (its sums are used as
// they are).
__host__ __device__ inline int red_blocks(int cells, int C, int splits) {
  if (splits == 1) return 0;
  const int per = kRedThreads / red_groups(splits);
  return (cells * C * kNodes + per - 1) / per;
}

template <int C>
__global__ __launch_bounds__(kRedThreads) void far_reduce_kernel(FarArgs A) {
  Frame& f = frame_of_block(&FarFrame::red_blk0, blockIdx.x);
  int b = blockIdx.x - f.red_blk0;
  long long part = f.part0, val = f.val0;
  int level = 0, values, groups, per;
  for (;;) {
    values = cells_at(f, level) * C * kNodes;
    groups = red_groups(f.splits[level]);
    per = kRedThreads / groups;
    const int nb = red_blocks(cells_at(f, level), C, f.splits[level]);
    if (b < nb) break;
    b -= nb;
    part += (long long)values * f.splits[level];
    val += values;
    ++level;
  }
  const int splits = f.splits[level];
  const int g = threadIdx.x / per, v = b * per + threadIdx.x % per;
  __shared__ double sh[kRedThreads];
  double s = 0.0;
  if (v < values) {
    const int cell = v / (C * kNodes), r = v - cell * C * kNodes;
    const double* p = A.part + part + (long long)cell * splits * C * kNodes + r;
#pragma unroll 8
    for (int i = g; i < splits; i += groups) s += p[(long long)i * C * kNodes];
  }
  if (groups > 1) {
    sh[threadIdx.x] = s;
    __syncthreads();
    if (g == 0) {
      s = 0.0;
      for (int i = 0; i < groups; ++i) s += sh[i * per + threadIdx.x];
    }
  }
  if (g == 0 && v < values) A.val[val + v] = s;
}

// ---- points --------------------------------------------------------------------

template <bool E, bool PHI, bool SOFT>
__global__ __launch_bounds__(kEvalThreads, E && PHI ? 3 : 4) void far_eval_kernel(FarArgs A) {
  constexpr int C = (E ? 3 : 0) + (PHI ? 1 : 0);
  constexpr int K = 3;  // points per thread along z
  constexpr int kPC = kPlanes * C;
  Frame& f = frame_of_block(&FarFrame::eval_blk0, blockIdx.x);
  const int b = blockIdx.x - f.eval_blk0;
  const int list = b / f.xblocks, leaf = f.leaf0 + list, xb = b % f.xblocks;
  const int bottom = f.levels - 1;
  int t[3];
  cell_parts(f, bottom, leaf, t);
  int lo[3], n[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    lo[i] = part_begin(f.n[i], f.l[i], t[i]);
    n[i] = part_begin(f.n[i], f.l[i], t[i] + 1) - lo[i];
  }
  const int x0 = lo[0] + xb * kPlanes;
  const int np = min(kPlanes, lo[0] + n[0] - x0);
  if (np <= 0) return;
  __shared__ double w1[kPC * kP * kP];
  __shared__ double w2[kPC * kLeafMax * kP];
  __shared__ double lz[kLeafMax * kP];
  // first the contracted planes of a level, then the near charges
  __shared__ union {
    double wt[kPC * kP * kP];
    double4 list[kNearLds];
  } u;
  __shared__ unsigned short redo[E ? kPlanes * kLeafMax * kLeafMax : 1];  // points to sum directly
  __shared__ int redos;
  double* const wt = u.wt;
  const int tid = threadIdx.x;
  if (E && tid == 0) redos = 0;
  const double* __restrict__ lagy =
      A.lag + f.lag0[1] + ((long long)f.l[1] * f.n[1] + lo[1]) * kP;
  const double* __restrict__ lagz =
      A.lag + f.lag0[2] + ((long long)f.l[2] * f.n[2] + lo[2]) * kP;
  for (int i = tid; i < n[2] * kP; i += kEvalThreads) lz[i] = lagz[i];
  for (int i = tid; i < kPC * kP * kP; i += kEvalThreads) w1[i] = 0.0;
  __syncthreads();
  // Every level's nodes: x contracted at the planes, y and z carried to the
  // leaf's nodes, summed in w1.
  long long val = f.val0, part = f.part0;
  for (int level = 0; level <= bottom; ++level) {
    const int ax = axis_level(f, 0, level), ay = axis_level(f, 1, level),
              az = axis_level(f, 2, level);
    const double* __restrict__ V = (f.splits[level] == 1 ? A.part + part : A.val + val) +
                                   (long long)ancestor(f, level, bottom, t) * C * kNodes;
    val += (long long)cells_at(f, level) * C * kNodes;
    part += (long long)cells_at(f, level) * f.splits[level] * C * kNodes;
    const double* __restrict__ lagx = A.lag + f.lag0[0] + ((long long)ax * f.n[0] + x0) * kP;
    const bool same = ay == f.l[1] && az == f.l[2];
    double* __restrict__ to = same ? w1 : wt;
    for (int i = tid; i < C * kP * kP; i += kEvalThreads) {
      const int comp = i / (kP * kP), r = i % (kP * kP);
      double s[kPlanes] = {};
#pragma unroll
      for (int k = 0; k < kP; ++k) {
        const double v = V[comp * kNodes + k * kP * kP + r];
#pragma unroll
        for (int p = 0; p < kPlanes; ++p)
          s[p] = fma(lagx[min(p, np - 1) * kP + k], v, s[p]);
      }
#pragma unroll
      for (int p = 0; p < kPlanes; ++p) {
        double* o = to + (p * C + comp) * kP * kP + r;
        *o = same ? *o + s[p] : s[p];
      }
    }
    __syncthreads();
    if (same) continue;
    if (ay != f.l[1]) {  // w2 <- Ty wt
      const double* __restrict__ T = A.lag + f.tr0[1] + ((long long)t[1] * f.l[1] + ay) * kP * kP;
      for (int i = tid; i < kPC * kP; i += kEvalThreads) {  // one (plane, comp, z) line
        const int pc = i / kP, c = i % kP;
        double v[kP];
#pragma unroll
        for (int k = 0; k < kP; ++k) v[k] = wt[pc * kP * kP + k * kP + c];
        for (int j = 0; j < kP; ++j) {
          double s = 0.0;
#pragma unroll
          for (int k = 0; k < kP; ++k) s = fma(T[j * kP + k], v[k], s);
          w2[pc * kP * kP + j * kP + c] = s;
        }
      }
    } else {
      for (int i = tid; i < kPC * kP * kP; i += kEvalThreads) w2[i] = wt[i];
    }
    __syncthreads();
    if (az != f.l[2]) {  // w1 += w2 Tz'
      const double* __restrict__ T = A.lag + f.tr0[2] + ((long long)t[2] * f.l[2] + az) * kP * kP;
      for (int i = tid; i < kPC * kP; i += kEvalThreads) {  // one (plane, comp, y) line
        double v[kP];
#pragma unroll
        for (int k = 0; k < kP; ++k) v[k] = w2[i * kP + k];
        for (int j = 0; j < kP; ++j) {
          double s = 0.0;
#pragma unroll
          for (int k = 0; k < kP; ++k) s = fma(T[j * kP + k], v[k], s);
          w1[i * kP + j] += s;
        }
      }
    } else {
      for (int i = tid; i < kPC * kP * kP; i += kEvalThreads) w1[i] += w2[i];
    }
    __syncthreads();
  }
  // contract y
  for (int i = tid; i < np * C * n[1] * kP; i += kEvalThreads) {
    const int c = i % kP, j = (i / kP) % n[1], pc = i / (kP * n[1]);
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kP; ++k) s = fma(lagy[j * kP + k], w1[pc * kP * kP + k * kP + c], s);
    w2[(pc * kLeafMax + j) * kP + c] = s;
  }
  const int* __restrict__ near = A.near + f.near0 + (long long)list * near_stride(f.nseg);
  const float4* __restrict__ ch = A.ch + f.ch0;
  const int total = near[0];
  const double least = E ? kCancel * (double)__int_as_float(near[1]) : 0.0;
  __syncthreads();
  // z, the near charges and the store
  const float* __restrict__ ax = A.ax[0] + f.ax0[0];
  const float* __restrict__ ay = A.ax[1] + f.ax0[1];
  const float* __restrict__ az = A.ax[2] + f.ax0[2];
  const double rclamp = pair_clamp();
  const int chunks = (n[2] + K - 1) / K, items = np * n[1] * chunks;
  for (int i0 = 0; i0 < items; i0 += kEvalThreads) {  // the same rounds for every thread
    const int i = min(i0 + tid, items - 1);
    const bool valid = i0 + tid < items;
    const int k0 = (i % chunks) * K, j = (i / chunks) % n[1], p = i / (chunks * n[1]);
    double acc[K][C];
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int c = 0; c < C; ++c) acc[k][c] = 0.0;
#pragma unroll
    for (int a = 0; a < kP; ++a)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const double v = w2[((p * C + c) * kLeafMax + j) * kP + a];
#pragma unroll
        for (int k = 0; k < K; ++k)
          acc[k][c] = fma(lz[min(k0 + k, n[2] - 1) * kP + a], v, acc[k][c]);
      }
    const double px = ax[x0 + p], py = ay[lo[1] + j];
    double pz[K];
#pragma unroll
    for (int k = 0; k < K; ++k) pz[k] = az[lo[2] + min(k0 + k, n[2] - 1)];
    for (int q0 = 0; q0 < total; q0 += kNearLds) {
      const int qn = min(kNearLds, total - q0);
      if (i0 == 0 || total > kNearLds) {  // a short list stays staged
        __syncthreads();
        if (tid < qn) {
          const float4 c = ch[near[kNearHead + q0 + tid]];
          u.list[tid] = make_double4(c.x, c.y, c.z, c.w);
        }
        __syncthreads();
      }
      for (int q = 0; q < qn; ++q) {
        const double4 c = u.list[q];
        const double dx = px - c.x, dy = py - c.y;
        const double dxy2 = fma(dy, dy, dx * dx);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const double dz = pz[k] - c.z;
          double re;
          const double y = pair_rsqrt<SOFT, !PHI>(fma(dz, dz, dxy2), rclamp, re);
          if constexpr (PHI) acc[k][C - 1] = fma(c.w, y, acc[k][C - 1]);
          if constexpr (E) {
            const double w = (c.w * re) * (re * re);
            acc[k][0] = fma(w, dx, acc[k][0]);
            acc[k][1] = fma(w, dy, acc[k][1]);
            acc[k][2] = fma(w, dz, acc[k][2]);
          }
        }
      }
    }
    if (!valid) continue;
    const long long m0 = f.out0 + ((long long)(x0 + p) * f.n[1] + lo[1] + j) * f.n[2] + lo[2] + k0;
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (k0 + k < n[2]) {
        if constexpr (E) {
          float* e = (float*)A.e + 3 * (m0 + k);
          e[0] = (float)(kCoulomb * acc[k][0]);
          e[1] = (float)(kCoulomb * acc[k][1]);
          e[2] = (float)(kCoulomb * acc[k][2]);
          if (fma(acc[k][2], acc[k][2], fma(acc[k][1], acc[k][1], acc[k][0] * acc[k][0])) <
              least * least)
            redo[atomicAdd(&redos, 1)] = (unsigned short)((p * n[1] + j) * n[2] + k0 + k);
        }
        if constexpr (PHI) ((float*)A.phi)[m0 + k] = (float)(kCoulomb * acc[k][C - 1]);
      }
  }
  if constexpr (E) {
    __syncthreads();
    const int again = redos;
    for (int i = 0; i < again; ++i) {  // the whole workgroup, charge by charge
      const int pt = redo[i];
      const int k = pt % n[2], j = pt / n[2] % n[1], p = pt / (n[1] * n[2]);
      const double px = ax[x0 + p], py = ay[lo[1] + j], pz = az[lo[2] + k];
      double e[3] = {0.0, 0.0, 0.0};
      for (int q = tid; q < 64 * f.nseg; q += kEvalThreads) {
        const float4 c = ch[q];
        const double dx = px - (double)c.x, dy = py - (double)c.y, dz = pz - (double)c.z;
        double re;
        pair_rsqrt<SOFT, !PHI>(fma(dz, dz, fma(dy, dy, dx * dx)), rclamp, re);
        const double w = ((double)c.w * re) * (re * re);
        e[0] = fma(w, dx, e[0]);
        e[1] = fma(w, dy, e[1]);
        e[2] = fma(w, dz, e[2]);
      }
#pragma unroll
      for (int d = 32; d > 0; d >>= 1)
#pragma unroll
        for (int c = 0; c < 3; ++c) e[c] += __shfl_xor(e[c], d);
      if ((tid & 63) == 0)
#pragma unroll
        for (int c = 0; c < 3; ++c) lz[(tid >> 6) * 3 + c] = e[c];
      __syncthreads();
      if (tid < 3) {
        double v = 0.0;
        for (int w = 0; w < kEvalThreads / 64; ++w) v += lz[w * 3 + tid];
        const long long m = f.out0 + ((long long)(x0 + p) * f.n[1] + lo[1] + j) * f.n[2] + lo[2] + k;
        ((float*)A.e)[3 * m + tid] = (float)(kCoulomb * v);
      }
      __syncthreads();
    }
  }
}

int halvings(int n) {
  int l = 0;
  while (((n + (1 << l) - 1) >> l) > kLeafMax) ++l;
  return l;
}

// Frames that share the four launches: workgroups of each, and the elements of
// the scratch arrays in FarArgs.
struct Group {
  int first = 0, count = 0;  // of the call's frames
  long long classify = 0, nodes = 0, reduce = 0, eval = 0;
  size_t lds = 0;  // of the classification
  // Leaves whose near lists are held at once, of the leaves of one frame whose lists
  // (room for every charge in each) would not fit the scratch bound; 0: all of them.
  int range = 0, leaves = 0;
  long long part = 0, val = 0, geo = 0, lag = 0, mask = 0, mag = 0, near = 0;
  size_t bytes() const {
    return (size_t)(part + val + geo + lag + mask) * 8 + (size_t)(mag + near) * 4;
  }
};

template <bool E, bool PHI>
void far_launch(hipStream_t st, FarArgs A, const Group& n, bool soft) {
  constexpr int C = (E ? 3 : 0) + (PHI ? 1 : 0);
  auto nodes = [&](long long blocks) {
    hipLaunchKernelGGL((far_nodes_kernel<E, PHI>), dim3((unsigned)blocks), dim3(kNodeThreads), 0, st,
                       A);
  };
  auto eval = [&](long long blocks) {
    if (soft)
      hipLaunchKernelGGL((far_eval_kernel<E, PHI, true>), dim3((unsigned)blocks),
                         dim3(kEvalThreads), 0, st, A);
    else
      hipLaunchKernelGGL((far_eval_kernel<E, PHI, false>), dim3((unsigned)blocks),
                         dim3(kEvalThreads), 0, st, A);
  };
  hipLaunchKernelGGL((far_classify_kernel<E>), dim3((unsigned)n.classify), dim3(kClassThreads), n.lds, st, A);
  nodes(n.nodes);
  if (n.reduce)
    hipLaunchKernelGGL((far_reduce_kernel<C>), dim3((unsigned)n.reduce), dim3(kRedThreads), 0, st,
                       A);
  eval(n.eval);
  // the other ranges of leaves: near lists alone (the workgroups behind those of
  // the nodes), in the memory of the previous range's, and their points
  if (n.range) A.one.node_blk0 = -(int)(n.nodes - n.range);
  for (int left = n.leaves - n.range; n.range && left > 0; left -= n.range) {
    A.one.leaf0 += n.range;
    const int now = std::min(n.range, left);
    nodes(now);
    eval((long long)now * A.one.xblocks);
  }
}

}  // namespace

bool far_grid_ok(int nx, int ny, int nz, int npad, double min_pairs) {
  const int n[3] = {nx, ny, nz};
  for (int i = 0; i < 3; ++i)
    if (n[i] < kFarMinAxis || n[i] > kMaxAxis) return false;
  return npad <= 64 * kMaxSegs && (double)nx * ny * nz * npad >= min_pairs;
}

struct FarPlan {
  std::vector<FarFrame> frames;
  std::vector<Group> groups;
  bool want_e, want_phi;
  void *buf = nullptr, *tab = nullptr;
};

// The frames in as few groups as the scratch bound allows.  The frames of all
// groups are one table, uploaded at once, so that a call of the same shapes finds
// it unchanged (and can be captured) whatever their number.
//
// The bound holds for one frame too: of the largest grid (4,681 cells) and charge
// count, node sums, masks and tables take 0.7 GB, and near lists are held for as
// many leaves at a time as the rest has room for (for all 4,096 they would take 2.1
// GB).  217 x 218 x 217 points, 45,000 charges: two ranges of leaves.
std::shared_ptr<const FarPlan> far_grid_plan(cpet_ctx* ctx, const std::vector<FarGrid>& grids,
                                             bool want_e, bool want_phi) {
  const int C = (want_e ? 3 : 0) + (want_phi ? 1 : 0);
  constexpr size_t kMaxScratch = (size_t)1 << 30;
  const int F = (int)grids.size();
  auto plan = std::make_shared<FarPlan>();
  plan->want_e = want_e;
  plan->want_phi = want_phi;
  std::vector<FarFrame>& frames = plan->frames;
  size_t bytes = 0;
  int done = 0;
  while (done < F) {
    Group n;
    n.first = done;
    // Node workgroups: two per CU over all frames, shared out by work.  A
    // level's far charges, over all its cells, are about the charges of the
    // frame (level 0) or twice that: with kRho, most charges of a level's
    // near region are far from its children.
    auto weight = [](int level) { return level ? 2.0 : 1.0; };
    double work = 0.0;
    for (int i = done; i < F; ++i) {
      int deep = 0;
      for (int k = 0; k < 3; ++k) deep = std::max(deep, halvings(grids[i].n[k]));
      for (int k = 0; k <= deep; ++k) work += weight(k) * grids[i].npad;
    }
    const double quantum = work * kThirds / (2.0 * ctx->num_cus);
    while (done < F) {
      const FarGrid& g = grids[done];
      FarFrame f = {};
      int values = 0;
      for (int i = 0; i < 3; ++i) {
        f.n[i] = g.n[i];
        f.l[i] = halvings(g.n[i]);
        f.ax0[i] = g.ax0[i];
        f.levels = std::max(f.levels, f.l[i] + 1);
        values += g.n[i];
      }
      f.nseg = g.npad / 64;
      f.ch0 = g.ch0;
      f.out0 = g.out0;
      f.class_blk0 = (int)n.classify;
      f.node_blk0 = (int)n.nodes;
      f.red_blk0 = (int)n.reduce;
      f.eval_blk0 = (int)n.eval;
      f.part0 = n.part;
      f.val0 = n.val;
      f.geo0 = n.geo;
      f.mask0 = n.mask;
      f.mag0 = n.mag;
      f.near0 = n.near;
      long long p = 0, nb = 0, rb = 0, leaves = 0;
      for (int k = 0; k < f.levels; ++k) {
        leaves = cells_at(f, k);
        f.cells += (int)leaves;
        f.splits[k] = std::max(1, std::min((f.nseg + 1) / 2,
                                           (int)(weight(k) * g.npad / (leaves * quantum) + 0.5)));
        nb += leaves * f.splits[k] * kThirds;
        p += leaves * f.splits[k] * C * kNodes;
        rb += red_blocks((int)leaves, C, f.splits[k]);
      }
      Group with = n;
      for (int i = 0; i < 3; ++i) {
        f.lag0[i] = with.lag;
        with.lag += (long long)(f.l[i] + 1) * f.n[i] * kP;
        f.tr0[i] = with.lag;
        with.lag += (long long)(1 << f.l[i]) * f.l[i] * kP * kP;
      }
      with.part += p;
      with.val += (long long)f.cells * C * kNodes;
      with.mask += (f.cells + leaves) * f.nseg;
      with.mag += (long long)f.cells * f.nseg;
      with.near += leaves * near_stride(f.nseg);
      with.geo += 3LL * kGeoPerAxis * 2;
      if (n.count && with.bytes() > kMaxScratch) break;
      long long lists = leaves;
      if (with.bytes() > kMaxScratch) {  // a frame alone
        const size_t list = (size_t)near_stride(f.nseg) * 4;
        const size_t rest = with.bytes() - leaves * list;
        lists = rest + list < kMaxScratch ? (long long)((kMaxScratch - rest) / list) : 1;
        with.range = (int)lists;
        with.leaves = (int)leaves;
        with.near = lists * near_stride(f.nseg);
      }
      const int widest = (f.n[0] + (1 << f.l[0]) - 1) >> f.l[0];
      f.xblocks = (widest + kPlanes - 1) / kPlanes;
      with.classify += f.nseg + 3 * kTableBlocks;
      with.nodes += nb + lists;
      with.reduce += rb;
      with.eval += lists * f.xblocks;
      with.lds = std::max(n.lds, (size_t)((values * 4 + 15) & ~15) + 6 * kGeoPerAxis * 8 +
                                     (size_t)f.cells * 20);
      ++with.count;
      n = with;
      frames.push_back(f);
      ++done;
      if (n.range) break;
    }
    bytes = std::max(bytes, n.bytes());
    plan->groups.push_back(n);
  }
  if (!(plan->buf = ctx_buf_try(ctx, kSlotFarGrid, bytes))) return nullptr;
  if (F > 1 && !(plan->tab = ctx_buf_try(ctx, kSlotFarTables, F * sizeof(FarFrame))))
    return nullptr;
  return plan;
}

int far_grid_run(cpet_ctx* ctx, const FarPlan& plan, const float* const (&ax)[3], const float4* ch,
                 bool soft, void* e, void* phi) {
  if (plan.tab) {
    const int rc = upload_table(ctx, kTabFarFrames, plan.tab, plan.frames.data(),
                                plan.frames.size() * sizeof(FarFrame));
    if (rc) return rc;
  }
  for (const Group& n : plan.groups) {
    FarArgs A = {};
    A.F = n.count;
    A.ch = ch;
    for (int i = 0; i < 3; ++i) A.ax[i] = ax[i];
    A.part = (double*)plan.buf;
    A.val = A.part + n.part;
    A.geo = A.val + n.val;
    A.lag = A.geo + n.geo;
    A.mask = (unsigned long long*)(A.lag + n.lag);
    A.mag = (float*)(A.mask + n.mask);
    A.near = (int*)(A.mag + n.mag);
    A.e = e;
    A.phi = phi;
    if (n.count == 1)
      A.one = plan.frames[n.first];
    else
      A.frames = (const FarFrame*)plan.tab + n.first;
    if (plan.want_e && plan.want_phi)
      far_launch<true, true>(ctx->stream, A, n, soft);
    else if (plan.want_e)
      far_launch<true, false>(ctx->stream, A, n, soft);
    else
      far_launch<false, true>(ctx->stream, A, n, soft);
    CPET_HIP_TRY(hipGetLastError());
  }
  return CPET_OK;
}

}  // namespace cpet
