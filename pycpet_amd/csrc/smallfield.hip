// Field and potential of few point-charge pairs, in one launch.
//
// A call of some 1e7 pairs is over in the time that launches, their gaps and a
// wave's serial chain take.  The direct path (field.hip) packs the charges,
// looks for charges near the grid, sums FP32 tiles split over the charges,
// adds the splits, and checks and recomputes points: six launches, of which
// the sums run with one or two waves per SIMD.  Here one kernel reads the
// caller's arrays, splits the charges over the lanes of a 1,024-thread
// workgroup, adds the splits in LDS and stores.  The pair terms are the
// "mixed" ones (FP64 displacement and r^2, FP32 rsq seed, FP64 correction, FP64
// sums) for E too: one evaluation serves E and phi, and nothing has to be
// checked or recomputed.  What bounds it is the FP64 pair term and its two
// conversions, about 170 cycles a pair and wave (9.2e11 pairs/s); the shorter
// correction y^3 (1 + 3e/2) with a test for the ends of the range saves 4 % of
// E and costs 25 % of phi.
//
// MI355X, whole calls on device tensors back to back (12.5 us of them is the
// host's side), direct -> here: one point x 8,000 charges 34 -> 13 us, 300
// points x 60,000 553 -> 34 us, 11^3 x 2,000 E and phi 41 -> 15 us, 21^3 x
// 2,000 44 -> 24 us.  The limits: kSmallMaxPairs.
//
// Every sum has a fixed order: results are reproducible bit for bit.

#include <algorithm>

#include "cpet_internal.h"
#include "pairterm.h"
#include "smallfield.h"

namespace cpet {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kStage = 1024;  // charges in LDS at once (32 KB)

struct SmallArgs {
  SmallBatch batch;         // many grids: blocks, sizes and offsets, or blk null
  int M, N;
  int ny, nz;               // grid
  const float *ax, *ay, *az;  // its axes, or null
  const float* pts;         // (M,3), when ax is null
  const float *x, *q;       // (N,3), (N)
  float *e, *phi;           // (M,3), (M)
};

// P points per workgroup: thread t has point t % P and every (1024 / P)-th
// charge from t / P on.
template <int P, bool E, bool PHI, bool SOFT, bool GRID, bool BATCH>
__global__ __launch_bounds__(kThreads) void small_field_kernel(SmallArgs a) {
  constexpr int S = kThreads / P;
  constexpr int C = (E ? 3 : 0) + (PHI ? 1 : 0);
  __shared__ double4 stage[P > 1 ? kStage : 1];
  __shared__ double sums[kWaves][C][P];
  const int tid = threadIdx.x, p = tid % P, s = tid / P;
  int block = blockIdx.x;
  const float4* __restrict__ ch = nullptr;
  if constexpr (BATCH) {
    const SmallBatch& t = a.batch;
    const int fr = t.blk[2 * block];
    block = t.blk[2 * block + 1];
    const int nx = t.geo[4 * fr];
    a.ny = t.geo[4 * fr + 1];
    a.nz = t.geo[4 * fr + 2];
    a.M = nx * a.ny * a.nz;
    a.ax = t.axes + t.ax_off[fr];
    a.ay = a.ax + nx;
    a.az = a.ay + a.ny;
    ch = t.ch + t.chg_off[fr];
    a.N = t.chg_off[fr + 1] - t.chg_off[fr];
    if constexpr (E) a.e += 3 * t.out_off[fr];
    if constexpr (PHI) a.phi += t.out_off[fr];
  }
  const int m = min(block * P + p, a.M - 1);
  double px, py, pz;
  if constexpr (GRID) {
    const int line = m / a.nz;
    px = a.ax[line / a.ny];
    py = a.ay[line % a.ny];
    pz = a.az[m - line * a.nz];
  } else {
    px = a.pts[3 * m];
    py = a.pts[3 * m + 1];
    pz = a.pts[3 * m + 2];
  }
  const double rclamp = pair_clamp();
  double acc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = 0.0;
  auto pair = [&](double cx, double cy, double cz, double q) __attribute__((always_inline)) {
    const double dx = px - cx, dy = py - cy, dz = pz - cz;
    double re;
    const double y =
        pair_rsqrt<SOFT, GRID && !PHI>(fma(dz, dz, fma(dy, dy, dx * dx)), rclamp, re);
    if constexpr (PHI) acc[C - 1] = fma(q, y, acc[C - 1]);
    if constexpr (E) {
      const double w = (q * re) * (re * re);
      acc[0] = fma(w, dx, acc[0]);
      acc[1] = fma(w, dy, acc[1]);
      acc[2] = fma(w, dz, acc[2]);
    }
  };
  auto charge = [&](int j) __attribute__((always_inline)) {
    if constexpr (BATCH) return ch[j];
    return make_float4(a.x[3 * j], a.x[3 * j + 1], a.x[3 * j + 2], a.q[j]);
  };
  if constexpr (P == 1) {
    // each charge is used once: straight from memory, coalesced
#pragma unroll 4
    for (int j = tid; j < a.N; j += kThreads) {
      const float4 c = charge(j);
      pair(c.x, c.y, c.z, c.w);
    }
  } else {
    for (int j0 = 0; j0 < a.N; j0 += kStage) {
      const int n = min(kStage, a.N - j0);
      __syncthreads();
      if (tid < n) {
        const float4 c = charge(j0 + tid);
        stage[tid] = make_double4(c.x, c.y, c.z, c.w);
      }
      __syncthreads();
#pragma unroll 2
      for (int j = s; j < n; j += S) {
        const double4 c = stage[j];
        pair(c.x, c.y, c.z, c.w);
      }
    }
  }
  // the lanes that share a point, then the waves, in order
#pragma unroll
  for (int off = P; off < 64; off <<= 1)
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] += __shfl_xor(acc[c], off);
  if ((tid & 63) < P)
#pragma unroll
    for (int c = 0; c < C; ++c) sums[tid >> 6][c][p] = acc[c];
  __syncthreads();
  if (tid >= P * C) return;
  const int c = tid / P, out = block * P + p;  // p = tid % P
  if (out >= a.M) return;
  double v = 0.0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) v += sums[w][c][p];
  const float r = (float)(kCoulomb * v);
  if (E && c < 3)
    a.e[3 * out + c] = r;
  else
    a.phi[out] = r;
}

template <int P, bool GRID, bool BATCH>
void launch(hipStream_t st, int blocks, const SmallArgs& a, bool soft) {
  const dim3 grid(blocks), block(kThreads);
  if (a.e && a.phi)
    hipLaunchKernelGGL((small_field_kernel<P, true, true, true, GRID, BATCH>), grid, block, 0, st, a);
  else if (a.phi)
    hipLaunchKernelGGL((small_field_kernel<P, false, true, false, GRID, BATCH>), grid, block, 0, st, a);
  else if (soft)
    hipLaunchKernelGGL((small_field_kernel<P, true, false, true, GRID, BATCH>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((small_field_kernel<P, true, false, false, GRID, BATCH>), grid, block, 0, st, a);
}

template <bool GRID, bool BATCH>
bool launch_p(int P, hipStream_t st, int blocks, const SmallArgs& a, bool soft) {
  switch (P) {
    case 1: launch<1, GRID, BATCH>(st, blocks, a, soft); return true;
    case 4: launch<4, GRID, BATCH>(st, blocks, a, soft); return true;
    case 16: launch<16, GRID, BATCH>(st, blocks, a, soft); return true;
    case 64: launch<64, GRID, BATCH>(st, blocks, a, soft); return true;
  }
  return false;
}

}  // namespace

bool small_field_ok(bool grid, long long M, int N) {
  const double pairs = (double)M * N;
  if (grid) return pairs <= kSmallMaxPairs;
  return pairs <= (M <= kSmallFewPoints ? 4 : 2) * kSmallMaxPairs;
}

bool small_batch_ok(double pairs, int most_charges, bool phi) {
  return pairs <= (phi ? 2.5e5 : 1.3e5) * most_charges;
}

// As many points per workgroup as leave about three workgroups per CU.
int small_field_points(const cpet_ctx* ctx, long long M) {
  const long long most = 3LL * ctx->num_cus;
  return M <= most ? 1 : M <= 4 * most ? 4 : M <= 16 * most ? 16 : 64;
}

int small_batch_launch(cpet_ctx* ctx, int P, int blocks, const SmallBatch& t, float* e, float* phi,
                       bool soft) {
  SmallArgs a = {};
  a.batch = t;
  a.e = e;
  a.phi = phi;
  if (!launch_p<true, true>(P, ctx->stream, blocks, a, soft)) {
    set_error("internal: %d points per workgroup", P);
    return CPET_ERR_ARG;
  }
  CPET_HIP_TRY(hipGetLastError());
  return CPET_OK;
}

int small_field_launch(cpet_ctx* ctx, int ny, int nz, const float* ax, const float* ay,
                       const float* az, long long M, const float* pts, int N, const float* x,
                       const float* q, float* e, float* phi, bool soft) {
  SmallArgs a = {};
  a.M = (int)M;
  a.N = N;
  a.ny = ny;
  a.nz = nz;
  a.ax = ax;
  a.ay = ay;
  a.az = az;
  a.pts = pts;
  a.x = x;
  a.q = q;
  a.e = e;
  a.phi = phi;
  ctx->fix_count = nullptr;
  ctx->all_f64 = e ? M : 0;
  int rc = prof_mark(ctx, 0);
  if (rc) return rc;
  const int P = small_field_points(ctx, M), blocks = (int)((M + P - 1) / P);
  if (ax)
    launch_p<true, false>(P, ctx->stream, blocks, a, soft);
  else
    launch_p<false, false>(P, ctx->stream, blocks, a, soft);
  CPET_HIP_TRY(hipGetLastError());
  for (int i = 1; i < 4; ++i)
    if ((rc = prof_mark(ctx, i))) return rc;
  return CPET_OK;
}

}  // namespace cpet
