// vplus.hpp - hypercube bookkeeping shared by the VEGAS+ kernels
// (vflowplus.py:37-80, 187-220): cube lookup from the event offsets, cube
// coordinates, per-cube segmented sums, and the fused producer's launcher.
//
// Events of an iteration are laid out cube after cube: cube c owns events
// offsets[c] .. offsets[c+1]-1 (offsets = exclusive prefix sum of n_ev,
// vflowplus.py:67).
#pragma once

#include "abi_util.hpp"
#include "device.hpp"
#include "rows.hpp"

namespace mv {

struct StrataK {
  int n_strat;
  int n_cubes;
  const int32_t* n_ev;
  const int32_t* off;
};

// largest c with off[c] <= e (off strictly increasing, off[0] = 0)
__device__ __forceinline__ int find_cube(const int32_t* __restrict__ off, int n_cubes, int e) {
  int lo = 0, hi = n_cubes;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= e) lo = mid;
    else hi = mid;
  }
  return lo;
}

// find_cube of a wave-uniform event by the whole wave: every step probes 64
// evenly spaced offsets at once (three loads one after the other for 1e4
// cubes, where a binary search takes fourteen). The whole wave must be active.
__device__ __forceinline__ int find_cube_wave(const int32_t* __restrict__ off, int n_cubes, int e) {
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = n_cubes;  // off[lo] <= e < off[hi]
  while (hi - lo > 1) {
    const int stride = (hi - lo + 63) >> 6;
    const int c = lo + lane * stride;
    const uint64_t below = __ballot(c < hi && off[min(c, hi)] <= e);  // a prefix of the lanes, lane 0 always
    const int i = __popcll(below) - 1;
    hi = min(hi, lo + (i + 1) * stride);
    lo = lo + i * stride;
  }
  return lo;
}

// q = c / n, r = c % n for 0 <= c < 2^24 through an FP32 reciprocal and
// one correction step
__device__ __forceinline__ void divmod_small(int c, int n, float rn, int& q, int& r) {
  q = (int)((float)c * rn);
  r = c - q * n;
  if (r < 0) {
    --q;
    r += n;
  } else if (r >= n) {
    ++q;
    r -= n;
  }
}

// t / n rounded correctly, for a positive integer n and 0 <= t < 2^31, from
// y = 1 / n rounded correctly (one division per launch): q = t y is within
// 1.5 ulp; one FMA residual correction makes it faithful, and a second,
// from a faithful quotient and a correctly rounded reciprocal, gives the
// correctly rounded quotient (Markstein's theorem). Five FP64 operations
// instead of a full division per dimension.
__device__ __forceinline__ double div_by_strat(double t, double n, double y) {
  double q = t * y;
  double r = fma(-q, n, t);
  q = fma(r, y, q);
  r = fma(-q, n, t);
  return fma(r, y, q);
}

// Segmented suffix sum over the wave's (sorted) cube ids; the first lane of
// each segment adds the segment total to ress / ress2 (vflowplus.py:213-214).
__device__ __forceinline__ void segment_add(int cube, double v, double v2, double* __restrict__ ress,
                                            double* __restrict__ ress2) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double ov = __shfl_down(v, off, 64);
    const double ov2 = __shfl_down(v2, off, 64);
    const int oc = __shfl_down(cube, off, 64);
    if (lane + off < 64 && oc == cube) {
      v += ov;
      v2 += ov2;
    }
  }
  const int pc = __shfl_up(cube, 1, 64);
  const bool head = lane == 0 || pc != cube;
  if (head && cube >= 0) {
    unsafeAtomicAdd(&ress[cube], v);
    unsafeAtomicAdd(&ress2[cube], v2);
  }
}

// The samplers with a compile-time n_dim (sample.hip) for Philox draws and
// n_dim <= MV_FUSED_MAX_DIM; false, with nothing launched, for anything else.
bool launch_plain_sample(const StepK& s, bool mixed, void* x, hipStream_t stream);
bool launch_vegas_sample(const StepK& s, bool mixed, const double* grid, void* x, void* w, uint8_t* idx,
                         hipStream_t stream);
bool launch_vplus_sample(const StepK& s, bool mixed, const StrataK& st, const double* grid, void* x, void* w,
                         uint8_t* idx, int32_t* seg, hipStream_t stream);

// The training digests with pair histograms (digest.hip), for the n_dim that
// digest_pairs_takes. Return the workgroups launched.
bool digest_pairs_takes(int n_dim);
int launch_digest_pairs(const StepK& s, bool mixed, const void* f, int64_t fstride, const void* w, int64_t wstride,
                        const uint8_t* idx, const RowsK& R, hipStream_t stream);
int launch_vplus_digest_pairs(const StepK& s, bool mixed, const StrataK& st, const void* f, const void* w,
                              const uint8_t* idx, const int32_t* seg, double* ress, double* ress2, const RowsK& R,
                              hipStream_t stream);

// The fused VEGAS+ producer (vplus_kernel.hpp), compiled per (integrand
// family, train, n_dim, injected draws) for 1 <= n_dim <= MV_FUSED_MAX_DIM,
// one launcher per precision. Return the workgroups launched or a negative
// error.
int launch_vplus_fused_mixed(int family, bool train, const StepK& k, const StrataK& st,
                             const mv_integrand& fn, const double* grid, double* ress, double* ress2,
                             const RowsK& R, hipStream_t s);
int launch_vplus_fused_f64(int family, bool train, const StepK& k, const StrataK& st,
                           const mv_integrand& fn, const double* grid, double* ress, double* ress2,
                           const RowsK& R, hipStream_t s);

// The batched VEGAS+ producer (batch_vplus.hpp) of one precision: 0 or a
// negative status.
int launch_batch_vplus_mixed(const mv_batch_vplus_item* items, const mv_batch_tile* tiles, int n_tiles, int family,
                             int min_dim, int max_dim, const int32_t* draws, const double* grids,
                             const int32_t* n_ev, const int32_t* offsets, double* ress, double* ress2, double* rows,
                             int blocks, hipStream_t stream);
int launch_batch_vplus_f64(const mv_batch_vplus_item* items, const mv_batch_tile* tiles, int n_tiles, int family,
                           int min_dim, int max_dim, const int32_t* draws, const double* grids,
                           const int32_t* n_ev, const int32_t* offsets, double* ress, double* ress2, double* rows,
                           int blocks, hipStream_t stream);

}  // namespace mv
