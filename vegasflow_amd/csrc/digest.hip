// digest.hip - the training digests of the unfused path with pair histograms
// (fused_event.hpp): weighted sums of a scalar integrand's values and the bin
// histograms (vflow.py:414-430), for VegasFlowPlus with sums per hypercube
// (vflowplus.py:209-218), for n_dim kPairMinDim .. kPairMaxDim. Vector
// integrands and other n_dim run the per-wave histograms of vegas.hip and
// vplus.hip.
//
// One LDS add per event and pair of dimensions into the workgroup's pair
// tables (pair_cells(n_dim) doubles of LDS, one workgroup per CU) leaves the
// kernels to their reads of values, weights, bins and cubes and to a fixed
// part of 5 us (tables zeroed, marginals added to the rows). With few waves per
// CU and few events per wave the reads are bound by latency: a wave issues the
// loads of kDigestU trips before it uses the first, and reads an event's row of
// bins in the widest pieces that its length (a compile-time n_dim) allows.
// VEGAS+ takes contiguous runs of trips, so that most trips lie in the cube
// whose sums the lanes hold; the others go round robin (runs were 1 us slower).
// Kernel times against per-wave histograms with a segmented scan per trip:
// VEGAS+ FP64 d = 6, 1e6 events 19.3 -> 10.2 us; against pair tables with
// bins read by byte unless n_dim was a multiple of four: VegasFlow mixed
// d = 8, steps of 1e6 and 5e5 on average 8.7 -> 8.1 us.
#include <array>
#include <type_traits>
#include <utility>

#include "abi_util.hpp"
#include "device.hpp"
#include "fused_event.hpp"
#include "rows.hpp"
#include "vplus.hpp"

namespace mv {

namespace {

constexpr int kDigestU = 4;

// Bins of one event, D bytes at any address, in words of four.
template <int D>
__device__ __forceinline__ void load_bins(const uint8_t* __restrict__ p, uint32_t (&v)[(D + 3) / 4]) {
#pragma unroll
  for (int g = 0; g < D / 4; ++g) __builtin_memcpy(&v[g], p + 4 * g, 4);
  if constexpr ((D & 3) != 0) {
    uint32_t rest = 0;
    if constexpr ((D & 2) != 0) {
      uint16_t h;
      __builtin_memcpy(&h, p + (D & ~3), 2);
      rest = h;
    }
    if constexpr ((D & 1) != 0) rest |= (uint32_t)p[D - 1] << (8 * ((D - 1) & 3));
    v[D / 4] = rest;
  }
}

// Adds the events' sums per cube, one trip of 64 at a time; the cubes of a
// trip are in ascending order, as the sampler lays them out, but any order
// gives the right sums (a run of equal cubes is one segment). The sums of the
// last cube are held in the lanes until another one comes.
struct CubeSums {
  double* ress;
  double* ress2;
  int held = -1;
  double v = 0.0, v2 = 0.0;

  __device__ __forceinline__ void flush() {
    if (held < 0) return;
    const double a = wave_sum(v), b = wave_sum(v2);
    if ((threadIdx.x & 63) == 0) {
      unsafeAtomicAdd(&ress[held], a);
      unsafeAtomicAdd(&ress2[held], b);
    }
    held = -1;
  }

  // every lane has a cube; lanes without an event carry the last event's cube
  // and zeros
  __device__ __forceinline__ void add(int cube, double t, double t2) {
    const int first = __builtin_amdgcn_readfirstlane(cube);
    if (__ballot(cube != first) == 0) {
      if (held != first) {
        flush();
        held = first;
        v = v2 = 0.0;
      }
      v += t;
      v2 += t2;
      return;
    }
    const int lane = threadIdx.x & 63;
    const int before = __shfl_up(cube, 1, 64);
    uint64_t heads = __ballot(lane > 0 && before != cube);  // lanes that start a further segment
    if (held != first) {
      flush();
      v = v2 = 0.0;
    }
    if (__popcll(heads) > 4) {
      if (held >= 0) {
        flush();
        v = v2 = 0.0;
      }
      segment_add(cube, t, t2, ress, ress2);
      return;
    }
    held = first;
    int lo = 0;
    for (; heads; heads &= heads - 1) {
      const int hi = __builtin_ctzll(heads);
      const bool in = lane >= lo && lane < hi;
      v += in ? t : 0.0;
      v2 += in ? t2 : 0.0;
      flush();
      held = __builtin_amdgcn_readlane(cube, hi);
      v = v2 = 0.0;
      lo = hi;
    }
    v = lane >= lo ? t : 0.0;
    v2 = lane >= lo ? t2 : 0.0;
  }
};

template <typename FT, int D, bool CUBES>
__global__ __launch_bounds__(kPairBlock) void digest_pairs(StepK s, StrataK st, const FT* __restrict__ f,
                                                           int64_t fstride, const FT* __restrict__ w,
                                                           int64_t wstride, const uint8_t* __restrict__ idx,
                                                           const int32_t* __restrict__ seg,
                                                           double* __restrict__ ress,
                                                           double* __restrict__ ress2, RowsK R) {
  constexpr int U = kDigestU, NW = (D + 3) / 4;
  constexpr int cells = pair_cells(D);
  __shared__ __align__(16) double H[cells];
  for (int i = threadIdx.x; i < cells / 2; i += kPairBlock)
    reinterpret_cast<double2*>(H)[i] = make_double2(0.0, 0.0);
  __syncthreads();
  const uint32_t top = kBins - 1;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int64_t n = CUBES ? (int64_t)st.off[st.n_cubes] : s.n_events;
  const int64_t trips = (n + 63) >> 6, waves = (int64_t)gridDim.x * (kPairBlock / 64);
  // consecutive waves in different workgroups: a remainder of trips falls on all CUs
  const int64_t g0 = (int64_t)wave * gridDim.x + blockIdx.x;
  // VEGAS+: a contiguous run, whose cubes' sums stay in the lanes; else every waves-th trip
  const int64_t t0 = CUBES ? trip_of(g0, trips, waves) : g0;
  const int64_t t1 = CUBES ? trip_of(g0 + 1, trips, waves) : trips;
  const int64_t next = CUBES ? 1 : waves;
  const int64_t last = min(t1 * 64, n) - 1;  // the last event this wave may read
  double acc = 0.0, acc2 = 0.0;
  CubeSums cs{ress, ress2};
  for (int64_t t = t0; t < t1; t += U * next) {
    FT fv[U], wv[U];
    uint32_t v[U][NW];
    int cube[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // past the run or the events: the last event again, not counted
      const int64_t e = min((t + u * next) * 64 + lane, last);
      fv[u] = f[e * fstride];
      wv[u] = w[e * wstride];
      load_bins<D>(idx + e * D, v[u]);
      cube[u] = CUBES ? seg[e] : 0;
    }
    // all loads are issued above this point: without it the compiler sinks those
    // of a trip into the branch that uses them, one latency after the other
#pragma unroll
    for (int u = 0; u < U; ++u) {
      asm volatile("" : "+v"(fv[u]), "+v"(wv[u]), "+v"(cube[u]));
#pragma unroll
      for (int g = 0; g < NW; ++g) asm volatile("" : "+v"(v[u][g]));
    }
    double tmp[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      tmp[u] = 0.0;
      if (t + u * next < t1 && (t + u * next) * 64 + lane < n) {
        tmp[u] = (double)wv[u] * (double)fv[u];  // vflow.py:416, vflowplus.py:209
        const double t2 = tmp[u] * tmp[u];
        if (!CUBES) {
          acc += tmp[u];
          acc2 += t2;
        }
#pragma unroll
        for (int p = 0; p < (D + 1) / 2; ++p) {
          const uint32_t x = v[u][p >> 1] >> (16 * (p & 1));
          const uint32_t b0 = min(x & 0xffu, top);
          const uint32_t b1 = 2 * p + 1 < D ? min((x >> 8) & 0xffu, top) : 0u;
          lds_add(&H[p * kPairBins + b0 * kBins + b1], t2);
        }
      }
    }
    if (CUBES) {
      const int run = (int)min((int64_t)U, t1 - t);
      // not unrolled: the segments' code once, not kDigestU times
#pragma unroll 1
      for (int u = 0; u < run; ++u) {
        double a = tmp[0];
        int c = cube[0];
#pragma unroll
        for (int k = 1; k < U; ++k) {
          a = u == k ? tmp[k] : a;
          c = u == k ? cube[k] : c;
        }
        cs.add(c, a, a * a);
      }
    }
  }
  if (CUBES) cs.flush();
  finish_pairs<kPairBlock, !CUBES>(acc, acc2, H, D, group_row(R));
}

template <typename FT>
using Kernel = void (*)(StepK, StrataK, const FT*, int64_t, const FT*, int64_t, const uint8_t*, const int32_t*,
                        double*, double*, RowsK);

template <typename FT, bool CUBES, int... Ds>
constexpr std::array<Kernel<FT>, sizeof...(Ds)> kernels_of(std::integer_sequence<int, Ds...>) {
  return {&digest_pairs<FT, Ds + kPairMinDim, CUBES>...};
}

template <typename FT, bool CUBES>
int launch(const StepK& s, const StrataK& st, const void* f, int64_t fstride, const void* w, int64_t wstride,
           const uint8_t* idx, const int32_t* seg, double* ress, double* ress2, const RowsK& R, hipStream_t stream) {
  static constexpr auto kernels =
      kernels_of<FT, CUBES>(std::make_integer_sequence<int, kPairMaxDim - kPairMinDim + 1>{});
  return launch_producer<kPairBlock>(kernels[s.n_dim - kPairMinDim], s.n_events, 0, stream, s, st,
                                     static_cast<const FT*>(f), fstride, static_cast<const FT*>(w), wstride, idx,
                                     seg, ress, ress2, R);
}

}  // namespace

bool digest_pairs_takes(int n_dim) {
  return n_dim >= kPairMinDim && n_dim <= kPairMaxDim &&
         (size_t)pair_cells(n_dim) * sizeof(double) + 2 * kPairBlock / 64 * sizeof(double) <= max_lds_per_block();
}

int launch_digest_pairs(const StepK& s, bool mixed, const void* f, int64_t fstride, const void* w, int64_t wstride,
                        const uint8_t* idx, const RowsK& R, hipStream_t stream) {
  return mixed ? launch<float, false>(s, StrataK{}, f, fstride, w, wstride, idx, nullptr, nullptr, nullptr, R, stream)
               : launch<double, false>(s, StrataK{}, f, fstride, w, wstride, idx, nullptr, nullptr, nullptr, R,
                                       stream);
}

int launch_vplus_digest_pairs(const StepK& s, bool mixed, const StrataK& st, const void* f, const void* w,
                              const uint8_t* idx, const int32_t* seg, double* ress, double* ress2, const RowsK& R,
                              hipStream_t stream) {
  return mixed ? launch<float, true>(s, st, f, 1, w, 1, idx, seg, ress, ress2, R, stream)
               : launch<double, true>(s, st, f, 1, w, 1, idx, seg, ress, ress2, R, stream);
}

}  // namespace mv
