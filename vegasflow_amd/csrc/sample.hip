// sample.hip - the samplers of the unfused path for Philox draws and n_dim
// 1 .. MV_FUSED_MAX_DIM: points, weights, bins and hypercubes of PlainFlow
// (monte_carlo.py:264-274), VegasFlow (vflow.py:87-126 + 33-83) and
// VegasFlowPlus (vflowplus.py:37-80). Injected draws and larger n_dim run the
// runtime-n_dim kernels of vegas.hip and vplus.hip, which give the same values
// bit by bit: FP64 keeps the reference's operation order, mixed precision is
// mixed_mirrored and an FP32 map.
//
// Bound by the draws and the writes (n_dim + 1 values, n_dim bins and, VEGAS+,
// a cube per event). Every wave works alone: it draws 64 consecutive events,
// stages their points and bins in its own part of the LDS and stores its
// contiguous piece of the row-major outputs, 16 bytes per lane, with no
// workgroup barrier between drawing and storing. Rows of the stage are an odd
// number of elements apart, so neither side conflicts on the LDS banks. The map
// is a table in LDS (one read per dimension instead of two gathers from the
// grid), and n_dim is a compile-time value, so the digits, the draws and the
// stage's addresses need no loops. Trips of VegasFlow and PlainFlow go round
// robin over the waves, so that the stores of all waves stay together (a
// contiguous run per wave was 10-20 % slower); VEGAS+ takes runs, because a
// trip's cube is searched from the last one's. Non-temporal stores made the
// sampler 4 % faster and the integrand that reads its points slower by more.
// Kernel times against the workgroup-staged kernels (VEGAS+: direct stores and
// a binary search per event): VegasFlow FP64 d = 6, 1e6 events 21.6 -> 15.8 us
// (3.9 TB/s); mixed d = 8, steps of 1e6 and 5e5 on average 17.3 -> 12.9 us;
// VEGAS+ FP64 d = 6, 1e6 events 42.9 -> 22.7 us.
#include <array>
#include <utility>

#include "abi_util.hpp"
#include "device.hpp"
#include "fused_event.hpp"
#include "rows.hpp"
#include "vplus.hpp"

namespace mv {

namespace {

constexpr int kPlain = 0, kVegas = 1, kVplus = 2;

// Stage rows: an odd number of elements.
template <int D>
constexpr int stage_row() {
  return D | 1;
}

// Element e of the stage's rows (row stride S) in row-major order.
template <int D, int S>
__device__ __forceinline__ int stage_at(int e) {
  return S == D ? e : (int)((uint32_t)e / D * S + (uint32_t)e % D);
}

// The n D elements of the stage's first n rows to the contiguous dst: for a
// whole trip and a 16-byte aligned dst (``wide``) 16 bytes per lane and store,
// at LDS addresses that do not change from trip to trip, else by element.
template <typename T, int D, int S>
__device__ __forceinline__ void store_rows(const T* st, T* __restrict__ dst, int n, bool wide) {
  constexpr int V = 16 / sizeof(T), vecs = 64 * D / V;
  const int lane = threadIdx.x & 63;
  if (wide && n == 64) {
#pragma unroll
    for (int k0 = 0; k0 < vecs; k0 += 64) {
      const int k = k0 + lane;
      if (k0 + 64 <= vecs || k < vecs) {
        struct alignas(16) Vec {
          T v[V];
        } o;
        if constexpr (S == D) {
          o = *reinterpret_cast<const Vec*>(st + k * V);
        } else if constexpr (D % V == 0) {  // a vector lies within one row
          const T* p = st + stage_at<D, S>(k * V);
#pragma unroll
          for (int i = 0; i < V; ++i) o.v[i] = p[i];
        } else {
#pragma unroll
          for (int i = 0; i < V; ++i) o.v[i] = st[stage_at<D, S>(k * V + i)];
        }
        *reinterpret_cast<Vec*>(dst + k * V) = o;
      }
    }
  } else {
    for (int e = lane; e < n * D; e += 64) dst[e] = st[stage_at<D, S>(e)];
  }
}

// The wave's LDS writes before, its reads after: one wave's LDS operations are
// in order, the fence keeps the compiler to that.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Largest c with off[c] <= e and its n_ev, for lanes whose events all lie at
// or after off[c0] (c0 wave-uniform): binary lifting over the 64 offsets from
// c0, held one per lane. 64 consecutive events starting in cube c0 lie in that
// window when cubes hold at least one event; a lane that reaches the window's
// last cube (only with empty cubes before it) searches all offsets instead.
__device__ __forceinline__ int window_cube(const StrataK& st, int c0, int e, int& nev) {
  const int lane = threadIdx.x & 63;
  const int lim = min(st.n_cubes - c0, 64);
  const int ok = lane < lim ? st.off[c0 + lane] : 0x7fffffff;
  const int nk = lane < lim ? st.n_ev[c0 + lane] : 0;
  int lo = 0;
#pragma unroll
  for (int stp = 32; stp >= 1; stp >>= 1) {
    const int probe = lo + stp;  // <= 63
    const int v = __shfl(ok, probe, 64);
    if (probe < lim && v <= e) lo = probe;
  }
  nev = __shfl(nk, lo, 64);
  int c = c0 + lo;
  if (lo == 63) {
    c = find_cube(st.off, st.n_cubes, e);
    nev = st.n_ev[c];
  }
  return c;
}

template <bool MIXED, int KIND, bool LIMITS, int D>
__global__ __launch_bounds__(kBlock) void sample(StepK s, StrataK st, const double* __restrict__ grid,
                                                 void* __restrict__ xo_, void* __restrict__ wo_,
                                                 uint8_t* __restrict__ io, int32_t* __restrict__ so,
                                                 int64_t events) {
  using T = typename std::conditional<MIXED, float, double>::type;
  constexpr int S = stage_row<D>(), groups = (D + 3) / 4;
  constexpr int nb = KIND == kPlain ? 0 : D * kBins;
  // {lower edge, width} per bin; mixed {edge, width, Jacobian factor} as floats
  using Entry = typename std::conditional<MIXED, float4, double2>::type;
  __shared__ __align__(16) Entry tab[nb > 0 ? nb : 1];
  __shared__ __align__(16) T xstage[kWaves * 64 * S];
  __shared__ __align__(16) uint8_t bstage[KIND == kPlain ? 16 : kWaves * 64 * D];
  T* xo = static_cast<T*>(xo_);
  T* wo = static_cast<T*>(wo_);
  const uint32_t draw = draw_of(s);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  if constexpr (KIND != kPlain) {
    for (int i = threadIdx.x; i < nb; i += kBlock) {
      const int j = i / kBins, b = i - j * kBins;
      const double lo = grid[j * (kBins + 1) + b];
      const double dx = grid[j * (kBins + 1) + b + 1] - lo;  // vflow.py:73
      if constexpr (MIXED)
        tab[i] = make_float4((float)lo, (float)dx, (float)(dx * kFBins), 0.0f);
      else
        tab[i] = make_double2(lo, dx);
    }
    __syncthreads();
  }
  // 64 rows are a multiple of 16 bytes: the base decides for every trip
  const bool xwide = ((uintptr_t)xo & 15u) == 0, iwide = ((uintptr_t)io & 15u) == 0;
  T* xs = xstage + wave * 64 * S;
  uint8_t* bs = bstage + (KIND == kPlain ? 0 : wave * 64 * D);
  const double fstrat = KIND == kVplus ? (double)st.n_strat : 1.0, ystrat = 1.0 / fstrat;
  const float rn = 1.0f / (float)fstrat;
  const int64_t n = KIND == kVplus ? (int64_t)st.off[st.n_cubes] : events;
  // this wave's trips of 64 events: VEGAS+ a contiguous run (the cube of one
  // trip is near that of the last), else every waves-th trip, which keeps the
  // stores of all waves together
  const int64_t trips = (n + 63) >> 6, waves = (int64_t)gridDim.x * kWaves;
  const int64_t g0 = KIND == kVplus ? (int64_t)blockIdx.x * kWaves + wave : (int64_t)wave * gridDim.x + blockIdx.x;
  const int64_t t0 = KIND == kVplus ? trip_of(g0, trips, waves) : g0;
  const int64_t t1 = KIND == kVplus ? trip_of(g0 + 1, trips, waves) : trips;
  const int64_t next = KIND == kVplus ? 1 : waves;
  int cube0 = 0;  // VEGAS+: the cube of the trip's first event
  if (KIND == kVplus && t0 < t1) cube0 = find_cube_wave(st.off, st.n_cubes, (int)(t0 * 64));
  for (int64_t t = t0; t < t1; t += next) {
    const int64_t base = t * 64;
    const int live = (int)min((int64_t)64, n - base);
    const int l = min(lane, live - 1);  // lanes past the end repeat the last event, and store nothing
    const uint64_t ge = (uint64_t)s.event_offset + (uint64_t)(base + l);
    const uint32_t c0 = (uint32_t)ge, c1 = (uint32_t)(ge >> 32);
    int cube = 0, nev = 1;
    uint32_t h[KIND == kVplus ? D : 1];
    if constexpr (KIND == kVplus) {
      cube = window_cube(st, cube0, (int)base + l, nev);
      cube0 = __builtin_amdgcn_readlane(cube, 63);
      int rest = cube;
#pragma unroll
      for (int j = D - 1; j >= 0; --j) {
        int q = 0, r = rest;
        if (j > 0) divmod_small(rest, st.n_strat, rn, q, r);
        h[j] = (uint32_t)r;
        rest = q;
      }
    }
    T w = (T)1;
    uint32_t bins[groups] = {};
    const auto group = [&](int g) {
      const uint4 hw = philox(c0, c1, draw, (uint32_t)g, s.key);
      uint4 lw = make_uint4(0, 0, 0, 0);
      if (!MIXED) lw = philox(c0, c1, draw, (uint32_t)(groups + g), s.key);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = 4 * g + q;
        if (j < D) {
          T x;
          int ind = 0;
          if constexpr (KIND == kPlain) {
            if constexpr (MIXED)
              x = fmaf((float)(word(hw, q) >> 9), 0x1p-23f, 0x1p-24f);
            else
              x = draw_f64(word(hw, q), word(lw, q));
          } else if constexpr (MIXED) {
            float frac;
            if constexpr (KIND == kVplus) {
              const double u = (double)word(hw, q) * 0x1p-32;
              const double xn = div_by_strat(((double)h[j] + u) * kFBins, fstrat, ystrat);
              ind = D == 1 ? clamp_bin((int)xn) : (int)xn;
              frac = (float)__builtin_amdgcn_fract(xn);
            } else {
              float f1;
              ind = kBins - 1 - mixed_mirrored(word(hw, q), f1);
              frac = 2.0f - f1;  // exact
            }
            const float4 e = tab[j * kBins + ind];
            x = fmaf(e.y, frac, e.x);
            w = w * e.z;
          } else {
            const double u = draw_f64(word(hw, q), word(lw, q));
            const double xn = KIND == kVplus ? div_by_strat(((double)h[j] + u) * kFBins, fstrat, ystrat)
                                             : kFBins * (1.0 - u);  // vflowplus.py:72, vflow.py:117
            ind = D == 1 ? clamp_bin((int)xn) : (int)xn;            // vflow.py:67
            const double2 e = tab[j * kBins + ind];
            x = e.x + e.y * __builtin_amdgcn_fract(xn);  // two roundings, as vflow.py:75-76
            w = w * (e.y * kFBins);            // vflow.py:78
          }
          if constexpr (LIMITS) {  // monte_carlo.py:273
            if constexpr (MIXED)
              x = fmaf(x, (float)s.xdelta[j], (float)s.xmin[j]);
            else
              x = s.xmin[j] + x * s.xdelta[j];
          }
          xs[lane * S + j] = x;
          bins[g] |= (uint32_t)ind << (8 * q);
        }
      }
    };
    // VEGAS+ multiplies the weights of the last group of four dimensions first,
    // as its runtime-n_dim kernel does
    if constexpr (KIND == kVplus) {
#pragma unroll
      for (int g = groups - 1; g >= 0; --g) group(g);
    } else {
#pragma unroll
      for (int g = 0; g < groups; ++g) group(g);
    }
    if (KIND != kPlain && io) {
#pragma unroll
      for (int j = 0; j < D;) {
        uint8_t* b = bs + lane * D + j;
        const uint32_t v = bins[j >> 2] >> (8 * (j & 3));
        if (D % 4 == 0) {
          *reinterpret_cast<uint32_t*>(b) = v;
          j += 4;
        } else if (D % 2 == 0) {
          *reinterpret_cast<uint16_t*>(b) = (uint16_t)v;
          j += 2;
        } else {
          *b = (uint8_t)v;
          j += 1;
        }
      }
    }
    wave_lds_order();
    store_rows<T, D, S>(xs, xo + base * D, live, xwide);
    if (KIND != kPlain && io) store_rows<uint8_t, D, D>(bs, io + base * D, live, iwide);
    if (KIND != kPlain && lane < live) {
      const double xj = LIMITS ? s.xjac * s.xdeltajac : s.xjac;
      if constexpr (KIND == kVplus) {
        if constexpr (MIXED) {
          wo[base + lane] = (float)(((double)w / (double)nev) * xj);
        } else {
          double wt = (w / (double)nev) * s.xjac;  // vflowplus.py:77, monte_carlo.py:270
          if (LIMITS) wt = wt * s.xdeltajac;
          wo[base + lane] = wt;
        }
        if (so) so[base + lane] = cube;
      } else if constexpr (MIXED) {
        wo[base + lane] = w * (float)xj;
      } else {
        double wt = w * s.xjac;  // monte_carlo.py:270
        if (LIMITS) wt = wt * s.xdeltajac;
        wo[base + lane] = wt;
      }
    }
    wave_lds_order();
  }
}

using Kernel = void (*)(StepK, StrataK, const double*, void*, void*, uint8_t*, int32_t*, int64_t);

template <bool MIXED, int KIND, bool LIMITS, int... Ds>
constexpr std::array<Kernel, sizeof...(Ds)> kernels_of(std::integer_sequence<int, Ds...>) {
  return {&sample<MIXED, KIND, LIMITS, Ds + 1>...};
}

template <int KIND>
Kernel kernel_of(bool mixed, bool limits, int d) {
  using Dims = std::make_integer_sequence<int, MV_FUSED_MAX_DIM>;
  static constexpr std::array<Kernel, MV_FUSED_MAX_DIM> k[2][2] = {
      {kernels_of<false, KIND, false>(Dims{}), kernels_of<false, KIND, true>(Dims{})},
      {kernels_of<true, KIND, false>(Dims{}), kernels_of<true, KIND, true>(Dims{})}};
  return k[mixed][limits][d - 1];
}

// false: the runtime-n_dim kernels take the call
bool launch(Kernel (*kernel)(bool, bool, int), const StepK& s, bool mixed, const StrataK& st, const double* grid, void* x,
            void* w, uint8_t* idx, int32_t* seg, hipStream_t stream) {
  if (s.inject || s.n_dim < 1 || s.n_dim > MV_FUSED_MAX_DIM) return false;
  launch_producer<kBlock>(kernel(mixed, s.xmin != nullptr, s.n_dim), s.n_events, 0, stream, s, st, grid, x, w, idx, seg, s.n_events);
  return true;
}

}  // namespace

bool launch_plain_sample(const StepK& s, bool mixed, void* x, hipStream_t stream) {
  return launch(kernel_of<kPlain>, s, mixed, StrataK{}, nullptr, x, nullptr, nullptr, nullptr, stream);
}

bool launch_vegas_sample(const StepK& s, bool mixed, const double* grid, void* x, void* w, uint8_t* idx,
                         hipStream_t stream) {
  return launch(kernel_of<kVegas>, s, mixed, StrataK{}, grid, x, w, idx, nullptr, stream);
}

bool launch_vplus_sample(const StepK& s, bool mixed, const StrataK& st, const double* grid, void* x, void* w,
                         uint8_t* idx, int32_t* seg, hipStream_t stream) {
  return launch(kernel_of<kVplus>, s, mixed, st, grid, x, w, idx, seg, stream);
}

}  // namespace mv
