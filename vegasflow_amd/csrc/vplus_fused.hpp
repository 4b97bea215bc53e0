// vplus_fused.hpp - the event body and the per-wave run loop of the fused
// VEGAS+ producers (vflowplus.py:37-80 + 187-220, monte_carlo.py:249-275),
// shared by the single-integral kernel (vplus_kernel.hpp) and the batched one
// (batch_vplus.hpp).
//
// The position of a draw in dimension j, xn = ((h + u) 50) / n_strat
// (vflowplus.py:72), is base_j + (50 / n_strat) u with base_j = (50 / n_strat) h
// formed once per lane and trip (or kept while the wave stays in one cube):
// one FMA per dimension instead of an addition, a product and a division, and
// nearer to the real number (against 80-bit arithmetic at n_strat = 10 rms
// 2.2e-15 for 2.4e-15, at most 6.5e-15 for 9.8e-15). FP64 throughout in FP64;
// mixed: u = hi * 2^-32 and the position in FP64, FP32 map and integrand, FP64
// sums. Injected draws keep the reference's three roundings, the division by
// n_strat as div_by_strat (vplus.hpp), correctly rounded.
//
// Every wave owns one contiguous run of the iteration's events, taken 64 at
// a time, and holds the ends of the next 64 cubes and their weights (jacobian
// over n_ev) one per lane, reloaded when a trip reaches past them. A trip
// inside one cube needs no lookup; a trip across boundaries gets the boundary
// bits of its 64 events by one lane scatter, and each lane its cube by counting
// the bits up to it. The sums of the cube a trip ends in stay in the lanes
// until the wave leaves it (one wave reduction and one FP64 global atomic per
// sum, cube and wave).
#pragma once

#include <array>
#include <type_traits>
#include <utility>

#include "abi_util.hpp"
#include "device.hpp"
#include "fused_event.hpp"
#include "rows.hpp"
#include "vplus.hpp"

namespace mv {

// Training at kPairMinDim <= n_dim <= kPairMaxDim keeps pair histograms
// (fused_event.hpp) in kPairBlock-thread workgroups: the events of a wave
// lie in one or two hypercubes, so per-dimension histograms would take most
// adds of a wave on the few bins a cube spans; the pair tables spread them
// over up to 2500 cells and need one add per pair of dimensions.
template <bool TRAIN, int D>
constexpr bool vplus_pairs() {
  return TRAIN && D >= kPairMinDim && D <= kPairMaxDim;
}
template <bool TRAIN, int D>
constexpr int vplus_block() {
  return vplus_pairs<TRAIN, D>() ? kPairBlock : kBlock;
}

namespace {

// One map table entry per (dimension, bin), 16 bytes read at once: (P, Q) in
// FP64 (the Jacobian from the slopes Q, JacGroups), (P, Q, W) in FP32.
template <bool MIXED>
using VplusEntry = typename std::conditional<MIXED, float4, double2>::type;

// Builds the map table (BS threads); integration limits folded in when xmin.
template <bool MIXED, int FAM, int BS>
__device__ __forceinline__ void vplus_table(const mv_integrand& fn, const double* __restrict__ grid, int d,
                                            const double* xmin, const double* xdelta, VplusEntry<MIXED>* tab) {
  for (int i = threadIdx.x; i < d * kBins; i += BS) {
    const int j = i / kBins, b = i - j * kBins;
    const double lo = grid[j * (kBins + 1) + b];
    const double dx = grid[j * (kBins + 1) + b + 1] - lo;  // vflow.py:73
    double P = lo, Q = dx;
    if (xmin) {  // monte_carlo.py:273
      P = xmin[j] + lo * xdelta[j];
      Q = dx * xdelta[j];
    }
    Integrand<double, FAM>::fold(fn, j, P, Q);
    if constexpr (MIXED)
      tab[i] = make_float4((float)P, (float)Q, (float)(dx * kFBins), 0.0f);  // vflow.py:78
    else
      tab[i] = make_double2(P, Q);
  }
}

// What the event body needs of the stratification: digits of a cube by
// multiplication (q = c / n as mulhi(c, magic) >> shift, exact for c < 2^24:
// magic = floor(2^(32 + shift) / n) + 1 exceeds 2^(32 + shift) / n by at most
// 1, and c < 2^24 <= 2^(32 + shift) / n) and the FP64 position constants.
template <bool MIXED, bool INJ>
struct StrataPos {
  int n;
  uint32_t magic, shift;
  double per_cube, per_draw, first;  // xn = per_cube h + first + per_draw (draw)
  __device__ __forceinline__ explicit StrataPos(int n_strat) : n(n_strat) {
    // shift = max(0, ceil(log2 n) - 8): 2^(24 + ceil(log2 n)) <= 2^(32 + shift)
    const int l = n > 1 ? 32 - __clz(n - 1) : 0;
    shift = l > 8 ? (uint32_t)(l - 8) : 0u;
    // the quotient's fraction is a multiple of 1 / n > 2^-25 and FP64 holds at
    // least 28 bits of it, so floor() of the rounded quotient is exact
    magic = (uint32_t)((uint64_t)(__longlong_as_double((int64_t)(1023 + 32 + shift) << 52) / (double)n) + 1u);
    per_cube = kFBins / (double)n;
    per_draw = per_cube * (MIXED ? 0x1p-32 : kSpan);
    first = MIXED ? 0.0 : per_cube * kTechCut;
  }
};

// base[j]: position of the lower corner of hypercube ``cube`` in dimension j
// (last dimension fastest, vflowplus.py:126-128); injected draws: the corner's
// digit itself.
template <int D, bool MIXED, bool INJ>
__device__ __forceinline__ void cube_base(int cube, const StrataPos<MIXED, INJ>& sp, double (&base)[D]) {
  uint32_t c = (uint32_t)cube;
#pragma unroll
  for (int j = D - 1; j >= 0; --j) {
    uint32_t h = c;
    if (j > 0) {
      const uint32_t q = __umulhi(c, sp.magic) >> sp.shift;
      h = c - __umul24(q, (uint32_t)sp.n);
      c = q;
    }
    base[j] = INJ ? (double)h : fma((double)h, sp.per_cube, sp.first);
  }
}

// One event with the corner positions ``base`` of its cube and the weight
// factor ``wev`` = jacobian / n_ev: returns tmp = w f / n_ev and, when
// training, adds tmp^2 to the histograms wh (the workgroup's pair tables if
// PAIRS, else the wave's per-dimension histogram). INJ: the draws come from
// s.inject (event i) instead of Philox.
template <int FAM, bool TRAIN, bool MIXED, int D, bool INJ, bool PAIRS, typename T>
__device__ __forceinline__ double vplus_event(Integrand<T, FAM>& F, const StepK& s, uint32_t ev_hi, uint32_t draw,
                                              int64_t i, const StrataPos<MIXED, INJ>& sp, const double (&base)[D],
                                              const VplusEntry<MIXED>* tab, const JacGroups<double>& cs,
                                              double wev, double* wh) {
  constexpr int groups = (D + 3) / 4;
  const uint32_t c0w = s.ev_lo + (uint32_t)i;
  F.begin();
  T w = (T)1;
  uint32_t pk[4] = {0u, 0u, 0u, 0u};
  uint32_t cell[kPairMaxDim / 2 + 1];
#pragma unroll
  for (int p = 0; p <= kPairMaxDim / 2; ++p) cell[p] = 0u;
#pragma unroll
  for (int g = 0; g < groups; ++g) {
    uint4 hw4 = make_uint4(0, 0, 0, 0), lw4 = make_uint4(0, 0, 0, 0);
    if (!INJ) {
      hw4 = philox(c0w, ev_hi, draw, (uint32_t)g, s.key);
      if (!MIXED) lw4 = philox(c0w, ev_hi, draw, (uint32_t)(groups + g), s.key);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = 4 * g + q;
      if (j < D) {
        double xn;
        if (INJ) {
          const double u = MIXED ? (double)static_cast<const uint32_t*>(s.inject)[i * D + j] * 0x1p-32
                                 : static_cast<const double*>(s.inject)[i * D + j];
          xn = div_by_strat((base[j] + u) * kFBins, (double)sp.n, 1.0 / (double)sp.n);  // vflowplus.py:72
        } else if (MIXED) {
          xn = fma((double)word(hw4, q), sp.per_draw, base[j]);
        } else {
          xn = fma(draw_mantissa(word(hw4, q), word(lw4, q)) - 1.0, sp.per_draw, base[j]);
        }
        // at n_dim >= 2 n_strat < 2^12, so xn < 50 (1 - 2^-32 / n_strat) stays
        // below 50 by more than its rounding
        const int ind = INJ || D == 1 ? clamp_bin((int)xn) : (int)xn;
        const double frac = __builtin_amdgcn_fract(xn);
        if constexpr (MIXED) {
          const float4 t = tab[j * kBins + ind];
          F.add_folded(j, fmaf(t.y, (float)frac, t.x));
          w = w * t.z;
        } else {
          const double2 t = tab[j * kBins + ind];
          F.add_folded(j, fma(t.y, frac, t.x));
          w = w * t.y;  // vflow.py:78, with cs
          if (q & 1) w = w * cs.g[2 * g + (q >> 1)];
        }
        if (TRAIN && PAIRS) cell[2 * g + (q >> 1)] += (uint32_t)ind * (q & 1 ? 8u : 8u * kBins);
        if (TRAIN && !PAIRS) pk[g] |= (uint32_t)ind << (8 * q);
      }
    }
  }
  if constexpr (!MIXED && (D & 1)) w = w * cs.g[D >> 1];
  // vflowplus.py:77, monte_carlo.py:270-274, vflowplus.py:209
  const double tmp = ((double)w * wev) * (double)F.value();
  if (TRAIN && PAIRS)
    pair_cell_adds(wh, cell, D, tmp * tmp);
  else if (TRAIN)
    hist_adds(wh, pk, D, tmp * tmp);
  return tmp;
}

// Adds the wave's sums of v and v2 to ress[cube], ress2[cube]: the two sums
// side by side, v in the lower 32 lanes and v2 in the upper ones after one
// exchange of the halves, then within each half as in wave_sum. One atomic
// instruction from lanes 31 and 63.
__device__ __forceinline__ void cube_flush(int cube, double v, double v2, double* __restrict__ ress,
                                           double* __restrict__ ress2) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v2), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v2), false, false);
  double a = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  a += dpp_f64<0xB1, 0xF, true>(a);   // quad_perm [1, 0, 3, 2]
  a += dpp_f64<0x4E, 0xF, true>(a);   // quad_perm [2, 3, 0, 1]
  a += dpp_f64<0x124, 0xF, true>(a);  // row_ror 4
  a += dpp_f64<0x128, 0xF, true>(a);  // row_ror 8
  a += dpp_f64<0x142, 0xA>(a);        // row_bcast 15 into rows 1 and 3
  const int lane = threadIdx.x & 63;
  if ((lane & 31) == 31) unsafeAtomicAdd((lane & 32 ? ress2 : ress) + cube, a);
}

// Inclusive sums of v within segments of lanes; seg: the first lane of this
// lane's segment. The whole wave must be active.
__device__ __forceinline__ double segment_scan(double v, int seg) {
  const int lane = threadIdx.x & 63;
  auto take = [&](double moved, bool same) { v += same ? moved : 0.0; };
  take(dpp_f64<0x111, 0xF>(v), lane - 1 >= seg);         // row_shr 1
  take(dpp_f64<0x112, 0xF>(v), lane - 2 >= seg);         // row_shr 2
  take(dpp_f64<0x114, 0xF>(v), lane - 4 >= seg);         // row_shr 4
  take(dpp_f64<0x118, 0xF>(v), lane - 8 >= seg);         // row_shr 8
  take(dpp_f64<0x142, 0xA>(v), (lane & 0x30) - 1 >= seg);  // row_bcast 15 into rows 1 and 3
  take(dpp_f64<0x143, 0xC>(v), seg <= 31);               // row_bcast 31 into rows 2 and 3
  return v;
}

// The wave's run of events first .. end - 1, 64 per trip, into the per-cube
// sums ress, ress2 (vflowplus.py:213-214) and the histograms. ``c0``: the
// cube of event ``first`` (find_cube_wave). Measured on the two-Gaussian
// mixture, d = 4, training: see vplus_kernel.hpp.
template <int FAM, bool TRAIN, bool MIXED, int D, bool INJ, bool PAIRS = vplus_pairs<TRAIN, D>(), typename T>
__device__ __forceinline__ void vplus_run(Integrand<T, FAM>& F, const StepK& s, uint32_t draw, const StrataK& st,
                                          const StrataPos<MIXED, INJ>& sp, int64_t first, int64_t end, int c0,
                                          const VplusEntry<MIXED>* tab, const JacGroups<double>& cs,
                                          double wscale, double* wh, double* __restrict__ ress,
                                          double* __restrict__ ress2) {
  if (first >= end) return;  // wave-uniform
  const int lane = threadIdx.x & 63;
  // the window: lane l holds the end of cube cw + l and wscale / its n_ev
  int cw = 0, wend = 0, k = 0;  // k: the trip's first cube is cw + k
  double wr = 0.0;
  const auto refill = [&](int c) {
    const bool in = c + lane < st.n_cubes;
    cw = c;
    k = 0;
    wend = in ? st.off[c + lane + 1] : 0x7fffffff;
    wr = wscale / (double)(in ? st.n_ev[c + lane] : 1);
  };
  refill(c0);
  int held = -1;  // the cube whose sums the lanes hold in hv, hv2
  double hv = 0.0, hv2 = 0.0;
  int based = -1;  // the cube that every lane's base and rn belong to, or -1
  double base[D], rn = 0.0;
  // one workgroup of 16 waves per CU (paced_trips): 95.1 -> 87.8 us mixed, 2e7
  // events, 19.5 -> 18.7 us FP64, 1e6 events
  constexpr bool PACED = PAIRS;
  int left = (int)((end - first + 63) >> 6), change = left;
  const int todo = left;
  // pieces of the run that do not cross a multiple of 2^32 in the event
  // counter (one, unless the run crosses it)
  for (int64_t from = first, to; from < end; from = to) {
    const uint64_t ge = (uint64_t)s.event_offset + (uint64_t)from;
    to = min(end, from + (int64_t)((1ull << 32) - (ge & 0xffffffffull)));
    const uint32_t ev_hi = (uint32_t)(ge >> 32);
    for (int64_t trip = from; trip < to; trip += 64) {
      if (PACED && left-- <= change) change = pace(todo, left + 1);
      const int b = (int)trip;                          // events of an iteration < 2^31
      const int n_live = (int)min((int64_t)64, to - trip);
      const int last = b + (n_live - 1);
      int e0 = __builtin_amdgcn_readlane(wend, k);  // the end of the first event's cube
      while (e0 <= b) {
        if (++k == 64) refill(cw + 64);
        e0 = __builtin_amdgcn_readlane(wend, k);
      }
      const bool live = lane < n_live;
      const bool inside = last < e0;
      int cube = cw + k, idx = k;
      uint64_t mask = 0;  // bit i: event b + i is the first of its cube (i >= 1)
      bool known = true;
      if (inside) {
        if (based != cube) {
          rn = bcast_lane(wr, k);
          cube_base<D>(cube, sp, base);
          based = cube;
        }
      } else {
        if (__builtin_amdgcn_readlane(wend, 63) <= last && cw + 64 < st.n_cubes) refill(cw + k);
        const int at = wend - b;
        const bool part = at >= 1 && at < n_live;
        mask = __ballot(__builtin_amdgcn_ds_permute(part ? at << 2 : 0, part ? 1 : 0) != 0) & ~1ull;
        // not so with empty cubes (two ends at one event, or a window that
        // still ends within the trip): each lane then searches the offsets
        known = __popcll(__ballot(part)) == __popcll(mask) &&
                (__builtin_amdgcn_readlane(wend, 63) > last || cw + 64 >= st.n_cubes);
        if (known) {
          idx = k + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 33),
                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)(mask >> 1), 0u));
          cube = cw + idx;
          rn = __shfl(wr, idx, 64);
        } else {
          cube = find_cube(st.off, st.n_cubes, b + min(lane, n_live - 1));
          rn = wscale / (double)st.n_ev[cube];
        }
        cube_base<D>(cube, sp, base);
        based = -1;
      }
      double tmp = 0.0;
      if (live)
        tmp = vplus_event<FAM, TRAIN, MIXED, D, INJ, PAIRS>(F, s, ev_hi, draw, (int64_t)b + lane, sp, base, tab, cs,
                                                            rn, wh);
      const double tmp2 = tmp * tmp;
      if (!known) {
        if (held >= 0) cube_flush(held, hv, hv2, ress, ress2);
        held = -1;
        hv = hv2 = 0.0;
        segment_add(cube, tmp, tmp2, ress, ress2);
        // the next trip starts in the cube of this trip's last event or later
        refill(__builtin_amdgcn_readlane(cube, n_live - 1));
        continue;
      }
      if (held != cw + k) {
        if (held >= 0) cube_flush(held, hv, hv2, ress, ress2);
        held = cw + k;
        hv = hv2 = 0.0;
      }
      if (inside) {
        hv += tmp;
        hv2 += tmp2;
        continue;
      }
      // the first cube ends here: its sums go out, the last cube's are held,
      // and those of any cube between are added at once
      int lo = __builtin_ctzll(mask);
      cube_flush(held, hv + (lane < lo ? tmp : 0.0), hv2 + (lane < lo ? tmp2 : 0.0), ress, ress2);
      const int n = __popcll(mask);
      if (n > 4) {
        const int prev = __shfl(wend, idx - 1, 64) - b;  // read where idx > k
        const int seg = idx > k ? prev : 0;
        const double a = segment_scan(tmp, seg), a2 = segment_scan(tmp2, seg);
        // the last lane of every cube between the first and the last one
        if (lane >= lo && lane < 63 && ((mask >> (lane + 1)) & 1)) {
          unsafeAtomicAdd(&ress[cube], a);
          unsafeAtomicAdd(&ress2[cube], a2);
        }
        lo = 63 - __builtin_clzll(mask);
      } else {
        for (uint64_t m = mask & (mask - 1); m; m &= m - 1) {
          const int hi = __builtin_ctzll(m);
          const bool in = lane >= lo && lane < hi;
          cube_flush(++held, in ? tmp : 0.0, in ? tmp2 : 0.0, ress, ress2);
          lo = hi;
        }
      }
      k += n;
      held = cw + k;
      hv = lane >= lo ? tmp : 0.0;
      hv2 = lane >= lo ? tmp2 : 0.0;
    }
  }
  if (held >= 0) cube_flush(held, hv, hv2, ress, ress2);
}

}  // namespace

}  // namespace mv
