// plain_fused.hip - the fused PlainFlow producer (plain.py:18-35,
// monte_carlo.py:249-275): uniform points from Philox, the built-in
// integrand, w f sums. Compiled per (integrand family, precision, n_dim,
// injected draws) for n_dim 1..MV_FUSED_MAX_DIM, where the event body is
// straight-line code; a runtime-n_dim instance takes larger n_dim (families
// that allow it).
#include <array>
#include <type_traits>
#include <utility>

#include "abi_util.hpp"
#include "device.hpp"
#include "rows.hpp"

namespace mv {

// One draw per dimension as FP64 integrand coordinate y_j = P_j + Q_j r, r the
// draw's 52 bits in [0, 1) (exact), for a compile-time n_dim: u = TECH_CUT +
// span r, the integration limits (LIM, monte_carlo.py:271-274) and the
// integrand's own affine map (Integrand::fold) in one FMA, where the separate
// steps take up to seven operations (d = 8 Gaussian: 248 -> 207 VALU
// instructions per 64 events, 75.2 -> 65.5 us at 1e7 events). P_j is held in scalar registers; without
// limits Q_j is the same for every dimension.
template <int FAM, int D, bool LIM>
struct PlainMap {
  double P[D], Q[LIM ? D : 1];
  __device__ __forceinline__ PlainMap(const StepK& s, const mv_integrand& fn) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      double p = kTechCut, q = kSpan;
      if (LIM) {
        p = s.xmin[j] + kTechCut * s.xdelta[j];
        q = kSpan * s.xdelta[j];
      }
      Integrand<double, FAM>::fold(fn, j, p, q);
      P[j] = bcast_lane(p, 0);
      if (LIM || j == 0) Q[LIM ? j : 0] = q;
    }
  }
  __device__ __forceinline__ double operator()(int j, uint32_t hi, uint32_t lo) const {
    return fma(draw_mantissa(hi, lo) - 1.0, Q[LIM ? j : 0], P[j]);
  }
};

// The FP64 events of this thread for a compile-time n_dim and Philox draws.
template <int FAM, int D, bool LIM>
__device__ __forceinline__ void plain_events_f64(const StepK& s, const mv_integrand& fn, uint32_t draw,
                                                 Integrand<double, FAM>& F, double wt, double& acc,
                                                 double& acc2) {
  const PlainMap<FAM, D, LIM> map(s, fn);
  constexpr int groups = (D + 3) / 4;
  event_trips<kBlock>(s, [&](uint32_t c0) {
    F.begin();
#pragma unroll
    for (int g = 0; g < groups; ++g) {
      const uint4 h = philox(c0, s.ev_hi, draw, (uint32_t)g, s.key);
      const uint4 l = philox(c0, s.ev_hi, draw, (uint32_t)(groups + g), s.key);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (4 * g + q < D) F.add_folded(4 * g + q, map(4 * g + q, word(h, q), word(l, q)));
    }
    const double tmp = F.value() * wt;  // plain.py:27
    acc += tmp;
    acc2 += tmp * tmp;
  });
}

// The events of this thread (plain.py:18-35): uniform points, with the
// integration limits (LIM, monte_carlo.py:271-274) or without, the
// integrand, and the sums of w f and (w f)^2. INJ: injected draws
// (s.inject, parity tests) instead of Philox. Both are compile-time choices,
// so that the event body has no test per dimension.
template <int FAM, bool MIXED, int D, bool INJ, bool LIM, typename T>
__device__ __forceinline__ void plain_events(const StepK& s, uint32_t draw, Integrand<T, FAM>& F, double wt,
                                             double& acc, double& acc2) {
  const int d = D ? D : s.n_dim;
  const int groups = D ? (D + 3) / 4 : s.groups;
  const uint32_t c1 = s.ev_hi;  // launch-uniform high word
  const auto event = [&](uint32_t c0, [[maybe_unused]] int64_t i) {
    F.begin();
#pragma unroll
    for (int g = 0; g < groups; ++g) {
      uint4 h = make_uint4(0, 0, 0, 0), l = make_uint4(0, 0, 0, 0);
      if (!INJ) {
        h = philox(c0, c1, draw, (uint32_t)g, s.key);
        if (!MIXED) l = philox(c0, c1, draw, (uint32_t)(groups + g), s.key);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = 4 * g + q;
        if (j < d) {
          T x;
          if (MIXED) {
            const uint32_t hw = INJ ? static_cast<const uint32_t*>(s.inject)[i * d + j] : word(h, q);
            float xf = fmaf((float)(hw >> 9), 0x1p-23f, 0x1p-24f);
            if (LIM) xf = fmaf(xf, (float)s.xdelta[j], (float)s.xmin[j]);
            x = (T)xf;
          } else {
            const double u = INJ ? static_cast<const double*>(s.inject)[i * d + j]
                                 : draw_f64(word(h, q), word(l, q));
            x = (T)(LIM ? s.xmin[j] + u * s.xdelta[j] : u);
          }
          F.add(j, x);
        }
      }
    }
    const double tmp = (double)F.value() * wt;  // plain.py:27
    acc += tmp;
    acc2 += tmp * tmp;
  };
  if (INJ) {
    const int64_t step = (int64_t)gridDim.x * kBlock;
    for (int64_t i = spread_first_event(); i < s.n_events; i += step) event(0u, i);
  } else {
    event_trips<kBlock>(s, [&](uint32_t c0) { event(c0, 0); });
  }
}

template <int FAM, bool MIXED, int D, bool INJ>
__global__ __launch_bounds__(kBlock) void plain_fused(StepK s, mv_integrand fn, RowsK R) {
  const uint32_t draw = iteration_draw(s);
  using T = typename std::conditional<MIXED, float, double>::type;
  Integrand<T, FAM> F(fn);
  const bool limits = s.xmin != nullptr;
  const double wt = limits ? s.xjac * s.xdeltajac : s.xjac;  // monte_carlo.py:270-274
  double acc = 0.0, acc2 = 0.0;
  if constexpr (!MIXED && !INJ && D > 0) {
    if (limits)
      plain_events_f64<FAM, D, true>(s, fn, draw, F, wt, acc, acc2);
    else
      plain_events_f64<FAM, D, false>(s, fn, draw, F, wt, acc, acc2);
  } else if (limits) {
    plain_events<FAM, MIXED, D, INJ, true>(s, draw, F, wt, acc, acc2);
  } else {
    plain_events<FAM, MIXED, D, INJ, false>(s, draw, F, wt, acc, acc2);
  }
  finish_block<false>(acc, acc2, nullptr, 0, iteration_rows(R));
}

namespace {

using Kernel = void (*)(StepK, mv_integrand, RowsK);

template <int FAM, bool MIXED, bool INJ, int... Ds>
constexpr std::array<Kernel, sizeof...(Ds)> kernels_of(std::integer_sequence<int, Ds...>) {
  return {&plain_fused<FAM, MIXED, Ds + 1, INJ>...};
}

template <int FAM, bool MIXED>
int launch_fam(const StepK& k, const mv_integrand& fn, const RowsK& R, hipStream_t st) {
  static constexpr auto table =
      kernels_of<FAM, MIXED, false>(std::make_integer_sequence<int, MV_FUSED_MAX_DIM>{});
  static constexpr auto table_inj =
      kernels_of<FAM, MIXED, true>(std::make_integer_sequence<int, MV_FUSED_MAX_DIM>{});
  const bool inj = k.inject != nullptr;
  const Kernel kern = k.n_dim >= 1 && k.n_dim <= MV_FUSED_MAX_DIM
                          ? (inj ? table_inj : table)[k.n_dim - 1]
                          : (inj ? &plain_fused<FAM, MIXED, 0, true> : &plain_fused<FAM, MIXED, 0, false>);
  return launch_iterations(kern, k, st, fn, R);
}

}  // namespace

int launch_plain_fused_dims(int family, bool mixed, const StepK& k, const mv_integrand& fn,
                            const RowsK& R, hipStream_t st) {
#define MV_PLAIN_FAM(F) \
  return mixed ? launch_fam<F, true>(k, fn, R, st) : launch_fam<F, false>(k, fn, R, st)
  switch (family) {
    case MV_FN_CONSTANT: MV_PLAIN_FAM(MV_FN_CONSTANT);
    case MV_FN_GAUSSIAN: MV_PLAIN_FAM(MV_FN_GAUSSIAN);
    case MV_FN_PRODUCT: MV_PLAIN_FAM(MV_FN_PRODUCT);
    case MV_FN_GAUSSMIX: MV_PLAIN_FAM(MV_FN_GAUSSMIX);
    case MV_FN_BWPOWER: MV_PLAIN_FAM(MV_FN_BWPOWER);
    default: return fail(MV_ERR_UNSUPPORTED, "fused plain kernel: unknown family %d", family);
  }
#undef MV_PLAIN_FAM
}

}  // namespace mv
