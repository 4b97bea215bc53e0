// vplus_kernel.hpp - the fused VEGAS+ producer (mv_vplus_fused): the kernel
// over one integral's events and its launcher, compiled per (integrand family,
// train, n_dim, injected draws) for n_dim 1..MV_FUSED_MAX_DIM, so that the
// event body (vplus_fused.hpp) is straight-line code; one precision per source
// file (vplus_fused_f64.hip, vplus_fused_mixed.hip), which compile in parallel.
//
// Bound by VALU issue at large event counts (some 150 instructions per 64
// mixed events inside a cube at d = 4, 36 of them Philox's) and by the latency
// of its few trips per wave at small ones. Measured on the two-Gaussian
// mixture, d = 4, adaptive training: positions by one FMA from the cube's
// corner, cube digits by multiplication, weights from one division per cube,
// boundary bits by a lane scatter and sums in pairs took the kernel from 152.6
// to 93.9 us (mixed, 2e7 events requested: 1e7 to 2e7 per iteration) and from
// 23.6 to 19.2 us (FP64, 1e6 requested), and the batched kernel of the serving
// mix from 451 to 276 us per tick.
#pragma once

#include "vplus_fused.hpp"

namespace mv {

template <int FAM, bool TRAIN, bool MIXED, int D, bool INJ>
__global__ __launch_bounds__((vplus_block<TRAIN, D>())) void vplus_fused(StepK s, StrataK st, mv_integrand fn,
                                                      const double* __restrict__ grid,
                                                      double* __restrict__ ress,
                                                      double* __restrict__ ress2, RowsK R) {
  constexpr bool PAIRS = vplus_pairs<TRAIN, D>();
  constexpr int BS = vplus_block<TRAIN, D>();
  constexpr int W = BS / 64;
  const uint32_t draw = draw_of(s);
  using T = typename std::conditional<MIXED, float, double>::type;
  constexpr int nb = D * kBins;
  constexpr int hist_len = PAIRS ? pair_cells(D) : (TRAIN ? kWaves * nb : 0);
  // static LDS: constant addresses
  __shared__ __align__(16) double smem[2 * nb + hist_len];
  VplusEntry<MIXED>* tab = reinterpret_cast<VplusEntry<MIXED>*>(smem);
  double* hist = smem + 2 * nb;
  // this wave's run: the iteration's 64-event trips split evenly over the
  // waves, wave g from trip_of(g) up to trip_of(g + 1) (not included)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t total = st.off[st.n_cubes];
  const int64_t trips = (total + 63) >> 6;
  const int64_t nwaves = (int64_t)gridDim.x * W;
  const int64_t gw = (int64_t)blockIdx.x * W + wave;
  const int64_t first = trip_of(gw, trips, nwaves) * 64;
  const int64_t end = min(trip_of(gw + 1, trips, nwaves) * 64, total);
  const int c0 = first < end ? find_cube_wave(st.off, st.n_cubes, (int)first) : 0;
  const bool limits = s.xmin != nullptr;
  vplus_table<MIXED, FAM, BS>(fn, grid, D, s.xmin, s.xdelta, tab);
  for (int i = threadIdx.x; i < hist_len / 2; i += BS) reinterpret_cast<double2*>(hist)[i] = make_double2(0.0, 0.0);
  const JacGroups<double> cs = MIXED ? JacGroups<double>{} : jacobian_groups<double, FAM>(fn, D, s.xdelta);
  __syncthreads();
  double* wh = PAIRS ? hist : hist + wave * nb;

  Integrand<T, FAM> F(fn);
  const double wscale = limits ? s.xjac * s.xdeltajac : s.xjac;
  const StrataPos<MIXED, INJ> sp(st.n_strat);
  vplus_run<FAM, TRAIN, MIXED, D, INJ>(F, s, draw, st, sp, first, end, c0, tab, cs, wscale, wh, ress, ress2);
  if (PAIRS)
    finish_pairs<BS, false>(0.0, 0.0, hist, D, group_row(R));
  else
    finish_block<TRAIN, false>(0.0, 0.0, hist, nb, R);
}

using VplusKernel = void (*)(StepK, StrataK, mv_integrand, const double*, double*, double*, RowsK);

template <int FAM, bool TRAIN, bool MIXED, bool INJ, int... Ds>
constexpr std::array<VplusKernel, sizeof...(Ds)> vplus_kernels_of(std::integer_sequence<int, Ds...>) {
  return {&vplus_fused<FAM, TRAIN, MIXED, Ds + 1, INJ>...};
}

template <int FAM, bool TRAIN, bool MIXED, bool INJ>
int launch_vplus_fam(const StepK& k, const StrataK& st, const mv_integrand& fn, const double* grid,
                     double* ress, double* ress2, const RowsK& R, hipStream_t s) {
  static constexpr auto table =
      vplus_kernels_of<FAM, TRAIN, MIXED, INJ>(std::make_integer_sequence<int, MV_FUSED_MAX_DIM>{});
  if (k.n_dim < 1 || k.n_dim > MV_FUSED_MAX_DIM)
    return fail(MV_ERR_UNSUPPORTED, "fused VEGAS+ kernel: n_dim %d outside 1..%d", k.n_dim,
                MV_FUSED_MAX_DIM);
  const bool pairs = TRAIN && k.n_dim >= kPairMinDim && k.n_dim <= kPairMaxDim;
  if (pairs)
    return launch_producer<kPairBlock>(table[k.n_dim - 1], k.n_events, 0, s, k, st, fn, grid, ress, ress2, R);
  return launch_producer(table[k.n_dim - 1], k.n_events, 0, s, k, st, fn, grid, ress, ress2, R);
}

template <int FAM, bool MIXED>
int launch_vplus_family(bool train, const StepK& k, const StrataK& st, const mv_integrand& fn,
                        const double* grid, double* ress, double* ress2, const RowsK& R, hipStream_t s) {
  const bool inj = k.inject != nullptr;
  if (train)
    return inj ? launch_vplus_fam<FAM, true, MIXED, true>(k, st, fn, grid, ress, ress2, R, s)
               : launch_vplus_fam<FAM, true, MIXED, false>(k, st, fn, grid, ress, ress2, R, s);
  return inj ? launch_vplus_fam<FAM, false, MIXED, true>(k, st, fn, grid, ress, ress2, R, s)
             : launch_vplus_fam<FAM, false, MIXED, false>(k, st, fn, grid, ress, ress2, R, s);
}

// The launcher of one precision: the kernel for (family, train, n_dim,
// injected draws). Returns the workgroups launched or a negative error.
template <bool MIXED>
int launch_vplus_precision(int family, bool train, const StepK& k, const StrataK& st,
                           const mv_integrand& fn, const double* grid, double* ress, double* ress2,
                           const RowsK& R, hipStream_t s) {
#define MV_VPF(F) return launch_vplus_family<F, MIXED>(train, k, st, fn, grid, ress, ress2, R, s)
  switch (family) {
    case MV_FN_CONSTANT: MV_VPF(MV_FN_CONSTANT);
    case MV_FN_GAUSSIAN: MV_VPF(MV_FN_GAUSSIAN);
    case MV_FN_PRODUCT: MV_VPF(MV_FN_PRODUCT);
    case MV_FN_GAUSSMIX: MV_VPF(MV_FN_GAUSSMIX);
    case MV_FN_BWPOWER: MV_VPF(MV_FN_BWPOWER);
    default: return fail(MV_ERR_UNSUPPORTED, "fused VEGAS+ kernel: unknown family %d", family);
  }
#undef MV_VPF
}

}  // namespace mv
