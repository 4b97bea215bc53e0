// batch_vplus.hpp - the producer of batched VegasFlowPlus integrals
// (mv_batch_vplus_fused): many VEGAS+ integrals advance one iteration in one
// persistent launch (vflowplus.py:37-80 + 187-220 per item). The iteration
// end of the items is in vplus.hip (mv_batch_vplus_finalize).
//
// Tiles of consecutive events of one item are split evenly over the
// workgroups (tiles.hpp; eight mixtures of d = 4, two of 2e7 and six of 1e6
// events requested: 276 us per launch with whole tiles dealt out in turn, 256
// with the split, 240 with paced waves too). Per span: the item's map table in
// LDS, histograms zeroed, then the span's 64-event trips split evenly over the
// waves, each wave walking its run with the single-integral event body
// (vplus_run: hypercube lookup over the item's offsets, draws, map, integrand,
// per-cube segmented sums into the item's ress / ress2). The histogram goes
// into the item's row with atomics. Tiles past the item's events of this iteration (tiles cover an
// upper bound of the adaptive event count) have none. Launches whose
// items share n_dim run a kernel compiled for it (the registers of one event
// body); mixed dimensions choose the body per tile.
#pragma once

#include <algorithm>
#include <array>
#include <type_traits>
#include <utility>

#include "abi_util.hpp"
#include "device.hpp"
#include "fused_event.hpp"
#include "rows.hpp"
#include "tiles.hpp"
#include "vplus.hpp"
#include "vplus_fused.hpp"

namespace mv {

// One wave's run of a tile for the tile's n_dim D: per-wave histograms
// (PAIRS false, hist + wave * 50 D) or the workgroup's pair tables (PAIRS,
// 2 <= D <= 14).
template <bool MIXED, int FAM, bool TRAIN, bool PAIRS, int D>
__device__ void vplus_tile_body(const mv_batch_vplus_item& it, const StepK& s, uint32_t draw,
                                const StrataK& st, int64_t first, int64_t end, int c0,
                                const VplusEntry<MIXED>* tab, double* hist, double* __restrict__ ress,
                                double* __restrict__ ress2) {
  using T = typename std::conditional<MIXED, float, double>::type;
  constexpr bool P = PAIRS && D >= kPairMinDim && D <= kPairMaxDim;
  if (PAIRS && !P) return;  // a pair launch holds only items it can pair
  Integrand<T, FAM> F(it.fn);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double* wh = P ? hist : hist + wave * (D * kBins);
  const JacGroups<double> cs = MIXED ? JacGroups<double>{} : jacobian_groups<double, FAM>(it.fn, D, nullptr);
  const StrataPos<MIXED, false> sp(st.n_strat);
  vplus_run<FAM, TRAIN, MIXED, D, false, P>(F, s, draw, st, sp, first, end, c0, tab, cs, s.xjac, wh, ress, ress2);
}

template <bool MIXED, int FAM, bool TRAIN, bool PAIRS, int... Ds>
__device__ void vplus_tile_dispatch(std::integer_sequence<int, Ds...>, int d, const mv_batch_vplus_item& it,
                                    const StepK& s, uint32_t draw, const StrataK& st, int64_t first,
                                    int64_t end, int c0, const VplusEntry<MIXED>* tab, double* hist,
                                    double* ress, double* ress2) {
  // one call for the tile's n_dim (d is workgroup-uniform)
  ((d == Ds + 1
        ? vplus_tile_body<MIXED, FAM, TRAIN, PAIRS, Ds + 1>(it, s, draw, st, first, end, c0, tab, hist, ress, ress2)
        : void()),
   ...);
}

// PAIRS: BS = kPairBlock threads and one set of pair tables per workgroup
// (items with 2 <= n_dim <= 14 only): a wave's events lie in one or two
// hypercubes, whose few bins per dimension would take most of a per-wave
// histogram's adds; the pair tables spread them over up to 2500 cells.
// DSPEC > 0: every tiled item has n_dim DSPEC (one event body, the
// registers of that n_dim only); 0: the body is chosen per tile.
template <bool MIXED, int FAM, bool PAIRS, int BS, int DSPEC>
__global__ __launch_bounds__(BS) void batch_vplus_fused(const mv_batch_vplus_item* __restrict__ items,
                                                        const mv_batch_tile* __restrict__ tiles,
                                                        int n_tiles, const int32_t* __restrict__ draws,
                                                        const double* __restrict__ grids,
                                                        const int32_t* __restrict__ n_ev,
                                                        const int32_t* __restrict__ offsets,
                                                        double* __restrict__ ress,
                                                        double* __restrict__ ress2,
                                                        double* __restrict__ rows, int nbmax) {
  constexpr int W = BS / 64;
  extern __shared__ double smem[];
  // LDS: the map table (nbmax 16-byte entries), then the histograms (per-wave,
  // or the pair tables)
  VplusEntry<MIXED>* tab = reinterpret_cast<VplusEntry<MIXED>*>(smem);
  double* hist = smem + 2 * nbmax;
  // the events that the tiles have in this iteration
  const auto work = [&](int i) {
    const mv_batch_tile t = tiles[i];
    const mv_batch_vplus_item& it = items[t.item];
    const int64_t left = (int64_t)offsets[it.off_offset + it.n_cubes] - t.first;
    const int groups = (it.n_dim + 3) >> 2;
    return TileWork{t.item, (int)max((int64_t)0, min((int64_t)t.count, left)), t.first,
                    MIXED ? 60 * groups + 21 * it.n_dim + 60 : 120 * groups + 33 * it.n_dim + 60,
                    tile_begins(tiles, i)};
  };
  for_each_span<BS>(n_tiles, work, [&](int item, int64_t first, int count) {
    const mv_batch_vplus_item& it = items[item];
    const StrataK st{it.n_strat, it.n_cubes, n_ev + it.cube_offset, offsets + it.off_offset};
    const int64_t end = first + count;
    const int d = it.n_dim;
    const int nb = d * kBins;
    // this wave's run: the span's trips split evenly over the waves
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t trips = (end - first + 63) >> 6;
    const int64_t a = first + trip_of(wave, trips, W) * 64;
    const int64_t b = min(first + trip_of(wave + 1, trips, W) * 64, end);
    const int c0 = a < b ? find_cube_wave(st.off, st.n_cubes, (int)a) : 0;
    __syncthreads();  // the previous tile is done with the LDS
    vplus_table<MIXED, FAM, BS>(it.fn, grids + it.grid_offset, d, nullptr, nullptr, tab);
    const int hist_len = PAIRS ? pair_cells(d) : W * nb;
    if (it.train)
      for (int i = threadIdx.x; i < hist_len; i += BS) hist[i] = 0.0;
    __syncthreads();
    StepK s{};
    s.n_dim = d;
    s.groups = (d + 3) / 4;
    s.n_events = end - first;
    s.key.k0 = (uint32_t)(it.seed & 0xffffffffu);
    s.key.k1 = (uint32_t)(it.seed >> 32);
    s.xjac = 1.0 / (double)it.n_cubes;  // vflowplus.py:139
    s.xdeltajac = 1.0;
    const uint32_t draw = (uint32_t)draws[item];
    double* cr = ress + it.cube_offset;
    double* cr2 = ress2 + it.cube_offset;
    if constexpr (DSPEC > 0) {
      if (it.train)
        vplus_tile_body<MIXED, FAM, true, PAIRS, DSPEC>(it, s, draw, st, a, b, c0, tab, hist, cr, cr2);
      else
        vplus_tile_body<MIXED, FAM, false, PAIRS, DSPEC>(it, s, draw, st, a, b, c0, tab, hist, cr, cr2);
    } else {
      constexpr auto dims = std::make_integer_sequence<int, MV_FUSED_MAX_DIM>{};
      if (it.train)
        vplus_tile_dispatch<MIXED, FAM, true, PAIRS>(dims, d, it, s, draw, st, a, b, c0, tab, hist, cr, cr2);
      else
        vplus_tile_dispatch<MIXED, FAM, false, PAIRS>(dims, d, it, s, draw, st, a, b, c0, tab, hist, cr, cr2);
    }
    // histogram bins into the item's row (its sum columns stay unused: the
    // VEGAS+ sums are per cube)
    if (it.train) {
      if (PAIRS)
        finish_pairs<BS, false>(0.0, 0.0, hist, d, rows + it.row_offset);
      else
        finish_row<true, false>(0.0, 0.0, hist, nb, rows + it.row_offset);
    }
  });
}

using BatchVplusKernel = void (*)(const mv_batch_vplus_item*, const mv_batch_tile*, int, const int32_t*,
                                  const double*, const int32_t*, const int32_t*, double*, double*, double*,
                                  int);

template <bool MIXED, int FAM, bool PAIRS, int D0, int... Ds>
constexpr std::array<BatchVplusKernel, sizeof...(Ds)> batch_vplus_table(std::integer_sequence<int, Ds...>) {
  return {&batch_vplus_fused<MIXED, FAM, PAIRS, PAIRS ? kPairBlock : kBlock, Ds + D0>...};
}

// The kernel for (family, histogram form): compiled for n_dim ``dspec``
// (1..MV_FUSED_MAX_DIM), or choosing the body per tile (dspec 0).
template <bool MIXED, int FAM, bool PAIRS>
BatchVplusKernel batch_vplus_family(int dspec) {
  // pair launches hold n_dim kPairMinDim..kPairMaxDim only, and on gfx950 the
  // others come to per-wave launches of one n_dim only outside that range
  if constexpr (PAIRS) {
    static constexpr auto table = batch_vplus_table<MIXED, FAM, true, kPairMinDim>(
        std::make_integer_sequence<int, kPairMaxDim - kPairMinDim + 1>{});
    if (dspec >= kPairMinDim && dspec <= kPairMaxDim) return table[dspec - kPairMinDim];
  } else {
    static constexpr auto low =
        batch_vplus_table<MIXED, FAM, false, 1>(std::make_integer_sequence<int, kPairMinDim - 1>{});
    static constexpr auto high = batch_vplus_table<MIXED, FAM, false, kPairMaxDim + 1>(
        std::make_integer_sequence<int, MV_FUSED_MAX_DIM - kPairMaxDim>{});
    if (dspec >= 1 && dspec < kPairMinDim) return low[dspec - 1];
    if (dspec > kPairMaxDim && dspec <= MV_FUSED_MAX_DIM) return high[dspec - kPairMaxDim - 1];
  }
  return &batch_vplus_fused<MIXED, FAM, PAIRS, PAIRS ? kPairBlock : kBlock, 0>;
}

template <bool MIXED, bool PAIRS>
BatchVplusKernel batch_vplus_kernel(int family, int dspec) {
  switch (family) {
    case MV_FN_CONSTANT: return batch_vplus_family<MIXED, MV_FN_CONSTANT, PAIRS>(dspec);
    case MV_FN_GAUSSIAN: return batch_vplus_family<MIXED, MV_FN_GAUSSIAN, PAIRS>(dspec);
    case MV_FN_PRODUCT: return batch_vplus_family<MIXED, MV_FN_PRODUCT, PAIRS>(dspec);
    case MV_FN_GAUSSMIX: return batch_vplus_family<MIXED, MV_FN_GAUSSMIX, PAIRS>(dspec);
    case MV_FN_BWPOWER: return batch_vplus_family<MIXED, MV_FN_BWPOWER, PAIRS>(dspec);
    default: return nullptr;
  }
}

// The producer of one precision (mv_batch_vplus_fused): picks the histogram
// form and the kernel, sizes the launch. Returns 0 or a negative status.
template <bool MIXED>
int launch_batch_vplus_precision(const mv_batch_vplus_item* items, const mv_batch_tile* tiles, int n_tiles,
                                 int family, int min_dim, int max_dim, const int32_t* draws, const double* grids,
                                 const int32_t* n_ev, const int32_t* offsets, double* ress, double* ress2,
                                 double* rows, int blocks, hipStream_t stream) {
  // pair tables whenever every tiled item can pair its dimensions and they
  // fit in a workgroup's LDS
  const int nbmax = max_dim * kBins;
  const size_t table = 2 * (size_t)nbmax;
  const bool pairs = min_dim >= kPairMinDim && max_dim <= kPairMaxDim &&
                     (table + (size_t)pair_cells(max_dim)) * sizeof(double) <= max_lds_per_block();
  const int dspec = min_dim == max_dim ? max_dim : 0;
  BatchVplusKernel k = pairs ? batch_vplus_kernel<MIXED, true>(family, dspec)
                             : batch_vplus_kernel<MIXED, false>(family, dspec);
  if (!k) return fail(MV_ERR_UNSUPPORTED, "mv_batch_vplus_fused: unknown family %d", family);
  const size_t hist = pairs ? (size_t)pair_cells(max_dim) : (size_t)kWaves * nbmax;
  const size_t lds = (table + hist) * sizeof(double);
  const int bs = pairs ? kPairBlock : kBlock;
  // at most the workgroups resident at once (a persistent launch)
  const int res = resident_blocks(reinterpret_cast<const void*>(k), lds, bs);
  if (res < 1) return fail(MV_ERR_UNSUPPORTED, "mv_batch_vplus_fused: a workgroup does not fit (n_dim %d)", max_dim);
  blocks = std::min(blocks, res);
  hipLaunchKernelGGL(k, dim3(blocks), dim3(bs), lds, stream, items, tiles, n_tiles, draws, grids, n_ev, offsets,
                     ress, ress2, rows, nbmax);
  return check_launch("mv_batch_vplus_fused");
}

}  // namespace mv
