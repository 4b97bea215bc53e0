// batch.hip - many independent VegasFlow integrals in one persistent launch.
//
// The events of every item of an iteration round are cut into tiles of
// consecutive events of one item. batch_fused: ``blocks`` workgroups stride
// over the tile list. batch_fused_pairs: the list is split evenly over the
// workgroups (tiles.hpp). A tile or span loads its item's map table into LDS,
// runs the same per-event body as the single-integral fused kernels
// (fused_event.hpp) and adds its sums and histogram into the item's row with
// FP64 atomics. The finalize kernel gives one wave per (item, sums) and per
// (item, dimension) job. Grids, rows, per-item draw counters, running weighted
// averages and the per-iteration history all stay on the device, so a round
// can be replayed from a captured HIP graph: nothing in it depends on host
// values.
//
// batch_fused_pairs is bound like the single pair kernel (VALU and LDS of one
// workgroup of 16 waves per CU) plus 17 us per launch (split 6, table and
// cleared histograms 2, marginals and row, launch). 256 Gaussians of d 2..12
// and 1e4..1e6 events, 5.3e7 events per round: 270 us with whole tiles dealt
// out in turn and the prologue and epilogue compiled per n_dim around the
// event loop (table reads issued one by one for want of scalar registers),
// 251 us with the split, 238 us with paced waves, 231 us with measured costs;
// the single kernel's rates for the same events come to 185 us.
#include <algorithm>
#include <type_traits>

#include "abi_util.hpp"
#include "device.hpp"
#include "fused_event.hpp"
#include "refine.hpp"
#include "rows.hpp"
#include "tiles.hpp"

namespace mv {

template <bool MIXED, int FAM, bool TRAIN>
__device__ __forceinline__ void batch_events(const mv_batch_item& it, const mv_batch_tile& tile,
                                             uint32_t draw, const void* tab,
                                             const JacGroups<typename std::conditional<MIXED, float, double>::type>& cs,
                                             double* hist, int nb, double* row) {
  using T = typename std::conditional<MIXED, float, double>::type;
  Integrand<T, FAM> F(it.fn);
  const Key key{(uint32_t)(it.seed & 0xffffffffu), (uint32_t)(it.seed >> 32)};
  const int d = it.n_dim;
  const int groups = (d + 3) / 4;
  const double wscale = 1.0 / (double)it.n_events;  // xjac, monte_carlo.py:224-227
  double* wh = hist + (threadIdx.x >> 6) * nb;
  double acc = 0.0, acc2 = 0.0;
  // a tile never crosses a multiple of 2^32 events (mv_batch_fused), so the
  // high counter word is uniform over the tile
  const uint32_t lo0 = (uint32_t)((uint64_t)tile.first & 0xffffffffu);
  const uint32_t hi = (uint32_t)((uint64_t)tile.first >> 32);
  for (int k = threadIdx.x; k < tile.count; k += kBlock) {
    double tmp;
    if constexpr (MIXED)
      tmp = event_mixed<FAM, TRAIN>(F, lo0 + (uint32_t)k, hi, draw, key, groups, d,
                                    static_cast<const float2*>(tab), cs, wh, nullptr, wscale);
    else
      tmp = event_f64<FAM, TRAIN>(F, lo0 + (uint32_t)k, hi, draw, key, groups, d,
                                  static_cast<const double2*>(tab), cs, wh, nullptr, wscale);
    acc += tmp;
    acc2 += tmp * tmp;
  }
  finish_row<TRAIN>(acc, acc2, hist, nb, row);
}

template <bool MIXED, int FAM>
__device__ __forceinline__ void batch_tile(const mv_batch_item& it, const mv_batch_tile& tile,
                                           uint32_t draw, const double* __restrict__ grids,
                                           double* __restrict__ rows, double* smem, int nbmax) {
  using T = typename std::conditional<MIXED, float, double>::type;
  using T2 = typename std::conditional<MIXED, float2, double2>::type;
  const int d = it.n_dim;
  const int nb = d * kBins;
  T2* tab = reinterpret_cast<T2*>(smem);
  double* hist = smem + (MIXED ? nbmax : 2 * nbmax);
  __syncthreads();  // the previous tile is done with the LDS
  build_table<T, FAM>(it.fn, grids + it.grid_offset, d, nullptr, nullptr, tab);
  if (it.train)
    for (int i = threadIdx.x; i < kWaves * nb; i += kBlock) hist[i] = 0.0;
  const JacGroups<T> cs = jacobian_groups<T, FAM>(it.fn, d, nullptr);
  __syncthreads();
  double* row = rows + it.row_offset;
  if (it.train)
    batch_events<MIXED, FAM, true>(it, tile, draw, tab, cs, hist, nb, row);
  else
    batch_events<MIXED, FAM, false>(it, tile, draw, tab, cs, hist, nb, row);
}

// FAM >= 0: every tile belongs to an item of that family (smaller register
// footprint); FAM < 0: dispatch on each tile's item.
template <bool MIXED, int FAM>
__global__ __launch_bounds__(kBlock) void batch_fused(const mv_batch_item* __restrict__ items,
                                                      const mv_batch_tile* __restrict__ tiles,
                                                      int n_tiles, int nbmax,
                                                      const int32_t* __restrict__ draws,
                                                      const double* __restrict__ grids,
                                                      double* __restrict__ rows) {
  extern __shared__ double smem[];
  for (int t = blockIdx.x; t < n_tiles; t += gridDim.x) {
    const mv_batch_tile tile = tiles[t];
    const mv_batch_item& it = items[tile.item];
    const uint32_t draw = (uint32_t)draws[tile.item];
    if constexpr (FAM >= 0) {
      batch_tile<MIXED, FAM>(it, tile, draw, grids, rows, smem, nbmax);
    } else {
      switch (it.fn.family) {
        case MV_FN_CONSTANT: batch_tile<MIXED, MV_FN_CONSTANT>(it, tile, draw, grids, rows, smem, nbmax); break;
        case MV_FN_GAUSSIAN: batch_tile<MIXED, MV_FN_GAUSSIAN>(it, tile, draw, grids, rows, smem, nbmax); break;
        case MV_FN_PRODUCT: batch_tile<MIXED, MV_FN_PRODUCT>(it, tile, draw, grids, rows, smem, nbmax); break;
        case MV_FN_GAUSSMIX: batch_tile<MIXED, MV_FN_GAUSSMIX>(it, tile, draw, grids, rows, smem, nbmax); break;
        default: batch_tile<MIXED, MV_FN_BWPOWER>(it, tile, draw, grids, rows, smem, nbmax); break;
      }
    }
  }
}

// ``body(k)`` for the events k = 0 .. count - 1 of a span, 64 consecutive ones
// per wave and trip; only the last, partial trip has a per-lane test.
template <int BS, bool PACED, typename Body>
__device__ __forceinline__ void span_trips(int count, Body&& body) {
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int full = count >> 6;
  uint32_t k = (uint32_t)(wave * 64 + lane);
  paced_trips<PACED, int>(wave, full, BS / 64, [&](int) {
    body(k);
    k += BS;
  });
  if (full % (BS / 64) == wave && k < (uint32_t)count) body(k);
}

// The events of a span for D = n_dim (0: it.n_dim, chosen at run time): sums
// into acc, acc2 and, for training items, the pair tables. Only this part is
// compiled per n_dim: with the map table and the row inside it, the addresses
// and masks of all its copies were hoisted out of the loop over spans, which
// left so few scalar registers that the table reads were issued one by one.
template <int FAM, int BS, bool MIXED, int D>
__device__ __forceinline__ void batch_span_events(const mv_batch_item& it, const mv_batch_tile& tile, uint32_t draw,
                                                  double* smem, double& acc, double& acc2) {
  using T = typename std::conditional<MIXED, float, double>::type;
  using T2 = typename std::conditional<MIXED, float2, double2>::type;
  const int d = D ? D : it.n_dim;
  const int groups = (d + 3) / 4;
  const Key key{(uint32_t)(it.seed & 0xffffffffu), (uint32_t)(it.seed >> 32)};
  const double wscale = 1.0 / (double)it.n_events;  // xjac, monte_carlo.py:224-227
  // a tile never crosses a multiple of 2^32 events: uniform high counter word
  const uint32_t lo0 = (uint32_t)((uint64_t)tile.first & 0xffffffffu);
  const uint32_t hi = (uint32_t)((uint64_t)tile.first >> 32);
  const T2* tab = reinterpret_cast<const T2*>(smem);
  double* H = smem + (MIXED ? 1 : 2) * d * kBins;  // a constant address where D is one
  const JacGroups<T> cs = jacobian_groups<T, FAM>(it.fn, d, nullptr);
  Integrand<T, FAM> F(it.fn);
  const auto add = [&](double tmp) {
    acc += tmp;
    acc2 += tmp * tmp;
  };
  if (it.train)
    span_trips<BS, MIXED>(tile.count, [&](uint32_t k) {
      if constexpr (MIXED)
        add(event_mixed_pairs<FAM, false>(F, lo0 + k, hi, draw, key, d, tab, cs, H, nullptr, wscale));
      else
        add(event_f64<FAM, true, true, 0>(F, lo0 + k, hi, draw, key, groups, d, tab, cs, H, nullptr, wscale));
    });
  else
    span_trips<BS, MIXED>(tile.count, [&](uint32_t k) {
      if constexpr (MIXED)
        add(event_mixed<FAM, false>(F, lo0 + k, hi, draw, key, groups, d, tab, cs, nullptr, nullptr, wscale));
      else
        add(event_f64<FAM, false, false, 0>(F, lo0 + k, hi, draw, key, groups, d, tab, cs, nullptr, nullptr, wscale));
    });
}

// One span with pair histograms (fused_event.hpp), BS threads. LDS = the map
// table (mixed: float2; FP64: double2 per bin), then the pair tables.
// PER_DIM: one event body per n_dim, chosen here.
template <int FAM, int BS, bool MIXED, bool PER_DIM>
__device__ __forceinline__ void batch_span_pairs(const mv_batch_item& it, const mv_batch_tile& tile, uint32_t draw,
                                                 const double* __restrict__ grids, double* __restrict__ rows,
                                                 double* smem) {
  using T = typename std::conditional<MIXED, float, double>::type;
  using T2 = typename std::conditional<MIXED, float2, double2>::type;
  const int d = it.n_dim;
  // 16-byte aligned: 50 d * 8 is a multiple of 400
  double2* H = reinterpret_cast<double2*>(smem + (MIXED ? 1 : 2) * d * kBins);
  __syncthreads();  // the previous span is done with the LDS
  build_table<T, FAM>(it.fn, grids + it.grid_offset, d, nullptr, nullptr, reinterpret_cast<T2*>(smem));
  if (it.train)
    for (int i = threadIdx.x; i < pair_cells(d) / 2; i += BS) H[i] = make_double2(0.0, 0.0);
  __syncthreads();
  double acc = 0.0, acc2 = 0.0;
#define MV_BTP(D) case D: batch_span_events<FAM, BS, MIXED, D>(it, tile, draw, smem, acc, acc2); break
  if constexpr (!PER_DIM) {
    batch_span_events<FAM, BS, MIXED, 0>(it, tile, draw, smem, acc, acc2);
  } else {
    switch (d) {
      MV_BTP(1); MV_BTP(2); MV_BTP(3); MV_BTP(4); MV_BTP(5); MV_BTP(6); MV_BTP(7);
      MV_BTP(8); MV_BTP(9); MV_BTP(10); MV_BTP(11); MV_BTP(12); MV_BTP(13);
      default: batch_span_events<FAM, BS, MIXED, kPairMaxDim>(it, tile, draw, smem, acc, acc2); break;
    }
  }
#undef MV_BTP
  static_assert(kPairMaxDim == 14, "the switch above covers n_dim 1..14");
  finish_pairs<BS, true, MIXED>(acc, acc2, reinterpret_cast<double*>(H), it.train ? d : 0, rows + it.row_offset);
}

// Cost of a training event for the split of the tiles (tiles.hpp), fitted to
// the times of Gaussian events of one n_dim without the launch's fixed part
// (17 us mixed, 22 us FP64): mixed, 5.12e7 events in 256 items, 79, 110, 99,
// 154, 152, 187, 182, 228, 268 us at d = 2, 3, 4, 5, 6, 7, 8, 10, 12; FP64,
// 1.28e7 events, 40, 50, 55, 79, 82, 91, 94, 122, 125, 138, 169 us at d = 2 ..
// 10, 12, 14; within 6 %. The unpaired dimension of an odd n_dim has 50 cells
// for all lanes.
template <bool MIXED>
__device__ __forceinline__ int batch_event_cost(int d) {
  const int groups = (d + 3) >> 2, odd = d & 1;
  return MIXED ? 23 * groups + 14 * d + 26 + 20 * odd : 56 * groups + 26 * d + 52 + 20 * odd;
}

template <int FAM, int BS, bool MIXED>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(4, 4))) void batch_fused_pairs(const mv_batch_item* __restrict__ items,
                                                        const mv_batch_tile* __restrict__ tiles,
                                                        int n_tiles,
                                                        const int32_t* __restrict__ draws,
                                                        const double* __restrict__ grids,
                                                        double* __restrict__ rows) {
  extern __shared__ double smem[];
  const auto work = [&](int i) {
    const mv_batch_tile t = tiles[i];
    return TileWork{t.item, t.count, t.first, batch_event_cost<MIXED>(items[t.item].n_dim),
                    tile_begins(tiles, i)};
  };
  for_each_span<BS>(n_tiles, work, [&](int item, int64_t first, int count) {
    const mv_batch_tile tile{item, count, first};
    const mv_batch_item& it = items[item];
    const uint32_t draw = (uint32_t)draws[item];
    if constexpr (FAM >= 0) {
      batch_span_pairs<FAM, BS, MIXED, true>(it, tile, draw, grids, rows, smem);
    } else {
      switch (it.fn.family) {
        case MV_FN_CONSTANT: batch_span_pairs<MV_FN_CONSTANT, BS, MIXED, false>(it, tile, draw, grids, rows, smem); break;
        case MV_FN_GAUSSIAN: batch_span_pairs<MV_FN_GAUSSIAN, BS, MIXED, false>(it, tile, draw, grids, rows, smem); break;
        case MV_FN_PRODUCT: batch_span_pairs<MV_FN_PRODUCT, BS, MIXED, false>(it, tile, draw, grids, rows, smem); break;
        case MV_FN_GAUSSMIX: batch_span_pairs<MV_FN_GAUSSMIX, BS, MIXED, false>(it, tile, draw, grids, rows, smem); break;
        default: batch_span_pairs<MV_FN_BWPOWER, BS, MIXED, false>(it, tile, draw, grids, rows, smem); break;
      }
    }
  });
}

__global__ __launch_bounds__(64) void batch_finalize_kernel(const mv_batch_item* __restrict__ items,
                                                            const int32_t* __restrict__ jobs,
                                                            double* __restrict__ grids,
                                                            double* __restrict__ rows,
                                                            int32_t* __restrict__ draws,
                                                            double* __restrict__ stats,
                                                            double* __restrict__ history,
                                                            int max_iter) {
  __shared__ double hb[kBins];
  const int item = jobs[2 * blockIdx.x], dim = jobs[2 * blockIdx.x + 1];
  const mv_batch_item& it = items[item];
  double* row = rows + it.row_offset;
  const int t = threadIdx.x;
  if (dim < 0) {
    if (t == 0) {
      const double N = (double)it.n_events;
      const double res = row[0], res2 = row[1];
      row[0] = 0.0;
      row[1] = 0.0;
      const double err = (N * res2 - res * res) / (N - 1.0);  // vflow.py:437
      const double sig = sqrt_clamped(err);                   // vflow.py:438
      double* st = stats + 4 * (int64_t)item;
      const double wgt = 1.0 / (sig * sig);                   // monte_carlo.py:718
      st[0] = res;
      st[1] = sig;
      st[2] += wgt;                                           // monte_carlo.py:720
      st[3] += res * wgt;                                     // monte_carlo.py:719
      const int k = draws[item];
      if (history && k < max_iter) {
        history[2 * ((int64_t)item * max_iter + k)] = res;
        history[2 * ((int64_t)item * max_iter + k) + 1] = sig;
      }
      draws[item] = k + 1;
    }
    return;
  }
  const int64_t c = 2 + (int64_t)dim * kBins + t;
  double* div = grids + it.grid_offset + (int64_t)dim * (kBins + 1);
  const double edge = t <= kBins ? div[t] : 0.0;
  if (t < kBins) {
    hb[t] = row[c];
    row[c] = 0.0;
  }
  __syncthreads();
  if (it.train && wave_hist_finite(hb)) refine_wave(hb, edge, div);
}

}  // namespace mv

using namespace mv;

extern "C" int mv_batch_fused(const mv_batch_item* items, int32_t n_items, const mv_batch_tile* tiles,
                              int32_t n_tiles, int32_t precision, int32_t family, int32_t max_dim,
                              const int32_t* draws, const double* grids, double* rows, int32_t blocks,
                              void* stream) {
  if (n_items < 0 || n_tiles < 0) return fail(MV_ERR_ARG, "mv_batch_fused: negative counts");
  if (n_tiles == 0) return MV_OK;
  if (!items || !tiles || !draws || !grids || !rows)
    return fail(MV_ERR_ARG, "mv_batch_fused: missing buffer");
  if (max_dim < 1 || max_dim > MV_FUSED_MAX_DIM)
    return fail(MV_ERR_UNSUPPORTED, "mv_batch_fused: max_dim must be 1..%d", MV_FUSED_MAX_DIM);
  if (precision != MV_F64 && precision != MV_MIXED)
    return fail(MV_ERR_ARG, "mv_batch_fused: unknown precision %d", precision);
  if (blocks < 1) return fail(MV_ERR_ARG, "mv_batch_fused: blocks < 1");
  const int nbmax = max_dim * kBins;
  hipStream_t s = as_stream(stream);
  const bool mixed = precision == MV_MIXED;
  const size_t lds = mixed ? (size_t)(nbmax + kWaves * nbmax) * sizeof(double)
                           : (size_t)(2 * nbmax + kWaves * nbmax) * sizeof(double);
#define MV_BF(MX, F)                                                                                \
  hipLaunchKernelGGL((batch_fused<MX, F>), dim3(blocks), dim3(kBlock), lds, s, items, tiles, n_tiles, \
                     nbmax, draws, grids, rows)
#define MV_BF_ALL(MX)                                             \
  switch (family) {                                               \
    case MV_FN_CONSTANT: MV_BF(MX, MV_FN_CONSTANT); break;        \
    case MV_FN_GAUSSIAN: MV_BF(MX, MV_FN_GAUSSIAN); break;        \
    case MV_FN_PRODUCT: MV_BF(MX, MV_FN_PRODUCT); break;          \
    case MV_FN_GAUSSMIX: MV_BF(MX, MV_FN_GAUSSMIX); break;        \
    case MV_FN_BWPOWER: MV_BF(MX, MV_FN_BWPOWER); break;          \
    default: MV_BF(MX, -1); break;                                \
  }
  if (mixed) { MV_BF_ALL(true) } else { MV_BF_ALL(false) }
#undef MV_BF_ALL
#undef MV_BF
  return check_launch("mv_batch_fused");
}

namespace {
constexpr int kBatchPairBlock = 1024;

size_t batch_pairs_lds(int max_dim, bool mixed) {
  if (max_dim < 1 || max_dim > kPairMaxDim) return 0;
  const size_t table = (size_t)max_dim * kBins * (mixed ? 1 : 2);
  const size_t lds = (table + pair_cells(max_dim)) * sizeof(double);
  return lds <= max_lds_per_block() ? lds : 0;
}

using BatchPairsKernel = void (*)(const mv_batch_item*, const mv_batch_tile*, int, const int32_t*, const double*,
                                  double*);

template <bool MIXED>
BatchPairsKernel batch_pairs_kernel(int family) {
  switch (family) {
    case MV_FN_CONSTANT: return batch_fused_pairs<MV_FN_CONSTANT, kBatchPairBlock, MIXED>;
    case MV_FN_GAUSSIAN: return batch_fused_pairs<MV_FN_GAUSSIAN, kBatchPairBlock, MIXED>;
    case MV_FN_PRODUCT: return batch_fused_pairs<MV_FN_PRODUCT, kBatchPairBlock, MIXED>;
    case MV_FN_GAUSSMIX: return batch_fused_pairs<MV_FN_GAUSSMIX, kBatchPairBlock, MIXED>;
    case MV_FN_BWPOWER: return batch_fused_pairs<MV_FN_BWPOWER, kBatchPairBlock, MIXED>;
    default: return batch_fused_pairs<-1, kBatchPairBlock, MIXED>;
  }
}

template <bool MIXED>
int32_t pairs_blocks(int32_t family, int32_t max_dim) {
  const size_t lds = batch_pairs_lds(max_dim, MIXED);
  if (!lds) return 0;
  return resident_blocks(reinterpret_cast<const void*>(batch_pairs_kernel<MIXED>(family)), lds,
                         kBatchPairBlock);
}

template <bool MIXED>
int fused_pairs(const mv_batch_item* items, int32_t n_items, const mv_batch_tile* tiles, int32_t n_tiles,
                int32_t family, int32_t max_dim, const int32_t* draws, const double* grids, double* rows,
                int32_t blocks, void* stream, const char* what) {
  if (n_items < 0 || n_tiles < 0) return fail(MV_ERR_ARG, "%s: negative counts", what);
  if (n_tiles == 0) return MV_OK;
  if (!items || !tiles || !draws || !grids || !rows) return fail(MV_ERR_ARG, "%s: missing buffer", what);
  const size_t lds = batch_pairs_lds(max_dim, MIXED);
  if (!lds) return fail(MV_ERR_UNSUPPORTED, "%s: max_dim must be 1..%d and fit the LDS", what, kPairMaxDim);
  if (blocks < 1) return fail(MV_ERR_ARG, "%s: blocks < 1", what);
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(batch_pairs_kernel<MIXED>(family), dim3(blocks), dim3(kBatchPairBlock), lds, s, items,
                     tiles, n_tiles, draws, grids, rows);
  return check_launch(what);
}
}  // namespace

extern "C" int32_t mv_batch_pairs_blocks(int32_t family, int32_t max_dim) {
  return pairs_blocks<true>(family, max_dim);
}

extern "C" int32_t mv_batch_pairs_blocks_f64(int32_t family, int32_t max_dim) {
  return pairs_blocks<false>(family, max_dim);
}

extern "C" int mv_batch_fused_pairs(const mv_batch_item* items, int32_t n_items,
                                    const mv_batch_tile* tiles, int32_t n_tiles, int32_t family,
                                    int32_t max_dim, const int32_t* draws, const double* grids,
                                    double* rows, int32_t blocks, void* stream) {
  return fused_pairs<true>(items, n_items, tiles, n_tiles, family, max_dim, draws, grids, rows, blocks, stream,
                           "mv_batch_fused_pairs");
}

extern "C" int mv_batch_fused_pairs_f64(const mv_batch_item* items, int32_t n_items,
                                        const mv_batch_tile* tiles, int32_t n_tiles, int32_t family,
                                        int32_t max_dim, const int32_t* draws, const double* grids,
                                        double* rows, int32_t blocks, void* stream) {
  return fused_pairs<false>(items, n_items, tiles, n_tiles, family, max_dim, draws, grids, rows, blocks, stream,
                            "mv_batch_fused_pairs_f64");
}

extern "C" int mv_batch_finalize(const mv_batch_item* items, const int32_t* jobs, int32_t n_jobs,
                                 double* grids, double* rows, int32_t* draws, double* stats,
                                 double* history, int32_t max_iter, void* stream) {
  if (n_jobs < 0) return fail(MV_ERR_ARG, "mv_batch_finalize: negative n_jobs");
  if (n_jobs == 0) return MV_OK;
  if (!items || !jobs || !grids || !rows || !draws || !stats)
    return fail(MV_ERR_ARG, "mv_batch_finalize: missing buffer");
  if (history && max_iter < 1) return fail(MV_ERR_ARG, "mv_batch_finalize: max_iter < 1");
  hipLaunchKernelGGL(batch_finalize_kernel, dim3(n_jobs), dim3(64), 0, as_stream(stream), items, jobs,
                     grids, rows, draws, stats, history, max_iter);
  return check_launch("mv_batch_finalize");
}
