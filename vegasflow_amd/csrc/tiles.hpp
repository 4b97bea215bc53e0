// tiles.hpp - the events of a batch's tile list split evenly over the
// workgroups of a persistent launch.
//
// A launch's tiles have different sizes and event costs, and a workgroup has
// only a few of them, so a grid stride over whole tiles leaves workgroups idle
// for up to the time of a heavy tile, and every tile pays for its map table,
// its cleared histograms and its row. Instead each workgroup finds the total
// cost of the list (two short passes over it), takes an equal interval of that
// cost, cuts tiles where the interval begins and ends, and joins what follows
// each other in one item: about one span per workgroup plus one per item. The
// cuts are at whole trips of 64 events from the tile's first. Measured: see
// batch.hip and batch_vplus.hpp.
#pragma once

#include "device.hpp"
#include "mivegas.h"

namespace mv {

// Costs are in units of which a workgroup does 200 000 in a microsecond. What
// comes with a span's table, histograms and row (about 5 us) is charged to a
// tile that does not continue the one before it in the list.
constexpr int64_t kSpanCost = 1000000;
// A workgroup gets at least this much, or stays out.
constexpr int64_t kMinShare = 200000;

// Events first .. first + count - 1 of an item, ``per_event`` each; begins: the
// tile does not continue the one before it.
struct TileWork {
  int item;
  int count;
  int64_t first;
  int per_event;
  bool begins;
  __device__ __forceinline__ int64_t fixed() const { return begins ? kSpanCost : 0; }
  __device__ __forceinline__ int64_t cost() const {
    return count > 0 ? fixed() + (int64_t)count * per_event : 0;
  }
  // the events before a share that ends x into this tile's cost
  __device__ __forceinline__ int cut(int64_t x) const {
    if (x <= fixed()) return 0;
    if (x >= cost()) return count;
    return (int)(((x - fixed()) / per_event) & ~63ll);
  }
};

// tiles[i] does not continue tiles[i - 1]
__device__ __forceinline__ bool tile_begins(const mv_batch_tile* __restrict__ tiles, int i) {
  return i == 0 || tiles[i - 1].item != tiles[i].item || tiles[i - 1].first + tiles[i - 1].count != tiles[i].first;
}

__device__ __forceinline__ int64_t uniform(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Runs body(item, first, count) for this workgroup's share of the tiles
// tile_of(0) .. tile_of(n_tiles - 1). tile_of(i) must give the same in every
// workgroup. A span stays within one item and one high word of the event
// index. The whole workgroup (BS threads) must call; body may use barriers.
template <int BS, typename TileOf, typename Body>
__device__ __forceinline__ void for_each_span(int n_tiles, TileOf&& tile_of, Body&& body) {
  constexpr int W = BS / 64;
  __shared__ int64_t part[W], found[2];
  const int tid = threadIdx.x, wave = tid >> 6;
  int64_t own = 0;
  for (int i = tid; i < n_tiles; i += BS) own += tile_of(i).cost();
  int64_t inc = wave_inclusive_scan(own);
  if ((tid & 63) == 63) part[wave] = inc;
  __syncthreads();
  int64_t total = 0;
  for (int k = 0; k < W; ++k) total += part[k];
  total = uniform(total);
  if (total == 0) return;
  const int64_t shares = max((int64_t)1, min((int64_t)gridDim.x, total / kMinShare));
  if ((int64_t)blockIdx.x >= shares) return;
  const int64_t lo = total * blockIdx.x / shares, hi = total * (blockIdx.x + 1) / shares;
  int64_t base = 0;
  for (int c = 0; c < n_tiles && base <= lo; c += BS) {
    int64_t v = own;
    if (n_tiles > BS) {
      v = c + tid < n_tiles ? tile_of(c + tid).cost() : 0;
      inc = wave_inclusive_scan(v);
      __syncthreads();  // part is read
      if ((tid & 63) == 63) part[wave] = inc;
      __syncthreads();
    }
    int64_t before = base + inc - v;
    for (int k = 0; k < W; ++k) {
      before += k < wave ? part[k] : 0;
      base += part[k];
    }
    base = uniform(base);
    if (before <= lo && lo < before + v) {  // one thread of the workgroup
      found[0] = c + tid;
      found[1] = before;
    }
  }
  __syncthreads();
  int t = __builtin_amdgcn_readfirstlane((int)found[0]);
  int64_t before = uniform(found[1]);
  for (;;) {
    int item = -1, count = 0;
    int64_t first = 0;
    for (; t < n_tiles && before < hi; ++t) {
      const TileWork w = tile_of(t);
      const int a = w.cut(lo - before), b = w.cut(hi - before);
      if (b > a) {
        const int64_t at = w.first + a;
        if (count == 0) {
          item = w.item;
          first = at;
        } else if (w.item != item || at != first + count || count >= 1 << 30 ||
                   ((at + (b - a) - 1) >> 32) != (first >> 32)) {
          break;  // the next span starts in this tile
        }
        count += b - a;
      }
      before += w.cost();
    }
    if (count == 0) return;
    body(item, first, count);
  }
}

}  // namespace mv
