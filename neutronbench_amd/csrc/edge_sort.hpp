// Stable radix sort of 64-bit elements by a run of their bits, for edge lists of 65,536 elements and more: a graph's
// edges by source and by destination (layout.hip), a schedule's edges by row and index (spmm.hip).
//
// Least significant digit first, digits of equal width of at most nine bits, so an 18-bit vertex id is two passes.
// A pass is bound by its bytes, eight read by the count, eight read and written by the scatter:
//   count    a block histograms its tile of 4,096 elements in LDS and writes one row of a [tiles, 512] table
//   prefix   the table's columns are added up, 128 tiles a block, then the blocks' totals and the digits by one block
//   scatter  a block ranks its tile, brings it into digit order in LDS and writes it out, eight elements of a digit on
//            average side by side
// Tiles that follow each other write neighbouring runs of every digit, so each XCD (blocks are dealt out to the eight in
// turn) takes an eighth of the tiles in order and its L2 puts the runs together to whole lines: 114.8 M edges, a
// scatter 0.90 ms with tiles in the blocks' order, 0.39 so (8,192 elements a tile, twice the run: 0.66 and 0.44), of which
// 0.33 are the bytes at a copy's rate.
// A tile is ranked as a sampled hop's chunk is (hop_sort_scatter_kernel): a wavefront's lanes with equal digits find each other
// with a ballot per digit bit, its own histogram in LDS counts the earlier rounds, and the wavefronts' histograms are
// added up in order.  42 KB of LDS, three blocks a CU, so that one block's loads run beside another's ranking.
#pragma once

#include "common.hpp"

namespace nts {

constexpr int kSortThreads = 512;
constexpr int kSortItems = 8;
constexpr uint32_t kSortTile = kSortThreads * kSortItems;
constexpr unsigned kSortDigitBits = 9;
constexpr uint32_t kSortBins = 1u << kSortDigitBits;
constexpr uint32_t kXcds = 8;
constexpr uint32_t kSortGroup = 128;  // tiles whose rows of the table one block of the prefix adds up

// Edges from which these passes are taken; the library's sort has fewer launches for shorter lists.  From an edge list to
// a chunk, us, the library's sort / these: 20 K edges 253 / 259, 100 K 342 / 311, 300 K 670 / 517, 1 M 1,067 / 833, 9 M with source
// ranges 2,658 / 2,041, 30 M 6,541 / 5,407, 114.8 M 15,492 / 10,025 (a pass of the library 0.6 ms for eight-byte pairs and 0.9 for a
// schedule's twelve, three of the former an order and five of the latter; here 0.42 and 0.20 for the count, two and four).
constexpr uint32_t kTiledSortEdges = 1u << 16;

using SortElement = unsigned long long;

// Where the last pass puts element v at position `at`: the element itself and its halves, each unless null.
struct SortSplit {
  SortElement *all;
  uint32_t *low, *high;
#if defined(__HIPCC__)
  __device__ __forceinline__ void operator()(uint32_t at, SortElement v) const {
    if (all) all[at] = v;
    if (low) low[at] = static_cast<uint32_t>(v);
    if (high) high[at] = static_cast<uint32_t>(v >> 32);
  }
#endif
};

inline uint32_t sort_tiles(uint32_t n) { return ceil_div(n, kSortTile); }
inline uint32_t sort_groups(uint32_t n) { return ceil_div(sort_tiles(n), kSortGroup); }
// Bytes of the count table: a row per tile and group, and one of the digits' first positions.
inline size_t sort_table_bytes(uint32_t n) {
  return (static_cast<size_t>(sort_tiles(n)) + sort_groups(n) + 1) * kSortBins * sizeof(uint32_t);
}

#if defined(__HIPCC__)
namespace {

__global__ __launch_bounds__(kSortThreads) void sort_count_kernel(uint32_t *__restrict__ table,
                                                                  const SortElement *__restrict__ in, uint32_t n,
                                                                  unsigned shift, uint32_t mask) {
  __shared__ uint32_t hist[kSortBins];
  const uint64_t first = static_cast<uint64_t>(blockIdx.x) * kSortTile;
  hist[threadIdx.x] = 0;
  __syncthreads();
  SortElement v[kSortItems];
#pragma unroll
  for (int j = 0; j < kSortItems; ++j) {
    const uint64_t e = first + j * kSortThreads + threadIdx.x;
    v[j] = e < n ? in[e] : 0;
  }
#pragma unroll
  for (int j = 0; j < kSortItems; ++j) {
    const bool active = first + j * kSortThreads + threadIdx.x < n;
    const uint32_t d = static_cast<uint32_t>(v[j] >> shift) & mask, d0 = wave_first(d);
    // Elements that come in order have one digit for whole wavefronts: one addition, not 64 to one counter.
    const uint64_t all = __ballot(active);
    if (__ballot(active && d == d0) == all) {
      if ((threadIdx.x & (kWave - 1)) == 0 && all) atomicAdd(&hist[d0], static_cast<uint32_t>(__popcll(all)));
    } else if (active) {
      atomicAdd(&hist[d], 1u);
    }
  }
  __syncthreads();
  table[static_cast<size_t>(blockIdx.x) * kSortBins + threadIdx.x] = hist[threadIdx.x];
}
static_assert(kSortThreads == static_cast<int>(kSortBins), "a thread per digit");

// rows [g * kSortGroup, ...) of the table become what the group's earlier tiles hold; sums[g] = the group's total.
__global__ __launch_bounds__(kSortThreads) void sort_prefix_kernel(uint32_t *__restrict__ table,
                                                                   uint32_t *__restrict__ sums, uint32_t tiles) {
  uint32_t *col = table + static_cast<size_t>(blockIdx.x) * kSortGroup * kSortBins + threadIdx.x;
  const uint32_t n = min(kSortGroup, tiles - blockIdx.x * kSortGroup);
  uint32_t run = 0;
  constexpr uint32_t U = 16;
  for (uint32_t t = 0; t < n; t += U) {
    uint32_t v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) v[u] = t + u < n ? col[static_cast<size_t>(t + u) * kSortBins] : 0u;
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      if (t + u < n) col[static_cast<size_t>(t + u) * kSortBins] = run;
      run += v[u];
    }
  }
  sums[static_cast<size_t>(blockIdx.x) * kSortBins + threadIdx.x] = run;
}

// sums[g] become what the earlier groups hold of each digit; first[d] = elements of the digits below d.
__global__ __launch_bounds__(kSortThreads) void sort_bases_kernel(uint32_t *__restrict__ sums,
                                                                  uint32_t *__restrict__ first, uint32_t groups) {
  __shared__ uint32_t wave_sums[kSortThreads / kWave];
  uint32_t run = 0;
  constexpr uint32_t U = 16;
  for (uint32_t g = 0; g < groups; g += U) {
    uint32_t v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) v[u] = g + u < groups ? sums[(g + u) * kSortBins + threadIdx.x] : 0u;
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      if (g + u < groups) sums[(g + u) * kSortBins + threadIdx.x] = run;
      run += v[u];
    }
  }
  uint32_t total;
  first[threadIdx.x] = block_prefix<kSortThreads>(run, wave_sums, &total);
}

template <typename Out>
__global__ __launch_bounds__(kSortThreads, 6) void sort_scatter_kernel(Out out, const SortElement *__restrict__ in,
                                                                    const uint32_t *__restrict__ table,
                                                                    const uint32_t *__restrict__ sums,
                                                                    const uint32_t *__restrict__ first, uint32_t n,
                                                                    unsigned shift, unsigned bits) {
  constexpr int kWaves = kSortThreads / kWave;
  __shared__ SortElement tile[kSortTile];
  __shared__ uint16_t wave_hist[kWaves][kSortBins];
  __shared__ uint32_t goes_to[kSortBins];  // position in the output, less the place in the tile, of a digit's elements
  __shared__ uint32_t wave_sums[kWaves];
  const uint32_t per_xcd = gridDim.x / kXcds, t = blockIdx.x % kXcds * per_xcd + blockIdx.x / kXcds;
  const uint64_t c0 = static_cast<uint64_t>(t) * kSortTile;
  if (c0 >= n) return;
  const uint32_t live = static_cast<uint32_t>(n - c0 < kSortTile ? n - c0 : kSortTile);
  const uint32_t mask = (1u << bits) - 1u;
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  SortElement v[kSortItems];
  uint32_t rank[kSortItems];
#pragma unroll
  for (int j = 0; j < kSortItems; ++j) {  // a wavefront's elements follow each other, 64 a round
    const uint32_t p = wave * (kWave * kSortItems) + j * kWave + lane;
    v[j] = p < live ? in[c0 + p] : 0;
  }
  const uint32_t start = first[threadIdx.x] + sums[static_cast<size_t>(t / kSortGroup) * kSortBins + threadIdx.x] +
                         table[static_cast<size_t>(t) * kSortBins + threadIdx.x];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) wave_hist[w][threadIdx.x] = 0;
  __syncthreads();
  uint16_t *hist = wave_hist[wave];
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (int j = 0; j < kSortItems; ++j) {
    const bool active = wave * (kWave * kSortItems) + j * kWave + lane < live;
    const uint32_t d = static_cast<uint32_t>(v[j] >> shift) & mask;
    uint64_t peers = __ballot(active);  // for an active lane: the active lanes with the same digit
    for (unsigned b = 0; b < bits; ++b) {
      const bool one = (d >> b) & 1u;
      const uint64_t votes = __ballot(one);
      peers &= one ? votes : ~votes;
    }
    const uint32_t seen = active ? hist[d] : 0u;
    rank[j] = seen + __popcll(peers & below);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // every lane has read its count before a leader raises it
    if (active && (peers & below) == 0) hist[d] = static_cast<uint16_t>(seen + __popcll(peers));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  __syncthreads();
  {  // a thread per digit: the wavefronts' counts become the place of their first element in the ordered tile
    uint32_t mine = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mine += wave_hist[w][threadIdx.x];
    uint32_t total;
    uint32_t run = block_prefix<kSortThreads>(mine, wave_sums, &total);
    goes_to[threadIdx.x] = start - run;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t c = wave_hist[w][threadIdx.x];
      wave_hist[w][threadIdx.x] = static_cast<uint16_t>(run);
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSortItems; ++j) {
    if (wave * (kWave * kSortItems) + j * kWave + lane < live)
      tile[hist[static_cast<uint32_t>(v[j] >> shift) & mask] + rank[j]] = v[j];
  }
  __syncthreads();
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < live; i += kSortThreads) {
    const SortElement e = tile[i];
    out(goes_to[static_cast<uint32_t>(e >> shift) & mask] + i, e);
  }
}

// Sorts in[0 .. n) by the bits [first_bit, first_bit + bits), stably, into `out`; `in` is kept.  a and b: n elements
// each, one of which may be `in` (it is then overwritten by the second pass); `table`: sort_table_bytes(n).  `finish`
// makes the last pass's output from the buffer that the pass does not read.
template <typename Finish>
hipError_t sort_elements(const SortElement *in, SortElement *a, SortElement *b, uint32_t n, unsigned first_bit,
                         unsigned bits, void *table, hipStream_t stream, Finish finish) {
  const uint32_t tiles = sort_tiles(n), groups = sort_groups(n);
  uint32_t *rows = static_cast<uint32_t *>(table);
  uint32_t *sums = rows + static_cast<size_t>(tiles) * kSortBins, *first = sums + static_cast<size_t>(groups) * kSortBins;
  const unsigned passes = (bits + kSortDigitBits - 1) / kSortDigitBits, width = (bits + passes - 1) / passes;
  const dim3 scatter_grid(ceil_div(tiles, kXcds) * kXcds);
  for (unsigned p = 0; p < passes; ++p) {
    const unsigned shift = first_bit + p * width, here = bits - p * width < width ? bits - p * width : width;
    SortElement *to = in == a ? b : a;
    hipLaunchKernelGGL(sort_count_kernel, dim3(tiles), dim3(kSortThreads), 0, stream, rows, in, n, shift, (1u << here) - 1u);
    hipLaunchKernelGGL(sort_prefix_kernel, dim3(groups), dim3(kSortThreads), 0, stream, rows, sums, tiles);
    hipLaunchKernelGGL(sort_bases_kernel, dim3(1), dim3(kSortThreads), 0, stream, sums, first, groups);
    if (p + 1 < passes) {
      hipLaunchKernelGGL(sort_scatter_kernel<SortSplit>, scatter_grid, dim3(kSortThreads), 0, stream,
                         SortSplit{to, nullptr, nullptr}, in, rows, sums, first, n, shift, here);
      in = to;
    } else {
      auto out = finish(to);
      hipLaunchKernelGGL(sort_scatter_kernel<decltype(out)>, scatter_grid, dim3(kSortThreads), 0, stream, out, in, rows, sums,
                         first, n, shift, here);
    }
    if (const hipError_t err = hipGetLastError(); err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace
#endif

}  // namespace nts
