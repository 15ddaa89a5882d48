// Edge <-> vertex movement, edge softmax and fused GAT attention kernels (replaces
// cuda/ntsCUDADistKernel.cuh:23-95, 166-260, cuda/ntsCUDAFuseKernel.cuh:492-506 and their
// launchers cuda/ntsCUDAGraphOP.cu:294-377, 449-474).
//
// Copies and per-edge products are edge-parallel (work per wavefront independent of any vertex's
// degree); per-destination reductions give one wavefront to one destination (or source) row, lanes
// spanning the feature / head dimension.  Sums run in edge order or through fixed-shape cross-lane
// butterflies, and nothing uses float atomics, so every result is bit-reproducible.
#include <algorithm>

#include "common.hpp"
#include "launch_size.hpp"

namespace nts {
namespace {

__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & (kWave - 1); }

// ---- vertex -> edge copies ------------------------------------------------------------------
//
// Edge-parallel: the edge count is read on the device (co[Vd]); a wavefront takes 64 consecutive
// edges per step, every lane looks up the feature row its edge copies from (the source id, or the
// destination that owns the edge, followed along the wavefront's contiguous span of edges), and
// sub-wavefront groups of G lanes then move 64/G rows at a time.  Work per wave does not depend on
// any vertex's degree.  Bound by the writes of the messages (1.27 GB: a fill takes 187 us; 412 -> 287 us from the
// destinations, 460 -> 367 from the sources, which also read as much from the caches): the next four
// rows are requested before these four are stored, because a wavefront's loads and stores complete in order and a load
// behind the stores would wait for them; and the stores leave the feature rows in the caches
// (outgrows_caches).

enum CopyMode { kFromSrc = 0, kFromDst = 1, kAddFromDst = 2 };

// owner_of by the whole wavefront (all 64 lanes call it, the result is the same on every lane): the lanes
// probe 64 evenly spaced offsets of the remaining range at once, so a search over 10^5 rows is three
// rounds of one load instead of seventeen dependent ones -- what a wavefront that walks only a step or
// two of a small edge list otherwise spends most of its time on.
__device__ __forceinline__ uint32_t owner_of_wave(const uint32_t *__restrict__ off, uint32_t n, uint32_t pos) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  uint32_t lo = 0, hi = n;  // answer in [lo, hi)
  while (hi - lo > 1) {
    const uint32_t step = (hi - lo + kWave - 1) / kWave;
    const uint64_t idx = static_cast<uint64_t>(lo) + static_cast<uint64_t>(lane + 1) * step;  // ascending probes
    const bool behind = idx < hi && off[idx] <= pos;
    const uint32_t k = __popcll(__ballot(behind));  // probes are ascending: the first k are not beyond pos
    lo += k * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo;
}

// Messages beyond half of the 256 MB last-level cache are gone from it before the next operator asks for them,
// and on their way they push out the feature rows and offsets that every operator reads: they are moved
// with non-temporal loads and stores.  Smaller ones stay in the cache for the next operator.  An operator chain
// (copies, softmax, sums, forward and backward), us, ordinary -> non-temporal: 26 MB of messages 528 -> 630,
// 51 MB 455 -> 489, 205 MB 950 -> 854, 1,024 MB 2,490 -> 2,306.
constexpr uint64_t kStreamedBytes = 128ull << 20;
constexpr uint32_t kTurnBytes = 32u << 10;
__device__ __forceinline__ bool outgrows_caches(uint64_t message_bytes) { return message_bytes > kStreamedBytes; }
__device__ __forceinline__ void store_streamed(float *p, float v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void store_streamed(float4 *p, float4 v) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 w = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(w, reinterpret_cast<f4 *>(p));
}

__device__ __forceinline__ void vsum(float &r, float a, float b) { r = a + b; }
__device__ __forceinline__ void vsum(float4 &r, float4 a, float4 b) {
  r = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float load_streamed(const float *p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ float4 load_streamed(const float4 *p) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 w = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(p));
  return make_float4(w.x, w.y, w.z, w.w);
}

template <typename V, int G>
__global__ __launch_bounds__(256) void edge_copy_kernel(V *__restrict__ msg, const V *__restrict__ feat,
                                                        const uint32_t *__restrict__ ri,
                                                        const uint32_t *__restrict__ co,
                                                        const uint32_t *__restrict__ mirror, uint32_t Vd, uint32_t Fv,
                                                        int mode) {
  const uint32_t E = co[Vd];
  const uint32_t lane = lane_id();
  const uint32_t gl = lane & (G - 1), grp = lane / G;
  constexpr uint32_t kEdgesPerStep = kWave / G;
  constexpr int U = G < 4 ? G : 4;  // rows of a group requested together
  const bool streamed = outgrows_caches(static_cast<uint64_t>(E) * Fv * sizeof(V));
  const uint64_t wave = wave_of_grid();
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  // A wavefront walks a contiguous span of wave steps: the destination that owns each step's edges
  // follows from the previous step's (owners_of_step) instead of a search per lane.  Messages that outgrow the caches are
  // walked in turns of some 32 KB, one wavefront's after the other's, so that those in flight write one stretch of
  // memory: from destinations 2.48 M edges of 128 floats 228 -> 200 us (a fill of as many bytes 184), 8 M 1,013 -> 934;
  // from sources 1,286 -> 1,224 (8 M of 128).
  const uint64_t total_steps = (static_cast<uint64_t>(E) + kWave - 1) / kWave;
  const uint64_t per_wave = (total_steps + n_waves - 1) / n_waves;
  // Rows of up to four vectors have no second loop: the edges are counted on the device, so messages of every size would pay
  // for its registers (rows of 16 floats: 64 -> 80, eight wavefronts per SIMD -> six; 1.2 M edges from sources 20.6 us and
  // 21.8 with it, of 12 floats 18.0, 20.4), and the order gives such rows little (8 M edges of 16 147, 147, from destinations
  // 91.8, 90.5; 40 M 487, 444).
  constexpr bool kTurns = sizeof(V) == 16 && G >= 8;
  uint64_t span = per_wave;
  if (kTurns && streamed) {
    const uint32_t turn_steps = Fv < kTurnBytes / (kWave * sizeof(V)) ? kTurnBytes / (kWave * sizeof(V)) / Fv : 1u;
    if (turn_steps < per_wave) span = turn_steps;
  }
  uint64_t first_step = wave * span;
  if (first_step >= total_steps) return;
  do {
    const uint64_t end_step = first_step + span < total_steps ? first_step + span : total_steps;
    uint32_t d0 = mode == kFromSrc ? 0u : owner_of_wave(co, Vd, static_cast<uint32_t>(first_step * kWave));
    for (uint64_t step = first_step; step < end_step; ++step) {
      const uint64_t base = step * kWave;
      const uint64_t e = base + lane;
      uint32_t row = 0;
      if (mode == kFromSrc) {
        if (e < E) {
          row = ri[e];
          if (mirror) row = mirror[row];
        }
      } else {
        row = owners_of_step(co, Vd, static_cast<uint32_t>(base), d0);
      }
      auto holder_of = [&](uint32_t j) { return j * kEdgesPerStep + grp; };  // lane that looked up this group's edge
      if (Fv <= G) {
        const bool col_live = gl < Fv;
        auto request = [&](uint32_t j0, V(&v)[U]) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint32_t holder = holder_of(j0 + u), r = __shfl(row, holder, kWave);
            if (base + holder < E && col_live) v[u] = feat[static_cast<size_t>(r) * Fv + gl];
          }
        };
        V cur[U], nxt[U];
        request(0, cur);
#pragma unroll
        for (uint32_t j0 = 0; j0 < G; j0 += U) {
          if (j0 + U < G) request(j0 + U, nxt);
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const uint64_t ee = base + holder_of(j0 + u);
            if (ee < E && col_live) {
              V *dst = msg + ee * Fv + gl;
              V v = cur[u];
              if (mode == kAddFromDst) vsum(v, *dst, v);
              if (streamed) store_streamed(dst, v);
              else *dst = v;
            }
          }
#pragma unroll
          for (int u = 0; u < U; ++u) cur[u] = nxt[u];
        }
        continue;
      }
      for (uint32_t j = 0; j < G; ++j) {
        const uint32_t holder = holder_of(j), r = __shfl(row, holder, kWave);
        const uint64_t ee = base + holder;
        if (ee < E) {
          const V *src = feat + static_cast<size_t>(r) * Fv;
          V *dst = msg + ee * Fv;
          for (uint32_t c = gl; c < Fv; c += G) {
            V v = src[c];
            if (mode == kAddFromDst) vsum(v, dst[c], v);
            if (streamed) store_streamed(dst + c, v);
            else dst[c] = v;
          }
        }
      }
    }
    first_step += n_waves * span;
  } while (kTurns && first_step < total_steps);
}

// ---- edge -> vertex sums ----------------------------------------------------------------------
//
// Rows with at most `long_limit` edges: a group of G lanes per row (64/G rows per wavefront) adds
// the row's edge rows in order; where the edge rows of consecutive vertices follow each other in
// memory (no permutation), a wavefront streams the edges of a run of rows through LDS instead (same
// sums).  Longer rows (power-law hubs) are listed first and summed by the first blocks of the same
// launch, which spread a row's edges over the slices of the block and add
// the slices' partial sums in a fixed order; calls of fewer than kLongMinVertices rows list none, and their first blocks
// find the hub rows themselves (few_long_edges).

constexpr uint32_t kNoLimit = 0xFFFFFFFFu;
constexpr uint32_t kLongRowEdges = 1024;    // edges of a row above which the block kernel takes over
constexpr uint64_t kGiantValues = 131072;   // softmax segments above this many values are cut into pieces, at most
constexpr uint64_t kGiantRowBytes = 1u << 20;  // row of edge rows above which it is cut into pieces for several blocks
constexpr uint32_t kLongRowValues = 32768;  // the same for softmax segments, in values (edges * heads), at most
constexpr uint32_t kLongRowMinValues = 2048;   // and at least
constexpr uint64_t kGiantMinValues = 32768;
constexpr uint32_t kByTotal = 0;               // in place of a line: long_segment_values of the call's values
constexpr uint32_t kByFewTotal = 1;            // few_long_values of them
constexpr uint32_t kLongMinVertices = 16384;  // vertex count below which the extra launches are not worth it
constexpr int kLongBlock = 1024;

// What the first blocks of a row launch do beside it when the rows above `long_limit` edges are summed
// in the same launch: the list of those rows, the piece table of the giant ones, where the pieces' sums
// go, the column tile of a 256-thread block, how many blocks are set aside (0: none), and whether hub rows are looked for
// where there is no list (few_long_edges); how many slices of a listed row a thread adds up.
template <typename V>
struct LongRowWork {
  const uint32_t *list, *count, *hdr;
  const uint4 *pieces;
  V *partial;
  uint32_t tile, blocks;
  bool own;
  uint32_t chains;
};

__device__ __forceinline__ void vadd(float &a, const float &b) { a += b; }
__device__ __forceinline__ void vadd(float4 &a, const float4 &b) {
  a.x += b.x;
  a.y += b.y;
  a.z += b.z;
  a.w += b.w;
}
template <typename V>
__device__ __forceinline__ V vnull();
template <>
__device__ __forceinline__ float vnull<float>() {
  return 0.f;
}
template <>
__device__ __forceinline__ float4 vnull<float4>() {
  return make_float4(0.f, 0.f, 0.f, 0.f);
}

// Sum of the columns [first_col, end_col) of the edge rows [e0, e1) by one block of 256 threads, added into dst (V = float, or
// float4 when rows are 16-byte aligned: a quarter of the load instructions and of the rounds a row
// takes).  They are at most `tile` vectors (a power of two <= 256); thread t owns
// column t % tile of C of the C * 256 / tile slices, a slice adds every so many-th edge of the range in ascending
// order (a round's loads together), and the slices' sums are then added pairwise in a fixed tree, the upper half to the lower.
// SKIP: nothing is requested beyond the range.
template <typename V, int U, int C, bool SKIP>
__device__ __forceinline__ void block_sum_edge_rows(V *__restrict__ dst, const V *__restrict__ msg,
                                                    const uint32_t *__restrict__ perm, uint32_t e0, uint32_t e1,
                                                    uint32_t Fv, uint32_t first_col, uint32_t end_col, uint32_t tile,
                                                    int accumulate, V *part) {
  const uint32_t slice = threadIdx.x / tile, n_slices = 256 / tile, col = first_col + (threadIdx.x & (tile - 1));
  static_assert(U % C == 0 && C <= 4, "a round's first load is the first slice's");
  V a[C];
#pragma unroll
  for (int j = 0; j < C; ++j) a[j] = vnull<V>();
  if (col < end_col && e1 - e0 > slice) {
    // The edge ids of the next round are requested while the rows of this one are on their way; beyond the range the last edge's, which
    // costs rows of a vector or two floats through a permutation, a line of memory a request, more than the rounds without a choice at each load give
    // (60 K rows, 4 M edges F = 1 109 -> 102 us, F = 4 119 -> 113; but F = 7 171 -> 230, 30 K, 3 M F = 47 230 -> 658).
    // Through a permutation, 2.48 M edges of 47 floats 704 -> 379 us.  Eight vectors a round took the kernels 98 registers instead of
    // 62 (30 K rows, 3 M edges F = 128 467, held to 72 with spills 502, four a round 467); narrow rows, whose kernels hold as many anyway,
    // have room for them.
    uint32_t k = e0 + slice, left = e1 - k, id[U];
    auto request_ids = [&] {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool there = u * n_slices < left;
        const uint32_t kk = k + (there ? u * n_slices : left - 1);
        if (SKIP) id[u] = 0;
        if (!SKIP || there) id[u] = perm ? perm[kk] : kk;
      }
    };
    request_ids();
    while (left) {
      V v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (SKIP) v[u] = vnull<V>();
        if (!SKIP || u * n_slices < left) v[u] = msg[static_cast<size_t>(id[u]) * Fv + col];
      }
      const uint32_t now = left;
      left = left > U * n_slices ? left - U * n_slices : 0u;
      if (left) {
        k += U * n_slices;
        request_ids();
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (u * n_slices < now) vadd(a[u % C], v[u]);
    }
  }
#pragma unroll
  for (int half = C / 2; half >= 1; half /= 2)
#pragma unroll
    for (int j = 0; j < half; ++j) vadd(a[j], a[j + half]);
  part[threadIdx.x] = a[0];
  __syncthreads();
  for (uint32_t stride = n_slices / 2; stride >= 1; stride >>= 1) {
    if (slice < stride) {
      V lo = part[threadIdx.x];
      vadd(lo, part[threadIdx.x + stride * tile]);
      part[threadIdx.x] = lo;
    }
    __syncthreads();
  }
  if (slice == 0 && col < end_col) {
    V total = part[threadIdx.x];
    if (accumulate) vadd(total, dst[col]);
    dst[col] = total;
  }
  __syncthreads();
}

// The same columns (tile vectors from first_col on, at most 32 floats) as one running sum in edge order: the block stages U vectors a
// thread in LDS while the next ones are on their way, and the threads that each own a float add them up.  some 12 ns an
// edge, what the additions take one after the other, where a lane group that loads and adds by itself takes 60 to 125.  `staged` holds 256 U vectors.
template <typename V, int U>
__device__ __forceinline__ void block_running_sum(V *__restrict__ dst, const V *__restrict__ msg, const uint32_t *__restrict__ perm,
                                                  uint32_t e0, uint32_t e1, uint32_t Fv, uint32_t first_col, uint32_t end_col, uint32_t tile,
                                                  int accumulate, V *staged) {
  constexpr uint32_t NF = sizeof(V) / 4;
  const uint32_t slice = threadIdx.x / tile, n_slices = 256 / tile, col = first_col + (threadIdx.x & (tile - 1));
  const uint32_t read_col = col < end_col ? col : end_col - 1;
  const uint32_t own = threadIdx.x, floats = tile * NF, live_floats = (end_col - first_col) * NF;
  uint32_t k = e0, left = e1 - e0, id[U];
  V v[U];
  auto request_ids = [&] {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t at = u * n_slices + slice, kk = k + (at < left ? at : left - 1);
      id[u] = perm ? perm[kk] : kk;
    }
  };
  auto request_rows = [&] {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = msg[static_cast<size_t>(id[u]) * Fv + read_col];
  };
  request_ids();
  request_rows();
  float a = 0.f;
  while (left) {
    const uint32_t now = left < U * n_slices ? left : U * n_slices;
    __syncthreads();  // the values before these have been added
#pragma unroll
    for (int u = 0; u < U; ++u) staged[u * 256 + threadIdx.x] = v[u];
    __syncthreads();
    k += now;
    left -= now;
    if (left) {
      request_ids();
      request_rows();
    }
    if (own < floats) {
      const float *f = reinterpret_cast<const float *>(staged) + own;
      uint32_t i = 0;
      for (; i + 16 <= now; i += 16) {
        float t[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) t[q] = f[(i + q) * floats];
#pragma unroll
        for (int q = 0; q < 16; ++q) a += t[q];
      }
      for (; i < now; ++i) a += f[i * floats];
    }
  }
  if (own < live_floats) {
    float *d = reinterpret_cast<float *>(dst + first_col) + own;
    *d = accumulate ? a + *d : a;
  }
  __syncthreads();
}

// Calls of fewer than kLongMinVertices rows, whose hub rows no launch lists: the edges of a row above which it is the first
// blocks', so that there are fewer than kFewLongRows of them.  Such rows stay one running sum in edge order, whoever adds them up (a
// sum in slices is three times as fast on dense graphs but 1.6e-6 of itself from what these calls returned before).  A lane group or a
// wavefront added a hub row up before, 8 or 16 edges a memory latency: contiguous / permuted sums, us, 2.9 K rows, 110 K edges F = 47 842 / 922
// -> 57 / 62, F = 128 903 / 945 -> 59 / 64; 10 K, 3 M F = 47 5,932 / 11,554 -> 939 / 1,074, F = 128 4,873 / 11,117 -> 1,225 / 1,364; 16 K, 1 M F = 128
// 1,604 / 3,746 -> 459 / 510; 16 K, 40 K F = 128 67 / 275 -> 33 / 38.  Rows of up to eight vectors, which a wavefront stages by itself, gain where
// there are few of them (kMaxNarrowHubRows): 4 K, 2 M F = 4 7,269 / 9,055 -> 1,001 / 1,054, but 16 K, 1 M 313 / 268 -> 329 / 351;
// through a permutation eight vectors do in any case: F = 32 10 K, 3 M 3,768 -> 1,625, 16 K, 1 M 976 -> 615.
constexpr uint32_t kMaxNarrowHubRows = 4096;
constexpr uint32_t kFewLongRows = 2048;
constexpr uint32_t kMinHubGroups = 64;
static_assert(kLongMinVertices <= 256 * kMinHubGroups && kLongMinVertices % 2 == 0, "a row a thread");
template <typename V, int G>
constexpr int kHubLoads = sizeof(V) == 16 && G > 8 ? 4 : 8;  // vectors that a thread of a hub block requests together
template <typename V, int OWN>
constexpr uint32_t kHubBytes = 256 * sizeof(V) * (OWN > 1 ? OWN : 1);  // scratch of a block that looks for them
__device__ __forceinline__ uint32_t few_long_edges(const uint32_t *__restrict__ off, uint32_t rows) {
  const uint32_t share = (off[rows] - off[0]) / kFewLongRows;
  return share < kLongRowEdges ? kLongRowEdges : share;
}
template <typename V>
__device__ __forceinline__ uint32_t long_limit_of(const LongRowWork<V> &lw, uint32_t limit, const uint32_t *__restrict__ off, uint32_t rows) {
  return lw.own ? few_long_edges(off, rows) : limit;
}

// The first blocks of a row launch take the listed long rows, one 256-thread block per row, and the
// pieces of the giant ones (their partial sums are combined by a launch of its own afterwards); the
// rows of the launch proper fill the chip meanwhile.
template <typename V, int U, int OWN, bool WIDE = false, bool SKIP = false>
__device__ __forceinline__ void sum_long_rows_in_this_block(V *__restrict__ out, const V *__restrict__ msg,
                                                            const uint32_t *__restrict__ off,
                                                            const uint32_t *__restrict__ perm, uint32_t rows, uint32_t Fv,
                                                            int accumulate, const LongRowWork<V> &lw, void *scratch) {
  V *part = static_cast<V *>(scratch);  // 256 of them, 256 OWN without a list
  if constexpr (OWN > 0) if (!lw.list) {
    // Few enough rows for these blocks to find the hubs among them: the rows are dealt out to groups of blocks in an order without
    // pattern (hubs of a generated graph have neighbouring numbers), a row a thread, and the blocks of a group take the column
    // tiles of the hub rows among its own.  (A list of all hub rows in every block took it 20 us where the offsets were not in its L2.)
    __shared__ uint32_t n_found;
    __shared__ uint16_t found[256];
    if (threadIdx.x == 0) n_found = 0;
    const uint32_t tiles = (Fv + lw.tile - 1) / lw.tile, most = lw.blocks / kMinHubGroups, sharers = tiles < most ? tiles : most;
    const uint32_t groups = lw.blocks / sharers, group = blockIdx.x / sharers;
    const uint32_t at = threadIdx.x * groups + group, r = at * 40503u % kLongMinVertices;  // (odd: every row once)
    uint32_t deg = 0;
    if (group < groups && at < kLongMinVertices && r < rows) deg = off[r + 1] - off[r];
    const uint32_t limit = few_long_edges(off, rows);
    __syncthreads();
    if (deg > limit) found[atomicAdd(&n_found, 1u)] = static_cast<uint16_t>(r);
    __syncthreads();
    const uint32_t n = n_found;
    for (uint32_t i = 0; i < n; ++i) {
      const uint32_t row = found[i];
      for (uint32_t t = blockIdx.x % sharers; t < tiles; t += sharers) {
        const uint32_t c0 = t * lw.tile, c1 = c0 + lw.tile < Fv ? c0 + lw.tile : Fv;
        block_running_sum<V, OWN>(out + static_cast<size_t>(row) * Fv, msg, perm, off[row], off[row + 1], Fv, c0, c1, lw.tile, accumulate, part);
      }
    }
    return;
  }
  // the column tiles of a listed row one after the other, then those of the pieces
  const uint32_t tiles = (Fv + lw.tile - 1) / lw.tile;
  const uint64_t n_rows = static_cast<uint64_t>(*lw.count) * tiles, n_all = n_rows + static_cast<uint64_t>(lw.hdr[1]) * tiles;
  for (uint64_t i = blockIdx.x; i < n_all; i += lw.blocks) {
    const uint64_t at = (i < n_rows ? i : i - n_rows) / tiles;
    const uint32_t c0 = static_cast<uint32_t>(i % tiles) * lw.tile, c1 = c0 + lw.tile < Fv ? c0 + lw.tile : Fv;
    uint32_t e0, e1;
    V *dst;
    if (i < n_rows) {
      const uint32_t r = lw.list[at];
      e0 = off[r];
      e1 = off[r + 1];
      dst = out + static_cast<size_t>(r) * Fv;
    } else {
      const uint4 pc = lw.pieces[at];
      e0 = pc.z;
      e1 = pc.w;
      dst = lw.partial + at * Fv;
    }
    const int add = i < n_rows && accumulate;
    if (WIDE && lw.chains == 4) block_sum_edge_rows<V, U, WIDE ? 4 : 1, false>(dst, msg, perm, e0, e1, Fv, c0, c1, lw.tile, add, part);
    else block_sum_edge_rows<V, U, 1, SKIP>(dst, msg, perm, e0, e1, Fv, c0, c1, lw.tile, add, part);
  }
}

// out[r,:] (+)= sum_{k in [off[r], off[r+1])} msg[perm ? perm[k] : k, :], added in k order: a group of G lanes for every row and
// every G vectors of it from first_group on.  The edge rows of a round are requested together and their ids a round ahead, so that a long row is a
// memory latency per U edges; the last, partial rounds are of eight, whose requests beyond the row are its last edge's again.
template <typename V, int G, int U>
__global__ __launch_bounds__(256, (U > 8 ? 4 : 8)) void gather_edge_to_row_kernel(V *__restrict__ out, const V *__restrict__ msg,
                                                                 const uint32_t *__restrict__ off,
                                                                 const uint32_t *__restrict__ perm, uint32_t rows,
                                                                 uint32_t Fv, int accumulate, uint32_t long_limit, uint32_t tiles,
                                                                 uint64_t first_group, LongRowWork<V> lw) {
  if (blockIdx.x < lw.blocks) {
    constexpr int kOwn = sizeof(V) == 16 ? 4 : U > 8 ? 16 : 0;  // (of floats, only the few rows' kernel has rows without a list)
    __shared__ V scratch[kHubBytes<V, kOwn> / sizeof(V)];
    sum_long_rows_in_this_block<V, sizeof(V) == 16 ? 4 : 8, kOwn, G == kWave && U == 8>(out, msg, off, perm, rows, Fv, accumulate, lw, scratch);
    return;
  }
  long_limit = long_limit_of(lw, long_limit, off, rows);
  const uint64_t group = first_group + (static_cast<uint64_t>(blockIdx.x - lw.blocks) * blockDim.x + threadIdx.x) / G;
  if (group >= static_cast<uint64_t>(rows) * tiles) return;
  const uint32_t r = static_cast<uint32_t>(group / tiles), c = static_cast<uint32_t>(group % tiles) * G + (threadIdx.x & (G - 1));
  if (c >= Fv) return;
  const uint32_t e0 = off[r], e1 = off[r + 1];
  if (e1 - e0 > long_limit) return;
  V a = vnull<V>();
  uint32_t k = e0, left = e1 - e0;
  if (left >= U) {
    uint32_t id[U];
    auto request_ids = [&] {
#pragma unroll
      for (int u = 0; u < U; ++u) id[u] = perm ? perm[k + u] : k + u;
    };
    request_ids();
    do {
      V v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = msg[static_cast<size_t>(id[u]) * Fv + c];
      k += U;
      left -= U;
      if (left >= U) request_ids();
#pragma unroll
      for (int u = 0; u < U; ++u) vadd(a, v[u]);
    } while (left >= U);
  }
  while (left) {
    V v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t kk = k + (u < left ? u : left - 1);
      v[u] = msg[static_cast<size_t>(perm ? perm[kk] : kk) * Fv + c];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (u < left) vadd(a, v[u]);
    k += 8;
    left = left > 8 ? left - 8 : 0u;
  }
  V *p = out + static_cast<size_t>(r) * Fv + c;
  if (accumulate) vadd(a, *p);
  *p = a;
}

// Smallest row r in [0, rows] whose weight before it, (off[r] - off0) + r, is at least x (x at most the
// weight before `rows`, the total), searched by the whole wavefront like owner_of_wave.
__device__ __forceinline__ uint32_t first_row_of_weight(const uint32_t *__restrict__ off, uint32_t rows, uint32_t off0,
                                                        uint64_t x) {
  if (x == 0) return 0;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint64_t pos = x - 1;
  uint32_t lo = 0, hi = rows + 1;  // the largest row whose weight is at most pos lies in [lo, hi)
  while (hi - lo > 1) {
    const uint32_t step = (hi - lo + kWave - 1) / kWave;
    const uint64_t idx = static_cast<uint64_t>(lo) + static_cast<uint64_t>(lane + 1) * step;
    const bool behind = idx < hi && static_cast<uint64_t>(off[idx] - off0) + idx <= pos;
    const uint32_t k = __popcll(__ballot(behind));
    lo += k * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo + 1 < rows ? lo + 1 : rows;  // at most `rows` for ascending offsets; never beyond them for any input
}

// Edge rows that lie one after the other in memory (no permutation: the sums over a destination's
// edges) and are at most one wavefront wide: a wavefront takes 64 consecutive rows, whose edges are one
// contiguous range, and streams that range through a tile of LDS private to it -- all 64 lanes load
// consecutive 4- or 16-byte vectors, the next round is requested before this one is added up -- while
// the lanes that each own one float of an output row (up to four from 32 lanes of 16 bytes on) walk the
// tile edge by edge and write a row out
// where it ends: the running fp32 sum in edge order, as in the kernel below, without a loop per lane
// group and its hand-out of rows.  Rows above `long_limit` edges are skipped (the first blocks of the
// launch sum them); empty rows are written as zeros (or left, when accumulating).
template <typename V, int G>
__global__ __launch_bounds__(256) void gather_edge_to_row_stream_kernel(V *__restrict__ out, const V *__restrict__ msg,
                                                                        const uint32_t *__restrict__ off,
                                                                        uint32_t rows, uint32_t Fv, int accumulate,
                                                                        uint32_t long_limit, LongRowWork<V> lw) {
  constexpr int NF = sizeof(V) / 4;
  constexpr int U = 8;                            // loads per lane and round
  __shared__ __align__(16) float tiles[4][kWave * U * NF];
  if (blockIdx.x < lw.blocks) {
    static_assert(sizeof(tiles) >= kHubBytes<V, 8>, "the hub blocks' scratch");
    sum_long_rows_in_this_block<V, kHubLoads<V, G>, G <= 8 ? 8 : 0>(out, msg, off, static_cast<const uint32_t *>(nullptr), rows, Fv, accumulate, lw, tiles);
    return;
  }
  long_limit = long_limit_of(lw, long_limit, off, rows);
  constexpr uint32_t kSlots = kWave / G;          // edge rows per load of the wavefront
  constexpr uint32_t kRound = kSlots * U;         // edge rows per round
  constexpr uint32_t kPitch = G * NF;             // floats of an edge row in the tile
  float *tile = tiles[wave_of_block()];
  const uint32_t lane = lane_id();
  const uint32_t col = lane & (G - 1), slot = lane / G;
  const bool col_live = col < Fv;
  const uint32_t comps = Fv * NF;  // floats of an output row: lane c owns the floats c + 64 k below comps
  constexpr int OWN = (G * NF + kWave - 1) / kWave;  // floats a lane owns at most (1 up to 16 lanes of 16 bytes)
  const uint64_t wave = wave_of_grid(lw.blocks);
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x - lw.blocks) * blockDim.x / kWave;
  // The wavefronts share the rows by weight, a row counting one plus its edges: wavefront w takes the
  // rows r with w C <= (off[r] - off[0]) + r < (w + 1) C.
  const uint32_t off0 = off[0];
  const bool streamed = outgrows_caches(static_cast<uint64_t>(off[rows] - off0) * Fv * sizeof(V));
  const uint64_t total = static_cast<uint64_t>(off[rows] - off0) + rows;
  const uint64_t share = (total + n_waves - 1) / n_waves;
  const uint64_t x0 = wave * share < total ? wave * share : total;
  const uint64_t x1 = x0 + share < total ? x0 + share : total;
  if (x0 == x1) return;
  const uint32_t r_begin = first_row_of_weight(off, rows, off0, x0);
  const uint32_t r_end = first_row_of_weight(off, rows, off0, x1);
  // The whole walk once per kind of load: a choice at each load keeps them from being in flight together.
  auto walk = [&](auto load) {
    for (uint64_t base = r_begin; base < r_end; base += kWave) {
      const uint32_t n_set = r_end - base < kWave ? static_cast<uint32_t>(r_end - base) : kWave;
      uint32_t my_e1 = 0;
      if (lane < n_set) my_e1 = off[base + lane + 1];
      uint32_t pos = off[base];                       // next edge to add (wave-uniform)
      const uint32_t range_end = wave_read(my_e1, n_set - 1);
      uint32_t j = 0;                                 // current row of the set
      float acc[OWN];
#pragma unroll
      for (int o = 0; o < OWN; ++o) acc[o] = 0.f;
      V cur[U];
      auto load_round = [&](uint32_t k) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          cur[u] = V{};
          const uint32_t idx = k + u * kSlots + slot;
          if (idx < range_end && col_live) cur[u] = load(msg + static_cast<size_t>(idx) * Fv + col);
        }
      };
      // Rows that end at `pos` are complete: written out (a skipped long row is not), next row.
      auto finish_rows = [&](bool skip_first) {
        bool skip = skip_first;
        while (j < n_set && wave_read(my_e1, j) == pos) {
          if (!skip) {
#pragma unroll
            for (int o = 0; o < OWN; ++o) {
              const uint32_t c = lane + o * kWave;
              if (c < comps) {
                float *p = reinterpret_cast<float *>(out) + (base + j) * comps + c;
                float v = acc[o];
                if (accumulate) v += *p;
                *p = v;
              }
            }
          }
          skip = false;
#pragma unroll
          for (int o = 0; o < OWN; ++o) acc[o] = 0.f;
          ++j;
        }
      };
      finish_rows(false);  // empty rows at the head of the set
      uint32_t loaded = 0xFFFFFFFFu;  // first edge of the round held in `cur`
      while (j < n_set) {
        const uint32_t row_end = wave_read(my_e1, j);
        if (row_end - pos > long_limit) {  // pos is this row's first edge: nothing of it has been added
          pos = row_end;
          finish_rows(true);
          continue;
        }
        const uint32_t ts = pos;  // this round covers [ts, ts + kRound)
        if (loaded != ts) load_round(ts);
        __builtin_amdgcn_wave_barrier();  // the previous round's reads of the tile are done
#pragma unroll
        for (int u = 0; u < U; ++u) reinterpret_cast<V *>(tile)[u * kWave + lane] = cur[u];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        loaded = ts + kRound;
        if (loaded < range_end) load_round(loaded);  // in flight while this round is added up
        const uint32_t tile_end = range_end - ts < kRound ? range_end : ts + kRound;
        while (pos < tile_end && j < n_set) {
          const uint32_t e1 = wave_read(my_e1, j);
          if (e1 - pos > long_limit) break;  // a long row starts here (a shorter one never has that much left)
          const uint32_t end = e1 < tile_end ? e1 : tile_end;
#pragma unroll
          for (int o = 0; o < OWN; ++o) {
            if (lane + o * kWave < comps) {
              const float *t = tile + (pos - ts) * kPitch + lane + o * kWave;
              float a = acc[o];
              uint32_t i = pos;
              for (; i + 4 <= end; i += 4, t += 4 * kPitch) {
                a += t[0];
                a += t[kPitch];
                a += t[2 * kPitch];
                a += t[3 * kPitch];
              }
              for (; i < end; ++i, t += kPitch) a += t[0];
              acc[o] = a;
            }
          }
          pos = end;
          if (pos == e1) finish_rows(false);
        }
      }
    }
  };
  if (streamed) walk([](const V *p) { return load_streamed(p); });
  else walk([](const V *p) { return *p; });
}

// The same sums for rows that fit one group (Fv <= G), with the rows of a wavefront handed out
// dynamically: a wavefront takes kFullSet consecutive rows (FEW: `few_rows`, see balanced_rows_per_wave), reads their offsets with one coalesced load,
// and its 64/G groups then pull rows from that set one after the other -- a group that finishes a
// short row takes the next pending one instead of idling until the longest row of a fixed
// assignment is done.  Every group adds its row's edge rows in order (eight loads in flight), so
// the result does not depend on which group happened to take which row.
//
// Narrow rows (G * sizeof(V) of 16 to 64 bytes) leave a lone lane or two with the whole row: a
// 1,000-edge row is then 125 dependent rounds of eight loads.  There S slices of G lanes share a
// row: together they load 8 S consecutive edge rows at once, and every lane of the group then adds
// those values in edge order, fetching each from the lane that loaded it.  The sum is the same
// running fp32 sum, bit for bit; only the loads are spread.
//
// Rows of more than `coop_limit` edges (G <= 8 only) are taken by the whole wavefront after the
// set's other rows: all 64 lanes load consecutive edge rows (256 values of type V per round), stage
// them in a tile of LDS private to the wavefront, and request the next round's rows before the
// lanes that each own one float of the output row add the staged values in edge order -- again the
// same running fp32 sum (the tile is padded with zeros, and a sum that starts at +0 is never -0, so
// the padding changes no bit).  A 1,000-edge row of 16-byte values is four such rounds instead of
// sixteen dependent ones.
template <int GG>  // lanes that share a row
constexpr uint32_t kFullSet = kWave / GG * 8u < kWave ? kWave / GG * 8u : static_cast<uint32_t>(kWave);
template <typename V, int G, int S, bool FEW>
__global__ __launch_bounds__(256, (sizeof(V) == 4 ? 8 : G <= 8 ? 5 : 1)) void gather_edge_to_row_balanced_kernel(V *__restrict__ out,
                                                                          const V *__restrict__ msg,
                                                                          const uint32_t *__restrict__ off,
                                                                          const uint32_t *__restrict__ perm,
                                                                          uint32_t rows, uint32_t Fv, int accumulate,
                                                                          uint32_t long_limit, uint32_t coop_limit,
                                                                          uint32_t few_rows, LongRowWork<V> lw) {
  constexpr bool kCoop = G <= 8;
  constexpr int kCoopU = sizeof(V) == 16 ? 4 : 8;           // loads per lane and round on the cooperative path
  constexpr uint32_t kCoopFloats = kWave * kCoopU * (sizeof(V) / 4);  // floats of a wavefront's tile
  __shared__ __align__(16) float coop_tile[kCoop ? 4 : 1][kCoop ? kCoopFloats : kHubBytes<V, 0> / 4];
  if (blockIdx.x < lw.blocks) {
    constexpr int kOwn = !kCoop ? 0 : sizeof(V) == 16 ? 4 : 8;  // (wider rows come in millions, with a list)
    static_assert(sizeof(coop_tile) >= kHubBytes<V, kOwn>, "the hub blocks' scratch");
    sum_long_rows_in_this_block<V, kHubLoads<V, G>, kOwn, false, G == 1 || (G == 2 && sizeof(V) == 4)>(out, msg, off, perm, rows, Fv, accumulate, lw, coop_tile);
    return;
  }
  long_limit = long_limit_of(lw, long_limit, off, rows);
  constexpr int NF = sizeof(V) / 4;
  const uint32_t lane = lane_id();
  constexpr int GG = G * S;  // lanes that share a row
  // A constant where it can be (1 M rows of 3 floats 137 us, 143 without); twice `few_rows` where most rows are a lane's own
  // business (see below), which eight rows a wavefront leave most lanes without (sampled layers' sums over their sources, four
  // heads, 236 K rows of 655 K edges 30.2 -> 25.9 us, 90 K of 156 K 13.8 -> 10.6; four times as many 25.2 and 10.2, but then
  // wavefronts with hub rows last longer: 76 K of 87 K with hubs 22 us, 26, 33, always 64 44).
  uint32_t set = FEW ? few_rows : kFullSet<GG>;
  if (FEW && G == 1 && sizeof(V) == 16 && off[rows] - off[0] < 4ull * rows) set = min(2u * few_rows, kFullSet<GG>);
  const uint32_t gl = lane & (GG - 1), grp = lane / GG;
  const uint32_t col = gl & (G - 1), slice = gl / G;
  const uint64_t wave = wave_of_grid(lw.blocks);
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x - lw.blocks) * blockDim.x / kWave;
  const bool col_live = col < Fv;
  const bool streamed = outgrows_caches(static_cast<uint64_t>(off[rows] - off[0]) * Fv * sizeof(V));
  for (uint64_t base = wave * set; base < rows; base += n_waves * set) {
    uint32_t my_e0 = 0, my_e1 = 0;
    bool mine = false;
    if (lane < set && base + lane < rows) {
      my_e0 = off[base + lane];
      my_e1 = off[base + lane + 1];
      mine = my_e1 - my_e0 <= long_limit;  // longer rows belong to the block kernels
    }
    uint64_t coop = 0;
    if (kCoop) {
      const bool shared = mine && my_e1 - my_e0 > coop_limit;
      coop = __ballot(shared);
      if (shared) mine = false;
    }
    if (G == 1) {
      // Rows one vector wide (the per-head values of an attention layer): a lane sums its own row when
      // the row has at most eight edges -- most rows of a sampled layer's transposed structure -- with
      // the eight loads in flight at once, added in edge order like everywhere else; only the longer
      // rows go through the sharing scheme below.
      const uint32_t deg = my_e1 - my_e0;
      if (mine && deg <= 8u) {
        V v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          v[u] = V{};
          if (static_cast<uint32_t>(u) < deg) {
            const uint32_t e = perm ? perm[my_e0 + u] : my_e0 + u;
            v[u] = msg[e];
          }
        }
        float s1[NF];
#pragma unroll
        for (int t = 0; t < NF; ++t) s1[t] = 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (static_cast<uint32_t>(u) < deg) {
            const float *vf = reinterpret_cast<const float *>(&v[u]);
#pragma unroll
            for (int t = 0; t < NF; ++t) s1[t] += vf[t];
          }
        }
        V *p = out + (base + lane);
        if (accumulate) {
          const V o = *p;
          const float *of = reinterpret_cast<const float *>(&o);
#pragma unroll
          for (int t = 0; t < NF; ++t) s1[t] += of[t];
        }
        V res;
        float *rf = reinterpret_cast<float *>(&res);
#pragma unroll
        for (int t = 0; t < NF; ++t) rf[t] = s1[t];
        *p = res;
        mine = false;
      }
    }
    uint64_t pending = __ballot(mine);  // rows of this set not handed out yet (wave-uniform)
    bool have = false;
    uint32_t row = 0, k = 0, e1 = 0;
    float a[NF];
    // The edge ids of a group's next round are requested while the rows of this one are on their way, so a
    // round is one memory latency and not two.
    uint32_t id[8];
    auto request_ids = [&](uint32_t from) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t idx = from + u * S + slice;
        id[u] = 0;
        if (idx < e1) id[u] = perm ? perm[idx] : idx;
      }
    };
    while (true) {
      // Groups without a row take the lowest pending rows, in group order.
      const uint64_t need_mask = __ballot(!have && gl == 0);
      bool took = false;
      if (!have) {
        const uint32_t rank = __popcll(need_mask & ((1ull << (grp * GG)) - 1ull));
        uint64_t m = pending;
        for (uint32_t t = 0; t < rank && m; ++t) m &= m - 1;
        if (m) {
          row = static_cast<uint32_t>(__builtin_ctzll(m));
          took = true;
        }
      }
      const uint32_t from = took ? row : lane;
      const uint32_t new_e0 = __shfl(my_e0, from, kWave), new_e1 = __shfl(my_e1, from, kWave);
      if (took) {
        have = true;
        k = new_e0;
        e1 = new_e1;
        request_ids(k);
#pragma unroll
        for (int t = 0; t < NF; ++t) a[t] = 0.f;
      }
      for (uint32_t t = __popcll(need_mask); t > 0 && pending; --t) pending &= pending - 1;  // handed out
      if (!__ballot(have)) break;
      if (have) {
        // up to 8 S edge rows of this group's row, loaded together (slice s takes the edges s, s + S,
        // ...), added in order
        V v[8];
        const uint32_t n = e1 - k < 8u * S ? e1 - k : 8u * S;
        auto request_rows = [&](auto load) {
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            v[u] = V{};
            const uint32_t idx = u * S + slice;
            if (idx < n && col_live) v[u] = load(msg + static_cast<size_t>(id[u]) * Fv + col);
          }
        };
        if (streamed) request_rows([](const V *p) { return load_streamed(p); });
        else request_rows([](const V *p) { return *p; });
        if (k + n < e1) request_ids(k + n);
        if (S == 1) {
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            if (static_cast<uint32_t>(u) < n && col_live) {
              const float *vf = reinterpret_cast<const float *>(&v[u]);
#pragma unroll
              for (int t = 0; t < NF; ++t) a[t] += vf[t];
            }
          }
        } else {
          const uint32_t first = lane - gl + col;  // the lane of slice 0 that holds this lane's column
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            if (!__ballot(static_cast<uint32_t>(u * S) < n)) break;  // no group of the wavefront has edges left
            const float *vf = reinterpret_cast<const float *>(&v[u]);
#pragma unroll
            for (int sl = 0; sl < S; ++sl) {
              float val[NF];
#pragma unroll
              for (int t = 0; t < NF; ++t) val[t] = __shfl(vf[t], first + sl * G, kWave);
              if (static_cast<uint32_t>(u * S + sl) < n) {
#pragma unroll
                for (int t = 0; t < NF; ++t) a[t] += val[t];
              }
            }
          }
        }
        k += n;
        if (k >= e1) {
          if (col_live && slice == 0) {
            V *p = out + (base + row) * Fv + col;
            if (accumulate) {
              const V o = *p;
              const float *of = reinterpret_cast<const float *>(&o);
#pragma unroll
              for (int t = 0; t < NF; ++t) a[t] += of[t];
            }
            V res;
            float *rf = reinterpret_cast<float *>(&res);
#pragma unroll
            for (int t = 0; t < NF; ++t) rf[t] = a[t];
            *p = res;
          }
          have = false;
        }
      }
    }
    if (kCoop) {
      // The long rows of this set, one after the other, by the whole wavefront.
      constexpr uint32_t kSlots = kWave / G;           // edge rows per load of the wavefront
      constexpr uint32_t kRound = kSlots * kCoopU;     // edge rows per round
      constexpr uint32_t kPitch = G * NF;              // floats of an edge row in the tile
      float *tile = coop_tile[wave_of_block()];
      const uint32_t slot = lane / G;
      const uint32_t comps = Fv * NF;                  // floats of an output row: lane c < comps owns float c
      while (coop) {
        const uint32_t j = static_cast<uint32_t>(__builtin_ctzll(coop));
        coop &= coop - 1;
        const uint32_t r0 = wave_read(my_e0, j), r1 = wave_read(my_e1, j);
        V cur[kCoopU];
        auto load_round = [&](uint32_t k) {
#pragma unroll
          for (int u = 0; u < kCoopU; ++u) {
            cur[u] = V{};
            const uint32_t idx = k + u * kSlots + slot;
            if (idx < r1 && col_live) {
              const uint32_t e = perm ? perm[idx] : idx;
              cur[u] = msg[static_cast<size_t>(e) * Fv + col];
            }
          }
        };
        load_round(r0);
        float acc = 0.f;
        for (uint32_t k = r0; k < r1; k += kRound) {
          __builtin_amdgcn_wave_barrier();  // the previous round's reads of the tile are done
#pragma unroll
          for (int u = 0; u < kCoopU; ++u) reinterpret_cast<V *>(tile)[u * kWave + lane] = cur[u];
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          if (k + kRound < r1) load_round(k + kRound);  // in flight while this round is added up
          const uint32_t n = r1 - k < kRound ? r1 - k : kRound;
          if (lane < comps) {
            for (uint32_t i = 0; i < n; i += 8) {  // whole groups of eight: the tile's tail holds zeros
#pragma unroll
              for (uint32_t t = 0; t < 8; ++t) acc += tile[(i + t) * kPitch + lane];
            }
          }
        }
        if (lane < comps) {
          float *p = reinterpret_cast<float *>(out) + static_cast<size_t>(base + j) * comps + lane;
          if (accumulate) acc += *p;
          *p = acc;
        }
      }
    }
  }
}

// Giant rows: a row so long that one block working through it alone would outlast the rest of the
// launch (a 300,000-edge hub next to 10^4 rows of a few thousand edges) is cut into pieces that
// separate blocks reduce, and a last kernel combines the pieces in order.  The caller's argument
// lists carry no edge count, so everything is sized by fixed capacities and decided on the device:
// a row is giant above the limit of its operator or above a 1/kGiantCap share of all edges, whichever
// is more, so there are never more than kGiantCap of them whatever order they are found in, and
// the piece length is chosen so that they need at most kPieceCap pieces.
constexpr uint32_t kGiantCap = 4096;
constexpr uint32_t kPieceCap = 8192;
constexpr uint32_t kGiantMinPiece = 4096;  // edges, for the softmax segments

// Values above which a softmax segment is a block's and not a wavefront's, and above which it is cut into pieces.
// A launch lasts at least as long as its longest segment, which a wavefront reads 512 values and a block 8,192 at a time,
// so the lines follow the values of the whole call: with both fixed at their upper ends the hub rows of a 2.48 M-edge
// graph (one head) took the wavefront launches 99 us forward and 96 backward, and now 4 and 25 beside a block launch of 19 and 18
// (attention layer of 47 columns, both directions: 844 -> 644 us).  From 33.5 M values up the ends are reached: a
// block's two barriers a segment then cost what it gains (126 M edges, four heads, 4,096 against 32,768 values
// for a wavefront: 1.43, 1.36 ms).
__device__ __forceinline__ uint32_t long_segment_values(uint64_t total_values) {
  const uint64_t v = total_values / 1024;
  return v < kLongRowMinValues ? kLongRowMinValues : v < kLongRowValues ? static_cast<uint32_t>(v) : kLongRowValues;
}
__device__ __forceinline__ uint64_t giant_segment_values(uint64_t total_values) {
  const uint64_t v = total_values / 256;
  return v < kGiantMinValues ? kGiantMinValues : v < kGiantValues ? v : kGiantValues;
}

// The same for a call of few rows (kFewRows), whose launch has blocks of 256 threads for both.
// The rows, by both sides' times in us, a call after the other, the kernels of many rows / these, for one, four and eight heads:
//   rows, edges    softmax fwd                  bwd                          attention fwd                bwd (eight heads always of many rows)
//   16 K, 200 K    78 / 34, 89 / 40, 91 / 40    84 / 34, 91 / 41, 91 / 40    94 / 34, 98 / 41, 97 / 42    96 / 39, 101 / 44
//   30 K, 1 M      76 / 33, 86 / 43, 84 / 50    79 / 33, 88 / 42, 86 / 53    86 / 38, 94 / 60, 107 / 72   89 / 44, 101 / 69
//   60 K, 4 M      79 / 43, 87 / 66, 116 / 106  79 / 42, 98 / 76, 176 / 159  92 / 71, 146 / 110, 191 / 164  93 / 85, 140 / 133
//   60 K, 10 M     84 / 55, 155 / 152, 294 / 300  86 / 57, 198 / 192, 388 / 385  149 / 121, 234 / 197, 513 / 473  140 / 139, 325 / 335
//   169 K, 2.48 M  90 / 42, 94 / 54, 96 / 71    93 / 38, 94 / 55, 101 / 84   104 / 57, 142 / 100, 186 / 134  108 / 76, 127 / 119
//   250 K, 3 M     91 / 47, 94 / 59, 97 / 74    94 / 43, 93 / 61, 121 / 101  107 / 67, 157 / 118, 201 / 150  107 / 87, 136 / 139
//   200 K, 20 M    100 / 80, 257 / 248, 448 / 428  108 / 80, 339 / 322, 648 / 608  329 / 194, 504 / 494, 732 / 712  405 / 305, 543 / 604
//   100 K, 40 M    166 / 133, 463 / 476         206 / 182, 638 / 666         462 / 398, 782 / 779         483 / 466, 836 / 908
//   beyond the line:
//   400 K, 2 M     68 / 49, 71 / 60, 79 / 71    68 / 48, 71 / 54, 84 / 69    92 / 70, 134 / 116, 183 / 146  95 / 100, 127 / 137
//   500 K, 20 M    98 / 82, 252 / 239, 446 / 453  102 / 78, 320 / 309, 616 / 618  297 / 187, 474 / 468, 826 / 792  368 / 307, 554 / 596
//   1 M, 8 M       93 / 90, 131 / 126, 251 / 227  82 / 76, 164 / 139, 279 / 263  196 / 176, 264 / 278, 453 / 489  187 / 226, 339 / 420
// What decides is how many edges a row has, which a call does not say.  Up to the line these kernels take a third to a half of sparse
// graphs' time off and cost the four-head calls of graphs of hundreds of edges a row 2 to 10 % of an operator (0.6 to 1.5 % of a layer:
// four heads, both directions, the backward of few / of many rows 100 K, 30 M 4,740 / 4,713, 200 K, 20 M 3,684 / 3,660, 60 K, 10 M 1,828 / 1,772,
// but 40 K, 1 M 342 / 350, 169 K, 2.48 M 707 / 712).  Sixteen heads 16 K, 1 M 105 / 72, 97 / 77, 159 / 86, 60 K, 4 M 238 / 249, 305 / 308, 372 / 334,
// 169 K, 2.48 M 171 / 142, 205 / 176, 290 / 203.  Beyond it the fused backward loses and the other three still gain a little; the line is not
// theirs alone.  The fused backward of more than four heads holds two arrays and the signs of the scores a lane, 114 registers for all of its paths
// together: above 32 K rows it is even in the operator (60 K, 4 M 256 / 257) and was slower in whole layers (60 K, 10 M 2,306 / 2,408, 50 K, 600 K 344 / 317).
constexpr uint32_t kFewRows = 1u << 18;
constexpr uint32_t kFewRowsManyHeads = 1u << 15;
constexpr uint32_t kFewPieceValues = 4096;
__device__ __forceinline__ uint64_t few_long_values(uint64_t total_values) {
  const uint64_t v = total_values / 2048;
  return v < 1024 ? 1024 : v < kLongRowValues ? v : kLongRowValues;
}
__device__ __forceinline__ uint64_t few_giant_values(uint64_t total_values) {
  const uint64_t v = total_values / 256;
  return v < 8192 ? 8192 : v < kGiantValues ? v : kGiantValues;
}

// hdr: [0] giant rows, [1] pieces,
//      [2] edges per piece, [4..5] edges of the listed giant rows (64-bit), [6] the long-row counter
//      (`count` points here, so that one fill clears all of them).
// list[0 .. *count) = rows r with (off[r+1] - off[r]) * width > limit that are not listed as giant
// (any order); giant_rows[0 .. hdr[0]) = rows above giant_limit values and above the share.  limit
// kByTotal and kByFewTotal: softmax calls, whose lines lie where their values put them.
__global__ __launch_bounds__(256) void collect_long_rows_kernel(uint32_t *__restrict__ list,
                                                                uint32_t *__restrict__ count,
                                                                uint32_t *__restrict__ giant_rows,
                                                                uint32_t *__restrict__ hdr,
                                                                const uint32_t *__restrict__ off, uint32_t rows,
                                                                uint32_t width, uint32_t limit,
                                                                uint64_t giant_limit) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const uint32_t deg = off[r + 1] - off[r];
  const uint64_t n = static_cast<uint64_t>(deg) * width;
  if (limit == kByTotal) {
    const uint64_t total = static_cast<uint64_t>(off[rows] - off[0]) * width;
    limit = long_segment_values(total);
    giant_limit = giant_segment_values(total);
  } else if (limit == kByFewTotal) {
    const uint64_t total = static_cast<uint64_t>(off[rows] - off[0]) * width;
    limit = static_cast<uint32_t>(few_long_values(total));
    giant_limit = few_giant_values(total);
  }
  if (n > giant_limit && deg > (off[rows] - off[0]) / kGiantCap) {
    const uint32_t gi = atomicAdd(&hdr[0], 1u);
    if (gi < kGiantCap) {
      giant_rows[gi] = r;
      atomicAdd(reinterpret_cast<unsigned long long *>(hdr + 4), static_cast<unsigned long long>(deg));
      return;
    }
  }
  if (n > limit) list[atomicAdd(count, 1u)] = r;
}

// One block: fixes the piece length, gives every listed giant row its first piece (every thread counts
// the pieces of a run of rows, then one prefix over the block) and writes the piece table (list
// position, row, first edge, end), a wavefront a row.
template <int BLOCK>
__device__ __forceinline__ void plan_giant_rows(uint32_t listed, unsigned long long edges, uint32_t *hdr, const uint32_t *giant_rows,
                                                uint32_t *first, uint4 *__restrict__ pieces, const uint32_t *__restrict__ off,
                                                uint32_t min_piece) {
  __shared__ uint32_t wave_sums[BLOCK / kWave];
  const uint32_t n = listed < kGiantCap ? listed : kGiantCap;
  const unsigned long long even = (edges + (kPieceCap - kGiantCap) - 1) / (kPieceCap - kGiantCap);
  const uint32_t len = even < min_piece ? min_piece : static_cast<uint32_t>(even);
  auto pieces_of = [&](uint32_t i) -> uint32_t {
    const uint32_t r = giant_rows[i];
    return (off[r + 1] - off[r] - 1) / len + 1;
  };
  const uint32_t per = (n + BLOCK - 1) / BLOCK;
  const uint32_t i0 = min(n, threadIdx.x * per), i1 = min(n, i0 + per);
  uint32_t mine = 0, total = 0;
  for (uint32_t i = i0; i < i1; ++i) mine += pieces_of(i);
  uint32_t p = block_prefix<BLOCK>(mine, wave_sums, &total);
  for (uint32_t i = i0; i < i1; ++i) {
    first[i] = p;
    p += pieces_of(i);
  }
  if (threadIdx.x == 0) {
    first[n] = total;
    hdr[0] = n;
    hdr[1] = total;
    hdr[2] = len;
  }
  __syncthreads();  // `first` is read by other threads of this block below
  for (uint32_t i = threadIdx.x / kWave; i < n; i += BLOCK / kWave) {
    const uint32_t r = giant_rows[i];
    const uint32_t e0 = off[r], e1 = off[r + 1], p0 = first[i], n_pieces = (e1 - e0 - 1) / len + 1;
    for (uint32_t q = lane_id(); q < n_pieces; q += kWave) {
      const uint32_t k = e0 + q * len;
      pieces[p0 + q] = make_uint4(i, r, k, e1 - k < len ? e1 : k + len);
    }
  }
}

__global__ __launch_bounds__(256) void giant_plan_kernel(uint32_t *__restrict__ hdr, const uint32_t *__restrict__ giant_rows,
                                                         uint32_t *__restrict__ first, uint4 *__restrict__ pieces,
                                                         const uint32_t *__restrict__ off, uint32_t min_piece) {
  plan_giant_rows<256>(hdr[0], *reinterpret_cast<const unsigned long long *>(hdr + 4), hdr, giant_rows, first, pieces, off, min_piece);
}

// look(row, edges) for every row, by one block: a thread loads the offsets of four rows at a time, and four times as many at once.
template <int BLOCK, typename Look>
__device__ __forceinline__ void each_row_by_block(const uint32_t *__restrict__ off, uint32_t rows, Look look) {
  typedef uint32_t Words4 __attribute__((ext_vector_type(4), aligned(4)));
  constexpr uint32_t kStep = 4 * BLOCK;
  constexpr int U = 4;
  for (uint32_t base = 0; base < rows; base += U * kStep) {
    Words4 w[U];
    uint32_t next[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t r = base + u * kStep + threadIdx.x * 4;
      w[u] = Words4{0u, 0u, 0u, 0u};
      next[u] = 0;
      if (r + 4 <= rows) {
        w[u] = *reinterpret_cast<const Words4 *>(off + r);
        next[u] = off[r + 4];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t r = base + u * kStep + threadIdx.x * 4;
      if (r + 4 <= rows) {
        look(r, w[u].y - w[u].x);
        look(r + 1, w[u].z - w[u].y);
        look(r + 2, w[u].w - w[u].z);
        look(r + 3, next[u] - w[u].w);
      } else {
        for (uint32_t t = r; t < rows; ++t) look(t, off[t + 1] - off[t]);
      }
    }
  }
}

// The lists, their counters and the piece table in one launch of one block, for up to kOneBlockRows rows: a fill, a launch that lists
// and one that plans are 14 us and as much of the host's time, this one 5 with 20 K rows, but a block reads the offsets of 169 K, from
// beyond its L2, in some 25 (attention layer of one head of 47, 2.48 M edges 527 -> 541).  limit: as in collect_long_rows_kernel.
constexpr uint32_t kOneBlockRows = 1u << 16;
__global__ __launch_bounds__(kLongBlock) void few_long_rows_kernel(uint32_t *__restrict__ list, uint32_t *__restrict__ count,
                                                                   uint32_t *giant_rows, uint32_t *hdr, uint32_t *first,
                                                                   uint4 *__restrict__ pieces, const uint32_t *__restrict__ off,
                                                                   uint32_t rows, uint32_t width, uint32_t limit_or_total,
                                                                   uint64_t most, uint32_t min_piece) {
  __shared__ uint32_t n_long, n_giant;
  __shared__ unsigned long long giant_edges;
  if (threadIdx.x == 0) {
    n_long = n_giant = 0;
    giant_edges = 0;
  }
  __syncthreads();
  const uint32_t edges = off[rows] - off[0];
  const uint64_t total = static_cast<uint64_t>(edges) * width;
  uint64_t limit = limit_or_total, giant_limit = most;
  if (limit_or_total == kByTotal) {
    limit = long_segment_values(total);
    giant_limit = giant_segment_values(total);
  } else if (limit_or_total == kByFewTotal) {
    limit = few_long_values(total);
    giant_limit = few_giant_values(total);
  }
  auto look = [&](uint32_t r, uint32_t deg) {
    const uint64_t n = static_cast<uint64_t>(deg) * width;
    if (n <= limit) return;
    if (n > giant_limit && deg > edges / kGiantCap) {
      const uint32_t gi = atomicAdd(&n_giant, 1u);
      if (gi < kGiantCap) {
        giant_rows[gi] = r;
        atomicAdd(&giant_edges, static_cast<unsigned long long>(deg));
        return;
      }
    }
    list[atomicAdd(&n_long, 1u)] = r;
  };
  each_row_by_block<kLongBlock>(off, rows, look);
  __syncthreads();
  if (threadIdx.x == 0) *count = n_long;
  plan_giant_rows<kLongBlock>(n_giant, giant_edges, hdr, giant_rows, first, pieces, off, min_piece);
}

// out[row, :] (+)= the row's piece sums, added in piece order.
__global__ __launch_bounds__(256) void giant_sum_combine_kernel(float *__restrict__ out,
                                                                const float *__restrict__ partial,
                                                                const uint32_t *__restrict__ hdr,
                                                                const uint32_t *__restrict__ giant_rows,
                                                                const uint32_t *__restrict__ first, uint32_t F,
                                                                int accumulate) {
  const uint32_t n = hdr[0];
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const uint32_t r = giant_rows[i];
    const uint32_t p0 = first[i], p1 = first[i + 1];
    for (uint32_t c = threadIdx.x; c < F; c += blockDim.x) {
      float a = 0.f;
      uint32_t p = p0;
      for (; p + 8 <= p1; p += 8) {  // eight pieces requested at once, added in order
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = partial[static_cast<size_t>(p + u) * F + c];
#pragma unroll
        for (int u = 0; u < 8; ++u) a += v[u];
      }
      for (; p < p1; ++p) a += partial[static_cast<size_t>(p) * F + c];
      float *dst = out + static_cast<size_t>(r) * F + c;
      *dst = accumulate ? *dst + a : a;
    }
  }
}

// ---- segment softmax --------------------------------------------------------------------------
//
// A destination's scores x[e0*H .. e1*H) are contiguous.  Lane l walks flat positions l, l+64, ...
// When H is a power of two <= 64 a lane always meets the same head (l mod H), so the per-head
// maximum and sum are a lane-local reduction followed by a butterfly over the lanes that share a
// head (xor masks 32 .. H).  Other head counts take one strided pass per head.

template <int MODE>  // 0 = max, 1 = sum
__device__ __forceinline__ float head_reduce(float v, uint32_t H) {
  for (uint32_t m = kWave / 2; m >= H; m >>= 1) {
    const float o = __shfl_xor(v, m, kWave);
    v = MODE == 0 ? fmaxf(v, o) : v + o;
  }
  return v;
}

__device__ __forceinline__ float leaky(float s, float slope) { return s > 0.f ? s : s * slope; }

// exp for the softmax kernels: the hardware's 2^x of x * log2(e), two instructions instead of the
// fourteen of the correctly rounded library routine -- these kernels are bound by their vector
// instructions for short segments.  Arguments are <= 0 (a value minus its segment's maximum); the
// product's rounding puts the relative error at |x| * 6e-8 (1e-6 at x = -20, where the result is
// 2e-9 of the segment's largest term), well inside the 1e-4 these operators are held to.
__device__ __forceinline__ float softmax_exp(float x) { return __expf(x); }

// Where the running maxima of a (maximum, sum of exp(v - maximum)) pair start: the lowest float and not -inf, so that a
// masked value (-inf) that comes first adds exp(-inf) = 0 and not exp(-inf + inf).  A head without any other value keeps
// a sum of 0 and becomes 0 / 0.
constexpr float kLowestMax = -3.402823466e38f;

// Multi-pass softmax forward of one segment with 16-byte lanes (H a multiple of 4, 16-byte aligned
// arrays): lane l of a group of WIDTH threads takes the vectors l, l + WIDTH, ... of the segment, i.e.
// four consecutive values = heads (4 l mod H) .. +3 of one edge, so a pass needs a quarter of the load
// rounds of the 4-byte version.  `load4(i)` fetches vector i (for the fused form: the four scores of
// its edge), `keep4(i, v)` may store it.  Leaves per-component running (max, sum) pairs in mx / sum.
template <int U, typename Load4, typename Keep4>
__device__ __forceinline__ void strided_max_sum_pass4(uint64_t first, uint64_t nv, uint64_t stride, Load4 load4,
                                                      Keep4 keep4, float (&mx)[4], float (&sum)[4]) {
  auto fold = [&](const float4 *v, int count) {
    float m[4] = {mx[0], mx[1], mx[2], mx[3]};
    for (int u = 0; u < count; ++u) {
      m[0] = fmaxf(m[0], v[u].x);
      m[1] = fmaxf(m[1], v[u].y);
      m[2] = fmaxf(m[2], v[u].z);
      m[3] = fmaxf(m[3], v[u].w);
    }
    float add[4] = {0.f, 0.f, 0.f, 0.f};
    for (int u = 0; u < count; ++u) {
      add[0] += softmax_exp(v[u].x - m[0]);
      add[1] += softmax_exp(v[u].y - m[1]);
      add[2] += softmax_exp(v[u].z - m[2]);
      add[3] += softmax_exp(v[u].w - m[3]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      sum[c] = sum[c] * softmax_exp(mx[c] - m[c]) + add[c];  // (at the start the old sum is 0 and stays 0)
      mx[c] = m[c];
    }
  };
  uint64_t i = first;
  for (; i + (U - 1) * stride < nv; i += U * stride) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = load4(i + u * stride);
#pragma unroll
    for (int u = 0; u < U; ++u) keep4(i + u * stride, v[u]);
    fold(v, U);
  }
  for (; i < nv; i += stride) {
    const float4 v = load4(i);
    keep4(i, v);
    fold(&v, 1);
  }
}

// Three kernels share a launch, by segment size n = degree * H (values):
//   short   n <= 128, power-of-two H <= 16: a group of 16 lanes per destination, the segment held
//           in registers -- one pass over memory, four destinations per wavefront in flight;
//   wave    up to long_segment_values of the call (or any size when the block kernel is not used): one wavefront per
//           destination; segments of at most 512 values are register-resident too, larger ones take
//           the three passes (max, sum, write) / two passes (dot, write) over memory;
//   block   longer segments (hub destinations), listed by collect_long_rows.
// The short and the wave kernel stride over the destinations (a wavefront of the wave kernel looks
// at 64 destinations at a time and visits only those that fall in its size class), so their launch
// size does not grow with the vertex count.

constexpr int kShortG = 16;        // lanes per destination in the short kernel
constexpr int kShortK = 8;         // values per lane held in registers there
constexpr uint32_t kShortValues = kShortG * kShortK;
constexpr int kWaveK = 8;          // values per lane the wave kernel can hold in registers
constexpr uint32_t kWaveRegValues = kWave * kWaveK;
constexpr uint32_t kWaveMidValues = kWave * 32;  // the fused forward's launch for the class above that: 32 per lane
static_assert(kWaveMidValues <= kLongRowMinValues, "the register classes lie below the block kernels' line");

// One strided pass over a segment with U loads in flight: positions first, first + stride, ...
// below n; `load(i)` fetches, `use(i, v)` consumes, in ascending position order.
template <int U, typename Load, typename Use>
__device__ __forceinline__ void strided_pass(uint64_t first, uint64_t n, uint64_t stride, Load load, Use use) {
  uint64_t i = first;
  for (; i + (U - 1) * stride < n; i += U * stride) {
    decltype(load(i)) v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = load(i + u * stride);
#pragma unroll
    for (int u = 0; u < U; ++u) use(i + u * stride, v[u]);
  }
  for (; i < n; i += stride) use(i, load(i));
}

// One strided pass that leaves a running (maximum, sum of exp(v - maximum)) pair, so that the maximum
// and the sum of a segment come out of a single read.  The U values in flight are folded in together:
// their maximum first, then one rescale of the old sum and U independent exponentials.
template <int U, typename Load, typename Seen>
__device__ __forceinline__ void strided_max_sum_pass(uint64_t first, uint64_t n, uint64_t stride, Load load,
                                                     Seen seen, float &mx, float &sum) {
  uint64_t i = first;
  for (; i + (U - 1) * stride < n; i += U * stride) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = load(i + u * stride);
    float m = mx;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      seen(i + u * stride, v[u]);
      m = fmaxf(m, v[u]);
    }
    float add = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) add += softmax_exp(v[u] - m);
    sum = sum * softmax_exp(mx - m) + add;  // (at the start the old sum is 0 and stays 0)
    mx = m;
  }
  for (; i < n; i += stride) {
    const float v = load(i);
    seen(i, v);
    const float m = fmaxf(mx, v);
    sum = sum * softmax_exp(mx - m) + softmax_exp(v - m);
    mx = m;
  }
}

// Reduction over the lanes of an aligned group of WIDTH lanes that share a head (lane mod H).
template <int MODE, int WIDTH>  // 0 = max, 1 = sum
__device__ __forceinline__ float head_reduce_w(float v, uint32_t H) {
  for (uint32_t m = WIDTH / 2; m >= H; m >>= 1) {
    const float o = __shfl_xor(v, m, WIDTH);
    v = MODE == 0 ? fmaxf(v, o) : v + o;
  }
  return v;
}

// Register-resident forward of one segment by WIDTH lanes (lane index gl), K values per lane;
// n <= WIDTH*K values, H a power of two <= WIDTH.
template <bool FUSED, int WIDTH, int K>
__device__ __forceinline__ void softmax_fwd_regs(float *__restrict__ ys, const float *__restrict__ xs,
                                                 const float *__restrict__ el, const float *__restrict__ er,
                                                 const uint32_t *__restrict__ ri, uint32_t d, uint32_t e0, uint32_t n,
                                                 uint32_t H, float slope, uint32_t gl) {
  const uint32_t h = gl & (H - 1);
  float erv = 0.f;
  if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
  float v[K];
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t i = gl + WIDTH * k;
    v[k] = -INFINITY;
    if (i < n) {
      if (FUSED) {
        const uint32_t src = ri[e0 + i / H];
        v[k] = leaky(el[static_cast<size_t>(src) * H + h] + erv, slope);
      } else {
        v[k] = xs[i];
      }
    }
    mx = fmaxf(mx, v[k]);
  }
  mx = head_reduce_w<0, WIDTH>(mx, H);
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    v[k] = (gl + WIDTH * k < n) ? softmax_exp(v[k] - mx) : 0.f;
    sum += v[k];
  }
  sum = head_reduce_w<1, WIDTH>(sum, H);
  const float inv = 1.f / sum;  // one division per lane instead of one per value
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t i = gl + WIDTH * k;
    if (i < n) ys[i] = v[k] * inv;
  }
}

// Register-resident backward, same shape.  Writes ger[d, :] when FUSED (zeros for an empty segment).
template <bool FUSED, int WIDTH, int K>
__device__ __forceinline__ void softmax_bwd_regs(float *__restrict__ gxs, float *__restrict__ ger,
                                                 const float *__restrict__ gys, const float *__restrict__ ys,
                                                 const float *__restrict__ el, const float *__restrict__ er,
                                                 const uint32_t *__restrict__ ri, uint32_t d, uint32_t e0, uint32_t n,
                                                 uint32_t H, float slope, uint32_t gl) {
  const uint32_t h = gl & (H - 1);
  float yv[K], gv[K];
  float dot = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t i = gl + WIDTH * k;
    yv[k] = 0.f;
    gv[k] = 0.f;
    if (i < n) {
      yv[k] = ys[i];
      gv[k] = gys[i];
    }
    dot += gv[k] * yv[k];
  }
  dot = head_reduce_w<1, WIDTH>(dot, H);
  float erv = 0.f, gsum = 0.f;
  if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t i = gl + WIDTH * k;
    if (i < n) {
      float g = yv[k] * (gv[k] - dot);
      if (FUSED) {
        const uint32_t src = ri[e0 + i / H];
        const float pre = el[static_cast<size_t>(src) * H + h] + erv;
        g *= pre > 0.f ? 1.f : slope;
        gsum += g;
      }
      gxs[i] = g;
    }
  }
  if (FUSED) {
    gsum = head_reduce_w<1, WIDTH>(gsum, H);
    if (gl < H) ger[static_cast<size_t>(d) * H + gl] = gsum;
  }
}

// These kernels are bound by their vector instructions, not by memory (253 per 256-value segment
// were counted, a wave64 instruction holding its SIMD for four cycles: 80 % of the launch time), and
// most of them served register slots beyond the segment's end.  The register paths are therefore
// instantiated for 1, 2, 4 and 8 slots per lane and called with the smallest count that covers
// every segment the wavefront is working on (`n`, the caller's segment size, must be in scope).
#define NTS_BY_SLOTS(WIDTH, FN, ...)                                        \
  do {                                                                      \
    if (!any_lane(n > 4u * (WIDTH))) {                                      \
      if (!any_lane(n > 2u * (WIDTH))) {                                    \
        if (!any_lane(n > 1u * (WIDTH))) FN<FUSED, WIDTH, 1>(__VA_ARGS__);  \
        else FN<FUSED, WIDTH, 2>(__VA_ARGS__);                              \
      } else {                                                              \
        FN<FUSED, WIDTH, 4>(__VA_ARGS__);                                   \
      }                                                                     \
    } else {                                                                \
      FN<FUSED, WIDTH, 8>(__VA_ARGS__);                                     \
    }                                                                       \
  } while (0)

// True if `pred` holds on any active lane of the wavefront.
__device__ __forceinline__ bool any_lane(bool pred) { return __ballot(pred) != 0; }

// Short segments (n <= kShortValues; power-of-two H <= kShortG): a group of kShortG lanes per
// destination, striding over the destinations.  BWD selects the backward formula.
// A segment of any length by one group of kShortG lanes, with plain strided passes (the safety net of a
// launch that was told no segment exceeds the short class: correct, not fast).
template <bool FUSED, bool BWD>
__device__ void softmax_group_any(float *__restrict__ outs, float *__restrict__ ger, const float *__restrict__ xs,
                                  const float *__restrict__ ys, const float *__restrict__ el,
                                  const float *__restrict__ er, const uint32_t *__restrict__ ri, uint32_t d,
                                  uint32_t e0, uint64_t n, uint32_t H, float slope, uint32_t gl) {
  const uint32_t h = gl & (H - 1);
  const float erv = FUSED ? er[static_cast<size_t>(d) * H + h] : 0.f;
  auto score = [&](uint64_t i) {
    if (!FUSED) return xs[i];
    return leaky(el[static_cast<size_t>(ri[e0 + i / H]) * H + h] + erv, slope);
  };
  if (!BWD) {
    float mx = -INFINITY;
    for (uint64_t i = gl; i < n; i += kShortG) mx = fmaxf(mx, score(i));
    mx = head_reduce_w<0, kShortG>(mx, H);
    float sum = 0.f;
    for (uint64_t i = gl; i < n; i += kShortG) sum += softmax_exp(score(i) - mx);
    sum = head_reduce_w<1, kShortG>(sum, H);
    const float inv = 1.f / sum;
    for (uint64_t i = gl; i < n; i += kShortG) outs[i] = softmax_exp(score(i) - mx) * inv;
  } else {
    float dot = 0.f;
    for (uint64_t i = gl; i < n; i += kShortG) dot += xs[i] * ys[i];
    dot = head_reduce_w<1, kShortG>(dot, H);
    float gsum = 0.f;
    for (uint64_t i = gl; i < n; i += kShortG) {
      float g = ys[i] * (xs[i] - dot);
      if (FUSED) {
        const float pre = el[static_cast<size_t>(ri[e0 + i / H]) * H + h] + erv;
        g *= pre > 0.f ? 1.f : slope;
        gsum += g;
      }
      outs[i] = g;
    }
    if (FUSED) {
      gsum = head_reduce_w<1, kShortG>(gsum, H);
      if (gl < H) ger[static_cast<size_t>(d) * H + gl] = gsum;
    }
  }
}

// ALL: the launch is the only one of its call (the caller bounded every segment by the short class), so
// a segment beyond the class is not skipped but computed by the group with plain strided passes.
template <bool FUSED, bool BWD, bool ALL = false>
__global__ __launch_bounds__(256) void edge_softmax_short_kernel(float *__restrict__ out, float *__restrict__ ger,
                                                                 const float *__restrict__ x_or_gy,
                                                                 const float *__restrict__ y,
                                                                 const float *__restrict__ el,
                                                                 const float *__restrict__ er,
                                                                 const uint32_t *__restrict__ co,
                                                                 const uint32_t *__restrict__ ri, uint32_t Vd,
                                                                 uint32_t H, float slope) {
  const uint32_t gl = threadIdx.x & (kShortG - 1);
  const uint64_t n_groups = static_cast<uint64_t>(gridDim.x) * (256 / kShortG);
  for (uint64_t d64 = (static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x) / kShortG; d64 < Vd; d64 += n_groups) {
    const uint32_t d = static_cast<uint32_t>(d64);
    const uint32_t e0 = co[d], e1 = co[d + 1];
    const uint64_t n64 = static_cast<uint64_t>(e1 - e0) * H;
    const size_t base = static_cast<size_t>(e0) * H;
    if (n64 > kShortValues) {  // the whole group takes the same way
      if (ALL)
        softmax_group_any<FUSED, BWD>(out + base, ger, x_or_gy ? x_or_gy + base : nullptr, y ? y + base : nullptr, el, er,
                                      ri, d, e0, n64, H, slope, gl);
      continue;
    }
    const uint32_t n = static_cast<uint32_t>(n64);
    if (BWD) {
      if (FUSED) {  // the four instances together would cost this kernel a wavefront per SIMD
        softmax_bwd_regs<FUSED, kShortG, kShortK>(out + base, ger, x_or_gy + base, y + base, el, er, ri, d, e0, n, H,
                                                  slope, gl);
      } else {
        NTS_BY_SLOTS(kShortG, softmax_bwd_regs, out + base, ger, x_or_gy + base, y + base, el, er, ri, d, e0, n, H,
                     slope, gl);
      }
    } else {
      if (n == 0) continue;
      NTS_BY_SLOTS(kShortG, softmax_fwd_regs, out + base, FUSED ? nullptr : x_or_gy + base, el, er, ri, d, e0, n, H,
                   slope, gl);
    }
  }
}

// The destinations of [base, base + set) whose segment size lies in [min_values, max_values], as a
// wave-uniform bit mask; every lane keeps the offsets of its own destination for the visit.
__device__ __forceinline__ uint64_t wave_rows_in_class(const uint32_t *__restrict__ co, uint32_t Vd, uint64_t base,
                                                       uint32_t set, uint32_t H, uint32_t min_values, uint32_t max_values,
                                                       uint32_t &my_e0, uint32_t &my_e1) {
  const uint32_t lane = lane_id();
  const uint64_t d = base + lane;
  my_e0 = 0;
  my_e1 = 0;
  bool mine = false;
  if (lane < set && d < Vd) {
    my_e0 = co[d];
    my_e1 = co[d + 1];
    const uint64_t n = static_cast<uint64_t>(my_e1 - my_e0) * H;
    mine = n >= min_values && n <= max_values;
  }
  return __ballot(mine);
}

// FUSED = false: y = softmax_seg(x).   FUSED = true: x is ignored and the score is
// leaky_relu(el[ri[e],h] + er[d,h], slope); in the three-pass path y first holds the raw score, then
// alpha.  Visits the destinations with min_values <= n <= max_values.
// PART: 0 = every segment size in one launch; 1 = the register-resident segments only, 2 = the
// longer ones only, 3 = segments of 513 .. 2,048 values held 16 or 32 per lane in registers -- launches
// of their own, each instance allotted the registers of its own path.  The fused form is launched in
// parts: its longer segments read el[src] with 16-byte lanes, which costs registers that the short
// ones should not pay for (Products-shaped graph: 3.05 -> 2.82 ms), and the class between them is
// still one pass over memory instead of writing raw scores and reading them back (2.76 -> 2.65 ms); for
// the plain softmax one launch is as fast as two or three (every variant runs at the rate of a copy).
template <bool FUSED, bool POW2, int PART>
__global__ __launch_bounds__(256) void edge_softmax_fwd_kernel(float *__restrict__ y, const float *__restrict__ x,
                                                               const float *__restrict__ el,
                                                               const float *__restrict__ er,
                                                               const uint32_t *__restrict__ co,
                                                               const uint32_t *__restrict__ ri, uint32_t Vd,
                                                               uint32_t H, float slope, uint32_t min_values,
                                                               uint32_t max_values, uint32_t vec4, uint32_t set) {
  if (max_values == kByTotal) max_values = long_segment_values(static_cast<uint64_t>(co[Vd] - co[0]) * H);
  const uint32_t lane = lane_id();
  const uint64_t wave = wave_of_grid();
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  for (uint64_t first = wave * set; first < Vd; first += n_waves * set) {
    uint32_t my_e0, my_e1;
    uint64_t todo = wave_rows_in_class(co, Vd, first, set, H, min_values < 1 ? 1 : min_values, max_values, my_e0, my_e1);
    while (todo) {
      const uint32_t j = static_cast<uint32_t>(__builtin_ctzll(todo));
      todo &= todo - 1;
      const uint32_t d = static_cast<uint32_t>(first) + j;
      const uint32_t e0 = wave_read(my_e0, j), e1 = wave_read(my_e1, j);
      const size_t base = static_cast<size_t>(e0) * H;
      const uint32_t n = (e1 - e0) * H;
      float *ys = y + base;
      const float *xs = FUSED ? nullptr : x + base;

      if (POW2) {
        if (PART <= 1 && n <= kWaveRegValues) {
          NTS_BY_SLOTS(kWave, softmax_fwd_regs, ys, xs, el, er, ri, d, e0, n, H, slope, lane);
          continue;
        }
        if (PART == 1) continue;
        if (PART == 3) {  // 513 .. 2,048 values: still one pass, 16 or 32 values per lane in registers
          if (n <= 16u * kWave) softmax_fwd_regs<FUSED, kWave, 16>(ys, xs, el, er, ri, d, e0, n, H, slope, lane);
          else softmax_fwd_regs<FUSED, kWave, 32>(ys, xs, el, er, ri, d, e0, n, H, slope, lane);
          continue;
        }
        if (PART == 2 && vec4 && n >= 2048u) {  // at least two full rounds of four vectors per lane
          const uint32_t h0 = (lane * 4u) & (H - 1);  // head of this lane's first value; 256 k = 0 mod H
          const uint32_t hq = H / 4;                  // lanes hq apart hold the same heads
          float4 erv = make_float4(0.f, 0.f, 0.f, 0.f);
          if (FUSED) erv = *reinterpret_cast<const float4 *>(er + static_cast<size_t>(d) * H + h0);
          const float4 *xs4 = reinterpret_cast<const float4 *>(xs);
          float4 *ys4 = reinterpret_cast<float4 *>(ys);
          float mx4[4] = {kLowestMax, kLowestMax, kLowestMax, kLowestMax}, sum4[4] = {0.f, 0.f, 0.f, 0.f};
          strided_max_sum_pass4<4>(
              lane, n / 4, kWave,
              [&](uint64_t i) -> float4 {
                if (!FUSED) return xs4[i];
                const uint32_t src = ri[e0 + static_cast<uint32_t>(i * 4 / H)];
                const float4 e = *reinterpret_cast<const float4 *>(el + static_cast<size_t>(src) * H + h0);
                return make_float4(leaky(e.x + erv.x, slope), leaky(e.y + erv.y, slope), leaky(e.z + erv.z, slope),
                                   leaky(e.w + erv.w, slope));
              },
              [&](uint64_t i, float4 sc) {
                if (FUSED) ys4[i] = sc;
              },
              mx4, sum4);
          float inv4[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float lane_mx = mx4[c];
            mx4[c] = head_reduce<0>(mx4[c], hq);
            sum4[c] = head_reduce<1>(sum4[c] * softmax_exp(lane_mx - mx4[c]), hq);
            inv4[c] = 1.f / sum4[c];
          }
          strided_pass<4>(lane, n / 4, kWave, [&](uint64_t i) -> float4 { return FUSED ? ys4[i] : xs4[i]; },
                          [&](uint64_t i, float4 sc) {
                            ys4[i] = make_float4(softmax_exp(sc.x - mx4[0]) * inv4[0], softmax_exp(sc.y - mx4[1]) * inv4[1],
                                                 softmax_exp(sc.z - mx4[2]) * inv4[2], softmax_exp(sc.w - mx4[3]) * inv4[3]);
                          });
          continue;
        }
        const uint32_t h = lane & (H - 1);
        float erv = 0.f;
        if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
        float mx = kLowestMax, sum = 0.f;
        strided_max_sum_pass<8>(
            lane, n, kWave,
            [&](uint64_t i) -> float {
              if (!FUSED) return xs[i];
              const uint32_t src = ri[e0 + i / H];
              return leaky(el[static_cast<size_t>(src) * H + h] + erv, slope);
            },
            [&](uint64_t i, float sc) {
              if (FUSED) ys[i] = sc;
            },
            mx, sum);
        // every lane's pair is brought to the head's maximum before the sums are added
        const float lane_mx = mx;
        mx = head_reduce<0>(mx, H);
        sum = head_reduce<1>(sum * softmax_exp(lane_mx - mx), H);
        const float inv = 1.f / sum;
        strided_pass<8>(lane, n, kWave, [&](uint64_t i) -> float { return FUSED ? ys[i] : xs[i]; },
                        [&](uint64_t i, float sc) { ys[i] = softmax_exp(sc - mx) * inv; });
      } else {
        const uint32_t deg = e1 - e0;
        for (uint32_t h = 0; h < H; ++h) {
          float erv = 0.f;
          if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
          float mx = -INFINITY;
          for (uint32_t k = lane; k < deg; k += kWave) {
            float sc;
            if (FUSED) {
              const uint32_t src = ri[e0 + k];
              sc = leaky(el[static_cast<size_t>(src) * H + h] + erv, slope);
              ys[static_cast<size_t>(k) * H + h] = sc;
            } else {
              sc = xs[static_cast<size_t>(k) * H + h];
            }
            mx = fmaxf(mx, sc);
          }
          mx = group_max<kWave>(mx);
          float sum = 0.f;
          for (uint32_t k = lane; k < deg; k += kWave) {
            const float sc = FUSED ? ys[static_cast<size_t>(k) * H + h] : xs[static_cast<size_t>(k) * H + h];
            sum += softmax_exp(sc - mx);
          }
          sum = group_sum<kWave>(sum);
          const float inv = 1.f / sum;
          for (uint32_t k = lane; k < deg; k += kWave) {
            const float sc = FUSED ? ys[static_cast<size_t>(k) * H + h] : xs[static_cast<size_t>(k) * H + h];
            ys[static_cast<size_t>(k) * H + h] = softmax_exp(sc - mx) * inv;
          }
        }
      }
    }
  }
}

// FUSED = false: gx = y * (gy - sum_seg gy*y).
// FUSED = true : additionally multiplies by leaky_relu'(el[src]+er[d]) and writes
//                ger[d,h] = sum_seg gx[e,h].
// Visits the destinations with min_values <= n <= max_values (empty segments included when
// min_values is 0, so that ger is written for every destination).
// PART as in the forward kernel: the fused form is launched in two parts.
template <bool FUSED, bool POW2, int PART>
__global__ __launch_bounds__(256) void edge_softmax_bwd_kernel(float *__restrict__ gx, float *__restrict__ ger,
                                                               const float *__restrict__ gy,
                                                               const float *__restrict__ y,
                                                               const float *__restrict__ el,
                                                               const float *__restrict__ er,
                                                               const uint32_t *__restrict__ co,
                                                               const uint32_t *__restrict__ ri, uint32_t Vd,
                                                               uint32_t H, float slope, uint32_t min_values,
                                                               uint32_t max_values, uint32_t vec4, uint32_t set) {
  if (max_values == kByTotal) max_values = long_segment_values(static_cast<uint64_t>(co[Vd] - co[0]) * H);
  const uint32_t lane = lane_id();
  const uint64_t wave = wave_of_grid();
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  for (uint64_t first = wave * set; first < Vd; first += n_waves * set) {
    uint32_t my_e0, my_e1;
    uint64_t todo = wave_rows_in_class(co, Vd, first, set, H, min_values, max_values, my_e0, my_e1);
    while (todo) {
      const uint32_t j = static_cast<uint32_t>(__builtin_ctzll(todo));
      todo &= todo - 1;
      const uint32_t d = static_cast<uint32_t>(first) + j;
      const uint32_t e0 = wave_read(my_e0, j), e1 = wave_read(my_e1, j);
      const size_t base = static_cast<size_t>(e0) * H;
      const uint32_t n = (e1 - e0) * H;
      const float *gys = gy + base;
      const float *ys = y + base;
      float *gxs = gx + base;

      if (POW2) {
        if (PART <= 1 && n <= kWaveRegValues) {
          NTS_BY_SLOTS(kWave, softmax_bwd_regs, gxs, ger, gys, ys, el, er, ri, d, e0, n, H, slope, lane);
          continue;
        }
        if (PART == 1) continue;

        if (PART == 2 && FUSED && vec4 && n >= 2048u) {
          // 16-byte lanes: four consecutive values = heads (4 lane mod H) .. +3 of one edge
          const uint32_t h0 = (lane * 4u) & (H - 1);
          const uint32_t hq = H / 4;
          const float4 *gys4 = reinterpret_cast<const float4 *>(gys);
          const float4 *ys4 = reinterpret_cast<const float4 *>(ys);
          float4 *gxs4 = reinterpret_cast<float4 *>(gxs);
          float dot4[4] = {0.f, 0.f, 0.f, 0.f};
          strided_pass<4>(lane, n / 4, kWave, [&](uint64_t i) -> float4 { return gys4[i]; },
                          [&](uint64_t i, float4 g) {
                            const float4 a = ys4[i];
                            dot4[0] += g.x * a.x;
                            dot4[1] += g.y * a.y;
                            dot4[2] += g.z * a.z;
                            dot4[3] += g.w * a.w;
                          });
#pragma unroll
          for (int c = 0; c < 4; ++c) dot4[c] = head_reduce<1>(dot4[c], hq);
          const float4 erv = *reinterpret_cast<const float4 *>(er + static_cast<size_t>(d) * H + h0);
          float gsum4[4] = {0.f, 0.f, 0.f, 0.f};
          strided_pass<4>(lane, n / 4, kWave,
                          [&](uint64_t i) -> float4 {
                            const uint32_t src = ri[e0 + static_cast<uint32_t>(i * 4 / H)];
                            return *reinterpret_cast<const float4 *>(el + static_cast<size_t>(src) * H + h0);
                          },
                          [&](uint64_t i, float4 e) {
                            const float4 g = gys4[i], a = ys4[i];
                            float4 r;
                            r.x = a.x * (g.x - dot4[0]) * (e.x + erv.x > 0.f ? 1.f : slope);
                            r.y = a.y * (g.y - dot4[1]) * (e.y + erv.y > 0.f ? 1.f : slope);
                            r.z = a.z * (g.z - dot4[2]) * (e.z + erv.z > 0.f ? 1.f : slope);
                            r.w = a.w * (g.w - dot4[3]) * (e.w + erv.w > 0.f ? 1.f : slope);
                            gsum4[0] += r.x;
                            gsum4[1] += r.y;
                            gsum4[2] += r.z;
                            gsum4[3] += r.w;
                            gxs4[i] = r;
                          });
#pragma unroll
          for (int c = 0; c < 4; ++c) gsum4[c] = head_reduce<1>(gsum4[c], hq);
          if (lane < hq) {
            *reinterpret_cast<float4 *>(ger + static_cast<size_t>(d) * H + h0) =
                make_float4(gsum4[0], gsum4[1], gsum4[2], gsum4[3]);
          }
          continue;
        }
        const uint32_t h = lane & (H - 1);
        float dot = 0.f;
        strided_pass<8>(lane, n, kWave, [&](uint64_t i) -> float2 { return make_float2(gys[i], ys[i]); },
                        [&](uint64_t, float2 v) { dot += v.x * v.y; });
        dot = head_reduce<1>(dot, H);
        float erv = 0.f, gsum = 0.f;
        if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
        strided_pass<8>(lane, n, kWave,
                        [&](uint64_t i) -> float4 {
                          float pre = 1.f;
                          if (FUSED) pre = el[static_cast<size_t>(ri[e0 + i / H]) * H + h] + erv;
                          return make_float4(gys[i], ys[i], pre, 0.f);
                        },
                        [&](uint64_t i, float4 v) {
                          float g = v.y * (v.x - dot);
                          if (FUSED) {
                            g *= v.z > 0.f ? 1.f : slope;
                            gsum += g;
                          }
                          gxs[i] = g;
                        });
        if (FUSED) {
          gsum = head_reduce<1>(gsum, H);
          if (lane < H) ger[static_cast<size_t>(d) * H + lane] = gsum;
        }
      } else {
        const uint32_t deg = e1 - e0;
        for (uint32_t h = 0; h < H; ++h) {
          float dot = 0.f;
          for (uint32_t k = lane; k < deg; k += kWave) {
            const size_t i = static_cast<size_t>(k) * H + h;
            dot += gys[i] * ys[i];
          }
          dot = group_sum<kWave>(dot);
          float erv = 0.f, gsum = 0.f;
          if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
          for (uint32_t k = lane; k < deg; k += kWave) {
            const size_t i = static_cast<size_t>(k) * H + h;
            float g = ys[i] * (gys[i] - dot);
            if (FUSED) {
              const uint32_t src = ri[e0 + k];
              const float pre = el[static_cast<size_t>(src) * H + h] + erv;
              g *= pre > 0.f ? 1.f : slope;
              gsum += g;
            }
            gxs[i] = g;
          }
          if (FUSED) {
            gsum = group_sum<kWave>(gsum);
            if (lane == 0) ger[static_cast<size_t>(d) * H + h] = gsum;
          }
        }
      }
    }
  }
}

// Block kernels for long segments (power-of-two H <= 64 only; other head counts stay on the wave
// kernels).  1024 threads walk the segment's values; thread t always meets head t mod H.  Per-head
// maxima / sums are reduced inside each wave with the head butterfly, then across the 16 waves
// through LDS in wave order.
template <int MODE, int BLOCK = kLongBlock>  // 0 = max, 1 = sum
__device__ __forceinline__ float block_head_reduce(float v, uint32_t H, float (*red)[kWave]) {
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  v = head_reduce<MODE>(v, H);
  if (lane < H) red[wave][lane] = v;
  __syncthreads();
  const uint32_t h = lane & (H - 1);
  float r = red[0][h];
  for (uint32_t wv = 1; wv < BLOCK / kWave; ++wv) r = MODE == 0 ? fmaxf(r, red[wv][h]) : r + red[wv][h];
  __syncthreads();
  return r;
}

// The segment of destination d by one block.
template <bool FUSED, int BLOCK>
__device__ __forceinline__ void softmax_fwd_by_block(float *__restrict__ y, const float *__restrict__ x,
                                                     const float *__restrict__ el, const float *__restrict__ er,
                                                     const uint32_t *__restrict__ co, const uint32_t *__restrict__ ri, uint32_t d,
                                                     uint32_t H, float slope, float (*red)[kWave]) {
  const uint32_t h = threadIdx.x & (H - 1);
  const uint32_t e0 = co[d], e1 = co[d + 1];
  const size_t base = static_cast<size_t>(e0) * H;
  const size_t n = static_cast<size_t>(e1 - e0) * H;
  float *ys = y + base;
  const float *xs = FUSED ? nullptr : x + base;
  float erv = 0.f;
  if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
  float mx = kLowestMax, sum = 0.f;
  strided_max_sum_pass<8>(
      threadIdx.x, n, BLOCK,
      [&](uint64_t j) -> float {
        if (!FUSED) return xs[j];
        const uint32_t src = ri[e0 + j / H];
        return leaky(el[static_cast<size_t>(src) * H + h] + erv, slope);
      },
      [&](uint64_t j, float sc) {
        if (FUSED) ys[j] = sc;
      },
      mx, sum);
  const float thread_mx = mx;
  mx = block_head_reduce<0, BLOCK>(mx, H, red);
  sum = block_head_reduce<1, BLOCK>(sum * softmax_exp(thread_mx - mx), H, red);
  const float inv = 1.f / sum;
  strided_pass<8>(threadIdx.x, n, BLOCK, [&](uint64_t j) -> float { return FUSED ? ys[j] : xs[j]; },
                  [&](uint64_t j, float sc) { ys[j] = softmax_exp(sc - mx) * inv; });
}

template <bool FUSED>
__global__ __launch_bounds__(kLongBlock) void edge_softmax_fwd_long_kernel(
    float *__restrict__ y, const float *__restrict__ x, const float *__restrict__ el, const float *__restrict__ er,
    const uint32_t *__restrict__ co, const uint32_t *__restrict__ ri, const uint32_t *__restrict__ list,
    const uint32_t *__restrict__ count, uint32_t H, float slope) {
  __shared__ float red[kLongBlock / kWave][kWave];
  const uint32_t n_rows = *count;
  for (uint32_t i = blockIdx.x; i < n_rows; i += gridDim.x)
    softmax_fwd_by_block<FUSED, kLongBlock>(y, x, el, er, co, ri, list[i], H, slope, red);
}

// gx over the edges [e0, e1) of destination d by one block, with their dot product given; returns with FUSED the sum of gx.
template <bool FUSED, int BLOCK>
__device__ __forceinline__ float softmax_bwd_pass(float *__restrict__ gx, const float *__restrict__ gy, const float *__restrict__ y,
                                                  const float *__restrict__ el, const float *__restrict__ er,
                                                  const uint32_t *__restrict__ ri, uint32_t d, uint32_t e0, uint32_t e1, uint32_t H,
                                                  float slope, float dot, float (*red)[kWave]) {
  const uint32_t h = threadIdx.x & (H - 1);
  const size_t base = static_cast<size_t>(e0) * H;
  const float *gys = gy + base;
  const float *ys = y + base;
  float *gxs = gx + base;
  float erv = 0.f, gsum = 0.f;
  if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
  strided_pass<8>(threadIdx.x, static_cast<uint64_t>(e1 - e0) * H, BLOCK,
                  [&](uint64_t j) -> float4 {
                    float pre = 1.f;
                    if (FUSED) pre = el[static_cast<size_t>(ri[e0 + j / H]) * H + h] + erv;
                    return make_float4(gys[j], ys[j], pre, 0.f);
                  },
                  [&](uint64_t j, float4 v) {
                    float g = v.y * (v.x - dot);
                    if (FUSED) {
                      g *= v.z > 0.f ? 1.f : slope;
                      gsum += g;
                    }
                    gxs[j] = g;
                  });
  return FUSED ? block_head_reduce<1, BLOCK>(gsum, H, red) : 0.f;
}

template <int BLOCK>
__device__ __forceinline__ float softmax_dot_by_block(const float *__restrict__ gy, const float *__restrict__ y, uint32_t e0,
                                                      uint32_t e1, uint32_t H, float (*red)[kWave]) {
  const size_t base = static_cast<size_t>(e0) * H;
  const float *gys = gy + base;
  const float *ys = y + base;
  float dot = 0.f;
  strided_pass<8>(threadIdx.x, static_cast<uint64_t>(e1 - e0) * H, BLOCK, [&](uint64_t j) -> float2 { return make_float2(gys[j], ys[j]); },
                  [&](uint64_t, float2 v) { dot += v.x * v.y; });
  return block_head_reduce<1, BLOCK>(dot, H, red);
}

template <bool FUSED, int BLOCK>
__device__ __forceinline__ void softmax_bwd_by_block(float *__restrict__ gx, float *__restrict__ ger, const float *__restrict__ gy,
                                                     const float *__restrict__ y, const float *__restrict__ el,
                                                     const float *__restrict__ er, const uint32_t *__restrict__ co,
                                                     const uint32_t *__restrict__ ri, uint32_t d, uint32_t H, float slope,
                                                     float (*red)[kWave]) {
  const uint32_t e0 = co[d], e1 = co[d + 1];
  const float dot = softmax_dot_by_block<BLOCK>(gy, y, e0, e1, H, red);
  const float gsum = softmax_bwd_pass<FUSED, BLOCK>(gx, gy, y, el, er, ri, d, e0, e1, H, slope, dot, red);
  if (FUSED && threadIdx.x < H) ger[static_cast<size_t>(d) * H + threadIdx.x] = gsum;
}

template <bool FUSED>
__global__ __launch_bounds__(kLongBlock) void edge_softmax_bwd_long_kernel(
    float *__restrict__ gx, float *__restrict__ ger, const float *__restrict__ gy, const float *__restrict__ y,
    const float *__restrict__ el, const float *__restrict__ er, const uint32_t *__restrict__ co,
    const uint32_t *__restrict__ ri, const uint32_t *__restrict__ list, const uint32_t *__restrict__ count, uint32_t H,
    float slope) {
  __shared__ float red[kLongBlock / kWave][kWave];
  const uint32_t n_rows = *count;
  for (uint32_t i = blockIdx.x; i < n_rows; i += gridDim.x)
    softmax_bwd_by_block<FUSED, kLongBlock>(gx, ger, gy, y, el, er, co, ri, list[i], H, slope, red);
}

// ---- giant segments of the softmax operators ----------------------------------------------------
//
// A piece of a giant destination is reduced by one block; per-head results of the pieces are
// combined in piece order.  Forward uses the online form: a piece keeps (m_p, s_p = sum exp(x - m_p));
// the destination's maximum is max_p m_p and its sum is sum_p s_p * exp(m_p - m).
// stats[piece, 0..H) / [H..2H) and rowstat[giant row, 0..H) / [H..2H) hold the two values per head.

template <bool FUSED, int BLOCK>
__device__ __forceinline__ void giant_softmax_stats(float *__restrict__ stats, float *__restrict__ y, const float *__restrict__ x,
                                                    const float *__restrict__ el, const float *__restrict__ er,
                                                    const uint32_t *__restrict__ ri, uint32_t p, uint4 pc, uint32_t H, float slope,
                                                    float (*red)[kWave]) {
  const uint32_t h = threadIdx.x & (H - 1);
  const uint32_t d = pc.y, e0 = pc.z;
  const size_t base = static_cast<size_t>(e0) * H;
  const uint64_t n = static_cast<uint64_t>(pc.w - e0) * H;
  float *ys = y + base;
  const float *xs = FUSED ? nullptr : x + base;
  float erv = 0.f;
  if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
  float mx = kLowestMax;
  strided_pass<8>(threadIdx.x, n, BLOCK,
                  [&](uint64_t j) -> float {
                    if (!FUSED) return xs[j];
                    const uint32_t src = ri[e0 + j / H];
                    return leaky(el[static_cast<size_t>(src) * H + h] + erv, slope);
                  },
                  [&](uint64_t j, float sc) {
                    if (FUSED) ys[j] = sc;
                    mx = fmaxf(mx, sc);
                  });
  mx = block_head_reduce<0, BLOCK>(mx, H, red);
  float sum = 0.f;
  strided_pass<8>(threadIdx.x, n, BLOCK, [&](uint64_t j) -> float { return FUSED ? ys[j] : xs[j]; },
                  [&](uint64_t, float sc) { sum += softmax_exp(sc - mx); });
  sum = block_head_reduce<1, BLOCK>(sum, H, red);
  if (threadIdx.x < H) {
    stats[static_cast<size_t>(p) * 2 * H + threadIdx.x] = mx;
    stats[static_cast<size_t>(p) * 2 * H + H + threadIdx.x] = sum;
  }
}

template <bool FUSED>
__global__ __launch_bounds__(kLongBlock) void giant_softmax_stats_kernel(
    float *__restrict__ stats, float *__restrict__ y, const float *__restrict__ x, const float *__restrict__ el,
    const float *__restrict__ er, const uint32_t *__restrict__ ri, const uint32_t *__restrict__ hdr,
    const uint4 *__restrict__ pieces, uint32_t H, float slope) {
  __shared__ float red[kLongBlock / kWave][kWave];
  const uint32_t n_pieces = hdr[1];
  for (uint32_t p = blockIdx.x; p < n_pieces; p += gridDim.x)
    giant_softmax_stats<FUSED, kLongBlock>(stats, y, x, el, er, ri, p, pieces[p], H, slope, red);
}

// MODE 0: online-softmax combine of (m_p, s_p).  MODE 1: plain sum of stats[piece, 0..H) in piece
// order (`width` floats of a piece from the next); the result goes to rowstat[giant row, 0..H) or, when `to_rows` is set, to to_rows[row, 0..H)
// (the per-destination gradient sum of the fused backward).
template <int MODE>
__global__ __launch_bounds__(64) void giant_softmax_combine_kernel(float *__restrict__ rowstat,
                                                                   float *__restrict__ to_rows,
                                                                   const float *__restrict__ stats,
                                                                   const uint32_t *__restrict__ hdr,
                                                                   const uint32_t *__restrict__ giant_rows,
                                                                   const uint32_t *__restrict__ first, uint32_t H, uint32_t width) {
  const uint32_t n = hdr[0];
  const uint32_t h = threadIdx.x;
  if (h >= H) return;
  for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
    const uint32_t p0 = first[i], p1 = first[i + 1];
    if (MODE == 0) {
      float m = -INFINITY;
      for (uint32_t p = p0; p < p1; ++p) m = fmaxf(m, stats[static_cast<size_t>(p) * width + h]);
      float sum = 0.f;
      for (uint32_t p = p0; p < p1; ++p)
        sum += stats[static_cast<size_t>(p) * width + H + h] * softmax_exp(stats[static_cast<size_t>(p) * width + h] - m);
      rowstat[static_cast<size_t>(i) * 2 * H + h] = m;
      rowstat[static_cast<size_t>(i) * 2 * H + H + h] = sum;
    } else {
      float sum = 0.f;
      for (uint32_t p = p0; p < p1; ++p) sum += stats[static_cast<size_t>(p) * width + h];
      if (to_rows) to_rows[static_cast<size_t>(giant_rows[i]) * H + h] = sum;
      else rowstat[static_cast<size_t>(i) * 2 * H + h] = sum;
    }
  }
}

template <bool FUSED>
__global__ __launch_bounds__(kLongBlock) void giant_softmax_apply_kernel(float *__restrict__ y,
                                                                         const float *__restrict__ x,
                                                                         const float *__restrict__ rowstat,
                                                                         const uint32_t *__restrict__ hdr,
                                                                         const uint4 *__restrict__ pieces,
                                                                         uint32_t H) {
  const uint32_t n_pieces = hdr[1];
  const uint32_t h = threadIdx.x & (H - 1);
  for (uint32_t p = blockIdx.x; p < n_pieces; p += gridDim.x) {
    const uint4 pc = pieces[p];
    const size_t base = static_cast<size_t>(pc.z) * H;
    const uint64_t n = static_cast<uint64_t>(pc.w - pc.z) * H;
    const float mx = rowstat[static_cast<size_t>(pc.x) * 2 * H + h];
    const float sum = rowstat[static_cast<size_t>(pc.x) * 2 * H + H + h];
    float *ys = y + base;
    const float *xs = FUSED ? ys : x + base;  // the fused forward left the raw score in y
    const float inv = 1.f / sum;
    strided_pass<8>(threadIdx.x, n, kLongBlock, [&](uint64_t j) -> float { return xs[j]; },
                    [&](uint64_t j, float sc) { ys[j] = softmax_exp(sc - mx) * inv; });
  }
}

// Backward, first stage: stats[piece, h] = sum over the piece of gy * y.
__global__ __launch_bounds__(kLongBlock) void giant_softmax_dot_kernel(float *__restrict__ stats,
                                                                       const float *__restrict__ gy,
                                                                       const float *__restrict__ y,
                                                                       const uint32_t *__restrict__ hdr,
                                                                       const uint4 *__restrict__ pieces, uint32_t H) {
  __shared__ float red[kLongBlock / kWave][kWave];
  const uint32_t n_pieces = hdr[1];
  for (uint32_t p = blockIdx.x; p < n_pieces; p += gridDim.x) {
    const uint4 pc = pieces[p];
    const float dot = softmax_dot_by_block<kLongBlock>(gy, y, pc.z, pc.w, H, red);
    if (threadIdx.x < H) stats[static_cast<size_t>(p) * H + threadIdx.x] = dot;
  }
}

// Backward, last stage: gx over the piece; with FUSED also stats[piece, h] = sum of the piece's gx.
template <bool FUSED>
__global__ __launch_bounds__(kLongBlock) void giant_softmax_bwd_apply_kernel(
    float *__restrict__ gx, float *__restrict__ stats, const float *__restrict__ gy, const float *__restrict__ y,
    const float *__restrict__ el, const float *__restrict__ er, const uint32_t *__restrict__ ri,
    const float *__restrict__ rowstat, const uint32_t *__restrict__ hdr, const uint4 *__restrict__ pieces, uint32_t H,
    float slope) {
  __shared__ float red[kLongBlock / kWave][kWave];
  const uint32_t n_pieces = hdr[1];
  const uint32_t h = threadIdx.x & (H - 1);
  for (uint32_t p = blockIdx.x; p < n_pieces; p += gridDim.x) {
    const uint4 pc = pieces[p];
    const float dot = rowstat[static_cast<size_t>(pc.x) * 2 * H + h];
    const float gsum = softmax_bwd_pass<FUSED, kLongBlock>(gx, gy, y, el, er, ri, pc.y, pc.z, pc.w, H, slope, dot, red);
    if (FUSED && threadIdx.x < H) stats[static_cast<size_t>(p) * H + threadIdx.x] = gsum;
  }
}

// ---- softmax operators on few rows ----------------------------------------------------------------
//
// Calls of at most kFewRows destinations, heads a power of two up to kShortG: what the kernels above do in nine to eleven
// launches on two streams, whose gaps and idle ends are most of the time there (and, below a million values, the host's
// launching them all of it), in one, or three to six where there are hub rows:
//   few_long_rows_kernel   lists the hub rows and cuts the giant ones (from kLongMinVertices rows up; above kOneBlockRows the three
//                          launches of many rows)
//   few_softmax_kernel     its first blocks take the listed rows and the pieces' statistics; every other wavefront a set of
//                          consecutive rows, short segments four at a time, each of the longer ones by the whole wavefront
//   few_giant_apply_kernel combines the statistics of a piece's row itself and writes the piece
//   giant_softmax_combine_kernel  (fused backward) the sums of the giant rows' gradients
// stats[piece, 0 .. 2H): (maximum, sum) forward; (dot product, sum of gx) backward.
constexpr uint64_t kDenseRow = 64;  // edges a row from which a wavefront takes kDenseSet rows together
constexpr uint32_t kDenseSet = 4;
template <bool FUSED>
__device__ __forceinline__ void softmax_fwd_by_wave(float *__restrict__ ys, const float *__restrict__ xs, const float *__restrict__ el,
                                                    const float *__restrict__ er, const uint32_t *__restrict__ ri, uint32_t d, uint32_t e0,
                                                    uint64_t n, uint32_t H, float slope, uint32_t lane) {
  if (n <= kWaveRegValues) {
    NTS_BY_SLOTS(kWave, softmax_fwd_regs, ys, xs, el, er, ri, d, e0, n, H, slope, lane);
    return;
  }
  const uint32_t h = lane & (H - 1);
  float erv = 0.f;
  if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
  float mx = kLowestMax, sum = 0.f;
  strided_max_sum_pass<8>(
      lane, n, kWave,
      [&](uint64_t i) -> float {
        if (!FUSED) return xs[i];
        const uint32_t src = ri[e0 + i / H];
        return leaky(el[static_cast<size_t>(src) * H + h] + erv, slope);
      },
      [&](uint64_t i, float sc) {
        if (FUSED) ys[i] = sc;
      },
      mx, sum);
  const float lane_mx = mx;
  mx = head_reduce<0>(mx, H);
  sum = head_reduce<1>(sum * softmax_exp(lane_mx - mx), H);
  const float inv = 1.f / sum;
  strided_pass<8>(lane, n, kWave, [&](uint64_t i) -> float { return FUSED ? ys[i] : xs[i]; },
                  [&](uint64_t i, float sc) { ys[i] = softmax_exp(sc - mx) * inv; });
}

template <bool FUSED>
__device__ __forceinline__ void softmax_bwd_by_wave(float *__restrict__ gxs, float *__restrict__ ger, const float *__restrict__ gys,
                                                    const float *__restrict__ ys, const float *__restrict__ el,
                                                    const float *__restrict__ er, const uint32_t *__restrict__ ri, uint32_t d, uint32_t e0,
                                                    uint64_t n, uint32_t H, float slope, uint32_t lane) {
  if (n <= kWaveRegValues) {
    NTS_BY_SLOTS(kWave, softmax_bwd_regs, gxs, ger, gys, ys, el, er, ri, d, e0, n, H, slope, lane);
    return;
  }
  const uint32_t h = lane & (H - 1);
  float dot = 0.f;
  strided_pass<8>(lane, n, kWave, [&](uint64_t i) -> float2 { return make_float2(gys[i], ys[i]); },
                  [&](uint64_t, float2 v) { dot += v.x * v.y; });
  dot = head_reduce<1>(dot, H);
  float erv = 0.f, gsum = 0.f;
  if (FUSED) erv = er[static_cast<size_t>(d) * H + h];
  strided_pass<8>(lane, n, kWave,
                  [&](uint64_t i) -> float4 {
                    float pre = 1.f;
                    if (FUSED) pre = el[static_cast<size_t>(ri[e0 + i / H]) * H + h] + erv;
                    return make_float4(gys[i], ys[i], pre, 0.f);
                  },
                  [&](uint64_t i, float4 v) {
                    float g = v.y * (v.x - dot);
                    if (FUSED) {
                      g *= v.z > 0.f ? 1.f : slope;
                      gsum += g;
                    }
                    gxs[i] = g;
                  });
  if (FUSED) {
    gsum = head_reduce<1>(gsum, H);
    if (lane < H) ger[static_cast<size_t>(d) * H + lane] = gsum;
  }
}

// The fused operators' segments above the register class with 16-byte lanes (heads a multiple of four, 16-byte aligned arrays), by
// a wavefront or a block: thread t of WIDTH takes the vectors t, t + WIDTH, ... of the segment, four consecutive heads of one
// edge each, and always meets the heads h0 = 4 t mod H .. + 3; threads H / 4 apart hold the same ones.  `most` and `all` reduce
// over these.
struct Attention4 {
  const float *el;
  const uint32_t *ri;
  uint32_t e0, H, h0;
  float4 er;
  float slope;
  __device__ __forceinline__ Attention4(const float *el_, const float *er_, const uint32_t *ri_, uint32_t d, uint32_t e0_, uint32_t H_,
                                        float slope_, uint32_t t)
      : el(el_), ri(ri_), e0(e0_), H(H_), h0((t * 4u) & (H_ - 1)), slope(slope_) {
    er = *reinterpret_cast<const float4 *>(er_ + static_cast<size_t>(d) * H + h0);
  }
  __device__ __forceinline__ float4 sum(uint64_t i) const {  // el + er of vector i
    const uint32_t src = ri[e0 + static_cast<uint32_t>(i * 4 / H)];
    const float4 e = *reinterpret_cast<const float4 *>(el + static_cast<size_t>(src) * H + h0);
    return make_float4(e.x + er.x, e.y + er.y, e.z + er.z, e.w + er.w);
  }
  __device__ __forceinline__ float4 score(uint64_t i) const {
    const float4 v = sum(i);
    return make_float4(leaky(v.x, slope), leaky(v.y, slope), leaky(v.z, slope), leaky(v.w, slope));
  }
};
// Raw scores to ys, and the (maximum, sum) of each of the four heads.
template <int WIDTH, typename Most, typename All>
__device__ __forceinline__ void attention_stats4(float4 *__restrict__ ys, const Attention4 &a, uint64_t nv, uint32_t t, Most most, All all,
                                                 float (&mx)[4], float (&sum)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    mx[c] = kLowestMax;
    sum[c] = 0.f;
  }
  strided_max_sum_pass4<4>(t, nv, WIDTH, [&](uint64_t i) { return a.score(i); }, [&](uint64_t i, float4 v) { ys[i] = v; }, mx, sum);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float own = mx[c];
    mx[c] = most(own);
    sum[c] = all(sum[c] * softmax_exp(own - mx[c]));
  }
}
template <int WIDTH>
__device__ __forceinline__ void attention_write4(float4 *__restrict__ ys, uint64_t nv, uint32_t t, const float (&mx)[4], const float (&sum)[4]) {
  const float inv[4] = {1.f / sum[0], 1.f / sum[1], 1.f / sum[2], 1.f / sum[3]};
  strided_pass<4>(t, nv, WIDTH, [&](uint64_t i) -> float4 { return ys[i]; },
                  [&](uint64_t i, float4 v) {
                    ys[i] = make_float4(softmax_exp(v.x - mx[0]) * inv[0], softmax_exp(v.y - mx[1]) * inv[1], softmax_exp(v.z - mx[2]) * inv[2],
                                        softmax_exp(v.w - mx[3]) * inv[3]);
                  });
}
template <int WIDTH, typename All>
__device__ __forceinline__ void attention_dot4(const float4 *__restrict__ gys, const float4 *__restrict__ ys, uint64_t nv, uint32_t t, All all,
                                               float (&dot)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) dot[c] = 0.f;
  struct Two {
    float4 g, a;
  };
  strided_pass<4>(t, nv, WIDTH, [&](uint64_t i) -> Two { return Two{gys[i], ys[i]}; },
                  [&](uint64_t, Two v) {
                    dot[0] += v.g.x * v.a.x;
                    dot[1] += v.g.y * v.a.y;
                    dot[2] += v.g.z * v.a.z;
                    dot[3] += v.g.w * v.a.w;
                  });
#pragma unroll
  for (int c = 0; c < 4; ++c) dot[c] = all(dot[c]);
}
// gx of the segment; gsum: its sum over each of the four heads.
template <int WIDTH, typename All>
__device__ __forceinline__ void attention_bwd4(float4 *__restrict__ gxs, const float4 *__restrict__ gys, const float4 *__restrict__ ys,
                                               const Attention4 &a, uint64_t nv, uint32_t t, All all, const float (&dot)[4], float (&gsum)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) gsum[c] = 0.f;
  strided_pass<4>(t, nv, WIDTH, [&](uint64_t i) -> float4 { return a.sum(i); },
                  [&](uint64_t i, float4 s) {
                    const float4 g = gys[i], y = ys[i];
                    const float4 r = make_float4(y.x * (g.x - dot[0]) * (s.x > 0.f ? 1.f : a.slope), y.y * (g.y - dot[1]) * (s.y > 0.f ? 1.f : a.slope),
                                                 y.z * (g.z - dot[2]) * (s.z > 0.f ? 1.f : a.slope), y.w * (g.w - dot[3]) * (s.w > 0.f ? 1.f : a.slope));
                    gsum[0] += r.x;
                    gsum[1] += r.y;
                    gsum[2] += r.z;
                    gsum[3] += r.w;
                    gxs[i] = r;
                  });
#pragma unroll
  for (int c = 0; c < 4; ++c) gsum[c] = all(gsum[c]);
}

struct FewHubs {
  const uint32_t *list, *count, *hdr, *first;
  const uint4 *pieces;
  float *stats;
  uint32_t blocks;  // of the launch, set aside for them (0: no hub rows are looked for)
};

// A hub row or a piece of a giant row by one block of 256 threads.
template <bool FUSED, bool BWD, bool VEC4>
__device__ __forceinline__ void few_hub_row(float *__restrict__ out, float *__restrict__ ger, const float *__restrict__ x_or_gy,
                                            const float *__restrict__ y, const float *__restrict__ el, const float *__restrict__ er,
                                            const uint32_t *__restrict__ co, const uint32_t *__restrict__ ri, uint32_t d, uint32_t H,
                                            float slope, float (*red)[kWave]) {
  if constexpr (!VEC4) {
    if (BWD) softmax_bwd_by_block<FUSED, 256>(out, ger, x_or_gy, y, el, er, co, ri, d, H, slope, red);
    else softmax_fwd_by_block<FUSED, 256>(out, x_or_gy, el, er, co, ri, d, H, slope, red);
  } else {
    const uint32_t t = threadIdx.x, e0 = co[d], hq = H / 4;
    const uint64_t nv = static_cast<uint64_t>(co[d + 1] - e0) * hq;
    const Attention4 a(el, er, ri, d, e0, H, slope, t);
    float4 *outs = reinterpret_cast<float4 *>(out + static_cast<size_t>(e0) * H);
    auto most = [&](float v) { return block_head_reduce<0, 256>(v, hq, red); };
    auto all = [&](float v) { return block_head_reduce<1, 256>(v, hq, red); };
    float s0[4], s1[4];
    if constexpr (BWD) {
      const float4 *gys = reinterpret_cast<const float4 *>(x_or_gy + static_cast<size_t>(e0) * H), *ys = reinterpret_cast<const float4 *>(y + static_cast<size_t>(e0) * H);
      attention_dot4<256>(gys, ys, nv, t, all, s0);
      attention_bwd4<256>(outs, gys, ys, a, nv, t, all, s0, s1);
      if (t < hq) *reinterpret_cast<float4 *>(ger + static_cast<size_t>(d) * H + a.h0) = make_float4(s1[0], s1[1], s1[2], s1[3]);
    } else {
      attention_stats4<256>(outs, a, nv, t, most, all, s0, s1);
      attention_write4<256>(outs, nv, t, s0, s1);
    }
  }
}
template <bool FUSED, bool BWD, bool VEC4>
__device__ __forceinline__ void few_giant_piece(float *__restrict__ stats, float *__restrict__ out, const float *__restrict__ x_or_gy,
                                                const float *__restrict__ y, const float *__restrict__ el, const float *__restrict__ er,
                                                const uint32_t *__restrict__ ri, uint32_t p, uint4 pc, uint32_t H, float slope,
                                                float (*red)[kWave]) {
  if constexpr (BWD) {
    const float dot = softmax_dot_by_block<256>(x_or_gy, y, pc.z, pc.w, H, red);
    if (threadIdx.x < H) stats[static_cast<size_t>(p) * 2 * H + threadIdx.x] = dot;
  } else if constexpr (!VEC4) {
    giant_softmax_stats<FUSED, 256>(stats, out, x_or_gy, el, er, ri, p, pc, H, slope, red);
  } else {
    const uint32_t t = threadIdx.x, hq = H / 4;
    const Attention4 a(el, er, ri, pc.y, pc.z, H, slope, t);
    float mx[4], sum[4];
    attention_stats4<256>(
        reinterpret_cast<float4 *>(out + static_cast<size_t>(pc.z) * H), a, static_cast<uint64_t>(pc.w - pc.z) * hq, t,
        [&](float v) { return block_head_reduce<0, 256>(v, hq, red); }, [&](float v) { return block_head_reduce<1, 256>(v, hq, red); }, mx, sum);
    if (t < hq) {
      float *st = stats + static_cast<size_t>(p) * 2 * H + a.h0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        st[c] = mx[c];
        st[H + c] = sum[c];
      }
    }
  }
}

template <bool FUSED, bool BWD, bool VEC4>
__global__ __launch_bounds__(256) void few_softmax_kernel(float *__restrict__ out, float *__restrict__ ger,
                                                          const float *__restrict__ x_or_gy, const float *__restrict__ y,
                                                          const float *__restrict__ el, const float *__restrict__ er,
                                                          const uint32_t *__restrict__ co, const uint32_t *__restrict__ ri,
                                                          uint32_t Vd, uint32_t H, float slope, uint32_t set, FewHubs hubs) {
  if (blockIdx.x < hubs.blocks) {
    __shared__ float red[256 / kWave][kWave];
    if (!hubs.list) {
      // Few enough rows for the hub blocks to find their own, a row a thread, dealt out in an order without pattern as in the edge
      // sums (sum_long_rows_in_this_block).
      __shared__ uint32_t n_found;
      __shared__ uint16_t found[256];
      if (threadIdx.x == 0) n_found = 0;
      const uint32_t at = threadIdx.x * hubs.blocks + blockIdx.x, r = at * 40503u % kLongMinVertices;  // (odd: every row once)
      uint32_t deg = 0;
      if (at < kLongMinVertices && r < Vd) deg = co[r + 1] - co[r];
      const uint64_t limit = few_long_values(static_cast<uint64_t>(co[Vd] - co[0]) * H);
      __syncthreads();
      if (static_cast<uint64_t>(deg) * H > limit) found[atomicAdd(&n_found, 1u)] = static_cast<uint16_t>(r);
      __syncthreads();
      const uint32_t n = n_found;
      for (uint32_t i = 0; i < n; ++i) few_hub_row<FUSED, BWD, VEC4>(out, ger, x_or_gy, y, el, er, co, ri, found[i], H, slope, red);
      return;
    }
    const uint32_t n_rows = *hubs.count, n_pieces = hubs.hdr[1];
    for (uint32_t i = blockIdx.x; i < n_rows + n_pieces; i += hubs.blocks) {
      if (i < n_rows) few_hub_row<FUSED, BWD, VEC4>(out, ger, x_or_gy, y, el, er, co, ri, hubs.list[i], H, slope, red);
      else few_giant_piece<FUSED, BWD, VEC4>(hubs.stats, out, x_or_gy, y, el, er, ri, i - n_rows, hubs.pieces[i - n_rows], H, slope, red);
    }
    return;
  }
  const uint32_t lane = lane_id();
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x - hubs.blocks) * (256 / kWave);
  const uint64_t limit = hubs.blocks ? few_long_values(static_cast<uint64_t>(co[Vd] - co[0]) * H) : ~0ull;
  if (co[Vd] - co[0] >= kDenseRow * Vd) set = set < kDenseSet ? set : kDenseSet;
  for (uint64_t first = wave_of_grid(hubs.blocks) * set; first < Vd; first += n_waves * set) {
    uint32_t my_e0 = 0, my_e1 = 0;
    const bool mine = lane < set && first + lane < Vd;
    if (mine) {
      my_e0 = co[first + lane];
      my_e1 = co[first + lane + 1];
    }
    const uint64_t my_n = static_cast<uint64_t>(my_e1 - my_e0) * H;
    uint64_t todo = __ballot(my_n > kShortValues && my_n <= limit);
    const uint64_t shorts = __ballot(mine && my_n <= kShortValues && (my_n || (BWD && FUSED)));
    {
      const uint32_t gl = lane & (kShortG - 1), grp = lane / kShortG;
      for (uint64_t left = shorts; left;) {
        // the next four short rows, one a group
        uint32_t j = kWave;
#pragma unroll
        for (uint32_t g = 0; g < kWave / kShortG; ++g) {
          if (left) {
            if (g == grp) j = static_cast<uint32_t>(__builtin_ctzll(left));
            left &= left - 1;
          }
        }
        const uint32_t e0 = __shfl(my_e0, j & (kWave - 1), kWave), e1 = __shfl(my_e1, j & (kWave - 1), kWave);
        const uint32_t n = j < kWave ? (e1 - e0) * H : 0u, d = static_cast<uint32_t>(first) + j;
        const size_t base = static_cast<size_t>(e0) * H;
        if (BWD) {
          if (j < kWave) {
            if (!any_lane(n > 2u * kShortG)) softmax_bwd_regs<FUSED, kShortG, 2>(out + base, ger, x_or_gy + base, y + base, el, er, ri, d, e0, n, H, slope, gl);
            else softmax_bwd_regs<FUSED, kShortG, kShortK>(out + base, ger, x_or_gy + base, y + base, el, er, ri, d, e0, n, H, slope, gl);
          }
        } else if (n) {
          NTS_BY_SLOTS(kShortG, softmax_fwd_regs, out + base, FUSED ? nullptr : x_or_gy + base, el, er, ri, d, e0, n, H, slope, gl);
        }
      }
    }
    while (todo) {
      const uint32_t j = static_cast<uint32_t>(__builtin_ctzll(todo));
      todo &= todo - 1;
      const uint32_t d = static_cast<uint32_t>(first) + j;
      const uint32_t e0 = wave_read(my_e0, j), e1 = wave_read(my_e1, j);
      const size_t base = static_cast<size_t>(e0) * H;
      const uint64_t n64 = static_cast<uint64_t>(e1 - e0) * H;
      if constexpr (VEC4) {
        if (n64 > kWaveRegValues) {
          const uint32_t hq = H / 4;
          const uint64_t nv = n64 / 4;
          const Attention4 a(el, er, ri, d, e0, H, slope, lane);
          float4 *outs = reinterpret_cast<float4 *>(out + base);
          auto most = [&](float v) { return head_reduce<0>(v, hq); };
          auto all = [&](float v) { return head_reduce<1>(v, hq); };
          float s0[4], s1[4];
          if constexpr (BWD) {
            const float4 *gys = reinterpret_cast<const float4 *>(x_or_gy + base), *ys = reinterpret_cast<const float4 *>(y + base);
            attention_dot4<kWave>(gys, ys, nv, lane, all, s0);
            attention_bwd4<kWave>(outs, gys, ys, a, nv, lane, all, s0, s1);
            if (lane < hq) *reinterpret_cast<float4 *>(ger + static_cast<size_t>(d) * H + a.h0) = make_float4(s1[0], s1[1], s1[2], s1[3]);
          } else {
            attention_stats4<kWave>(outs, a, nv, lane, most, all, s0, s1);
            attention_write4<kWave>(outs, nv, lane, s0, s1);
          }
          continue;
        }
      }
      if (BWD) softmax_bwd_by_wave<FUSED>(out + base, ger, x_or_gy + base, y + base, el, er, ri, d, e0, n64, H, slope, lane);
      else softmax_fwd_by_wave<FUSED>(out + base, FUSED ? nullptr : x_or_gy + base, el, er, ri, d, e0, n64, H, slope, lane);
    }
  }
}

template <bool FUSED, bool BWD, bool VEC4>
__global__ __launch_bounds__(256) void few_giant_apply_kernel(float *__restrict__ out, const float *__restrict__ x_or_gy,
                                                              const float *__restrict__ y, const float *__restrict__ el,
                                                              const float *__restrict__ er, const uint32_t *__restrict__ ri,
                                                              uint32_t H, float slope, FewHubs hubs) {
  __shared__ float red[256 / kWave][kWave];
  const uint32_t n_pieces = hubs.hdr[1];
  const uint32_t lane = lane_id(), h = lane & (H - 1);
  for (uint32_t p = blockIdx.x; p < n_pieces; p += gridDim.x) {
    const uint4 pc = hubs.pieces[p];
    // lane l takes the pieces l / H, l / H + 64 / H, ... of the row, then the lanes of a head are combined
    const uint32_t q0 = hubs.first[pc.x] + lane / H, q1 = hubs.first[pc.x + 1];
    const float *st = hubs.stats + h;
    if (BWD) {
      float dot = 0.f;
      for (uint32_t q = q0; q < q1; q += kWave / H) dot += st[static_cast<size_t>(q) * 2 * H];
      dot = head_reduce<1>(dot, H);
      if constexpr (VEC4) {
        const uint32_t t = threadIdx.x, hq = H / 4;
        const Attention4 a(el, er, ri, pc.y, pc.z, H, slope, t);
        const size_t base = static_cast<size_t>(pc.z) * H;
        float d4[4], gsum[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) d4[c] = __shfl(dot, a.h0 + c, kWave);  // (lane h holds head h)
        attention_bwd4<256>(reinterpret_cast<float4 *>(out + base), reinterpret_cast<const float4 *>(x_or_gy + base),
                            reinterpret_cast<const float4 *>(y + base), a, static_cast<uint64_t>(pc.w - pc.z) * hq, t,
                            [&](float v) { return block_head_reduce<1, 256>(v, hq, red); }, d4, gsum);
        if (t < hq) *reinterpret_cast<float4 *>(hubs.stats + static_cast<size_t>(p) * 2 * H + H + a.h0) = make_float4(gsum[0], gsum[1], gsum[2], gsum[3]);
        continue;
      }
      const float gsum = softmax_bwd_pass<FUSED, 256>(out, x_or_gy, y, el, er, ri, pc.y, pc.z, pc.w, H, slope, dot, red);
      if (FUSED && threadIdx.x < H) hubs.stats[static_cast<size_t>(p) * 2 * H + H + threadIdx.x] = gsum;
      continue;
    }
    float mx = kLowestMax, sum = 0.f;
    for (uint32_t q = q0; q < q1; q += kWave / H) mx = fmaxf(mx, st[static_cast<size_t>(q) * 2 * H]);
    mx = head_reduce<0>(mx, H);
    for (uint32_t q = q0; q < q1; q += kWave / H)
      sum += st[static_cast<size_t>(q) * 2 * H + H] * softmax_exp(st[static_cast<size_t>(q) * 2 * H] - mx);
    sum = head_reduce<1>(sum, H);
    const float inv = 1.f / sum;
    const size_t base = static_cast<size_t>(pc.z) * H;
    float *ys = out + base;
    const float *xs = FUSED ? ys : x_or_gy + base;  // the fused forward left the raw score in y
    strided_pass<8>(threadIdx.x, static_cast<uint64_t>(pc.w - pc.z) * H, 256, [&](uint64_t j) -> float { return xs[j]; },
                    [&](uint64_t j, float sc) { ys[j] = softmax_exp(sc - mx) * inv; });
  }
}

// ---- gradient of the attention-weighted aggregation with respect to alpha ----------------------
//
// galpha[e,h] = < in[ri[e], h-th slice], gout[d, h-th slice] > for e in CSC(d).  Edge-parallel like
// the copies: 64 consecutive edges per wave step, (source, owner) looked up per lane.

// Fast path: G = (H*Fh)/VEC lanes cover one edge's row (G a power of two <= 64), the Fh/VEC lanes of
// a head add their products with an xor butterfly.  A wave step takes 64 consecutive edges and each
// of the 64/G lane groups G consecutive ones of them, so a group's destination changes rarely and
// its gout row stays in registers until it does: one gathered row per edge instead of two.
template <int VEC>
__global__ __launch_bounds__(256) void sddmm_edge_kernel(float *__restrict__ galpha, const float *__restrict__ in,
                                                         const float *__restrict__ gout,
                                                         const uint32_t *__restrict__ co,
                                                         const uint32_t *__restrict__ ri, uint32_t Vd, uint32_t H,
                                                         uint32_t Fh, uint32_t G, uint32_t lanes_per_head) {
  const uint32_t E = co[Vd];
  const uint32_t F = H * Fh;
  const uint32_t lane = lane_id();
  const uint32_t gl = lane & (G - 1), grp = lane / G;
  const uint64_t wave = wave_of_grid();
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  uint32_t d_held = 0xFFFFFFFFu;
  float4 y4 = make_float4(0.f, 0.f, 0.f, 0.f);
  float y1 = 0.f;
  // A wavefront walks a contiguous span of wave steps, so that the owner of each step's edges is
  // found from the previous step's instead of by a search per lane.
  const uint64_t total_steps = (static_cast<uint64_t>(E) + kWave - 1) / kWave;
  const uint64_t per_wave = (total_steps + n_waves - 1) / n_waves;
  const uint64_t first_step = wave * per_wave;
  const uint64_t end_step = first_step + per_wave < total_steps ? first_step + per_wave : total_steps;
  if (first_step >= end_step) return;
  uint32_t d0 = owner_of_wave(co, Vd, static_cast<uint32_t>(first_step * kWave));
  for (uint64_t step = first_step; step < end_step; ++step) {
    const uint64_t base = step * kWave;
    const uint64_t e = base + lane;
    const uint32_t own = owners_of_step(co, Vd, static_cast<uint32_t>(base), d0);
    const uint32_t src = e < E ? ri[e] : 0u;
    // Eight edges at a time: their gathered rows -- and the destination rows of the edges at which the
    // destination changes -- are requested before the first is used (four measure the same on a whole
    // graph; on a sampled layer of 410 k edges, where the launch is a few dependent rounds long, eight
    // take the mini-batch epoch's backward stage from 8.2 to 8.0 ms).
    constexpr uint32_t U = 8;
    for (uint32_t j0 = 0; j0 < G; j0 += U) {
      uint32_t d[U];
      bool valid[U], fresh[U];
      float4 x4[U], w4[U];
      float x1[U], w1[U];
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        const uint32_t holder = grp * G + j0 + u;
        const uint32_t s = __shfl(src, holder & (kWave - 1), kWave);
        d[u] = __shfl(own, holder & (kWave - 1), kWave);
        valid[u] = j0 + u < G && base + holder < E;
        fresh[u] = valid[u] && d[u] != (u ? d[u - 1] : d_held);  // an edge is valid only if the one before it is
        x4[u] = w4[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        x1[u] = w1[u] = 0.f;
        if (valid[u]) {
          const float *a = in + static_cast<size_t>(s) * F + gl * VEC;
          if (VEC == 4) x4[u] = *reinterpret_cast<const float4 *>(a); else x1[u] = a[0];
        }
        if (fresh[u]) {
          const float *b = gout + static_cast<size_t>(d[u]) * F + gl * VEC;
          if (VEC == 4) w4[u] = *reinterpret_cast<const float4 *>(b); else w1[u] = b[0];
        }
      }
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        float p = 0.f;
        if (valid[u]) {
          if (fresh[u]) {
            if (VEC == 4) y4 = w4[u]; else y1 = w1[u];
            d_held = d[u];
          }
          p = VEC == 4 ? fmaf(x4[u].w, y4.w, fmaf(x4[u].z, y4.z, fmaf(x4[u].y, y4.y, x4[u].x * y4.x))) : x1[u] * y1;
        }
        for (uint32_t m = lanes_per_head / 2; m >= 1; m >>= 1) p += __shfl_xor(p, m, kWave);
        if (valid[u] && (gl & (lanes_per_head - 1)) == 0)
          galpha[(base + grp * G + j0 + u) * H + gl / lanes_per_head] = p;
      }
    }
  }
}

// General shapes: the 64 edges of a step are taken one after the other; for each edge and head the
// lanes stride over the head's slice and a full-wave butterfly adds the partial products.
__global__ __launch_bounds__(256) void sddmm_edge_generic_kernel(float *__restrict__ galpha,
                                                                 const float *__restrict__ in,
                                                                 const float *__restrict__ gout,
                                                                 const uint32_t *__restrict__ co,
                                                                 const uint32_t *__restrict__ ri, uint32_t Vd,
                                                                 uint32_t H, uint32_t Fh) {
  const uint32_t E = co[Vd];
  const uint32_t F = H * Fh;
  const uint32_t lane = lane_id();
  const uint64_t wave = wave_of_grid();
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  for (uint64_t base = wave * kWave; base < E; base += n_waves * kWave) {
    const uint64_t e = base + lane;
    uint32_t src = 0, own = 0;
    if (e < E) {
      src = ri[e];
      own = owner_of(co, Vd, static_cast<uint32_t>(e));
    }
    const uint32_t n = static_cast<uint32_t>(min(static_cast<uint64_t>(kWave), E - base));
    for (uint32_t j = 0; j < n; ++j) {
      const float *a = in + static_cast<size_t>(wave_read(src, j)) * F;
      const float *b = gout + static_cast<size_t>(wave_read(own, j)) * F;
      for (uint32_t h = 0; h < H; ++h) {
        float p = 0.f;
        for (uint32_t f = lane; f < Fh; f += kWave) p = fmaf(a[h * Fh + f], b[h * Fh + f], p);
        p = group_sum<kWave>(p);
        if (lane == 0) galpha[(base + j) * H + h] = p;
      }
    }
  }
}

inline bool is_pow2(uint32_t v) { return v && !(v & (v - 1)); }

}  // namespace
}  // namespace nts

using namespace nts;

namespace {
// Grid for the edge-parallel kernels: the edge count lives on the device, so the grid is sized from
// the vertex count (assuming a few dozen edges per vertex) and the kernels stride over the edges.
inline dim3 edge_grid(uint32_t Vd) {
  uint64_t blocks = (static_cast<uint64_t>(Vd) * 32 + 255) / 256;
  if (blocks < 64) blocks = 64;
  if (blocks > 8192) blocks = 8192;
  return dim3(static_cast<unsigned>(blocks));
}

// Lanes per row for a row of Fv vector elements: the smallest power of two >= Fv, at most 64.
inline int lanes_for(uint32_t Fv) {
  int g = 1;
  while (g < 64 && static_cast<uint32_t>(g) < Fv) g <<= 1;
  return g;
}

template <typename V>
void launch_edge_copy(V *msg, const V *feat, const uint32_t *ri, const uint32_t *co, const uint32_t *mirror,
                      uint32_t Vd, uint32_t Fv, int mode, hipStream_t stream) {
  const dim3 grid = edge_grid(Vd), block(256);
#define NTS_COPY(GG)                                                                                              \
  hipLaunchKernelGGL((edge_copy_kernel<V, GG>), grid, block, 0, stream, msg, feat, ri, co, mirror, Vd, Fv, mode)
  switch (lanes_for(Fv)) {
    case 1: NTS_COPY(1); break;
    case 2: NTS_COPY(2); break;
    case 4: NTS_COPY(4); break;
    case 8: NTS_COPY(8); break;
    case 16: NTS_COPY(16); break;
    case 32: NTS_COPY(32); break;
    default: NTS_COPY(64); break;
  }
#undef NTS_COPY
}

int edge_copy_impl(float *msg, const float *feat, const uint32_t *ri, const uint32_t *co, const uint32_t *mirror,
                   uint32_t Vd, uint32_t F, int mode, hipStream_t stream, const char *who) {
  if (F == 0) return fail(NTS_ERR_INVALID, who);
  if (Vd == 0) return NTS_OK;
  if (!msg || !feat || !co || (mode == kFromSrc && !ri)) return fail(NTS_ERR_INVALID, who);
  if (F % 4 == 0 && aligned_to(msg, 16) && aligned_to(feat, 16))
    launch_edge_copy(reinterpret_cast<float4 *>(msg), reinterpret_cast<const float4 *>(feat), ri, co, mirror, Vd,
                     F / 4, mode, stream);
  else
    launch_edge_copy(msg, feat, ri, co, mirror, Vd, F, mode, stream);
  NTS_LAUNCH_CHECK(who);
  return NTS_OK;
}

// Scratch of the long-row path in one stream-ordered allocation: list[rows], its counter, and the
// tables of the giant rows (header, row list, first-piece prefix, piece table).
struct LongRows {
  ScratchBlock block;  // owns the allocation: returned to the pool on every way out of the caller
  uint32_t *list = nullptr;
  uint32_t *count = nullptr;
  uint32_t *hdr = nullptr;
  uint32_t *giant_rows = nullptr;
  uint32_t *first = nullptr;
  uint4 *pieces = nullptr;
};

// Collects the rows whose segment holds more than `limit` values (edges * width) when the vertex
// count makes hubs likely, the ones above `giant_limit` values separately (with their piece table);
// returns with lr.list == nullptr when the long path is not used.
int take_long_rows(LongRows &lr, uint32_t rows, hipStream_t stream) {
  if (rows < kLongMinVertices) return NTS_OK;
  const size_t list_bytes = (static_cast<size_t>(rows) + 7) / 8 * 8 * sizeof(uint32_t);  // list, 32-byte multiple
  const size_t small_bytes = (8 + kGiantCap + kGiantCap + 8) * sizeof(uint32_t);  // hdr (with the counter), rows, first
  NTS_HIP_TRY(lr.block.alloc(list_bytes + small_bytes + kPieceCap * sizeof(uint4), stream));
  unsigned char *buf = static_cast<unsigned char *>(lr.block.ptr);
  lr.list = reinterpret_cast<uint32_t *>(buf);
  lr.hdr = reinterpret_cast<uint32_t *>(buf + list_bytes);
  lr.count = lr.hdr + 6;
  lr.giant_rows = lr.hdr + 8;
  lr.first = lr.giant_rows + kGiantCap;
  lr.pieces = reinterpret_cast<uint4 *>(buf + list_bytes + small_bytes);
  return NTS_OK;
}
int collect_long_rows(const LongRows &lr, const uint32_t *off, uint32_t rows, uint32_t width, uint32_t limit,
                      uint64_t giant_limit, uint32_t min_piece, hipStream_t stream) {
  if (!lr.list) return NTS_OK;
  if (rows <= kOneBlockRows) {
    hipLaunchKernelGGL(few_long_rows_kernel, dim3(1), dim3(kLongBlock), 0, stream, lr.list, lr.count, lr.giant_rows, lr.hdr, lr.first,
                       lr.pieces, off, rows, width, limit, giant_limit, min_piece);
    NTS_LAUNCH_CHECK("few_long_rows_kernel");
    return NTS_OK;
  }
  if (int rc = nts_memset_zero(lr.hdr, 8 * sizeof(uint32_t), stream)) return rc;  // counters
  hipLaunchKernelGGL(collect_long_rows_kernel, dim3(ceil_div(rows, 256)), dim3(256), 0, stream, lr.list, lr.count,
                     lr.giant_rows, lr.hdr, off, rows, width, limit, giant_limit);
  NTS_LAUNCH_CHECK("collect_long_rows_kernel");
  hipLaunchKernelGGL(giant_plan_kernel, dim3(1), dim3(256), 0, stream, lr.hdr, lr.giant_rows, lr.first, lr.pieces, off,
                     min_piece);
  NTS_LAUNCH_CHECK("giant_plan_kernel");
  return NTS_OK;
}

int release_long_rows(LongRows &lr) {
  lr.list = nullptr;
  NTS_HIP_TRY(lr.block.release());
  return NTS_OK;
}

constexpr unsigned kLongGrid = 512;  // blocks of the long-row kernels; they stride over the list

// Edges of a row above which the whole wavefront takes it (rows up to eight lanes wide); NTS_EDGE_SUM_COOP
// in the environment overrides it (0 = never).
uint32_t coop_limit() {
  static const uint32_t value = [] {
    const char *env = getenv("NTS_EDGE_SUM_COOP");
    if (!env) return 64u;
    const long v = atol(env);
    return v <= 0 ? kNoLimit : static_cast<uint32_t>(v);
  }();
  return value;
}

// Blocks of a row launch set aside for the listed long rows and the pieces of the giant ones.
constexpr uint32_t kMergedLongBlocks = 2048;

// The same for calls of fewer than kLongMinVertices rows, which find them themselves; not where rows are so few that each has a
// block's worth of wavefronts beside it anyway.
constexpr uint32_t kOwnHubBlocks = 512;

// Whether a group of lanes takes a row of its own and of 64 vectors at most (gather_edge_to_row_kernel), and not wavefronts sets of
// rows.  us, sets / a row each, contiguous and permuted sums of edge rows:
//                   contiguous: F = 47, 128, 200      permuted: F = 47, 64, 100, 128, 200
//   2.9 K, 110 K      56 / 56, 78 / 59, 110 / 69        472 / 62, 150 / 62, 305 / 63, 296 / 63, 564 / 77
//   6 K, 12 K         17 / 9, 16 / 11, 28 / 10          36 / 10, 36 / 10, 38 / 12, 38 / 12, 41 / 11
//   16 K, 100 K       54 / 29, 52 / 45, 100 / 46        216 / 34, 178 / 32, 211 / 51, 207 / 51, 250 / 49
//   16 K, 1 M         303 / 317, 427 / 386, 515 / 576   372 / 346, 462 / 318, 523 / 358, 500 / 426, 584 / 622
//   10 K, 3 M         881 / 909, 1,667 / 1,349, 2,191 / 2,201   1,098 / 995, 1,776 / 1,156, 1,936 / 1,345, 1,920 / 1,508, 2,410 / 2,429
//                   contiguous: F = 47, 128    permuted: F = 47, 64, 100, 128, 200
//   30 K, 3 M         213 / 175, 361 / 348       534 / 221, 298 / 240, 447 / 335, 463 / 366
//   169 K, 2.48 M     186 / 188, 310 / 319       381 / 229, 258 / 226, 374 / 309, 388 / 343, 639 / 523
//   400 K, 2 M        187 / 223, 301 / 298       337 / 263, 294 / 214, 391 / 285, 409 / 312
//   1 M, 8 M          508 / 639, 1,021 / 1,004   943 / 786, 689 / 645, 1,109 / 961, 1,133 / 1,061
//   1.5 M, 6 M                                   763 / 791, 545 / 568, 888 / 809, 889 / 876
//   2.4 M, 5 M                                   807 / 978, 508 / 629, 840 / 946, 861 / 976, 1,437 / 1,519
// so a row each for the permuted sums up to a million rows, for the contiguous ones below 16,384 (there hub rows are one running sum on
// either side, and dense graphs lose up to a tenth at some widths to what sparse ones gain several times).  Rows of up to eight vectors leave
// a lane or two a whole row there: 2.9 K, 110 K F = 4 34 / 46 with a row each, sets 15 / 18; but eight permuted vectors 30 K, 3 M 224
// sets, 164, 169 K 191, 170 (400 K 161, 171; 16 K, 100 K 38, 49).
constexpr uint32_t kMinHubRows = 64;  // (fewer rows have a block's worth of wavefronts beside each anyway: no hub blocks)
bool group_takes_a_row(uint32_t rows, uint32_t Fv, bool vectors, bool permuted) {
  if (rows < kMinHubRows || Fv > kWave) return true;
  if (Fv <= 8) return permuted && vectors && Fv > 4 && rows >= kLongMinVertices && rows <= 1u << 18;
  return rows < (permuted ? 1u << 20 : kLongMinVertices);
}
// Rows that are few leave the chip idle, and floats spread them over four times as many lanes, each with 32 loads in flight where
// vectors have room for eight.  us, vectors / floats, contiguous and permuted: F = 64 4 K, 200 K 148 / 102, 159 / 110, 16 K, 1 M 443 / 290, 484 /
// 318; F = 128 153 / 103, 164 / 111 and 518 / 384, 558 / 426, 6 K, 12 K 9.6 / 10.9, 10.7 / 12.2.  From three wavefronts of floats a row on only
// where these do not fill the chip twice: F = 200 40 rows, 3 K 26 / 18, 2 K, 8 K 12 / 10, but 16 K, 100 K 46 / 67, 16 K, 1 M 576 / 759.
bool floats_for_few_rows(uint32_t rows, uint32_t F) {
  return F > 32 && rows < kLongMinVertices && (F <= 128 || static_cast<uint64_t>(rows) * ceil_div(F, kWave) <= 16384);
}

// NTS_EDGE_SUM_STREAM=0 in the environment: contiguous edge rows take the lane-group kernel like permuted ones.
bool stream_contiguous_rows() {
  static const bool value = [] {
    const char *env = getenv("NTS_EDGE_SUM_STREAM");
    return !(env && atol(env) == 0);
  }();
  return value;
}

// A wavefront streams the contiguous edges of up to 64 rows at a time, and of fewer where that would leave it without
// the 8,192 wavefronts that the chip holds: whatever the width, 64 rows cost a small vertex set its parallelism and 16
// cost a large one a wavefront's start-up per four rows' worth of work.  us, 64 / 16 rows a wavefront: 50 K rows, 5 M
// edges F = 4 191 / 95, F = 128 833 / 599; 169 K, 2.48 M F = 4 88 / 80, F = 32 117 / 108, F = 128 348 / 307; 1 M, 2.5 M F = 4
// 135 / 168, F = 32 166 / 211, F = 64 224 / 259, F = 128 436 / 439; 2.4 M, 60 M within 3 %.  16 / 8: 30 K, 3 M F = 4 68 / 59, F = 47 264 /
// 214, 16 K, 1 M F = 4 34 / 24, F = 128 149 / 131; 50 K, 500 K F = 4 45 / 45, F = 128 110 / 112, with four 117.
uint32_t streamed_rows_per_wave(uint32_t rows) {
  constexpr uint32_t kChipWaves = 8192;
  uint32_t per = kWave;
  while (per > 8 && rows / per < kChipWaves) per /= 2;
  return per;
}

// Rows that a wavefront of the permuted sums hands out at a time: eight per lane group, so that a wavefront with two
// groups (128-byte-wide vectors) is not left with 32 rows per group while others have finished, and fewer, down to eight,
// where that leaves the chip without its 8,192 wavefronts.  us, always eight per group / so: 16.5 K rows, 300 K edges F = 4
// 69 / 46, F = 16 133 / 54, F = 128 214 / 206; 100 K, 8 M F = 1 209 / 172, F = 32 682 / 411; 169 K, 2.48 M F = 1 78 / 67, F = 32
// 193 / 145 (not below 16 rows: 16.5 K F = 16 68, 100 K F = 32 441); from 524,288 rows up the same.
uint32_t balanced_rows_per_wave(uint32_t rows, uint32_t set) {
  constexpr uint32_t kChipWaves = 8192;
  while (set > 8 && rows / set < kChipWaves) set /= 2;
  return set;
}

template <typename V>
void launch_gather_rows(V *out, const V *msg, const uint32_t *off, const uint32_t *perm, uint32_t rows, uint32_t Fv,
                        int accumulate, uint32_t limit, const LongRowWork<V> &lw, hipStream_t stream) {
  const bool row_each = group_takes_a_row(rows, Fv, sizeof(V) == 16, perm != nullptr);
  if (!row_each && !perm && stream_contiguous_rows()) {
    const uint32_t blocks = ceil_div(rows, 4 * streamed_rows_per_wave(rows));
    const dim3 grid((blocks < 16384u ? blocks : 16384u) + lw.blocks);
#define NTS_STREAM(GG)                                                                                          \
  hipLaunchKernelGGL((gather_edge_to_row_stream_kernel<V, GG>), grid, dim3(256), 0, stream, out, msg, off, rows, Fv, \
                     accumulate, limit, lw)
    switch (lanes_for(Fv)) {
      case 1: NTS_STREAM(1); break;
      case 2: NTS_STREAM(2); break;
      case 4: NTS_STREAM(4); break;
      case 8: NTS_STREAM(8); break;
      case 16: NTS_STREAM(16); break;
      case 32: NTS_STREAM(32); break;
      default: NTS_STREAM(64); break;
    }
#undef NTS_STREAM
    return;
  }
  if (!row_each) {
    // One group covers a row: wavefronts hand their 64 rows out dynamically (strided launch).
#define NTS_BALANCED(GG, SS)                                                                                    \
  do {                                                                                                          \
    const uint32_t set = balanced_rows_per_wave(rows, kFullSet<(GG) * (SS)>);                                  \
    const uint32_t blocks = ceil_div(rows, 4 * set); /* at most `set` rows per wavefront at a time */          \
    const dim3 grid((blocks < 16384u ? blocks : 16384u) + lw.blocks);                                          \
    if (set < kFullSet<(GG) * (SS)>)                                                                            \
      hipLaunchKernelGGL((gather_edge_to_row_balanced_kernel<V, GG, SS, (kFullSet<(GG) * (SS)> > 8)>), grid, dim3(256), 0, stream, out, msg, \
                         off, perm, rows, Fv, accumulate, limit, coop_limit(), set, lw);                        \
    else                                                                                                        \
      hipLaunchKernelGGL((gather_edge_to_row_balanced_kernel<V, GG, SS, false>), grid, dim3(256), 0, stream, out, msg, \
                         off, perm, rows, Fv, accumulate, limit, coop_limit(), set, lw);                        \
  } while (0)
    switch (lanes_for(Fv)) {  // rows narrower than eight lanes are shared by eight lanes all the same
      case 1: NTS_BALANCED(1, 8); break;
      case 2: NTS_BALANCED(2, 4); break;
      case 4: NTS_BALANCED(4, 2); break;
      case 8: NTS_BALANCED(8, 1); break;
      case 16: NTS_BALANCED(16, 1); break;
      case 32: NTS_BALANCED(32, 1); break;
      default: NTS_BALANCED(64, 1); break;
    }
#undef NTS_BALANCED
    return;
  }
  // One launch up to 2^32 threads; the hub rows are the first one's.
#define NTS_GATHER(GG)                                                                                            \
  do {                                                                                                            \
    const uint32_t tiles = ceil_div(Fv, GG);                                                                      \
    const uint64_t groups = static_cast<uint64_t>(rows) * tiles;                                                  \
    LongRowWork<V> hubs = lw;                                                                                     \
    for (uint64_t first = 0; first < groups;) {                                                                   \
      const uint32_t blocks = blocks_of_groups(groups - first, GG, hubs.blocks);                                  \
      if (sizeof(V) == 4 && rows < kLongMinVertices)                                                              \
        hipLaunchKernelGGL((gather_edge_to_row_kernel<V, GG, sizeof(V) == 16 ? 8 : 32>), dim3(blocks), dim3(256), 0, \
                           stream, out, msg, off, perm, rows, Fv, accumulate, limit, tiles, first, hubs);         \
      else                                                                                                        \
        hipLaunchKernelGGL((gather_edge_to_row_kernel<V, GG, 8>), dim3(blocks), dim3(256), 0, stream, out, msg, off, \
                           perm, rows, Fv, accumulate, limit, tiles, first, hubs);                                \
      first += static_cast<uint64_t>(blocks - hubs.blocks) * (256 / GG);                                          \
      hubs.blocks = 0;                                                                                            \
    }                                                                                                             \
  } while (0)
  switch (lanes_for(Fv)) {
    case 1: NTS_GATHER(1); break;
    case 2: NTS_GATHER(2); break;
    case 4: NTS_GATHER(4); break;
    case 8: NTS_GATHER(8); break;
    case 16: NTS_GATHER(16); break;
    case 32: NTS_GATHER(32); break;
    default: NTS_GATHER(64); break;
  }
#undef NTS_GATHER
}

int gather_edge_impl(float *out, const float *msg, const uint32_t *off, const uint32_t *perm, uint32_t rows,
                     uint32_t F, int accumulate, hipStream_t stream, const char *who) {
  if (F == 0) return fail(NTS_ERR_INVALID, who);
  if (rows == 0) return NTS_OK;
  if (!out || !msg || !off) return fail(NTS_ERR_INVALID, who);
  LongRows lr;
  // A block reads a row at 20 to 40 GB/s, whatever the rest of the chip does, so the bound is one on bytes: up
  // to 64 bytes an edge row it is 16,384 edges in pieces of 4,096; at 512 bytes 2,048 in pieces of 512
  // (one block and up to 8 MB before: the sums over 1.27 GB of edge rows 463 -> 422 us, through a
  // permutation 669 -> 605).
  uint64_t giant_edges = kGiantRowBytes / (4ull * F);
  giant_edges = giant_edges > 16384 ? 16384 : giant_edges < kLongRowEdges ? kLongRowEdges : giant_edges;
  if (int rc = take_long_rows(lr, rows, stream)) return rc;
  if (int rc = collect_long_rows(lr, off, rows, 1u, kLongRowEdges, giant_edges, static_cast<uint32_t>(giant_edges / 4),
                                 stream))
    return rc;
  const uint32_t limit = lr.list ? kLongRowEdges : kNoLimit;
  // 16-byte vectors for the row kernels and the block kernels alike
  bool v4 = F % 4 == 0 && aligned_to(out, 16) && aligned_to(msg, 16);
  if (v4 && floats_for_few_rows(rows, F)) v4 = false;
  const uint32_t Fv = v4 ? F / 4 : F;
  // Long rows, and giant rows in pieces: in the first blocks of the row launch; the pieces' sums go to stream-ordered scratch and a
  // launch of its own combines them in order.  Few rows: the first blocks find the hub rows themselves and take columns of 128 bytes of one each,
  // of 64 where that leaves a row's blocks a tile each.
  const uint32_t hub_lanes = v4 ? 8u : F > 32 && F <= 128 ? 16u : 32u;
  const bool own = !lr.list && rows >= kMinHubRows && (Fv > 8 || (perm && Fv > 4 && v4) || rows < kMaxNarrowHubRows);
  const uint32_t hub_blocks = lr.list ? kMergedLongBlocks : !own ? 0u : Fv <= hub_lanes ? kOwnHubBlocks / 2 : kOwnHubBlocks;
  const uint32_t most_lanes = own ? hub_lanes : 256u;
  uint32_t tile = 1;
  while (tile < Fv && tile < most_lanes) tile <<= 1;
  // Listed rows of more than 64 vectors are added by as many slices as 1,024 threads have beside the whole row: eight or four, four of
  // them a thread; two, of a thread each, beside 128 vectors of a row of up to 512; one above.  With tiles of 256 and a slice a thread a chain of
  // additions was two to four times as many edges, and rows of 65 to 127 floats were 2.7 times as far from their sums in 64 bits (1.8e-7
  // instead of 6.7e-8, values in [0, 1), 16.5 K rows, 1 M edges).  us, so / as it is, 30 K rows, 3 M edges F = 65 229 / 218, 127 362 / 342, 257 747 /
  // 695 (two slices a thread 818), 512 1,217 / 1,220, 169 K, 2.48 M F = 602 1,608 / 1,573; the first of these as four tiles with a slice a thread 277.
  const uint32_t chains = !own && Fv > kWave && Fv <= 256 ? 4 : 1;
  if (!own && Fv > 256 && Fv <= 512) tile = 128;
  ScratchBlock partial_block;
  float *partial = nullptr;
  if (lr.list) {
    NTS_HIP_TRY(partial_block.alloc(static_cast<size_t>(kPieceCap) * F * sizeof(float), stream));
    partial = static_cast<float *>(partial_block.ptr);
  }
  if (v4) {
    LongRowWork<float4> lw{lr.list, lr.count, lr.hdr, lr.pieces, reinterpret_cast<float4 *>(partial), tile,
                           hub_blocks, own, chains};
    launch_gather_rows(reinterpret_cast<float4 *>(out), reinterpret_cast<const float4 *>(msg), off, perm, rows, Fv,
                       accumulate, limit, lw, stream);
  } else {
    LongRowWork<float> lw{lr.list, lr.count, lr.hdr, lr.pieces, partial, tile, hub_blocks, own, chains};
    launch_gather_rows(out, msg, off, perm, rows, Fv, accumulate, limit, lw, stream);
  }
  hipError_t launch_err = hipGetLastError();
  if (lr.list && launch_err == hipSuccess) {
    hipLaunchKernelGGL(giant_sum_combine_kernel, dim3(kGiantCap / 4), dim3(256), 0, stream, out, partial, lr.hdr,
                       lr.giant_rows, lr.first, F, accumulate);
    launch_err = hipGetLastError();
  }
  if (lr.list) NTS_HIP_TRY(partial_block.release());
  if (launch_err != hipSuccess) {
    (void)release_long_rows(lr);
    return fail_hip(launch_err, who);
  }
  return release_long_rows(lr);
}

// A second stream per host thread and device, for launches that a call runs beside those on the
// caller's stream (the block kernels of the few hub rows, which leave most of the chip idle, beside the
// kernels of all other rows).  Created at first use and kept until the process ends; a thread that
// ends leaves its stream and events behind (destroying them from a thread-exit hook could run after the
// runtime has shut down).  NTS_SOFTMAX_SIDE_STREAM=0 in the environment: everything on the caller's stream.
struct SideLane {
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
SideLane *side_lane() {
  static const bool enabled = [] {
    const char *env = getenv("NTS_SOFTMAX_SIDE_STREAM");
    return !(env && atol(env) == 0);
  }();
  if (!enabled) return nullptr;
  constexpr int kDevices = 16;
  thread_local SideLane lanes[kDevices];
  thread_local bool tried[kDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return nullptr;
  SideLane &l = lanes[dev];
  if (!tried[dev]) {
    tried[dev] = true;
    hipStream_t st = nullptr;
    hipEvent_t a = nullptr, b = nullptr;
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) == hipSuccess &&
        hipEventCreateWithFlags(&a, hipEventDisableTiming) == hipSuccess &&
        hipEventCreateWithFlags(&b, hipEventDisableTiming) == hipSuccess) {
      l.stream = st;
      l.fork = a;
      l.join = b;
    } else {
      if (a) (void)hipEventDestroy(a);
      if (st) (void)hipStreamDestroy(st);
      (void)hipGetLastError();
    }
  }
  return l.stream ? &l : nullptr;
}

// The side lane between a fork (it waits for everything enqueued on `main` so far) and the join (`main`
// waits for it), which also happens on every way out of the scope.
class SideWork {
 public:
  SideWork(hipStream_t main, bool wanted) : main_(main), lane_(wanted ? side_lane() : nullptr) {
    // a stream that is recording a graph keeps all of the call's launches: the side stream is shared by
    // the thread's calls and must not become part of a recording
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (lane_ && (hipStreamIsCapturing(main_, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone)) {
      (void)hipGetLastError();
      lane_ = nullptr;
    }
    if (lane_ && (hipEventRecord(lane_->fork, main_) != hipSuccess ||
                  hipStreamWaitEvent(lane_->stream, lane_->fork, 0) != hipSuccess)) {
      (void)hipGetLastError();
      lane_ = nullptr;  // nothing has been enqueued on the side stream: the caller's stream takes the work
    }
  }
  SideWork(const SideWork &) = delete;
  SideWork &operator=(const SideWork &) = delete;
  hipStream_t stream() const { return lane_ ? lane_->stream : main_; }
  hipError_t join() {
    if (!lane_) return hipSuccess;
    SideLane *l = lane_;
    lane_ = nullptr;
    const hipError_t e = hipEventRecord(l->join, l->stream);
    return e != hipSuccess ? e : hipStreamWaitEvent(main_, l->join, 0);
  }
  ~SideWork() { (void)join(); }

 private:
  hipStream_t main_;
  SideLane *lane_;
};

// Destinations that a wavefront of the softmax wave kernels looks at together: it visits those of its class one after the other, so
// as few as leave the chip its 8,192 wavefronts.  us, 64 / so, fused backward, H = 1 and 4: 60 K rows, 4 M edges 134 / 99, 232 / 123; 169 K,
// 2.48 M 90 / 84, 145 / 121; from 524,288 rows up 64 (600 K, 3 M forward 115, 16 129).
uint32_t softmax_rows_per_wave(uint32_t Vd) {
  constexpr uint32_t kChipWaves = 8192;
  uint32_t per = kWave;
  while (per > 8 && Vd / per < kChipWaves) per /= 2;
  return per;
}

constexpr uint32_t kFewHubBlocks = 128;  // that look for their hub rows themselves
static_assert(kLongMinVertices <= 256 * kFewHubBlocks, "a row a thread");
// Destinations that a wavefront takes together in a call of few rows (kDenseSet where these are long): 64 / 16 / 4 fused forward
// 169 K rows, 2.48 M edges H = 1 74 / 66 / 76, 30 K, 1 M 64 / 39 / 35, 200 K, 20 M 235 / 192 / 179.
uint32_t few_rows_per_wave(uint32_t Vd) {
  constexpr uint32_t kChipWaves = 8192;
  uint32_t per = kWave;
  while (per > 4 && Vd / per < kChipWaves) per /= 2;
  return per;
}

template <bool FUSED, bool BWD, bool VEC4>
int few_softmax(float *out, float *ger, const float *x_or_gy, const float *y, const float *el, const float *er, const uint32_t *co,
                const uint32_t *ri, uint32_t Vd, uint32_t H, float slope, bool look_for_hubs, hipStream_t stream, const char *who) {
  LongRows lr;
  ScratchBlock stats_block;
  FewHubs hubs{};
  if (look_for_hubs) {
    if (int rc = take_long_rows(lr, Vd, stream)) return rc;
    hubs.blocks = lr.list ? kLongGrid : kFewHubBlocks;
  }
  if (lr.list) {
    NTS_HIP_TRY(stats_block.alloc(static_cast<size_t>(kPieceCap) * 2 * H * sizeof(float), stream));
    hubs = FewHubs{lr.list, lr.count, lr.hdr, lr.first, lr.pieces, static_cast<float *>(stats_block.ptr), kLongGrid};
    if (int rc = collect_long_rows(lr, co, Vd, H, kByFewTotal, 0, kFewPieceValues / H, stream)) return rc;
  }
  const uint32_t set = few_rows_per_wave(Vd);
  hipLaunchKernelGGL((few_softmax_kernel<FUSED, BWD, VEC4>), dim3(hubs.blocks + ceil_div(Vd, 4 * (set < kDenseSet ? set : kDenseSet))), dim3(256), 0, stream, out,
                     ger, x_or_gy, y, el, er, co, ri, Vd, H, slope, set, hubs);
  NTS_LAUNCH_CHECK(who);
  if (!lr.list) return NTS_OK;
  hipLaunchKernelGGL((few_giant_apply_kernel<FUSED, BWD, VEC4>), dim3(kLongGrid), dim3(256), 0, stream, out, x_or_gy, y, el, er, ri, H, slope, hubs);
  if (FUSED && BWD)
    hipLaunchKernelGGL(giant_softmax_combine_kernel<1>, dim3(kGiantCap / 4), dim3(64), 0, stream, static_cast<float *>(nullptr), ger,
                       hubs.stats + H, lr.hdr, lr.giant_rows, lr.first, H, 2 * H);
  NTS_LAUNCH_CHECK(who);
  NTS_HIP_TRY(stats_block.release());
  return release_long_rows(lr);
}

// Edge softmax / fused attention, forward (gy == nullptr) or backward; x / el / er / ri / ger are
// null where the variant does not use them.
int softmax_impl(bool backward, bool fused, float *out, float *ger, const float *x_or_gy, const float *y,
                 const float *el, const float *er, const uint32_t *co, const uint32_t *ri, uint32_t Vd, uint32_t H,
                 float slope, hipStream_t stream, const char *who, uint32_t max_degree = 0) {
  const bool pow2 = is_pow2(H) && H <= kWave;
  LongRows lr;
  // A caller that bounds every segment below the block kernels' class where it begins highest (a sampled layer: at most
  // `fanout` edges per destination) needs none of the launches that look for hub rows: every segment is a wavefront's,
  // also one that a call without a bound would hand to a block because its values are few in all.  A longer segment than
  // stated is still computed, by one wavefront.
  const bool no_hubs = max_degree != 0 && static_cast<uint64_t>(max_degree) * H <= kLongRowValues;
  const bool one_short_launch = fused && max_degree != 0 && static_cast<uint64_t>(max_degree) * H <= kShortValues;
  if (pow2 && H <= static_cast<uint32_t>(kShortG) && Vd <= (fused && backward && H > 4 ? kFewRowsManyHeads : kFewRows) && !one_short_launch) {
    const bool vec4 = fused && H % 4 == 0 && aligned_to(out, 16) && aligned_to(x_or_gy, 16) && aligned_to(y, 16) && aligned_to(el, 16) &&
                      aligned_to(er, 16) && aligned_to(ger, 16);
    auto call = [&](auto f) { return f(out, ger, x_or_gy, y, el, er, co, ri, Vd, H, slope, !no_hubs, stream, who); };
    if (!fused) return backward ? call(few_softmax<false, true, false>) : call(few_softmax<false, false, false>);
    if (vec4) return backward ? call(few_softmax<true, true, true>) : call(few_softmax<true, false, true>);
    return backward ? call(few_softmax<true, true, false>) : call(few_softmax<true, false, false>);
  }
  if (pow2 && !no_hubs)
    if (int rc = take_long_rows(lr, Vd, stream)) return rc;
  const uint32_t max_values = lr.list ? kByTotal : kNoLimit;
  // The block kernels of the hub rows and the kernels of the giant ones' pieces run on the side lane,
  // beside the launches for all other rows below (they write other rows); their scratch is taken
  // before the fork, so that whatever the pool ordered for it on `stream` lies before it too.
  const size_t stats_floats = static_cast<size_t>(kPieceCap) * 2 * H, row_floats = static_cast<size_t>(kGiantCap) * 2 * H;
  ScratchBlock stats_block;
  if (lr.list) NTS_HIP_TRY(stats_block.alloc((stats_floats + row_floats) * sizeof(float), stream));
  SideWork side(stream, lr.list != nullptr);
  const hipStream_t hub_stream = side.stream();
  // (listing them too: the launches of the other rows do not need it; 169 K rows, 2.48 M edges, one head 86 -> 76 us)
  if (int rc = collect_long_rows(lr, co, Vd, H, kByTotal, 0, kGiantMinPiece, hub_stream)) return rc;
  // 16-byte lanes for the segments that do not fit the register paths: whole heads per lane and
  // every array 16-byte aligned (a segment starts at e0 * H floats).
  const uint32_t vec4 = pow2 && H % 4 == 0 && aligned_to(out, 16) && aligned_to(x_or_gy, 16) && aligned_to(y, 16) &&
                        aligned_to(el, 16) && aligned_to(er, 16) && aligned_to(ger, 16);
  const bool use_short = pow2 && H <= static_cast<uint32_t>(kShortG);
  const uint32_t min_values = use_short ? kShortValues + 1 : 0u;
  // Both strided kernels: enough wavefronts to fill the chip several times, never more than the work.
  const dim3 block(256);
  const uint32_t short_blocks = ceil_div(static_cast<uint64_t>(Vd) * kShortG, 256);
  const dim3 short_grid(short_blocks < 16384u ? short_blocks : 16384u);
  const uint32_t wave_blocks = ceil_div(Vd, 4);  // at most one destination per wavefront
  const dim3 grid(wave_blocks < 8192u ? wave_blocks : 8192u);
  const uint32_t set = softmax_rows_per_wave(Vd);
  if (lr.list) {
    // The hub rows first: their few large blocks take their places on the chip before the launches for
    // all other rows fill it.
    if (!backward) {
      if (fused)
        hipLaunchKernelGGL(edge_softmax_fwd_long_kernel<true>, dim3(kLongGrid), dim3(kLongBlock), 0, hub_stream, out,
                           x_or_gy, el, er, co, ri, lr.list, lr.count, H, slope);
      else
        hipLaunchKernelGGL(edge_softmax_fwd_long_kernel<false>, dim3(kLongGrid), dim3(kLongBlock), 0, hub_stream, out,
                           x_or_gy, el, er, co, ri, lr.list, lr.count, H, slope);
    } else {
      if (fused)
        hipLaunchKernelGGL(edge_softmax_bwd_long_kernel<true>, dim3(kLongGrid), dim3(kLongBlock), 0, hub_stream, out, ger,
                           x_or_gy, y, el, er, co, ri, lr.list, lr.count, H, slope);
      else
        hipLaunchKernelGGL(edge_softmax_bwd_long_kernel<false>, dim3(kLongGrid), dim3(kLongBlock), 0, hub_stream, out, ger,
                           x_or_gy, y, el, er, co, ri, lr.list, lr.count, H, slope);
    }
    NTS_LAUNCH_CHECK(who);
    // Giant segments: per-piece statistics, ordered combine, apply (see the kernels above).
    float *stats = static_cast<float *>(stats_block.ptr);
    float *rowstat = stats + stats_floats;
    const dim3 pgrid(kLongGrid), pblock(kLongBlock), cgrid(kGiantCap / 4), cblock(64);
    if (!backward) {
      if (fused)
        hipLaunchKernelGGL(giant_softmax_stats_kernel<true>, pgrid, pblock, 0, hub_stream, stats, out, x_or_gy, el, er, ri,
                           lr.hdr, lr.pieces, H, slope);
      else
        hipLaunchKernelGGL(giant_softmax_stats_kernel<false>, pgrid, pblock, 0, hub_stream, stats, out, x_or_gy, el, er, ri,
                           lr.hdr, lr.pieces, H, slope);
      hipLaunchKernelGGL(giant_softmax_combine_kernel<0>, cgrid, cblock, 0, hub_stream, rowstat,
                         static_cast<float *>(nullptr), stats, lr.hdr, lr.giant_rows, lr.first, H, 2 * H);
      if (fused)
        hipLaunchKernelGGL(giant_softmax_apply_kernel<true>, pgrid, pblock, 0, hub_stream, out, x_or_gy, rowstat, lr.hdr,
                           lr.pieces, H);
      else
        hipLaunchKernelGGL(giant_softmax_apply_kernel<false>, pgrid, pblock, 0, hub_stream, out, x_or_gy, rowstat, lr.hdr,
                           lr.pieces, H);
    } else {
      hipLaunchKernelGGL(giant_softmax_dot_kernel, pgrid, pblock, 0, hub_stream, stats, x_or_gy, y, lr.hdr, lr.pieces, H);
      hipLaunchKernelGGL(giant_softmax_combine_kernel<1>, cgrid, cblock, 0, hub_stream, rowstat,
                         static_cast<float *>(nullptr), stats, lr.hdr, lr.giant_rows, lr.first, H, H);
      if (fused) {
        hipLaunchKernelGGL(giant_softmax_bwd_apply_kernel<true>, pgrid, pblock, 0, hub_stream, out, stats, x_or_gy, y, el, er,
                           ri, rowstat, lr.hdr, lr.pieces, H, slope);
        hipLaunchKernelGGL(giant_softmax_combine_kernel<1>, cgrid, cblock, 0, hub_stream, rowstat, ger, stats, lr.hdr,
                           lr.giant_rows, lr.first, H, H);
      } else {
        hipLaunchKernelGGL(giant_softmax_bwd_apply_kernel<false>, pgrid, pblock, 0, hub_stream, out, stats, x_or_gy, y, el, er,
                           ri, rowstat, lr.hdr, lr.pieces, H, slope);
      }
    }
    NTS_LAUNCH_CHECK(who);
  }
  if (use_short && one_short_launch) {
    // Every segment fits the short class by the caller's word: one launch (which still computes a
    // longer segment, slowly, should there be one).
    if (backward)
      hipLaunchKernelGGL((edge_softmax_short_kernel<true, true, true>), short_grid, block, 0, stream, out, ger, x_or_gy,
                         y, el, er, co, ri, Vd, H, slope);
    else
      hipLaunchKernelGGL((edge_softmax_short_kernel<true, false, true>), short_grid, block, 0, stream, out, ger, x_or_gy,
                         y, el, er, co, ri, Vd, H, slope);
    NTS_LAUNCH_CHECK(who);
    return NTS_OK;
  }
  if (use_short) {
#define NTS_SHORT(FU, BW)                                                                                          \
  hipLaunchKernelGGL((edge_softmax_short_kernel<FU, BW>), short_grid, block, 0, stream, out, ger, x_or_gy, y, el, er, \
                     co, ri, Vd, H, slope)
    if (fused) { if (backward) NTS_SHORT(true, true); else NTS_SHORT(true, false); }
    else       { if (backward) NTS_SHORT(false, true); else NTS_SHORT(false, false); }
#undef NTS_SHORT
    NTS_LAUNCH_CHECK(who);
  }
  if (!backward) {
#define NTS_FWD(FU, P2, PART, LO, HI)                                                                             \
  hipLaunchKernelGGL((edge_softmax_fwd_kernel<FU, P2, PART>), grid, block, 0, stream, out, x_or_gy, el, er, co, ri, \
                     Vd, H, slope, LO, HI, vec4, set)
    if (pow2 && fused) {
      // the register-resident segments, then the longer ones
      NTS_FWD(true, true, 1, min_values, kWaveRegValues);
      // 513 .. 2,048 values in a launch of their own: 16 or 32 values per lane in registers, one pass over
      // memory, and the registers that costs are not the other classes' (64 per lane measured slower)
      NTS_FWD(true, true, 3, kWaveRegValues + 1, kWaveMidValues);
      NTS_FWD(true, true, 2, kWaveMidValues + 1, max_values);
    } else if (pow2) {
      NTS_FWD(false, true, 0, min_values, max_values);
    } else {
      if (fused) NTS_FWD(true, false, 0, min_values, max_values); else NTS_FWD(false, false, 0, min_values, max_values);
    }
#undef NTS_FWD
    NTS_LAUNCH_CHECK(who);
  } else {
#define NTS_BWD(FU, P2, PART, LO, HI)                                                                            \
  hipLaunchKernelGGL((edge_softmax_bwd_kernel<FU, P2, PART>), grid, block, 0, stream, out, ger, x_or_gy, y, el, er, co, \
                     ri, Vd, H, slope, LO, HI, vec4, set)
    if (pow2 && fused) {
      NTS_BWD(true, true, 1, min_values, kWaveRegValues);
      // (a launch of its own for the class above that, held in registers as in the forward pass, measured no
      // gain up to 1,024 values and 3.36 -> 3.57 ms up to 2,048: the backward holds two arrays per lane)
      NTS_BWD(true, true, 2, kWaveRegValues + 1, max_values);
    } else if (pow2) {
      NTS_BWD(false, true, 0, min_values, max_values);
    } else {
      if (fused) NTS_BWD(true, false, 0, min_values, max_values); else NTS_BWD(false, false, 0, min_values, max_values);
    }
#undef NTS_BWD
    NTS_LAUNCH_CHECK(who);
  }
  if (lr.list) {
    const hipError_t join_err = side.join();  // `stream` waits for the hub rows before their scratch goes back
    NTS_HIP_TRY(stats_block.release());
    if (join_err != hipSuccess) return fail_hip(join_err, who);
  }
  return release_long_rows(lr);
}
}  // namespace

extern "C" {

int nts_scatter_src_to_edge(float *msg, const float *feat, const uint32_t *ri, const uint32_t *co,
                            const uint32_t *mirror, uint32_t Vd, uint32_t F, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_scatter_src_to_edge");
  return edge_copy_impl(msg, feat, ri, co, mirror, Vd, F, kFromSrc, stream, "nts_scatter_src_to_edge: bad argument");
}

int nts_scatter_dst_to_edge(float *msg, const float *feat, const uint32_t *co, uint32_t Vd, uint32_t F,
                            nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_scatter_dst_to_edge");
  return edge_copy_impl(msg, feat, nullptr, co, nullptr, Vd, F, kFromDst, stream,
                        "nts_scatter_dst_to_edge: bad argument");
}

int nts_scatter_grad_to_edge(float *msg_grad, const float *gout, const uint32_t *co, uint32_t Vd, uint32_t F,
                             nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_scatter_grad_to_edge");
  return edge_copy_impl(msg_grad, gout, nullptr, co, nullptr, Vd, F, kAddFromDst, stream,
                        "nts_scatter_grad_to_edge: bad argument");
}

int nts_gather_edge_to_dst(float *out, const float *msg, const uint32_t *co, uint32_t Vd, uint32_t F, int accumulate,
                           nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_gather_edge_to_dst");
  return gather_edge_impl(out, msg, co, nullptr, Vd, F, accumulate, stream, "nts_gather_edge_to_dst: bad argument");
}

int nts_gather_edge_to_src(float *out, const float *msg, const uint32_t *ro, const uint32_t *perm, uint32_t Vs,
                           uint32_t F, int accumulate, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_gather_edge_to_src");
  if (Vs != 0 && !perm) return fail(NTS_ERR_INVALID, "nts_gather_edge_to_src: null perm");
  return gather_edge_impl(out, msg, ro, perm, Vs, F, accumulate, stream, "nts_gather_edge_to_src: bad argument");
}

int nts_edge_softmax_fwd(float *y, const float *x, const uint32_t *co, uint32_t Vd, uint32_t H,
                         nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_edge_softmax_fwd");
  if (H == 0) return fail(NTS_ERR_INVALID, "nts_edge_softmax_fwd: H is 0");
  if (Vd == 0) return NTS_OK;
  if (!y || !x || !co) return fail(NTS_ERR_INVALID, "nts_edge_softmax_fwd: null pointer");
  return softmax_impl(false, false, y, nullptr, x, nullptr, nullptr, nullptr, co, nullptr, Vd, H, 0.f, stream,
                      "nts_edge_softmax_fwd");
}

int nts_edge_softmax_bwd(float *gx, const float *gy, const float *y, const uint32_t *co, uint32_t Vd, uint32_t H,
                         nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_edge_softmax_bwd");
  if (H == 0) return fail(NTS_ERR_INVALID, "nts_edge_softmax_bwd: H is 0");
  if (Vd == 0) return NTS_OK;
  if (!gx || !gy || !y || !co) return fail(NTS_ERR_INVALID, "nts_edge_softmax_bwd: null pointer");
  return softmax_impl(true, false, gx, nullptr, gy, y, nullptr, nullptr, co, nullptr, Vd, H, 0.f, stream,
                      "nts_edge_softmax_bwd");
}

int nts_gat_attention_fwd(float *alpha, const float *el, const float *er, const uint32_t *co, const uint32_t *ri,
                          uint32_t Vd, uint32_t H, float slope, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_gat_attention_fwd");
  if (H == 0) return fail(NTS_ERR_INVALID, "nts_gat_attention_fwd: H is 0");
  if (Vd == 0) return NTS_OK;
  if (!alpha || !el || !er || !co || !ri) return fail(NTS_ERR_INVALID, "nts_gat_attention_fwd: null pointer");
  return softmax_impl(false, true, alpha, nullptr, nullptr, nullptr, el, er, co, ri, Vd, H, slope, stream,
                      "nts_gat_attention_fwd");
}

int nts_gat_attention_fwd_bounded(float *alpha, const float *el, const float *er, const uint32_t *co,
                                  const uint32_t *ri, uint32_t Vd, uint32_t H, float slope, uint32_t max_degree,
                                  nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_gat_attention_fwd_bounded");
  if (H == 0) return fail(NTS_ERR_INVALID, "nts_gat_attention_fwd_bounded: H is 0");
  if (Vd == 0) return NTS_OK;
  if (!alpha || !el || !er || !co || !ri) return fail(NTS_ERR_INVALID, "nts_gat_attention_fwd_bounded: null pointer");
  return softmax_impl(false, true, alpha, nullptr, nullptr, nullptr, el, er, co, ri, Vd, H, slope, stream,
                      "nts_gat_attention_fwd_bounded", max_degree);
}

int nts_gat_attention_bwd_bounded(float *gs, float *ger, const float *galpha, const float *alpha, const float *el,
                                  const float *er, const uint32_t *co, const uint32_t *ri, uint32_t Vd, uint32_t H,
                                  float slope, uint32_t max_degree, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_gat_attention_bwd_bounded");
  if (H == 0) return fail(NTS_ERR_INVALID, "nts_gat_attention_bwd_bounded: H is 0");
  if (Vd == 0) return NTS_OK;
  if (!gs || !ger || !galpha || !alpha || !el || !er || !co || !ri)
    return fail(NTS_ERR_INVALID, "nts_gat_attention_bwd_bounded: null pointer");
  return softmax_impl(true, true, gs, ger, galpha, alpha, el, er, co, ri, Vd, H, slope, stream,
                      "nts_gat_attention_bwd_bounded", max_degree);
}

int nts_gat_attention_bwd(float *gs, float *ger, const float *galpha, const float *alpha, const float *el,
                          const float *er, const uint32_t *co, const uint32_t *ri, uint32_t Vd, uint32_t H,
                          float slope, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_gat_attention_bwd");
  if (H == 0) return fail(NTS_ERR_INVALID, "nts_gat_attention_bwd: H is 0");
  if (Vd == 0) return NTS_OK;
  if (!gs || !ger || !galpha || !alpha || !el || !er || !co || !ri)
    return fail(NTS_ERR_INVALID, "nts_gat_attention_bwd: null pointer");
  return softmax_impl(true, true, gs, ger, galpha, alpha, el, er, co, ri, Vd, H, slope, stream,
                      "nts_gat_attention_bwd");
}

int nts_sddmm_heads(float *galpha, const float *in, const float *gout, const uint32_t *co, const uint32_t *ri,
                    uint32_t Vd, uint32_t H, uint32_t Fh, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_sddmm_heads");
  if (H == 0 || Fh == 0) return fail(NTS_ERR_INVALID, "nts_sddmm_heads: H or Fh is 0");
  if (static_cast<uint64_t>(H) * Fh > 0xFFFFFFFFull) return fail(NTS_ERR_INVALID, "nts_sddmm_heads: H*Fh overflows");
  if (Vd == 0) return NTS_OK;
  if (!galpha || !in || !gout || !co || !ri) return fail(NTS_ERR_INVALID, "nts_sddmm_heads: null pointer");
  const uint32_t F = H * Fh;
  const dim3 grid = edge_grid(Vd), block(256);
  uint32_t vec = 1;
  if (sddmm_by_lanes(in, gout, H, Fh, &vec)) {
    const uint32_t lanes = F / vec, lanes_per_head = Fh / vec;
    if (vec == 4)
      hipLaunchKernelGGL(sddmm_edge_kernel<4>, grid, block, 0, stream, galpha, in, gout, co, ri, Vd, H, Fh, lanes,
                         lanes_per_head);
    else
      hipLaunchKernelGGL(sddmm_edge_kernel<1>, grid, block, 0, stream, galpha, in, gout, co, ri, Vd, H, Fh, lanes,
                         lanes_per_head);
  } else {
    hipLaunchKernelGGL(sddmm_edge_generic_kernel, grid, block, 0, stream, galpha, in, gout, co, ri, Vd, H, Fh);
  }
  NTS_LAUNCH_CHECK("nts_sddmm_heads");
  return NTS_OK;
}

}  // extern "C"
