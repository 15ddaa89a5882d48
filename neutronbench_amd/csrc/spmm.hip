// Aggregation kernels: weighted / unweighted SpMM executed as a row gather, forward over CSC and
// backward over CSR (replaces cuda/ntsCUDAFuseKernel.cuh:147-290, 327-487 and their launchers
// cuda/ntsCUDAGraphOP.cu:186-292).
//
// Mapping.  One wavefront (64 lanes) owns one work item = one output row, or one chunk of a long
// row.  The 64 lanes span the feature dimension: lane l holds NACC register accumulators of VEC
// consecutive floats at columns (l + 64*k)*VEC (VEC = 4 when rows are 16-byte aligned, else 1), so
// every row read is a fully coalesced 64*VEC*4-byte wave load and each output element is written
// exactly once, without atomics.
// Neighbour (index, weight) pairs are fetched 64 at a time with one coalesced load per wave, staged
// in a wave-private LDS tile and read back one pair at a time by all lanes at once (a broadcast
// read), then moved to scalar registers, so the source-row base address is scalar and every
// index/weight is read from memory once per row instead of once per lane.
// Narrow rows (F <= 32*VEC) use sub-wavefront groups of G lanes per row (spmm_group_kernel).
//
// Accumulation order within a row is the edge order of the offsets array, one fused multiply-add
// per edge and element -- the order of the CPU operators (core/ntsMiniBatchGraphOp.hpp:154-240),
// so unsplit rows reproduce an FMA-contracted CPU build bit for bit.
#include <stdlib.h>
#include <string.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include <algorithm>
#include <array>
#include <atomic>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "common.hpp"
#include "edge_sort.hpp"
#include "plan_scratch.hpp"

// Fixed scratch of nts_spmm_gather_static_scratch, the entry point for callers that must not allocate:
// each device that loads this library holds one copy of the array until the process ends.  Host code
// never passes the array's name to a kernel (on the host the name is only a stand-in for the symbol):
// its device address is looked up once per device and kept in g_static_scratch_ptr.
constexpr size_t kStaticScratchBytes = NTS_SPMM_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace nts {
namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_static_scratch_mutex;
unsigned char *g_static_scratch_ptr[kMaxScratchDevices] = {};

// Device address of `scratch` on the current device (looked up on the first call per device).
int static_scratch_address(unsigned char **out) {
  int dev = -1;
  NTS_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxScratchDevices) return fail(NTS_ERR_INVALID, "static scratch: device ordinal out of range");
  std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
  if (!g_static_scratch_ptr[dev]) {
    unsigned char *p = nullptr;
    NTS_HIP_TRY(hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch)));
    if (!p) return fail(NTS_ERR_HIP, "static scratch: hipGetSymbolAddress returned a null address");
    g_static_scratch_ptr[dev] = p;
  }
  *out = g_static_scratch_ptr[dev];
  return NTS_OK;
}

template <int VEC>
struct Vec;
template <>
struct Vec<1> {
  using type = float;
};
template <>
struct Vec<2> {
  using type = float2;
};
template <>
struct Vec<4> {
  using type = float4;
};

// Vectors of a row that starts at any float (SHARED): the memory path takes 16-byte lanes at multiples of four bytes.
typedef float Floats4 __attribute__((ext_vector_type(4), aligned(4)));
template <int VEC, bool SHARED>
__device__ __forceinline__ typename Vec<VEC>::type load_row(const float *p) {
  if constexpr (VEC == 4 && SHARED) {
    const Floats4 v = *reinterpret_cast<const Floats4 *>(p);
    return make_float4(v.x, v.y, v.z, v.w);
  } else {
    return *reinterpret_cast<const typename Vec<VEC>::type *>(p);
  }
}
// The floats `skip` .. VEC - 1 of r, to p + skip on; with `accumulate` added to what is there.
template <int VEC>
__device__ __forceinline__ void store_row(float *p, typename Vec<VEC>::type r, uint32_t skip, bool accumulate) {
  if constexpr (VEC == 4) {
    if (skip == 0) {
      if (accumulate) {
        const Floats4 o = *reinterpret_cast<const Floats4 *>(p);
        r = make_float4(r.x + o.x, r.y + o.y, r.z + o.z, r.w + o.w);
      }
      *reinterpret_cast<Floats4 *>(p) = Floats4{r.x, r.y, r.z, r.w};
      return;
    }
  }
  const float *f = reinterpret_cast<const float *>(&r);
#pragma unroll
  for (uint32_t i = 0; i < VEC; ++i)
    if (i >= skip) p[i] = accumulate ? f[i] + p[i] : f[i];
}

template <int VEC>
__device__ __forceinline__ typename Vec<VEC>::type vzero();
template <>
__device__ __forceinline__ float vzero<1>() {
  return 0.f;
}
template <>
__device__ __forceinline__ float2 vzero<2>() {
  return make_float2(0.f, 0.f);
}
template <>
__device__ __forceinline__ float4 vzero<4>() {
  return make_float4(0.f, 0.f, 0.f, 0.f);
}

__device__ __forceinline__ void vfma(float &a, float x, float w) { a = fmaf(x, w, a); }
__device__ __forceinline__ void vfma(float2 &a, float2 x, float w) {
  a.x = fmaf(x.x, w, a.x);
  a.y = fmaf(x.y, w, a.y);
}
__device__ __forceinline__ void vfma(float4 &a, float4 x, float w) {
  a.x = fmaf(x.x, w, a.x);
  a.y = fmaf(x.y, w, a.y);
  a.z = fmaf(x.z, w, a.z);
  a.w = fmaf(x.w, w, a.w);
}
// Zero in place of the first `skip` floats: the columns that the lane before has too count once in a product.
__device__ __forceinline__ void drop_first(float &, uint32_t) {}
__device__ __forceinline__ void drop_first(float4 &a, uint32_t skip) {
  a.x = skip > 0 ? 0.f : a.x;
  a.y = skip > 1 ? 0.f : a.y;
  a.z = skip > 2 ? 0.f : a.z;
}
__device__ __forceinline__ float vdot(float a, float b) { return a * b; }
__device__ __forceinline__ float vdot(float4 a, float4 b) {
  return fmaf(a.w, b.w, fmaf(a.z, b.z, fmaf(a.y, b.y, a.x * b.x)));
}
__device__ __forceinline__ void vadd(float &a, float x) { a += x; }
__device__ __forceinline__ void vadd(float2 &a, float2 x) {
  a.x += x.x;
  a.y += x.y;
}
__device__ __forceinline__ void vadd(float4 &a, float4 x) {
  a.x += x.x;
  a.y += x.y;
  a.z += x.z;
  a.w += x.w;
}

// Edges processed per inner step: keeps 8..16 independent row loads in flight per lane.
// With 4-byte lanes and six to ten accumulators (F = 602: ten) four edges per step were measured
// against one, two and three: 11.04 ms against 11.54 / 11.13 / 11.13 for the Reddit-shaped F=602 pass --
// a step's loads are all requested before the first is used, so a wavefront then has 40 row loads in
// flight instead of 10.  With 16-byte lanes the same count would cost 160 registers.
__host__ __device__ constexpr int unroll_for(int nacc, int vec) {
  return nacc >= 6 ? (vec == 1 ? 4 : 1) : nacc >= 4 ? 2 : nacc >= 2 ? 4 : 8;
}

// Work item of a planned launch: row, first edge, one-past-last edge, partial slot (kNoSlot = the
// item is a whole row and writes `out` directly).
using Item = uint4;

// Per-head edge weights (attention-weighted aggregation): w is alpha [E_csc, H], a column belongs
// to head column / Fh, and the weight of edge position e is alpha[(perm ? perm[e] : e) * H + head].
struct HeadArgs {
  const uint32_t *perm;
  uint32_t H;
  uint32_t Fh;
};

template <int VEC, int NACC, bool LDS_TILE, bool HEADS, bool REMAP, bool RUNS>
__global__ __launch_bounds__(256) void spmm_wave_kernel(const float *__restrict__ in, float *__restrict__ out,
                                                        const float *__restrict__ w,
                                                        const uint32_t *__restrict__ offsets,
                                                        const uint32_t *__restrict__ indices, uint32_t index_base,
                                                        uint32_t n_items, uint32_t n_list, uint32_t F,
                                                        uint32_t first_col, uint32_t panels, const Item *__restrict__ items,
                                                        float *__restrict__ partial,
                                                        int accumulate, HeadArgs heads, uint32_t row_edge_limit,
                                                        const uint32_t *__restrict__ edge_ids, uint32_t in_ld,
                                                        uint32_t partial_ld, int out_scalar) {
  using V = typename Vec<VEC>::type;
  constexpr int U = unroll_for(NACC, VEC);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t col_base = first_col + blockIdx.x % panels * (kWave * VEC * NACC);
  const uint32_t item = blockIdx.x / panels * (blockDim.x / kWave) + (threadIdx.x / kWave);
  if (item >= n_items) return;

  // Work items [0, n_list) come from the list, the ones after it are the rows 0, 1, ... themselves
  // (a launch may hold both: the pieces of long rows first, then every row that fits one wavefront).
  uint32_t row, e0, e1, slot;
  if (item < n_list) {
    const Item it = items[item];
    row = wave_first(it.x);
    e0 = wave_first(it.y);
    e1 = wave_first(it.z);
    slot = wave_first(it.w);
  } else {
    row = item - n_list;
    e0 = wave_first(offsets[row]);
    e1 = wave_first(offsets[row + 1]);
    slot = kNoSlot;
    if (e1 - e0 > row_edge_limit) return;  // a long row: its pieces are separate work items
  }

  // Lanes past the end of the row (in the last accumulator; where one launch covers all panels, in any of the last
  // panel's) read the row's last VEC columns instead, so that loads need no predication; their sums are never stored.
  uint32_t col[NACC];
  uint32_t lcol[NACC];
  uint32_t head[NACC];
  bool live[NACC];
  V acc[NACC];
#pragma unroll
  for (int k = 0; k < NACC; ++k) {
    col[k] = col_base + (lane + kWave * k) * VEC;
    live[k] = col[k] < F;
    lcol[k] = live[k] ? col[k] : in_ld - VEC;
    head[k] = HEADS ? lcol[k] / heads.Fh : 0u;
    acc[k] = vzero<VEC>();
  }

  // Tile of up to 64 neighbour (index, weight) pairs, fetched with one coalesced load per wave; the
  // next tile is fetched while the current one is consumed.  The pairs are then handed to the whole
  // wave one at a time as scalars: either straight from the registers that hold them (readlane), or
  // (LDS_TILE) through a wave-private LDS tile that every lane reads at the same address.  The LDS
  // region belongs to one wave and LDS operations of a wave complete in order, so no block barrier
  // is needed -- which matters because waves of a block run different trip counts.
  __shared__ uint2 lds_tile[LDS_TILE ? 4 : 1][LDS_TILE ? kWave : 1];
  uint2 *tile = lds_tile[LDS_TILE ? (threadIdx.x / kWave) : 0];
  // Second component of a pair: the edge weight (as bits), or with per-head weights the id of the
  // edge in alpha's (CSC) order.
  // edge_ids (a schedule that gathers through its own, re-ordered copy of the indices): position of
  // edge e in the caller's weight / alpha order.
  auto second_of = [&](uint32_t e) -> uint32_t {
    const uint32_t id = REMAP ? edge_ids[e] : e;
    if (HEADS) return heads.perm ? heads.perm[id] : id;
    return w ? __float_as_uint(w[id]) : __float_as_uint(1.f);
  };
  uint32_t nxt_i = 0;
  uint32_t nxt_s = HEADS ? 0u : __float_as_uint(1.f);
  if (e0 + lane < e1) {
    nxt_i = indices[e0 + lane] - index_base;
    nxt_s = second_of(e0 + lane);
  }
  for (uint32_t eb = e0; eb < e1; eb += kWave) {
    const uint32_t n = min(static_cast<uint32_t>(kWave), e1 - eb);
    const uint32_t my_i = nxt_i;
    const uint32_t my_s = nxt_s;
    if (LDS_TILE) {
      __builtin_amdgcn_wave_barrier();  // earlier reads of the tile are done before it is overwritten
      tile[lane] = make_uint2(my_i, my_s);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    const uint32_t en = eb + kWave + lane;
    if (en < e1) {
      nxt_i = indices[en] - index_base;
      nxt_s = second_of(en);
    }
    auto pair_at = [&](uint32_t j, uint32_t &idx, uint32_t &second) {
      if (LDS_TILE) {
        const uint2 p = tile[j];
        idx = wave_first(p.x);
        second = wave_first(p.y);
      } else {
        idx = wave_read(my_i, j);
        second = wave_read(my_s, j);
      }
    };
    if (RUNS && LDS_TILE && !HEADS) {
      // Runs of consecutive edges with the same neighbour (a multigraph's parallel edges, adjacent in
      // sorted rows): the row is loaded once and added once per edge of the run, in edge order with
      // each edge's own weight, so the result is the same bit for bit.  Up to U runs per step.
      const uint32_t prev = tile[lane ? lane - 1 : 0].x;
      uint64_t starts = __ballot(lane < n && (lane == 0 || my_i != prev));
      while (starts) {
        uint32_t rs[U + 1];
        int nr = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          rs[u] = n;
          if (starts) {
            rs[u] = static_cast<uint32_t>(__builtin_ctzll(starts));
            starts &= starts - 1;
            nr = u + 1;
          }
        }
        rs[U] = starts ? static_cast<uint32_t>(__builtin_ctzll(starts)) : n;
        V v[U][NACC];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (u < nr) {
            const float *src = in + static_cast<size_t>(wave_first(tile[rs[u]].x)) * in_ld;
#pragma unroll
            for (int k = 0; k < NACC; ++k) v[u][k] = *reinterpret_cast<const V *>(src + lcol[k]);
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (u < nr) {
            const uint32_t end = (u + 1 < U) ? rs[u + 1] : rs[U];
            for (uint32_t q = rs[u]; q < end; ++q) {
              const float wgt = __uint_as_float(wave_first(tile[q].y));
#pragma unroll
              for (int k = 0; k < NACC; ++k) vfma(acc[k], v[u][k], wgt);
            }
          }
        }
      }
      continue;
    }
    uint32_t j = 0;
    for (; j + U <= n; j += U) {
      const float *src[U];
      uint32_t ss[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        uint32_t si;
        pair_at(j + u, si, ss[u]);
        src[u] = in + static_cast<size_t>(si) * in_ld;
      }
      V v[U][NACC];
      float wv[U][HEADS ? NACC : 1];
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int k = 0; k < NACC; ++k) {
          v[u][k] = *reinterpret_cast<const V *>(src[u] + lcol[k]);
          if (HEADS) wv[u][k] = w[static_cast<size_t>(ss[u]) * heads.H + head[k]];
        }
        if (!HEADS) wv[u][0] = __uint_as_float(ss[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int k = 0; k < NACC; ++k) {
          vfma(acc[k], v[u][k], wv[u][HEADS ? k : 0]);
        }
      }
    }
    for (; j < n; ++j) {
      uint32_t si, ss;
      pair_at(j, si, ss);
      const float *src = in + static_cast<size_t>(si) * in_ld;
#pragma unroll
      for (int k = 0; k < NACC; ++k) {
        const float wgt = HEADS ? w[static_cast<size_t>(ss) * heads.H + head[k]] : __uint_as_float(ss);
        vfma(acc[k], *reinterpret_cast<const V *>(src + lcol[k]), wgt);
      }
    }
  }

  if (VEC > 1 && out_scalar && slot == kNoSlot) {
    // Output rows that do not start on a 16-byte boundary (F not a multiple of four while the gather
    // runs over a padded copy of the input): the row is stored one float at a time.
    float *dst = out + static_cast<size_t>(row) * F;
#pragma unroll
    for (int k = 0; k < NACC; ++k) {
      const float *r = reinterpret_cast<const float *>(&acc[k]);
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        const uint32_t cc = col[k] + c;
        if (cc < F) dst[cc] = accumulate ? r[c] + dst[cc] : r[c];
      }
    }
    return;
  }
  float *dst =
      (slot == kNoSlot) ? out + static_cast<size_t>(row) * F : partial + static_cast<size_t>(slot) * partial_ld;
  const bool add = accumulate && slot == kNoSlot;
#pragma unroll
  for (int k = 0; k < NACC; ++k) {
    if (live[k]) {
      V *p = reinterpret_cast<V *>(dst + col[k]);
      V r = acc[k];
      if (add) vadd(r, *p);
      *p = r;
    }
  }
}

// Sub-wavefront variant for narrow rows: G lanes per row, 64/G rows per wavefront, one VEC-wide accumulator per lane.
// Neighbour pairs are fetched G at a time per group and broadcast inside the group with cross-lane shuffles.
// A lane's vector never crosses the end of its head (or row): where the width is no multiple of VEC the last lane's starts
// earlier, shares columns with the lane before it and stores only its own.  16-byte lanes at any float instead of a
// wavefront of 4-byte ones for a row of 47 floats: 500 K rows, 20 M edges with source ranges 809 -> 416 us, and from 33 to 127
// floats 800-1,046 -> 343-861; 1 M, 3 M without a schedule 306 -> 210.
// With per-head weights the registers are held down to what six wavefronts per SIMD have (90-96 -> 75-77; the gather waits
// for memory): four heads of 32 on 169 K rows, 2.48 M edges 175 -> 146 us, 1 M, 3 M 499 -> 403, 500 K, 20 M 1,066 -> 970; eight
// wavefronts 157, 419 and 1,028.  Without, groups of up to 16 lanes are held to eight (72 -> 63 registers: 1 M, 3 M without a
// schedule F = 64 219 -> 208, F = 47 211 -> 201); 32 lanes would spill in the loop (2.45 M, 126 M F = 100 and 128 20.4 -> 21.1 ms a
// step), and rows with runs, held to seven, lose the overlap of their loads (60 K, 600 K F = 17 48 -> 101 us).
constexpr uint32_t kXcds = 8;
template <int G, bool HEADS, bool RUNS>
constexpr int group_waves() {
  return HEADS ? 6 : !RUNS && G <= 16 ? 8 : 1;
}
template <bool SHARED, bool PANELS, int G, int VEC, int U, bool HEADS, bool REMAP, bool RUNS>
__global__ __launch_bounds__(256, (group_waves<G, HEADS, RUNS>())) void spmm_group_kernel(const float *__restrict__ in, float *__restrict__ out,
                                                         const float *__restrict__ w,
                                                         const uint32_t *__restrict__ offsets,
                                                         const uint32_t *__restrict__ indices, uint32_t index_base,
                                                         uint32_t n_items, uint32_t n_list, uint32_t F,
                                                         const Item *__restrict__ items, float *__restrict__ partial,
                                                         int accumulate, HeadArgs heads,
                                                         uint32_t row_edge_limit,
                                                         const uint32_t *__restrict__ edge_ids, uint32_t panels,
                                                         int panel_bits, uint32_t in_ld, uint32_t partial_ld) {
  using V = typename Vec<VEC>::type;
  static_assert(U <= G, "a step's pairs come from one tile");  // U edges per step: their rows are requested together
  const uint32_t gl = threadIdx.x & (G - 1);
  // Blocks are dealt out to the eight XCDs in turn.  1 << panel_bits panels (two or four; one needs no turns) alternate and an XCD
  // meets one of them.  Of other numbers, eight blocks of items are 8 * panels units of work, panel by panel, and XCD x takes the units
  // x * panels and on: an XCD meets two panels, three where there are eleven (641 to 704 floats).  (The alternating panels too by that rule: 169 K rows, 2.48 M edges
  // F = 128 97 -> 100 us.)
  uint32_t panel = 0, block = blockIdx.x;
  if (PANELS) {
    if (panel_bits >= 0) {
      panel = blockIdx.x & (panels - 1);
      block = blockIdx.x >> panel_bits;
    } else {
      const uint32_t turn = blockIdx.x / kXcds, unit = blockIdx.x % kXcds * panels + turn % panels;
      panel = unit / kXcds;
      block = turn / panels * kXcds + unit % kXcds;
    }
  } else {
    in_ld = partial_ld = F;
  }
  const uint32_t item = (block * blockDim.x + threadIdx.x) / G;
  if (item >= n_items) return;  // whole groups leave together; shuffles stay inside a group

  uint32_t row, e0, e1, slot;
  if (item < n_list) {  // listed work items first, then the rows themselves
    const Item it = items[item];
    row = it.x;
    e0 = it.y;
    e1 = it.z;
    slot = it.w;
  } else {
    row = item - n_list;
    e0 = offsets[row];
    e1 = offsets[row + 1];
    slot = kNoSlot;
    if (e1 - e0 > row_edge_limit) return;  // a long row: its pieces are separate work items
  }
  // This lane's first column, the one its loads start at, and its head.  SHARED: of `per_head` lanes a head the last one
  // starts earlier where the head ends; otherwise idle lanes re-read the last columns and never store.
  uint32_t col = (panel * G + gl) * VEC, lcol, head = 0;
  bool live;
  if (SHARED) {
    const uint32_t q = panel * G + gl, Fh = HEADS ? heads.Fh : F, per_head = (Fh + VEC - 1) / VEC;
    if (HEADS) head = min(q / per_head, heads.H - 1);
    const uint32_t first = (q - head * per_head) * VEC;
    live = first < Fh;
    col = head * Fh + first;
    lcol = head * Fh + min(first, Fh - VEC);
  } else {
    live = col < F;
    lcol = live ? col : F - VEC;
    if (HEADS) head = lcol / heads.Fh;
  }
  V acc = vzero<VEC>();

  // The (index, weight) pairs of the next G edges are requested while the current ones are used, so
  // that a group does not wait for them at the start of every tile.
  auto fetch_pair = [&](uint32_t e, uint32_t &pi, uint32_t &ps) {
    pi = 0;
    ps = HEADS ? 0u : __float_as_uint(1.f);  // weight bits, or the edge's id in alpha's order
    if (e < e1) {
      pi = indices[e] - index_base;
      const uint32_t id = REMAP ? edge_ids[e] : e;
      if (HEADS)
        ps = heads.perm ? heads.perm[id] : id;
      else if (w)
        ps = __float_as_uint(w[id]);
    }
  };
  uint32_t nxt_i, nxt_s;
  fetch_pair(e0 + gl, nxt_i, nxt_s);
  V held = vzero<VEC>();            // RUNS: the row loaded last and its index
  uint32_t held_i = 0xFFFFFFFFu;
  for (uint32_t eb = e0; eb < e1; eb += G) {
    const uint32_t n = min(static_cast<uint32_t>(G), e1 - eb);
    const uint32_t my_i = nxt_i, my_s = nxt_s;
    fetch_pair(eb + G + gl, nxt_i, nxt_s);
    uint32_t j = 0;
    for (; j + U <= n; j += U) {
      uint32_t si[U];
      uint32_t ss[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        si[u] = __shfl(my_i, j + u, G);
        ss[u] = __shfl(my_s, j + u, G);
      }
      V v[U];
      float wv[U];
      if (RUNS) {
        // An edge that repeats its predecessor's index (a parallel edge) does not load the row again:
        // the group keeps the last row it loaded in `held` and adds it with the edge's own weight.
        bool fresh[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          fresh[u] = si[u] != (u ? si[u - 1] : held_i);
          v[u] = vzero<VEC>();
          if (fresh[u]) v[u] = load_row<VEC, SHARED>(in + static_cast<size_t>(si[u]) * in_ld + lcol);
          wv[u] = HEADS ? w[static_cast<size_t>(ss[u]) * heads.H + head] : __uint_as_float(ss[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (fresh[u]) held = v[u];
          vfma(acc, held, wv[u]);
        }
        held_i = si[U - 1];
        continue;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        v[u] = load_row<VEC, SHARED>(in + static_cast<size_t>(si[u]) * in_ld + lcol);
        wv[u] = HEADS ? w[static_cast<size_t>(ss[u]) * heads.H + head] : __uint_as_float(ss[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        vfma(acc, v[u], wv[u]);
      }
    }
    if (!RUNS && j < n) {
      // The last, partial step: its rows are requested together like a full step's (a sampled layer's
      // rows are a step or two long; one edge after the other, each waited for, doubled their time),
      // and added in the same order.
      const uint32_t left = n - j;
      V v[U];
      float wv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t si = __shfl(my_i, (j + u) & (G - 1), G);
        const uint32_t ss = __shfl(my_s, (j + u) & (G - 1), G);
        v[u] = vzero<VEC>();
        wv[u] = 0.f;
        if (static_cast<uint32_t>(u) < left) {
          v[u] = load_row<VEC, SHARED>(in + static_cast<size_t>(si) * in_ld + lcol);
          wv[u] = HEADS ? w[static_cast<size_t>(ss) * heads.H + head] : __uint_as_float(ss);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (static_cast<uint32_t>(u) < left) vfma(acc, v[u], wv[u]);
      }
      j = n;
    }
    for (; j < n; ++j) {
      const uint32_t si = __shfl(my_i, j, G);
      const uint32_t ss = __shfl(my_s, j, G);
      const float wgt = HEADS ? w[static_cast<size_t>(ss) * heads.H + head] : __uint_as_float(ss);
      if (RUNS) {
        if (si != held_i) held = load_row<VEC, SHARED>(in + static_cast<size_t>(si) * in_ld + lcol);
        held_i = si;
        vfma(acc, held, wgt);
        continue;
      }
      vfma(acc, load_row<VEC, SHARED>(in + static_cast<size_t>(si) * in_ld + lcol), wgt);
    }
  }

  if (live) {
    float *dst = (slot == kNoSlot) ? out + static_cast<size_t>(row) * F : partial + static_cast<size_t>(slot) * partial_ld;
    if (SHARED) {
      store_row<VEC>(dst + lcol, acc, col - lcol, accumulate && slot == kNoSlot);
    } else {
      V *p = reinterpret_cast<V *>(dst + col);
      V r = acc;
      if (accumulate && slot == kNoSlot) vadd(r, *p);
      *p = r;
    }
  }
}

// Backward of the attention-weighted aggregation over the transposed structure, both gradients from one
// pass over the gathered rows: for source row s and its edges k (destination d = indices[k], edge id
// e = perm[k] in alpha's order)
//   out[s, h, :]  = sum_k alpha[e, h] * gout[d, h, :]          (the aggregation, in edge order)
//   galpha[e, h]  = < x[s, h, :], gout[d, h, :] >
// The row gout[d] is what either gradient gathers, so the second costs the products and a 4 * H byte
// store per edge instead of a pass of its own over E rows (126 M edges, 4 heads of 32: an attention layer's
// forward and backward 32.5 -> 27.2 ms, of which nts_sddmm_heads was 8.1; 2.48 M edges, one head of 47: 1,115 -> 853 us).
// A group of G lanes owns a row (or a piece of one) and G / LH heads of it: LH lanes per head, each with
// NJ vectors of VEC floats at (sub + LH * j) * VEC of the head's slice, so that a head never shares a lane
// with another whatever its width (41 or 47 floats: 16 lanes with three floats each).  x[s] stays in
// registers.  The products of U edges are added over a head's lanes together: each butterfly step
// halves the edges a lane still holds (U - 1 exchanges for U edges instead of U log2 LH), which leaves
// lane `sub` with edge sub's sum and spreads the stores over the lanes.
// A wavefront's loads and stores complete in order, and a load behind stores would wait for them: the sums of a step
// are stored when the rows of the next one are on their way, in a loop whose accesses depend on no condition (so that
// the wait for the rows can leave the stores out).  A long row's step is then one memory latency and not two: 5 K
// vertices, 40 K edges, four heads of 4 135 -> 70 us; 30 K, 300 K, of 16 66 -> 47.  Where throughput bounds it the figures are close: 1 M, 20 M, four of 32 1,911 -> 1,863 us.
// Requesting the rows of two steps ahead was slower everywhere (0.85 times: a third fewer wavefronts fit).
//
// Wavefronts per SIMD that the registers are held down for.  The rows of wide groups come from memory, and six
// wavefronts with one or two spilled values outside the loop beat four (1.5 M vertices, 5 M edges, four heads of 32 1,050 -> 854
// us); narrower ones lose more by the spills than they gain (30 K, 300 K, eight of 4 with six 93, without 52 us).  The forms
// that share columns spill two to four, and six still beat five, whose spills are one or two (1 M, 4 M 8 x 17 786, 859 us, 4 x 25 590, 636,
// 2 x 47 575, 600; 169 K, 2.48 M 304, 316, 235, 236, 235, 223).
template <int G, int LH, int NJ, int VEC>
constexpr int grad_waves() {
  if (VEC != 4 || NJ != 1 || LH == 1) return 1;
  return LH < 8 ? 5 : G >= 32 ? 6 : 1;
}
template <int G, int LH, int NJ, int VEC, bool SHARED>
__global__ __launch_bounds__(256, (grad_waves<G, LH, NJ, VEC>())) void attention_grad_kernel(const float *__restrict__ gout, float *__restrict__ out,
                                                             const float *__restrict__ alpha,
                                                             const uint32_t *__restrict__ offsets,
                                                             const uint32_t *__restrict__ indices, uint32_t n_items,
                                                             uint32_t n_list, uint32_t F,
                                                             const Item *__restrict__ items,
                                                             float *__restrict__ partial, int accumulate,
                                                             HeadArgs heads, uint32_t row_edge_limit,
                                                             const float *__restrict__ x, float *__restrict__ galpha) {
  using V = typename Vec<VEC>::type;
  constexpr int U = NJ * VEC >= 8 ? 4 : 8;   // edges per step
  constexpr int S = LH < U ? LH : U;         // lanes of a head that end up with a sum to store
  const uint32_t gl = threadIdx.x & (G - 1), sub = gl & (LH - 1);
  const uint32_t item = (blockIdx.x * blockDim.x + threadIdx.x) / G;
  if (item >= n_items) return;  // whole groups leave together; shuffles stay inside a group
  uint32_t row, e0, e1, slot;
  if (item < n_list) {
    const Item it = items[item];
    row = it.x;
    e0 = it.y;
    e1 = it.z;
    slot = it.w;
  } else {
    row = item - n_list;
    e0 = offsets[row];
    e1 = offsets[row + 1];
    slot = kNoSlot;
    if (e1 - e0 > row_edge_limit) return;  // a long row: its pieces are separate work items
  }
  const uint32_t H = heads.H, Fh = heads.Fh;
  const uint32_t my_head = blockIdx.y * (G / LH) + gl / LH;
  const bool head_live = my_head < H;
  const uint32_t head = head_live ? my_head : H - 1;
  uint32_t col[NJ], skip[NJ];
  bool live[NJ];
  V acc[NJ], xr[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const uint32_t c = (sub + LH * j) * VEC, from = SHARED ? min(c, Fh - VEC) : c;
    live[j] = c < Fh;
    skip[j] = live[j] ? c - from : 0u;
    col[j] = head * Fh + (c < Fh ? from : 0u);  // idle lanes re-read the head's first columns
    acc[j] = vzero<VEC>();
    xr[j] = vzero<VEC>();
    if (e0 < e1) xr[j] = load_row<VEC, SHARED>(x + static_cast<size_t>(row) * F + col[j]);  // (no edge: x need not hold the row)
    if (SHARED) drop_first(xr[j], skip[j]);
  }
  const uint32_t n_edges = e1 - e0;
  // Lane l of a group holds the pair of edge l % U of a step, one step ahead; beyond the row the last edge's.
  uint32_t my_i, my_s, nxt_i, nxt_s;
  auto fetch_pair = [&](uint32_t k, uint32_t &pi, uint32_t &ps) {
    const uint32_t at = e0 + min(k + (gl & (U - 1)), n_edges - 1);
    pi = indices[at];
    ps = heads.perm[at];
  };
  V v[U][NJ];
  float p[U];
  // Lane `sub` of a head answers for the edges S * i + sub % S of a step: it loads their weights and stores their sums.
  const uint32_t mine = sub & (S - 1);
  uint32_t id[U / S];
  float w[U / S];
  auto gather_row = [&](int u, bool there) {
    const uint32_t si = __shfl(my_i, u, G);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (there) v[u][j] = load_row<VEC, SHARED>(gout + static_cast<size_t>(si) * F + col[j]);
  };
  auto gather_weight = [&](int i, bool there) {
    id[i] = __shfl(my_s, S * i + mine, G);
    if (there) w[i] = alpha[static_cast<size_t>(id[i]) * H + head];
  };
  auto products = [&](uint32_t left) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float wu = LH == 1 ? w[u / S] : __shfl(w[u / S], u % S, LH);
      p[u] = 0.f;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if (static_cast<uint32_t>(u) < left) vfma(acc[j], v[u][j], wu);
        V own = v[u][j];
        if (SHARED) drop_first(own, skip[j]);  // (also here: zero times an infinity is no zero)
        const float q = vdot(own, xr[j]);
        p[u] += live[j] ? q : 0.f;
      }
    }
    int cnt = U;
#pragma unroll
    for (int m = 1; m < LH; m <<= 1) {
      if (cnt > 1) {
        const bool upper = sub & m;
#pragma unroll
        for (int i = 0; i < U / 2; ++i) {
          if (i < cnt / 2) {
            const float keep = upper ? p[2 * i + 1] : p[2 * i];
            const float send = upper ? p[2 * i] : p[2 * i + 1];
            p[i] = keep + __shfl_xor(send, m, kWave);
          }
        }
        cnt /= 2;
      } else {
        p[0] += __shfl_xor(p[0], m, kWave);
      }
    }
  };
  uint32_t k = 0;
  if (n_edges) fetch_pair(0, my_i, my_s);
  if (n_edges >= U) {
    fetch_pair(U, nxt_i, nxt_s);
    uint32_t done[U / S];
#pragma unroll
    for (int i = 0; i < U / S; ++i) done[i] = __shfl(my_s, S * i + mine, G);
#pragma unroll
    for (int u = 0; u < U; ++u) p[u] = 0.f;
    do {
#pragma unroll
      for (int i = 0; i < U / S; ++i) gather_weight(i, true);
#pragma unroll
      for (int u = 0; u < U; ++u) gather_row(u, true);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < U / S; ++i) {
        galpha[static_cast<size_t>(done[i]) * H + head] = p[i];
        done[i] = id[i];
      }
      k += U;
      my_i = nxt_i;
      my_s = nxt_s;
      fetch_pair(k + U, nxt_i, nxt_s);
      __builtin_amdgcn_sched_barrier(0);
      products(U);
    } while (n_edges - k >= U);
#pragma unroll
    for (int i = 0; i < U / S; ++i) galpha[static_cast<size_t>(done[i]) * H + head] = p[i];
  }
  const uint32_t left = n_edges - k;
  if (left) {
#pragma unroll
    for (int i = 0; i < U / S; ++i) {
      w[i] = 0.f;
      gather_weight(i, S * i + mine < left);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) v[u][j] = vzero<VEC>();
      gather_row(u, static_cast<uint32_t>(u) < left);
    }
    products(left);
#pragma unroll
    for (int i = 0; i < U / S; ++i)
      if (head_live && sub < S && S * i + mine < left) galpha[static_cast<size_t>(id[i]) * H + head] = p[i];
  }
  float *dst = (slot == kNoSlot) ? out + static_cast<size_t>(row) * F : partial + static_cast<size_t>(slot) * F;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if (head_live && live[j]) {
      if (SHARED) {
        store_row<VEC>(dst + col[j], acc[j], skip[j], accumulate && slot == kNoSlot);
        continue;
      }
      V *q = reinterpret_cast<V *>(dst + col[j]);
      V r = acc[j];
      if (accumulate && slot == kNoSlot) vadd(r, *q);
      *q = r;
    }
  }
}

// a[j] = the columns c[j] of n >= 1 consecutive partial rows of stride ld, added one after the other from the first on.  Up to U of
// them are requested together (a row's sum is a memory latency per round, and the launch lasts as long as its longest row; U = 8 before:
// 8 K rows, 2 M edges F = 47 19 -> 8 us, F = 300 26 -> 18, 169 K, 2.48 M F = 128 5.2 -> 3.7, 233 K, 50 M with source ranges F = 128 104 ->
// 74; F = 602, 359 us, is bound by the 1.1 GB that it reads), the last ones eight at a time, whose requests
// beyond the end are the last row's again.
template <int J, int U>
__device__ __forceinline__ void add_partial_rows(const float *__restrict__ src, size_t ld, uint32_t n, const uint32_t (&c)[J], float (&a)[J]) {
#pragma unroll
  for (int j = 0; j < J; ++j) a[j] = src[c[j]];
  uint32_t k = 1;
  for (; n - k >= U; k += U) {
    float v[U][J];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < J; ++j) v[u][j] = src[(k + u) * ld + c[j]];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < J; ++j) a[j] += v[u][j];
  }
  for (; k < n; k += 8) {
    float v[8][J];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int j = 0; j < J; ++j) v[u][j] = src[(k + u < n ? k + u : n - 1) * ld + c[j]];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (k + u < n) a[j] += v[u][j];
  }
}
template <int J>
constexpr int kPartialRows = J == 1 ? 32 : J == 2 ? 16 : 8;

// Second stage for split rows: out[row,:] (+)= partial[first,:] + partial[first+1,:] + ... in slot
// order.  Block (x, y) owns 256 columns (tile y) of split row x; `splits[i]` = (row, first slot,
// slot count, unused).
__global__ __launch_bounds__(256) void spmm_reduce_partials_kernel(float *__restrict__ out,
                                                                   const float *__restrict__ partial,
                                                                   const uint4 *__restrict__ splits, uint32_t F,
                                                                   int accumulate, uint32_t ld) {
  const uint4 s = splits[blockIdx.x];
  const uint32_t c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= F) return;
  const uint32_t col[1] = {c};
  float a[1];
  add_partial_rows<1, kPartialRows<1>>(partial + static_cast<size_t>(s.y) * ld, ld, s.z, col, a);
  float *dst = out + static_cast<size_t>(s.x) * F + c;
  *dst = accumulate ? a[0] + *dst : a[0];
}

// The same for rows of up to 1,024 columns: one block per split row covers all columns (thread t
// adds columns t, t + 256, ...), so that a block reads whole, contiguous partial rows.
template <int J>
__global__ __launch_bounds__(256) void spmm_reduce_partials_wide_kernel(float *__restrict__ out,
                                                                        const float *__restrict__ partial,
                                                                        const uint4 *__restrict__ splits, uint32_t F,
                                                                        int accumulate, uint32_t ld) {
  const uint4 s = splits[blockIdx.x];
  const float *src = partial + static_cast<size_t>(s.y) * ld;
  uint32_t c[J];
  bool live[J];
  float a[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    c[j] = threadIdx.x + 256u * j;
    live[j] = c[j] < F;
    if (!live[j]) c[j] = F - 1;  // re-read the last column, never stored
  }
  add_partial_rows<J, kPartialRows<J>>(src, ld, s.z, c, a);
  float *dst = out + static_cast<size_t>(s.x) * F;
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (live[j]) dst[c[j]] = accumulate ? a[j] + dst[c[j]] : a[j];
}

// Launches the second stage for a plan's split rows.
inline void launch_reduce_partials(float *out, const float *partial, const uint4 *splits, uint32_t n_splits, uint32_t F,
                                   int accumulate, hipStream_t stream, uint32_t ld = 0) {
  if (!ld) ld = F;  // row stride of the partial sums
  // Up to 1,024 columns one block adds whole rows (contiguous reads: 29.6 -> 29.2 ms per step on the
  // Reddit-shaped F=602 workload); wider rows are tiled 256 columns per block.
#define NTS_REDUCE_WIDE(J)                                                                                          \
  hipLaunchKernelGGL(spmm_reduce_partials_wide_kernel<J>, dim3(n_splits), dim3(256), 0, stream, out, partial, splits, \
                     F, accumulate, ld)
  if (F > 256 && F <= 512)
    NTS_REDUCE_WIDE(2);
  else if (F > 512 && F <= 768)
    NTS_REDUCE_WIDE(3);
  else if (F > 768 && F <= 1024)
    NTS_REDUCE_WIDE(4);
  else
    hipLaunchKernelGGL(spmm_reduce_partials_kernel, dim3(n_splits, ceil_div(F, 256)), dim3(256), 0, stream, out, partial,
                       splits, F, accumulate, ld);
#undef NTS_REDUCE_WIDE
}

// Copy of a [rows, F] matrix with the row stride padded to `ld` floats (a multiple of four; the pad
// columns are zero), so that every row starts on a 16-byte boundary and the gather can use 16-byte
// lanes.  One thread per 16 bytes written.
__global__ __launch_bounds__(256) void pad_rows_kernel(float4 *__restrict__ dst, const float *__restrict__ src,
                                                       uint32_t rows, uint32_t F, uint32_t ld) {
  const uint32_t per_row = ld / 4;
  const uint64_t total = static_cast<uint64_t>(rows) * per_row;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint32_t r = static_cast<uint32_t>(i / per_row);
    const uint32_t c = static_cast<uint32_t>(i % per_row) * 4;
    const float *p = src + static_cast<size_t>(r) * F + c;
    float4 v;
    v.x = c + 0 < F ? p[0] : 0.f;
    v.y = c + 1 < F ? p[1] : 0.f;
    v.z = c + 2 < F ? p[2] : 0.f;
    v.w = c + 3 < F ? p[3] : 0.f;
    dst[i] = v;
  }
}

struct LaunchArgs {
  const float *in;
  float *out;
  const float *w;
  const uint32_t *offsets;
  const uint32_t *indices;
  uint32_t index_base;
  uint32_t n_items;
  uint32_t F;
  const Item *items;
  float *partial;
  int accumulate;
  hipStream_t stream;
  HeadArgs heads = HeadArgs{nullptr, 0u, 0u};  // H == 0: one weight per edge
  uint32_t row_edge_limit = 0xFFFFFFFFu;       // whole-row launches skip rows with more edges than this
  const uint32_t *edge_ids = nullptr;          // schedules with their own index copy: edge -> caller's edge position
  uint32_t in_ld = 0;                          // row stride of `in` in floats (0 = F)
  uint32_t partial_ld = 0;                     // row stride of `partial` in floats (0 = F)
  bool dup_runs = false;                       // rows hold runs of equal indices worth loading once per run
  uint32_t scheduled_rows = 0;                 // rows of the schedule that `items` comes from (0: no schedule)
  bool ranged = false;                         // a schedule with source ranges: rows are cut where these end
  uint32_t edges = 0;                          // edges of the rows, as the caller or the schedule has them
  bool bounded = false;                        // the caller knows that no row has more than kAutoChunk edges
  uint32_t rows_after_items = 0;               // with items: this many whole rows follow the listed items in the launch
  const float *dot_rows = nullptr;             // with dot_out: the rows whose products with the gathered ones
  float *dot_out = nullptr;                    // are the gradient of alpha (attention_grad_kernel)
};

// Lanes per head and vectors per lane of attention_grad_kernel for heads of `vecs` vectors; 16 lanes with up to
// four vectors each cover 64 vectors, wider heads are not its business.
constexpr uint32_t kGradMaxVecs = 64;
bool attention_grad_takes(const LaunchArgs &a) { return ceil_div(a.heads.Fh, a.heads.Fh >= 4 ? 4 : 1) <= kGradMaxVecs; }

// Rows off 16-byte boundaries: lanes of one float or of four that start at any float.  One float a lane spreads a step's
// products over more lanes, four take fewer registers and instructions for wide rows.  us, one float / four:
//   heads x floats   5 K rows, 40 K edges   20 K, 300 K   169 K, 2.48 M   1 M, 4 M     500 K, 20 M
//   1 x 5            62 / 99                40 / 48       113 / 120       195 / 219    928 / 950
//   1 x 17           86 / 94                47 / 49       130 / 135       277 / 235    1,031 / 1,014
//   4 x 10           66 / 91                47 / 49       175 / 161       614 / 404    1,575 / 1,266
//   1 x 47           --                     50 / 49       167 / 164       405 / 400    1,227 / 1,201
//   8 x 13           73 / 92                64 / 51       432 / 254       1,311 / 649  3,298 / 1,746
//   8 x 47           96 / 104               87 / 93       704 / 714       2,012 / 2,052
// Two and three heads of 33 to 48 floats take one float a lane where rows are short: 2 x 47 sampled layers 90 K rows, 156 K edges
// 46 / 48, 54 K, 118 K 44 / 45, but 169 K, 2.48 M 242 / 235; 3 x 47 60 / 63, 54 / 57, 1 M, 4 M 800 / 817, but 169 K 312 / 306.
// Heads of 65 to 256 floats of such rows took a pass per gradient: 1 x 101 127 -> 65 on 20 K, 622 -> 245, 1,458 -> 640, 4,713 -> 1,679.
bool grad_floats_are_faster(const LaunchArgs &a) {
  const uint32_t Fh = a.heads.Fh, rows = a.n_items + (a.items ? a.rows_after_items : 0u);
  if (Fh > kGradMaxVecs) return false;
  const uint64_t lanes = static_cast<uint64_t>(a.heads.H) * (Fh <= 4 ? 4 : Fh <= 8 ? 8 : ceil_div(Fh, 16) * 16);
  if (Fh < 4 || lanes <= 16 || (lanes <= 32 && rows <= 1u << 19)) return true;
  if (Fh > 32) return Fh <= 48 && (a.heads.H >= 4 || (a.heads.H >= 2 && a.edges < 8ull * rows));
  return rows <= (lanes <= 64 ? 1u << 15 : 1u << 13);
}

template <int G, int LH, int NJ, int VEC, bool SHARED>
void launch_attention_grad_as(const LaunchArgs &a) {
  const uint32_t n_list = a.items ? a.n_items : 0u, n_total = a.n_items + (a.items ? a.rows_after_items : 0u);
  const dim3 grid(ceil_div(n_total, 256 / G), ceil_div(a.heads.H, G / LH));
  hipLaunchKernelGGL((attention_grad_kernel<G, LH, NJ, VEC, SHARED>), grid, dim3(256), 0, a.stream, a.in, a.out, a.w, a.offsets,
                     a.indices, n_total, n_list, a.F, a.items, a.partial, a.accumulate, a.heads, a.row_edge_limit,
                     a.dot_rows, a.dot_out);
}

template <int LH, int NJ, int VEC, bool SHARED>
void launch_attention_grad_lanes(const LaunchArgs &a) {
  // As many heads side by side as there are, in groups of 8 (a tile of edge pairs is one per lane) to 64 lanes.
  const uint32_t H = a.heads.H;
  if constexpr (LH <= 8) {
    if (H * LH <= 8) return launch_attention_grad_as<8, LH, NJ, VEC, SHARED>(a);
  }
  if (H * LH <= 16) return launch_attention_grad_as<16, LH, NJ, VEC, SHARED>(a);
  if (H * LH <= 32) return launch_attention_grad_as<32, LH, NJ, VEC, SHARED>(a);
  return launch_attention_grad_as<64, LH, NJ, VEC, SHARED>(a);
}

template <int VEC, bool SHARED = false>
void launch_attention_grad(const LaunchArgs &a) {
  const uint32_t vecs = ceil_div(a.heads.Fh, VEC);
  // Lanes that a narrow head leaves idle are rows that the wavefront does not work on: eight heads of four floats
  // with four lanes each instead of one, 1.5 M vertices, 5 M edges 704 us, 459 now; two lanes for eight floats 762, 652.
  // (Not for heads of one or two floats: 30 K vertices, 300 K edges, eight heads of one 59 us, 70 with a lane each.)
  if constexpr (VEC == 4) {
    if (vecs <= 1) return launch_attention_grad_lanes<1, 1, VEC, SHARED>(a);
    if (vecs <= 2) return launch_attention_grad_lanes<2, 1, VEC, SHARED>(a);
  }
  if (vecs <= 4) return launch_attention_grad_lanes<4, 1, VEC, SHARED>(a);
  if (vecs <= 8) return launch_attention_grad_lanes<8, 1, VEC, SHARED>(a);
  if (vecs <= 16) return launch_attention_grad_lanes<16, 1, VEC, SHARED>(a);
  if (vecs <= 32) return launch_attention_grad_lanes<16, 2, VEC, SHARED>(a);
  if (vecs <= 48) return launch_attention_grad_lanes<16, 3, VEC, SHARED>(a);
  return launch_attention_grad_lanes<16, 4, VEC, SHARED>(a);
}

template <int VEC, int NACC>
void launch_wave(const LaunchArgs &a, uint32_t col_base, uint32_t panels) {
  constexpr int kWavesPerBlock = 4;
  const uint32_t n_list = a.items ? a.n_items : 0u, n_total = a.n_items + (a.items ? a.rows_after_items : 0u);
  const uint32_t blocks = ceil_div(n_total, kWavesPerBlock);
  const dim3 grid(blocks * panels), block(kWavesPerBlock * kWave);
  // Neighbour pairs always go through the wave-private LDS tile (a register-broadcast variant measured
  // the same: 12.44 ms against 12.40 ms for the 114.8 M-edge F=602 gather).
#define NTS_LAUNCH_WAVE(HD, RM, RUNS)                                                                                  \
  hipLaunchKernelGGL((spmm_wave_kernel<VEC, NACC, true, HD, RM, RUNS>), grid, block, 0, a.stream, a.in, a.out, a.w,    \
                     a.offsets, a.indices, a.index_base, n_total, n_list, a.F, col_base, panels, a.items, a.partial, \
                     a.accumulate,                                                                                     \
                     a.heads, a.row_edge_limit, a.edge_ids, a.in_ld ? a.in_ld : a.F,                                  \
                     a.partial_ld ? a.partial_ld : a.F,                                                                \
                     (VEC > 1 && (a.F % VEC != 0 || !aligned_to(a.out, 4 * VEC))) ? 1 : 0)
  if (a.edge_ids) {
    if (a.heads.H) NTS_LAUNCH_WAVE(true, true, false);
    else if (a.dup_runs) NTS_LAUNCH_WAVE(false, true, true);
    else NTS_LAUNCH_WAVE(false, true, false);
  } else {
    if (a.heads.H) NTS_LAUNCH_WAVE(true, false, false);
    else if (a.dup_runs) NTS_LAUNCH_WAVE(false, false, true);
    else NTS_LAUNCH_WAVE(false, false, false);
  }
#undef NTS_LAUNCH_WAVE
}

template <int G, int VEC, int U = 8, bool SHARED = false, bool PANELS = false>
void launch_group(const LaunchArgs &a, uint32_t panels = 1) {
  const uint32_t per_block = 256 / G;
  const uint32_t n_list = a.items ? a.n_items : 0u, n_total = a.n_items + (a.items ? a.rows_after_items : 0u);
  int panel_bits = -1;
  for (uint32_t bits = 0; bits < 3; ++bits)
    if (panels == 1u << bits) panel_bits = static_cast<int>(bits);
  // where panels do not alternate, whole turns of the XCDs (the last ones' surplus blocks leave at once)
  const uint32_t turn = PANELS && panel_bits < 0 ? kXcds : 1u;
  const uint32_t blocks = ceil_div(n_total, per_block * turn) * turn * panels;
#define NTS_LAUNCH_GROUP(HD, RM, RUNS)                                                                                  \
  hipLaunchKernelGGL((spmm_group_kernel<SHARED, PANELS, G, VEC, U, HD, RM, RUNS>), dim3(blocks), dim3(256), 0, a.stream, a.in, a.out, a.w, \
                     a.offsets, a.indices, a.index_base, n_total, n_list, a.F, a.items, a.partial, a.accumulate,        \
                     a.heads,                                                                                          \
                     a.row_edge_limit, a.edge_ids, panels, panel_bits, a.in_ld ? a.in_ld : a.F, a.partial_ld ? a.partial_ld : a.F)
  if constexpr (PANELS) {  // neither heads nor repeated indices (panel_lanes)
    if (a.edge_ids) NTS_LAUNCH_GROUP(false, true, false);
    else NTS_LAUNCH_GROUP(false, false, false);
  } else if (a.edge_ids) {
    if (a.heads.H) NTS_LAUNCH_GROUP(true, true, false);
    else if (a.dup_runs) NTS_LAUNCH_GROUP(false, true, true);
    else NTS_LAUNCH_GROUP(false, true, false);
  } else {
    if (a.heads.H) NTS_LAUNCH_GROUP(true, false, false);
    else if (a.dup_runs) NTS_LAUNCH_GROUP(false, false, true);
    else NTS_LAUNCH_GROUP(false, false, false);
  }
#undef NTS_LAUNCH_GROUP
}

constexpr uint32_t kChipWaves = 8192;                      // wavefronts that the chip holds
constexpr uint64_t kAllL2Bytes = 8ull * (4 << 20);         // the L2s of its eight XCDs

template <int VEC>
void launch_wave_vec(const LaunchArgs &a) {
  // Column panels of at most 10 accumulators per lane, balanced; wider rows are covered by several
  // launches over disjoint column ranges (each panel re-walks the edge list; outputs are disjoint), or, where one
  // panel does not fill the chip, by one launch whose blocks alternate between them.  us, apart / together, F = 1,433: 2.7 K
  // items 32 / 18, 5.2 K 35 / 23, 8.8 K 44 / 40, 21 K 78 / 86 (all panels of a row at once need more of the caches), 172 K 1,733 / 2,067.
  constexpr uint32_t kMaxAcc = 10;
  const uint32_t per_acc = kWave * VEC;
  const uint32_t total_acc = ceil_div(a.F, per_acc);
  const uint32_t panels = ceil_div(total_acc, kMaxAcc);
  const uint32_t acc_per_panel = ceil_div(total_acc, panels);
  const uint32_t n_total = a.n_items + (a.items ? a.rows_after_items : 0u);
  const bool together = panels > 1 && n_total <= kChipWaves;
  uint32_t col_base = 0;
  while (col_base < a.F) {
    const uint32_t remaining = a.F - col_base;
    uint32_t nacc = ceil_div(remaining, per_acc);
    if (nacc > acc_per_panel) nacc = acc_per_panel;
    switch (nacc) {
      case 1: launch_wave<VEC, 1>(a, col_base, together ? panels : 1u); break;
      case 2: launch_wave<VEC, 2>(a, col_base, together ? panels : 1u); break;
      case 3: launch_wave<VEC, 3>(a, col_base, together ? panels : 1u); break;
      case 4: launch_wave<VEC, 4>(a, col_base, together ? panels : 1u); break;
      case 5: launch_wave<VEC, 5>(a, col_base, together ? panels : 1u); break;
      case 6: launch_wave<VEC, 6>(a, col_base, together ? panels : 1u); break;
      case 7: launch_wave<VEC, 7>(a, col_base, together ? panels : 1u); break;
      case 8: launch_wave<VEC, 8>(a, col_base, together ? panels : 1u); break;
      case 9: launch_wave<VEC, 9>(a, col_base, together ? panels : 1u); break;
      default: launch_wave<VEC, 10>(a, col_base, together ? panels : 1u); break;
    }
    if (together) return;
    col_base += nacc * per_acc;
  }
}

// Vector width of the row loads: 16-byte lanes when every row starts 16-byte aligned (rows start
// at multiples of F floats from the base pointers), otherwise 4-byte lanes.  8-byte lanes are not
// used: measured on MI355X, dwordx2 gathers run ~20 % slower than either dword or dwordx4 gathers of
// the same bytes (F=512: 15.4 ms vs 12.8 / 11.7 ms; F=602: 18.8 ms vs 15.3 ms with dword lanes).
int pick_vec(const LaunchArgs &a) {
  const bool heads_ok = a.heads.H == 0 || a.heads.Fh % 4 == 0;  // a 16-byte lane must stay inside one head
  if (a.in_ld) {
    // Gather over a padded copy of the input (row stride a multiple of four floats): 16-byte lanes
    // whatever F is; output rows off a 16-byte boundary are stored float by float.
    const uint32_t pld = a.partial_ld ? a.partial_ld : a.F;
    if (a.in_ld % 4 == 0 && aligned_to(a.in, 16) && (!a.partial || (pld % 4 == 0 && aligned_to(a.partial, 16))) &&
        a.heads.H == 0)
      return 4;
    return 1;
  }
  const bool a16 = aligned_to(a.in, 16) && aligned_to(a.out, 16) && (!a.partial || aligned_to(a.partial, 16));
  if (a.F % 4 == 0 && a16 && heads_ok) return 4;
  return 1;
}

// Lanes of a column panel (16 or 32, of four floats each: panels of 256 or 512 bytes), or 0 for rows that are not cut into panels.
// An XCD meets one or two panels of a row only (three of eleven), so that its 4 MB L2 holds a share of the gathered matrix that is as many times
// smaller.  us without / with, panels of whole lines (the last one may be shorter):
//   rows          169 K, 2.48 M   60 K, 4 M   1 M, 6 M        20 M of 500 K   233 K, 114.8 M simple   2.45 M, 126 M (40 M)
//   128  2 x 16   111 / 98                                    722 / 690       2,651 / 2,660           5,221 / 5,108
//   192  3 x 16                   171 / 146                                                           (80 M 6,082 / 5,495)
//   256  2 x 32   251 / 221                                   1,437 / 1,388   4,871 / 4,852           11,255 / 10,386
//   320  5 x 16                   318 / 241   700 K, 7.5 M 1,316 / 1,157                              (80 M 10,590 / 9,121)
//   384  3 x 32   409 / 344       407 / 304   1,468 / 1,383   2,255 / 2,051   8,183 / 7,291           (7,496 / 6,924)
//   512  4 x 32   584 / 451                                   3,137 / 2,746
//   640  5 x 32                   773 / 523                                   1 M, 40 M 9,217 / 7,301 (80 M 23,238 / 19,127)
// Rows off whole lines are gathered from a copy padded to them where that pays (padded_stride), the copy included:
//   300  5 x 16   1 M, 40 M 4,226 / 4,275                     1,963 / 1,947   7,536 / 6,392           15,003 / 14,410
//   450  4 x 32   200 K, 12 M 1,587 / 1,518                   3,365 / 2,975   9,674 / 9,236           (80 M 16,989 / 16,514)
//   500  4 x 32   200 K, 12 M 1,803 / 1,588                   3,271 / 3,143   10,629 / 9,531          26,582 / 23,291
//   602  5 x 32   1 M, 24 M 6,430 / 6,062                     4,414 / 3,879   12,992 / 11,767         31,848 / 28,922
//   700  11 x 16  200 K, 12 M 2,562 / 2,261; 1 M, 40 M 10,888 / 9,437
// and without a copy, panels that share a line, by schedules without source ranges whose rows are wide and long: 450 60 K, 4 M
// 535 / 474, 500 20 K, 4 M 416 / 326, 602 757 / 651, 30 K, 600 K 129 / 108, 700 145 / 126; but 300 60 K, 4 M 330 / 376, 602 300 K, 3 M
// 1,036 / 1,098, 1 M, 6 M 2,573 / 2,915.  Shorter panels cost more than they give (64 bytes: 2.8 times the time, 128: as much as
// without), longer ones of 64 lanes lose too (602 233 K 15,300, 500 9,900).  Without them stay:
//   rows of 512 bytes that the L2s hold together (20 K rows, 4 M edges 93 / 95; wider rows gain there too: F = 256 and 512 2 K, 8 K
//     11.4 / 11.5, 12.0 / 11.1, 5 K, 60 K 14.3 / 14.2, 18.1 / 16.9, 20 K, 300 K 33 / 32, 58 / 51, 60 K, 600 K 60 / 55, 124 / 96)
//   rows of 160 and 224 floats, whose last panel is half idle: 2.45 M, 40 M 3,111 / 3,302, 1 M, 40 M 2,764 / 2,825
//   rows with fewer than five edges each once they fill the chip, which are read once or twice whatever the caches hold,
//     while every panel walks the short rows again: F = 512 32 K, 100 K 34 / 37, 130 K, 300 K 126 / 139, 300 K, 600 K 267 / 290, 2.45 M, 5 M
//     2,402 / 2,667, 10 M 3,782 / 4,042; but 2 K, 8 K 12 / 10, 300 K, 1.5 M 492 / 438, 600 K, 3 M 1,008 / 985; and rows of other widths
//     that do not fill it (2 K, 16 K F = 192 to 640 13 / 14)
//   rows loaded once per run of equal indices (233 K, 114.8 M F = 128 2,277 / 2,346; 100 K, 40 M F = 602 3,399 / 3,707), heads (169 K
//     155 / 199: the weights are read once a panel) and calls without a schedule (133 / 149: mostly short rows)
constexpr uint32_t kMinPanelEdges = 5;                     // edges a row
// Panels of 512 bytes, or of 256 where they leave fewer lanes idle.
uint32_t lanes_for_lines(uint32_t lines) { return lines % 4 == 1 || lines % 4 == 2 ? 16u : 32u; }
constexpr uint32_t kMaxPanelLines = 24;                    // (wider rows were not measured)
uint32_t panel_lanes(const LaunchArgs &a, int vec) {
  if (!a.scheduled_rows || a.heads.H || a.dup_runs) return 0;
  const uint32_t lines = ceil_div(a.F, 32);
  if (static_cast<uint64_t>(a.n_items) * (lines + 4) * 8 >= 0xF0000000ull) return 0;  // (a launch has fewer than 2^32 threads)
  const bool full = a.n_items > kChipWaves, sparse = a.edges < static_cast<uint64_t>(kMinPanelEdges) * a.scheduled_rows;
  if (a.in_ld) return lines <= kMaxPanelLines ? lanes_for_lines(lines) : 0u;
  if (vec == 4 && a.F % 32 == 0) {
    if (a.F == 128) return static_cast<uint64_t>(a.scheduled_rows) * a.F * sizeof(float) > kAllL2Bytes ? 16u : 0u;
    if (a.F == 256) return 32;
    if (a.F == 512) return full && sparse ? 0u : 32u;
    return lines >= 6 && lines != 7 && lines <= kMaxPanelLines && full && !sparse ? lanes_for_lines(lines) : 0u;
  }
  return !a.ranged && a.F >= 448 && lines <= kMaxPanelLines && a.n_items > 2 * kChipWaves && a.edges >= 20ull * a.scheduled_rows ? 32u : 0u;
}

// Lanes of a narrow row.  A group of G lanes fetches G edge pairs at a time and works on one row, so what counts is how
// long the rows are and how many of them there are:
//   lanes of one float (16 or 32 a row, 64 up to 64 floats) put fewer rows into a wavefront and request more edges of a
//     row at once: for launches that last as long as their longest rows or pieces, or that do not fill the chip;
//   lanes of four floats take fewer instructions a row: where there are many rows.
// Rows off 16-byte boundaries take the latter too (SHARED), a wavefront of 4-byte lanes otherwise.
enum NarrowLanes {
  kFloats4, kFloats8, kFloats16, kFloats16x16, kFloats32, kFloats32x16, kFloats64, kVectors4, kVectors8, kVectors16, kVectors32, kVectors64, kWide
};
struct RowShape {
  uint32_t rows, F, lanes;          // lanes: of four floats that a row takes
  uint64_t edges;
  bool vectors, aligned;            // rows (heads) of four floats and more; of 16-byte boundaries throughout
  bool longer(uint64_t n) const { return edges >= n * rows; }  // rows of n edges and more on average
};
NarrowLanes fewest_lanes(const RowShape &s) {
  if (!s.vectors) return s.F <= 4 ? kFloats4 : s.F <= 8 ? kFloats8 : s.F <= 16 ? kFloats16 : s.F <= 32 ? kFloats32 : kWide;
  if (s.lanes <= 4) return kVectors4;
  if (s.lanes <= 8) return kVectors8;
  if (s.lanes <= 16) return kVectors16;
  return s.lanes <= 32 ? kVectors32 : kWide;
}

// Rows of a schedule, whose long rows are pieces of their own.  Every line below was measured over 24 graphs of 2 K to 2.4 M
// rows and 2 to 200 edges a row, in turn over several sets of arrays; us, four floats a lane (the fewest lanes) / others:
//   F = 16   eight lanes of four (each row's half idle): 100 K rows, 300 K edges 18 -> 16, 1 M, 3 M 89 -> 59, 2.4 M, 6 M 256 -> 174; from
//            eight edges a row 16 lanes of one float: 60 K, 600 K 25 -> 18, 169 K, 2.48 M 70 -> 33, and there 16 edges a step from
//            twelve edges a row (169 K 35 -> 33, 300 K, 4.5 M 63 -> 53; 1 M, 8 M 112 -> 118); up to 65,536 rows one float in any case
//            (20 K, 60 K 11.6 -> 10.5, but 169 K, 500 K 18.6 -> 21)
//   F = 7    8 lanes of one float, 16 from eight edges a row: 300 K, 900 K 24, 27, 300 K, 4.5 M 79, 62; 5 K, 1 M 28, 30
//   F = 32   8 lanes of four.  16 lanes 300 K, 4.5 M 98 -> 80, 169 K, 2.48 M 50 -> 44, but 500 K, 20 M 244 -> 262, 500 K, 1.5 M 49 -> 52; 32
//            of one float 20 K, 60 K 11.9 -> 10.9, but 100 K, 300 K 16 -> 21, 300 K, 900 K 34 -> 43, 500 K, 1.5 M 49 -> 65
//   F = 31   32 lanes of one float 20 K, 60 K 11.7, eight of four 13.3, 16 12.5; 100 K, 300 K 22, 19, 20; 300 K, 4.5 M 100, 127, 104; 50 K,
//            8 M 103, 106, 100; 200 K, 1.7 M 51, 55, 49, 200 K, 7 M 112, 149, 123, 50 K, 4.5 M 65, 80, 71 (F = 21 101, 126, 107 and 64, 74, 66,
//            but 100 K, 4 M 61, 60, 54); with repeated edges 100 K, 20 M F = 17 276, 238, 256
//   F = 64   16 lanes of four; a wavefront 100 K, 300 K 21 -> 32, 60 K, 600 K 24 -> 32
//   F = 47   a wavefront of 4-byte lanes / 16 of four: 300 K, 900 K 75, 44, 120 K, 7.5 M 134, 128, 50 K, 3.2 M 59, 60, 50 K, 4.5 M 69, 80, 20 K,
//            2.3 M 40, 43, 50 K, 8 M 102, 110; with source ranges 20 K, 1.8 M 41, 45, 34 K, 6.5 M 115, 117 (F = 33 106, 102), 120 K, 6.4 M 145,
//            141, 100 K, 16.4 M 283, 264, with repeated edges too 100 K, 20 M 650, 261
//   F = 127  a wavefront / 32 of four: 169 K, 500 K 77, 69, 50 K, 2 M 80, 79, 120 K, 7.5 M 272, 292, 90 K, 8 M 267, 286, 50 K, 8 M 207, 221 (F = 90
//            120 K, 7.5 M 195, 200, 90 K, 8 M 195, 197); with source ranges 34 K, 6.5 M 206, 192, 500 K, 20 M with repeated edges 1,050, 861
//   F = 201  64 lanes of four 8 K, 30 K 15.6 -> 12.8, 20 K, 3 M 130 -> 119; but 50 K, 8 M 324 -> 363, and F = 129 20 K, 3 M 88 -> 103
NarrowLanes scheduled_lanes(const RowShape &s, bool ranged, bool dup_runs) {
  const bool large = s.edges > 1u << 20, few = s.rows <= 1u << 15;
  if (s.F <= 16) {
    if (s.longer(8)) return s.F <= 8 && !large && s.longer(64) ? kFloats8 : large && s.longer(12) ? kFloats16x16 : kFloats16;
    if (s.rows <= 1u << 16) return kFloats16;
    return s.F <= 8 ? kFloats8 : s.vectors ? kVectors8 : kFloats16;
  }
  if (!s.vectors) return fewest_lanes(s);
  if (s.F <= 32) {
    const bool one = few || (s.lanes > 6 && s.longer(16) && !dup_runs);
    if ((few && !s.longer(8)) || (one && !s.aligned && !s.longer(128))) return kFloats32;
    const bool sixteen = large && s.longer(8) && (s.aligned ? !s.longer(32) : !dup_runs || !s.longer(64));
    return sixteen || s.lanes > 8 ? kVectors16 : kVectors8;
  }
  if (s.lanes <= 16) return !s.aligned && s.longer(64) && (few ? !dup_runs : !ranged) ? kWide : kVectors16;
  if (s.lanes <= 32) return !s.aligned && s.longer(32) && s.lanes > 24 && !ranged ? kWide : kVectors32;
  return !s.aligned && few && s.lanes >= 48 && s.lanes <= 64 ? kVectors64 : kWide;
}

// Calls without a schedule.  `bounded`: the caller knows that no row is long (sampled layers), so one launch of whole rows;
// `pieces` > 0: rows above 256 edges are cut into up to so many; otherwise a launch of whole rows among which one may be
// long, and lasts as long as that one.  Measured on sampled layers of R-MAT graphs, their transposed structures, and whole
// graphs; us, the fewest lanes / others:
//   bounded     F = 16 1 K rows, 5 K edges 6.2 -> 4.1 with 16 of one float, 28 K, 272 K 7.3 -> 6.8; but 133 K, 655 K 12 -> 14; F = 64 1 K
//               4.9 -> 4.2 with a wavefront; but 16 K, 156 K 8.2 -> 10.2, 32 K of five 6.9 -> 14; F = 32 with 32 of one 5 K, 118 K 6.9 ->
//               5.1; but 28 K 7.8 -> 8.4, 32 K of five 6.0 -> 6.5; F = 201 64 of four 133 K 97 -> 93, but 5 K, 118 K 15 -> 16
//   whole rows  F = 16 5 K, 40 K 107 -> 41 with 16 of one float and 16 edges a step; F = 32 68 -> 36 with 32; F = 64 56 -> 37 with a
//               wavefront; sources of a sampled layer 28 K, 37 K 8.9 -> 10.6; F = 201 78 -> 30 with 64 of four
//   pieces      F = 16 60 K, 600 K 63 -> 41, 300 K, 4.5 M 177 -> 166; 1 M, 3 M 131 -> 133; F = 8 255 K, 343 K 59 -> 37; F = 7 eight lanes
//               of one 169 K, 2.48 M 67, 16 73; F = 32 60 K, 600 K 51 -> 45 with 32 of one; but 169 K 82 -> 90; F = 17 100 K, 300 K with
//               eight of four 41 -> 47, 256 K, 343 K 46 -> 47, 1 M, 3 M 172 -> 131; F = 47 32 K, 100 K with 16 of four 32 -> 39, 54 K, 118 K
//               33 -> 30, 300 K, 900 K 102 -> 69; F = 201 64 of four 89 K, 156 K 69 -> 51, but rows of 1.4 edges 117 -> 124
NarrowLanes plain_lanes(const RowShape &s, bool bounded, uint32_t pieces) {
  const uint32_t items = s.rows + pieces;
  const bool mostly_pieces = pieces > s.rows;
  if (s.F <= 16) {
    if (bounded) {
      if (s.rows <= 1u << 15) return kFloats16;
      return s.F <= 4 ? kFloats4 : s.F <= 8 ? kFloats8 : s.aligned ? fewest_lanes(s) : kFloats16;
    }
    if (s.F <= 8 && pieces && (mostly_pieces || items > 1u << 18 || s.edges > 1u << 20)) return s.F <= 4 ? kFloats4 : kFloats8;
    if (s.vectors && (mostly_pieces || items > 1u << 19)) return fewest_lanes(s);
    return items <= 1u << 14 ? kFloats16x16 : kFloats16;
  }
  if (!s.vectors) return fewest_lanes(s);
  if (s.F <= 32) {
    if (bounded) {
      if (s.rows <= 1u << (s.aligned ? 14 : 15)) return kFloats32;
      return !s.aligned && s.rows <= 1u << 16 ? kVectors16 : fewest_lanes(s);
    }
    const bool floats = items <= 1u << (pieces ? 16 : 15) ||
                        (!s.aligned && !mostly_pieces && s.rows <= 1u << (s.longer(2) ? 17 : 18));
    return !floats ? fewest_lanes(s) : items <= 1u << 14 && s.longer(2) ? kFloats32x16 : kFloats32;
  }
  if (s.F <= 64) {
    const bool floats = bounded ? s.rows <= 1u << 11 : pieces ? s.rows <= 1u << 15 && (!s.aligned || s.longer(8)) : s.rows <= 3u << 13;
    return floats ? kFloats64 : fewest_lanes(s);
  }
  if (s.lanes <= 32 || s.lanes > 64 || s.aligned || mostly_pieces || items > 3u << 17) return fewest_lanes(s);
  return (bounded ? !s.longer(16) : pieces ? 2 * s.edges >= 3ull * s.rows : s.rows <= 1u << 15) ? kVectors64 : kWide;
}

NarrowLanes narrow_lanes(const LaunchArgs &a, int vec) {
  const uint32_t H = a.heads.H ? a.heads.H : 1u, width = a.heads.H ? a.heads.Fh : a.F;
  const uint32_t n_total = a.n_items + (a.items ? a.rows_after_items : 0u);
  RowShape s{n_total, a.F, 0u, a.edges, width >= 4, vec == 4};
  const uint64_t lanes = static_cast<uint64_t>(H) * ceil_div(width, 4);
  s.lanes = lanes > 64 ? 65u : static_cast<uint32_t>(lanes);
  if (n_total >= 1u << 28) return fewest_lanes(s);  // 16 lanes a row would be more threads than a launch can have
  if (a.scheduled_rows) {
    s.rows = a.scheduled_rows;
    return scheduled_lanes(s, a.ranged, a.dup_runs);
  }
  const uint32_t pieces = a.items ? a.n_items : 0u;
  s.rows = n_total - pieces;
  return plain_lanes(s, a.bounded, pieces);
}

void launch_spmm(const LaunchArgs &a) {
  if (a.n_items == 0) return;
  if (a.dot_out) {
    const bool a16 = aligned_to(a.in, 16) && aligned_to(a.out, 16) && aligned_to(a.dot_rows, 16);
    if (a.heads.Fh % 4 == 0 && a16) return launch_attention_grad<4>(a);
    return grad_floats_are_faster(a) ? launch_attention_grad<1>(a) : launch_attention_grad<4, true>(a);
  }
  const int vec = pick_vec(a);
  const uint32_t F = a.F;
  if (const uint32_t lanes = panel_lanes(a, vec)) {
    const uint32_t panels = ceil_div(F, lanes * 4);
    if (F % 4 == 0 && vec == 4 && aligned_to(a.out, 16)) return lanes == 16 ? launch_group<16, 4, 8, false, true>(a, panels) : launch_group<32, 4, 8, false, true>(a, panels);
    return lanes == 16 ? launch_group<16, 4, 8, true, true>(a, panels) : launch_group<32, 4, 8, true, true>(a, panels);
  }
  if (!a.in_ld) {
    switch (narrow_lanes(a, vec)) {
      case kFloats4: return launch_group<4, 1, 4>(a);
      case kFloats8: return launch_group<8, 1>(a);
      case kFloats16: return launch_group<16, 1>(a);
      case kFloats16x16: return launch_group<16, 1, 16>(a);
      case kFloats32: return launch_group<32, 1>(a);
      case kFloats32x16: return launch_group<32, 1, 16>(a);
      case kVectors4: return vec == 4 ? launch_group<4, 4, 4>(a) : launch_group<4, 4, 4, true>(a);
      case kVectors8: return vec == 4 ? launch_group<8, 4>(a) : launch_group<8, 4, 8, true>(a);
      case kVectors16: return vec == 4 ? launch_group<16, 4>(a) : launch_group<16, 4, 8, true>(a);
      case kVectors32: return vec == 4 ? launch_group<32, 4>(a) : launch_group<32, 4, 8, true>(a);
      case kVectors64: return launch_group<64, 4, 8, true>(a);
      case kFloats64: return launch_wave_vec<1>(a);
      case kWide: break;
    }
  }
  // Wave per row.
  if (vec == 4) return launch_wave_vec<4>(a);
  return launch_wave_vec<1>(a);
}

// ---- launches without a plan: hub rows are cut into pieces on the device ---------------------------
//
// A call that brings no plan still must not let one wavefront walk a 10^5-edge row alone.  For edge
// counts where that can matter, the pieces are derived on the device in the same stream, without
// any copy to the host: pieces[r] = ceil(deg/chunk) for rows longer than `chunk` = 256 edges (else 0), an
// exclusive scan gives each long row its first partial slot, one thread per possible piece writes
// the work item (binary search of the scan), whole-row wavefronts skip the long rows, the piece
// wavefronts write partial sums and a last kernel adds each long row's partials in slot order.
// The number of pieces is not known on the host, so grids and buffers are sized for its upper bound
// E/chunk + min(rows, E/chunk); surplus work items are empty.  Scratch is stream-ordered
// (hipMallocAsync / hipFreeAsync).  Calls below kAutoLargeEdges take the pieces' slots from a counter
// instead of a scan (launch_spmm_cut_small).

constexpr uint32_t kAutoMinEdges = 1u << 16;  // below this a serial hub row costs less than the set-up
// Piece length.  Shorter pieces mean more partial rows but also narrower index spans per piece
// (rows ascend), hence better locality once the pieces are ordered by source, and more parallelism
// for calls with few long rows: on the 114.8 M-edge graph at F=602 1,024-edge pieces take 18.9 ms,
// 256-edge pieces 16.3 ms; a 2.3 M-edge sampled layer has only 2,300 pieces of 1,024 edges.
constexpr uint32_t kAutoChunk = 256;
// Calls below this many edges (sampled layers) skip the ordering of the pieces by source: their
// source rows fit the caches anyway and every launch saved counts at this size.
constexpr uint32_t kAutoLargeEdges = 1u << 22;

// Pieces of row r: 0 for a row that fits one wavefront, else ceil(degree / chunk); 0 for r == rows,
// so that the exclusive scan's last entry is the total.  Evaluated inside the scan (no launch and no
// array of its own).
struct PieceCount {
  const uint32_t *off;
  uint32_t rows, chunk;
  __host__ __device__ uint32_t operator()(uint32_t r) const {
    if (r >= rows) return 0u;
    const uint32_t deg = off[r + 1] - off[r];
    return deg > chunk ? (deg + chunk - 1) / chunk : 0u;
  }
};
using PieceCountIterator = rocprim::transform_iterator<rocprim::counting_iterator<uint32_t>, PieceCount, uint32_t>;

// Also writes keys[i] = the gather index of the piece's first edge (0xFFFFFFFF for an empty item):
// the pieces are then issued in ascending key order, so that wavefronts resident at the same time
// gather from nearby source rows (with sorted adjacency a piece covers a narrow index range).
__global__ __launch_bounds__(256) void auto_items_kernel(Item *__restrict__ items, uint32_t *__restrict__ keys,
                                                         const uint32_t *__restrict__ base,
                                                         const uint32_t *__restrict__ off,
                                                         const uint32_t *__restrict__ indices, uint32_t index_base,
                                                         uint32_t rows, uint32_t chunk, uint32_t p_max) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p_max) return;
  if (i >= base[rows]) {
    items[i] = make_uint4(0u, 0u, 0u, i);  // empty item: writes zeros to its own unused slot
    keys[i] = 0xFFFFFFFFu;
    return;
  }
  const uint32_t r = owner_of(base, rows, i);  // the last row whose first slot is <= i is the long row itself
  const uint32_t e0 = off[r] + (i - base[r]) * chunk;
  items[i] = make_uint4(r, e0, min(off[r + 1], e0 + chunk), i);
  keys[i] = indices[e0] - index_base;
}

__global__ __launch_bounds__(256) void auto_order_items_kernel(Item *__restrict__ ordered,
                                                               const Item *__restrict__ items,
                                                               const uint32_t *__restrict__ order, uint32_t p_max) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < p_max) ordered[j] = items[order[j]];
}

// Block (x, y): if work item x is the first piece of its row, adds that row's partials in slot order
// into out (256 columns per block, tile y).
__global__ __launch_bounds__(256) void auto_reduce_kernel(float *__restrict__ out, const float *__restrict__ partial,
                                                          const Item *__restrict__ items,
                                                          const uint32_t *__restrict__ base, uint32_t F,
                                                          int accumulate, uint32_t p_max) {
  const uint32_t i = blockIdx.x;
  const uint32_t r = items[i].x;
  if (base[r] != i) return;
  // Slots at or beyond p_max were never written (only possible when the caller's edge count is
  // smaller than offsets[rows]): they are not read.
  const uint32_t n = min(base[r + 1], p_max) - i;
  if (n == 0) return;
  const uint32_t c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= F) return;
  const uint32_t col[1] = {c};
  float a[1];
  add_partial_rows<1, kPartialRows<1>>(partial + static_cast<size_t>(i) * F, F, n, col, a);
  float *dst = out + static_cast<size_t>(r) * F + c;
  *dst = accumulate ? a[0] + *dst : a[0];
}

// The same with one block per work item covering all columns (rows of up to 1,024 columns): whole,
// contiguous partial rows are read, and a third or a quarter as many blocks are launched.
template <int J>
__global__ __launch_bounds__(256) void auto_reduce_wide_kernel(float *__restrict__ out,
                                                               const float *__restrict__ partial,
                                                               const Item *__restrict__ items,
                                                               const uint32_t *__restrict__ base, uint32_t F,
                                                               int accumulate, uint32_t p_max) {
  const uint32_t i = blockIdx.x;
  const uint32_t r = items[i].x;
  if (base[r] != i) return;
  const uint32_t n = min(base[r + 1], p_max) - i;  // as in auto_reduce_kernel
  if (n == 0) return;
  const float *src = partial + static_cast<size_t>(i) * F;
  uint32_t c[J];
  bool live[J];
  float a[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    c[j] = threadIdx.x + 256u * j;
    live[j] = c[j] < F;
    if (!live[j]) c[j] = F - 1;  // re-read the last column, never stored
  }
  add_partial_rows<J, kPartialRows<J>>(src, F, n, c, a);
  float *dst = out + static_cast<size_t>(r) * F;
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (live[j]) dst[c[j]] = accumulate ? a[j] + dst[c[j]] : a[j];
}

inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }

// Calls below kAutoLargeEdges (sampled layers) need no order among the pieces, so they need no scan
// either: a long row takes its consecutive partial slots from a counter (integer atomic: which slots a
// row gets varies from call to call, the order of its pieces inside them and therefore every sum does
// not), and lists itself for the second stage.
//   ctr[0] = slots handed out, ctr[1] = rows listed (one 64-bit counter).  Items are pre-filled as empty, so the slots beyond
//   the live count cost a wavefront that writes zeros to a slot nobody reads.
__global__ __launch_bounds__(256) void auto_fill_kernel(Item *__restrict__ items, uint32_t *__restrict__ ctr,
                                                        uint32_t p_max) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 2) ctr[i] = 0;
  if (i < p_max) items[i] = make_uint4(0u, 0u, 0u, i);
}

// A block asks for the slots of its 1,024 rows at once, because requests to one counter are served some 10 ns apart, and
// the lanes of a wavefront write its rows' pieces one each, wherever they belong: a hub row of 20,000 edges is 80
// pieces, which one thread wrote one after the other (2.48 M edges, 169 K rows: 20.7 -> 4.9 us; a request per
// wavefront is slower).  Most blocks and wavefronts of a sampled layer have no row to cut and leave after one look:
// with a prefix over the block for every one of them 90 K rows took 5.0 us instead of 3.9.
constexpr int kCutBlock = 1024;
__global__ __launch_bounds__(kCutBlock) void auto_cut_kernel(Item *__restrict__ items, uint4 *__restrict__ splits,
                                                             uint32_t *__restrict__ ctr,
                                                             const uint32_t *__restrict__ off, uint32_t rows,
                                                             uint32_t chunk, uint32_t p_max, uint32_t s_max) {
  // Slots (low half) and rows (high half) that the block's wavefronts ask for, and where the block's start.
  __shared__ unsigned long long asked, places_of_block;
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & (kWave - 1);
  const uint32_t b = off[r < rows ? r : rows], e = off[r < rows ? r + 1 : rows], deg = e - b;
  const uint32_t n = deg > chunk ? (deg + chunk - 1) / chunk : 0u;
  if (threadIdx.x == 0) asked = 0;
  __syncthreads();
  const uint64_t cut = __ballot(n != 0);
  uint32_t upto = n;  // pieces of the wavefront's rows up to this one
  unsigned long long before_wave = 0;
  if (cut) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const uint32_t up = __shfl_up(upto, d, kWave);
      if (lane >= static_cast<uint32_t>(d)) upto += up;
    }
    if (lane == kWave - 1) before_wave = atomicAdd(&asked, static_cast<unsigned long long>(__popcll(cut)) << 32 | upto);
  }
  __syncthreads();
  if (asked == 0) return;
  if (threadIdx.x == 0)  // both counters at once: rows are listed in the order of their slots
    places_of_block = atomicAdd(reinterpret_cast<unsigned long long *>(ctr), asked);
  __syncthreads();
  if (!cut) return;
  const unsigned long long places = places_of_block + before_wave;  // (the last lane's)
  const uint32_t wave_slot = wave_read(static_cast<uint32_t>(places), kWave - 1);
  const uint32_t wave_place = wave_read(static_cast<uint32_t>(places >> 32), kWave - 1);
  const uint32_t first = wave_slot + upto - n, s = wave_place + __popcll(cut & ((1ull << lane) - 1ull));
  // Slots at or beyond p_max do not exist (only possible when the caller's edge count is smaller than
  // offsets[rows]): such pieces are not created, and a row without any is listed with none, so that every entry that
  // the second stage reads was written.  A row with a slot always finds a place: the rows before it in the list took
  // two slots each at least, and p_max <= 2 s_max - 1 or every row has a place.
  if (n != 0 && s < s_max)
    splits[s] = first < p_max ? make_uint4(r, first, min(n, p_max - first), 0u) : make_uint4(0u, 0u, 0u, 0u);
  const uint32_t total = wave_read(upto, kWave - 1);
  for (uint32_t t0 = 0; t0 < total; t0 += kWave) {
    const uint32_t t = t0 + lane;
    uint32_t own = 0;  // lanes whose pieces all lie before piece t
#pragma unroll
    for (uint32_t step = kWave / 2; step >= 1; step >>= 1)
      if (__shfl(upto, own + step - 1, kWave) <= t) own += step;
    const uint32_t before = __shfl(upto - n, own, kWave), rb = __shfl(b, own, kWave), re = __shfl(e, own, kWave);
    const uint32_t at = wave_slot + t, e0 = rb + (t - before) * chunk;
    if (t < total && at < p_max) items[at] = make_uint4(r - lane + own, e0, min(re, e0 + chunk), at);
  }
}

// Block (x, y): adds the partials of listed row x in slot order into out (256 columns per block, tile y).
__global__ __launch_bounds__(256) void auto_reduce_listed_kernel(float *__restrict__ out,
                                                                 const float *__restrict__ partial,
                                                                 const uint4 *__restrict__ splits,
                                                                 const uint32_t *__restrict__ ctr, uint32_t F,
                                                                 int accumulate, uint32_t s_max) {
  const uint32_t live = ctr[1] < s_max ? ctr[1] : s_max;
  if (blockIdx.x >= live) return;
  const uint4 sp = splits[blockIdx.x];
  const uint32_t c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= F || sp.z == 0) return;
  const uint32_t col[1] = {c};
  float a[1];
  add_partial_rows<1, kPartialRows<1>>(partial + static_cast<size_t>(sp.y) * F, F, sp.z, col, a);
  float *dst = out + static_cast<size_t>(sp.x) * F + c;
  *dst = accumulate ? a[0] + *dst : a[0];
}

int launch_spmm_cut_small(const LaunchArgs &a, uint32_t edges, unsigned char *fixed, size_t fixed_cap) {
  const uint32_t rows = a.n_items;
  const uint32_t chunk = kAutoChunk;
  const uint32_t by_edges = edges / chunk;
  const uint32_t s_max = (rows < by_edges ? rows : by_edges) + 1;  // rows of more than `chunk` edges
  const uint32_t p_max = by_edges + s_max;
  const size_t n_items_b = up256(static_cast<size_t>(p_max) * sizeof(Item));
  const size_t n_splits_b = up256(static_cast<size_t>(s_max) * sizeof(uint4));
  const size_t n_partial = up256(static_cast<size_t>(p_max) * a.F * sizeof(float));
  const size_t need = 256 + n_items_b + n_splits_b + n_partial;
  unsigned char *buf = fixed;
  if (fixed) {
    if (need > fixed_cap) {
      char msg[200];
      snprintf(msg, sizeof msg, "spmm: the call needs %zu bytes of scratch, the fixed scratch holds %zu", need,
               fixed_cap);
      return fail(NTS_ERR_INVALID, msg);
    }
  } else {
    NTS_HIP_TRY(scratch_alloc(reinterpret_cast<void **>(&buf), need, a.stream));
  }
  uint32_t *ctr = reinterpret_cast<uint32_t *>(buf);
  Item *items = reinterpret_cast<Item *>(buf + 256);
  uint4 *splits = reinterpret_cast<uint4 *>(buf + 256 + n_items_b);
  float *partial = reinterpret_cast<float *>(buf + 256 + n_items_b + n_splits_b);
  hipLaunchKernelGGL(auto_fill_kernel, dim3(ceil_div(p_max, 256)), dim3(256), 0, a.stream, items, ctr, p_max);
  hipLaunchKernelGGL(auto_cut_kernel, dim3(ceil_div(rows, kCutBlock)), dim3(kCutBlock), 0, a.stream, items, splits, ctr, a.offsets,
                     rows, chunk, p_max, s_max);
  LaunchArgs pc = a;
  pc.n_items = p_max;
  pc.items = items;
  pc.partial = partial;
  pc.rows_after_items = rows;
  pc.row_edge_limit = chunk;
  launch_spmm(pc);
  hipLaunchKernelGGL(auto_reduce_listed_kernel, dim3(s_max, ceil_div(a.F, 256)), dim3(256), 0, a.stream, a.out, partial,
                     splits, ctr, a.F, a.accumulate, s_max);
  const hipError_t err = hipGetLastError();
  if (!fixed) {
    const hipError_t freed = scratch_free(buf, a.stream);
    if (err == hipSuccess && freed != hipSuccess) return fail_hip(freed, "spmm: scratch");
  }
  if (err != hipSuccess) return fail_hip(err, "spmm: balanced launch");
  return NTS_OK;
}

// `a` describes the whole-row launch (a.n_items = rows, no items).  Scratch comes from the library's
// stream-ordered pool, or, when `fixed` is set, from that caller-held region of `fixed_cap` bytes
// (nothing is allocated or freed then; a call that needs more is refused).
int launch_spmm_balanced(LaunchArgs a, uint32_t edges, unsigned char *fixed = nullptr, size_t fixed_cap = 0) {
  const uint32_t rows = a.n_items;
  a.edges = edges;
  if (edges < kAutoMinEdges) {
    launch_spmm(a);
    return NTS_OK;
  }
  const bool large = edges >= kAutoLargeEdges;
  if (!large) return launch_spmm_cut_small(a, edges, fixed, fixed_cap);
  const uint32_t chunk = kAutoChunk;
  const uint32_t by_edges = edges / chunk;
  const uint32_t p_max = by_edges + (rows < by_edges ? rows : by_edges) + 1;
  size_t scan_bytes = 0, sort_bytes = 0;
  {
    uint32_t *nul = nullptr;
    PieceCountIterator none(rocprim::counting_iterator<uint32_t>(0u), PieceCount{nullptr, 0u, chunk});
    NTS_HIP_TRY(rocprim::exclusive_scan(nullptr, scan_bytes, none, nul, 0u, static_cast<size_t>(rows) + 1,
                                        rocprim::plus<uint32_t>(), a.stream, false));
    NTS_HIP_TRY(rocprim::radix_sort_pairs(nullptr, sort_bytes, nul, nul, rocprim::counting_iterator<uint32_t>(0u), nul,
                                          p_max, 0u, 32u, a.stream, false));
  }
  const size_t tmp_bytes = up256(scan_bytes > sort_bytes ? scan_bytes : sort_bytes);
  const size_t n_off = up256((static_cast<size_t>(rows) + 1) * sizeof(uint32_t));
  const size_t n_items_b = up256(static_cast<size_t>(p_max) * sizeof(Item));
  const size_t n_keys_b = up256(static_cast<size_t>(p_max) * sizeof(uint32_t));
  const size_t n_partial = up256(static_cast<size_t>(p_max) * a.F * sizeof(float));
  const size_t need = n_off + 2 * n_items_b + 3 * n_keys_b + tmp_bytes + n_partial;
  unsigned char *buf = fixed;
  if (fixed) {
    if (need > fixed_cap) {
      char msg[200];
      snprintf(msg, sizeof msg, "spmm: the call needs %zu bytes of scratch, the fixed scratch holds %zu", need,
               fixed_cap);
      return fail(NTS_ERR_INVALID, msg);
    }
  } else {
    NTS_HIP_TRY(scratch_alloc(reinterpret_cast<void **>(&buf), need, a.stream));
  }
  unsigned char *cursor = buf;
  auto take = [&cursor](size_t bytes) {
    unsigned char *p = cursor;
    cursor += bytes;
    return p;
  };
  uint32_t *base = reinterpret_cast<uint32_t *>(take(n_off));
  Item *items = reinterpret_cast<Item *>(take(n_items_b));
  Item *ordered = reinterpret_cast<Item *>(take(n_items_b));
  uint32_t *keys = reinterpret_cast<uint32_t *>(take(n_keys_b));
  uint32_t *keys_sorted = reinterpret_cast<uint32_t *>(take(n_keys_b));
  uint32_t *order = reinterpret_cast<uint32_t *>(take(n_keys_b));
  void *tmp = take(tmp_bytes);
  float *partial = reinterpret_cast<float *>(take(n_partial));
  auto bail = [&](hipError_t err, const char *what) {
    if (!fixed) (void)scratch_free(buf, a.stream);
    return fail_hip(err, what);
  };
  PieceCountIterator counts(rocprim::counting_iterator<uint32_t>(0u), PieceCount{a.offsets, rows, chunk});
  hipError_t err = rocprim::exclusive_scan(tmp, scan_bytes, counts, base, 0u, static_cast<size_t>(rows) + 1,
                                           rocprim::plus<uint32_t>(), a.stream, false);
  if (err != hipSuccess) return bail(err, "spmm: scan of piece counts");
  hipLaunchKernelGGL(auto_items_kernel, dim3(ceil_div(p_max, 256)), dim3(256), 0, a.stream, items, keys, base, a.offsets,
                     a.indices, a.index_base, rows, chunk, p_max);
  err = hipGetLastError();
  if (err != hipSuccess) return bail(err, "auto_items_kernel");
  if (large) {
    err = rocprim::radix_sort_pairs(tmp, sort_bytes, keys, keys_sorted, rocprim::counting_iterator<uint32_t>(0u), order,
                                    p_max, 0u, 32u, a.stream, false);
    if (err != hipSuccess) return bail(err, "spmm: ordering of the pieces");
    hipLaunchKernelGGL(auto_order_items_kernel, dim3(ceil_div(p_max, 256)), dim3(256), 0, a.stream, ordered, items,
                       order, p_max);
    err = hipGetLastError();
    if (err != hipSuccess) return bail(err, "auto_order_items_kernel");
  }
  // One launch: the pieces first (the heavy, uniform work), then the rows that fit one wavefront,
  // so that the rows fill the chip while the last pieces, each a serial chain, finish.
  LaunchArgs pc = a;
  pc.n_items = p_max;
  pc.items = large ? ordered : items;
  pc.partial = partial;
  pc.rows_after_items = rows;
  pc.row_edge_limit = chunk;
  launch_spmm(pc);
#define NTS_AUTO_REDUCE_WIDE(J)                                                                                     \
  hipLaunchKernelGGL(auto_reduce_wide_kernel<J>, dim3(p_max), dim3(256), 0, a.stream, a.out, partial, items, base, a.F, \
                     a.accumulate, p_max)
  if (a.F > 256 && a.F <= 512)
    NTS_AUTO_REDUCE_WIDE(2);
  else if (a.F > 512 && a.F <= 768)
    NTS_AUTO_REDUCE_WIDE(3);
  else if (a.F > 768 && a.F <= 1024)
    NTS_AUTO_REDUCE_WIDE(4);
  else
    hipLaunchKernelGGL(auto_reduce_kernel, dim3(p_max, ceil_div(a.F, 256)), dim3(256), 0, a.stream, a.out, partial, items,
                       base, a.F, a.accumulate, p_max);
#undef NTS_AUTO_REDUCE_WIDE
  err = hipGetLastError();
  if (err != hipSuccess) return bail(err, "spmm: balanced launch");
  if (!fixed) NTS_HIP_TRY(scratch_free(buf, a.stream));
  return NTS_OK;
}

// Where a pass per gradient is faster although it gathers the rows twice: graphs of few edges, whose hub rows no
// wavefront shares the work of (kAutoMinEdges), so that a launch lasts as long as the longest row.  A step of eight edges
// of the fused kernel, with its sums across the lanes, takes longer than one of the gather of wide rows; the other pass
// has no such chain.  Fused and separate, us: 5 K vertices, 40 K edges, eight heads of 8 91, 65; one of 64 81, 68;
// of 128 121, 73; two of 64 97, 73; but four of 4 70, 106, one of 32 75, 81 (rows below 64 floats stay fused)
// and four of 64 97, 100.  For widths that nts_sddmm_heads is slow at, only one head off 16-byte boundaries is affected: 5 K, 40 K, 47
// floats 94, 80, 201 209, 143; two of 47 97, 142; 2.7 K, 13 K, 47 floats 39, 58 (and 5 K, 20 K 43, 60: the line could lie higher).  With fewer than four edges a row on average there are
// no such rows, or they matter less: 10 K, 25 K, two of 64 36, 45; a sampled layer of 4 K destinations, 41 K edges, eight
// heads of 8 7, 14.
bool separate_gradients_are_faster(const LaunchArgs &a, uint32_t edges) {
  if (edges >= kAutoMinEdges || edges / 4 < a.n_items) return false;
  const uint32_t H = a.heads.H, Fh = a.heads.Fh;
  uint32_t vec = 1;
  if (sddmm_by_lanes(a.dot_rows, a.in, H, Fh, &vec)) return a.F >= 64;
  return H == 1 && vec == 1 && Fh > 32 && edges >= kAutoMinEdges / 4;
}

// ---- the same schedule built on the device -----------------------------------------------------------
//
// nts_spmm_plan_create_slabs needs the index array to cut rows at source-range boundaries; copying it
// to the host and scheduling there costs seconds per 10^8 edges.  The kernels below build the item
// list of make_schedule -- the same pieces, slots, order of pieces, order of whole rows and order of
// split rows, entry for entry -- from the arrays where they lie:
//   plan_cut_rows_kernel      16 lanes per row: the row's range count by its length, a lower_bound per
//                             range boundary, pieces per (row, range) into a [rows, n_slabs] table
//   exclusive scan of the table = first partial slot of every (row, range); its total = slots
//   plan_emit_pieces_kernel   one thread per non-empty (row, range): its pieces and their sort keys
//                             (range id, then longer pieces first); slot order is creation order, so a
//                             stable radix sort by key reproduces the host's stable_sort
//   plan_row_keys_kernel      per row: key of the whole rows (descending length, stable by row) and of
//                             the split rows (descending slot count, stable by row)
//   plan_finish_kernel        whole rows behind the pieces; the split-row table
// Rows long enough to be cut must ascend.  plan_scan_edges_kernel flags the ones that do not; if there are
// any, a stable radix sort of (row, index) keys orders them in a copy of the index array that the schedule
// then cuts and gathers through, with the caller's position of every edge beside it (an edge list in
// random order, 114.8 M edges: 3.2 ms, where sorting the rows on 16 host threads took 0.9 s).

struct PlanShape {
  uint32_t chunk, n_slabs, wide_ranges;
  uint64_t fine_width;
  // Ranges a row of `deg` edges is cut at (0 = the row stays whole): see make_schedule.
  __host__ __device__ uint32_t ranges_for(uint32_t deg) const {
    if (deg <= chunk) return (wide_ranges && deg > chunk / 4) ? wide_ranges : 0u;
    return (wide_ranges && deg <= 4ull * chunk) ? n_slabs / 2 : n_slabs;
  }
};

struct PlanCounters {  // device words read back to the host
  unsigned long long repeated;  // edges whose index equals that of the edge before them in their row
  uint32_t largest_index;
  uint32_t unsorted_long_row;   // a row that would be cut does not ascend
  uint32_t n_splits;
  uint32_t bad_offsets, bad_total;
  uint32_t first_edge;          // offsets[0]
  uint32_t longest_row;
};

__device__ __forceinline__ uint32_t lower_bound_index(const uint32_t *__restrict__ idx, uint32_t lo, uint32_t hi,
                                                      uint64_t lim, uint32_t base) {
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (static_cast<uint64_t>(idx[mid] - base) < lim) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// kCutLanes lanes per row, each searching the whole row for the end of its range: one thread that searched range after
// range from where the last one ended was 32 searches in a row (114.8 M edges, 233 K rows: 280 -> 80 us).
constexpr uint32_t kCutLanes = 16;
__global__ __launch_bounds__(256) void plan_cut_rows_kernel(uint32_t *__restrict__ counts, uint32_t *__restrict__ stops,
                                                            const uint32_t *__restrict__ off,
                                                            const uint32_t *__restrict__ idx, uint32_t index_base,
                                                            uint32_t rows, PlanShape sh) {
  const uint32_t gl = threadIdx.x & (kCutLanes - 1), group = (threadIdx.x & (kWave - 1)) / kCutLanes;
  const uint32_t per_block = blockDim.x / kCutLanes;
  for (uint64_t r64 = static_cast<uint64_t>(blockIdx.x) * per_block + threadIdx.x / kCutLanes; r64 < rows;
       r64 += static_cast<uint64_t>(gridDim.x) * per_block) {
    const uint32_t r = static_cast<uint32_t>(r64);
    const uint32_t b = off[r], e = off[r + 1], deg = e - b;
    const uint32_t R = sh.ranges_for(deg);
    if (R == 0) continue;  // the table was cleared: a whole row has no pieces
    uint32_t *cnt = counts + static_cast<size_t>(r) * sh.n_slabs;
    uint32_t *stp = stops + static_cast<size_t>(r) * sh.n_slabs;
    const uint32_t per = sh.n_slabs / R;
    uint32_t cut = b, nonempty = 0;
    for (uint32_t c0 = 0; c0 < R; c0 += kCutLanes) {
      const uint32_t c = c0 + gl;
      const uint64_t hi = static_cast<uint64_t>(c + 1) * per * sh.fine_width;  // first index of the next range
      const uint32_t stop = c + 1 >= R ? e : lower_bound_index(idx, cut, e, hi, index_base);
      const uint32_t up = __shfl_up(stop, 1, kCutLanes), n = stop - (gl ? up : cut);
      if (c < R) {
        cnt[c] = deg > sh.chunk ? (n + sh.chunk - 1) / sh.chunk : (n ? 1u : 0u);
        stp[c] = stop;
      }
      nonempty += __popcll(__ballot(c < R && n) >> (group * kCutLanes) & ((1ull << kCutLanes) - 1));
      cut = __shfl(stop, kCutLanes - 1, kCutLanes);
    }
    if (deg <= sh.chunk && nonempty <= 1)  // all edges in one wide range: the row stays whole
      for (uint32_t c = gl; c < R; c += kCutLanes) cnt[c] = 0;
  }
}

__global__ __launch_bounds__(256) void plan_emit_pieces_kernel(Item *__restrict__ pieces, uint32_t *__restrict__ keys,
                                                               const uint32_t *__restrict__ counts,
                                                               const uint32_t *__restrict__ stops,
                                                               const uint32_t *__restrict__ slot_base,
                                                               const uint32_t *__restrict__ off, uint32_t rows,
                                                               PlanShape sh) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<uint64_t>(rows) * sh.n_slabs) return;
  const uint32_t n = counts[i];
  if (!n) return;
  const uint32_t r = static_cast<uint32_t>(i / sh.n_slabs), c = static_cast<uint32_t>(i % sh.n_slabs);
  const uint32_t b = off[r], deg = off[r + 1] - b;
  const uint32_t per = sh.n_slabs / sh.ranges_for(deg);
  const uint32_t lo = c ? stops[i - 1] : b, hi = stops[i];
  const uint32_t first = slot_base[i];
  for (uint32_t j = 0; j < n; ++j) {
    const uint32_t e0 = lo + j * sh.chunk, e1 = min(hi, e0 + sh.chunk);
    pieces[first + j] = make_uint4(r, e0, e1, first + j);
    keys[first + j] = c * per * (sh.chunk + 1) + (sh.chunk - (e1 - e0));
  }
}

__global__ __launch_bounds__(256) void plan_row_keys_kernel(uint32_t *__restrict__ whole_key,
                                                            uint32_t *__restrict__ split_key,
                                                            const uint32_t *__restrict__ slot_base,
                                                            const uint32_t *__restrict__ off, uint32_t rows,
                                                            PlanShape sh, PlanCounters *__restrict__ counters) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t split = 0;
  if (r < rows) {
    const uint32_t P = slot_base[static_cast<size_t>(r + 1) * sh.n_slabs] - slot_base[static_cast<size_t>(r) * sh.n_slabs];
    const uint32_t deg = off[r + 1] - off[r];
    whole_key[r] = P == 0 ? sh.chunk - deg : sh.chunk + 1;  // whole rows by descending length, cut rows last
    split_key[r] = ~P;                                      // split rows by descending slot count, whole rows last
    split = P ? 1u : 0u;
  }
  const uint32_t n = __popcll(__ballot(split));
  if ((threadIdx.x & (kWave - 1)) == 0 && n) atomicAdd(&counters->n_splits, n);
}

__global__ __launch_bounds__(256) void plan_finish_kernel(Item *__restrict__ items, uint4 *__restrict__ splits,
                                                          const uint32_t *__restrict__ whole_order,
                                                          const uint32_t *__restrict__ split_order,
                                                          const uint32_t *__restrict__ slot_base,
                                                          const uint32_t *__restrict__ off, uint32_t n_pieces,
                                                          uint32_t n_whole, uint32_t n_splits, uint32_t n_slabs) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n_whole) {
    const uint32_t r = whole_order[j];
    items[n_pieces + j] = make_uint4(r, off[r], off[r + 1], kNoSlot);
  }
  if (j < n_splits) {
    const uint32_t r = split_order[j];
    const uint32_t first = slot_base[static_cast<size_t>(r) * n_slabs];
    splits[j] = make_uint4(r, first, slot_base[static_cast<size_t>(r + 1) * n_slabs] - first, 0u);
  }
}

// A few blocks that stride over the rows: one request a block for the longest row, because requests to one word are served
// some 10 ns apart (a block per 256 rows: 2.4 M rows 114 us, 5 without the longest row).
constexpr uint32_t kCheckBlocks = 512;
__global__ __launch_bounds__(256) void plan_check_offsets_kernel(const uint32_t *__restrict__ off, uint32_t rows,
                                                                 uint32_t edges, PlanCounters *__restrict__ counters) {
  const uint64_t t = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  uint32_t longest = 0;
  for (uint64_t r = t; r < rows; r += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint32_t b = off[r], e = off[r + 1];
    if (e < b) counters->bad_offsets = 1u;
    else longest = max(longest, e - b);
  }
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1)
    longest = max(longest, static_cast<uint32_t>(__shfl_xor(static_cast<int>(longest), m, kWave)));
  __shared__ uint32_t wave_longest[256 / kWave];
  if ((threadIdx.x & (kWave - 1)) == 0) wave_longest[threadIdx.x / kWave] = longest;
  __syncthreads();
  if (threadIdx.x == 0)
    atomicMax(&counters->longest_row, max(max(wave_longest[0], wave_longest[1]), max(wave_longest[2], wave_longest[3])));
  if (t == 0) {
    if (off[rows] != edges) counters->bad_total = 1u;
    counters->first_edge = off[0];
  }
}

// One pass over the edges: every wavefront walks a contiguous span of edges and carries the row along
// (owners_of_row_step), so the position of a row start inside the span costs no search.  Counts the edges
// that repeat the index before them in their row, finds the largest index, and flags the rows of more
// than `cut_above` edges whose indices do not ascend.  Bound by the one read of the index array; an edge
// list in random order has a descent at every second edge, so nothing is listed or counted per descent
// (the list's counter alone took 42 ms for 114.8 M edges; the pass takes 0.23 to 0.3 ms whatever the order).
__global__ __launch_bounds__(256) void plan_scan_edges_kernel(const uint32_t *__restrict__ off,
                                                              const uint32_t *__restrict__ idx, uint32_t rows,
                                                              uint32_t edges, uint32_t cut_above,
                                                              unsigned char *__restrict__ unsorted,
                                                              PlanCounters *__restrict__ counters) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  const uint64_t total_steps = (static_cast<uint64_t>(edges) + kWave - 1) / kWave;
  const uint64_t per_wave = (total_steps + n_waves - 1) / n_waves;
  const uint64_t first_step = wave * per_wave;
  const uint64_t end_step = first_step + per_wave < total_steps ? first_step + per_wave : total_steps;
  uint32_t row = 0, row_begin = 0, row_end = 0;  // a wavefront without a span still takes part in the block's sums
  if (first_step < end_step) row = owner_of(off, rows, static_cast<uint32_t>(first_step * kWave));
  unsigned long long equal = 0;
  uint32_t largest = 0, descends = 0, flagged = 0;  // flagged: the row at hand is
  uint32_t before = 0;
  if (first_step && first_step < end_step) before = idx[first_step * kWave - 1];
  for (uint64_t step4 = first_step; step4 < end_step; step4 += kWalkSteps) {
    uint32_t v[kWalkSteps];
#pragma unroll
    for (int u = 0; u < kWalkSteps; ++u) {
      const uint64_t k = (step4 + u) * kWave + lane;
      v[u] = step4 + u < end_step && k < edges ? idx[k] : 0u;
    }
#pragma unroll
    for (int u = 0; u < kWalkSteps; ++u) {
      if (step4 + u >= end_step) break;
      const uint32_t base = static_cast<uint32_t>((step4 + u) * kWave), k = base + lane, b = v[u];
      uint32_t a = __shfl_up(b, 1, kWave);
      if (lane == 0) a = before;
      before = wave_read(b, kWave - 1);
      if (step_inside_row(base, row_end)) {  // no row starts here
        largest = max(largest, b);
        equal += a == b ? 1u : 0u;
        if (!flagged && row_end - row_begin > cut_above && __ballot(a > b)) {
          flagged = descends = 1;
          if (lane == 0) unsorted[row] = 1;
        }
        continue;
      }
      flagged = 0;
      const uint32_t own = owners_of_row_step(off, rows, base, row, row_begin, row_end);
      if (k >= edges) continue;
      largest = max(largest, b);
      const uint32_t start = off[own];
      if (k == start) continue;
      equal += a == b ? 1u : 0u;
      if (a > b && off[own + 1] - start > cut_above) {
        unsorted[own] = 1;  // the same value from every lane that finds one
        descends = 1;
      }
    }
  }
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) {
    equal += __shfl_xor(equal, m, kWave);
    largest = max(largest, static_cast<uint32_t>(__shfl_xor(static_cast<int>(largest), m, kWave)));
  }
  if (__ballot(descends) != 0 && lane == 0) counters->unsorted_long_row = 1u;
  // One addition per block to the shared counters: with one per wavefront of 4,096 blocks the pass took 0.77 ms.
  __shared__ unsigned long long block_equal[4];
  __shared__ uint32_t block_largest[4];
  const uint32_t w = threadIdx.x / kWave;
  if (lane == 0) {
    block_equal[w] = equal;
    block_largest[w] = largest;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    equal = block_equal[0] + block_equal[1] + block_equal[2] + block_equal[3];
    if (equal) atomicAdd(&counters->repeated, equal);
    atomicMax(&counters->largest_index, max(max(block_largest[0], block_largest[1]), max(block_largest[2], block_largest[3])));
  }
}

// Keys of the stable sort that orders the flagged rows by index and leaves every other row as it is:
// (row, index) for an edge of a flagged row, (row, 0) otherwise; local_bits: the edge's place in its row below that, so that
// the element sorted is all there is to move.
__global__ __launch_bounds__(256) void plan_sort_keys_kernel(unsigned long long *__restrict__ keys,
                                                             const uint32_t *__restrict__ off,
                                                             const uint32_t *__restrict__ idx, uint32_t index_base,
                                                             uint32_t rows, uint32_t edges,
                                                             const unsigned char *__restrict__ unsorted,
                                                             unsigned index_bits, unsigned local_bits) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * blockDim.x / kWave;
  const uint64_t total_steps = (static_cast<uint64_t>(edges) + kWave - 1) / kWave;
  const uint64_t per_wave = (total_steps + n_waves - 1) / n_waves;
  const uint64_t first_step = wave * per_wave;
  const uint64_t end_step = first_step + per_wave < total_steps ? first_step + per_wave : total_steps;
  if (first_step >= end_step) return;
  const uint32_t mask = static_cast<uint32_t>((1ull << index_bits) - 1);
  uint32_t row = owner_of(off, rows, static_cast<uint32_t>(first_step * kWave)), row_begin = 0, row_end = 0;
  uint32_t flagged = 0;  // the row at hand is
  auto put = [&](uint32_t k, uint32_t own, uint32_t own_begin, uint32_t is_unsorted, uint32_t index) {
    const unsigned long long key =
        (static_cast<unsigned long long>(own) << index_bits) | (is_unsorted ? (index - index_base) & mask : 0u);
    keys[k] = local_bits ? key << local_bits | (k - own_begin) : key;
  };
  for (uint64_t step4 = first_step; step4 < end_step; step4 += kWalkSteps) {
    uint32_t v[kWalkSteps];
#pragma unroll
    for (int u = 0; u < kWalkSteps; ++u) {
      const uint64_t k = (step4 + u) * kWave + lane;
      v[u] = step4 + u < end_step && k < edges ? idx[k] : 0u;
    }
#pragma unroll
    for (int u = 0; u < kWalkSteps; ++u) {
      if (step4 + u >= end_step) break;
      const uint32_t base = static_cast<uint32_t>((step4 + u) * kWave), k = base + lane;
      if (step_inside_row(base, row_end)) {
        put(k, row, row_begin, flagged, v[u]);
        continue;
      }
      const uint32_t own = owners_of_row_step(off, rows, base, row, row_begin, row_end);
      flagged = row_end ? unsorted[row] : 0u;
      if (k < edges) put(k, own, off[own], unsorted[own], v[u]);
    }
  }
}

// The last pass of the sort of (row, index, place in the row) elements: the index array in the new order and every edge's
// position in the caller's.  An edge of a row that is left as it is stays where it was.
struct TakeSorted {
  uint32_t *sorted_idx, *edge_ids;
  const uint32_t *off, *idx;
  const unsigned char *unsorted;
  uint32_t index_base, index_mask;
  unsigned index_bits, local_bits;
  __device__ __forceinline__ void operator()(uint32_t at, SortElement v) const {
    const uint32_t row = static_cast<uint32_t>(v >> local_bits >> index_bits);
    edge_ids[at] = off[row] + (static_cast<uint32_t>(v) & ((1u << local_bits) - 1u));
    sorted_idx[at] = unsorted[row] ? static_cast<uint32_t>(v >> local_bits) & index_mask : idx[at] - index_base;
  }
};

// The index array in the new order.  An edge of an ordered row carries its index in its key; only the
// other rows' are fetched through the edge ids (all of them: 1.0 ms for 114.8 M edges, scattered within
// each row).
__global__ __launch_bounds__(256) void plan_take_indices_kernel(uint32_t *__restrict__ sorted_idx,
                                                                const unsigned long long *__restrict__ keys,
                                                                const uint32_t *__restrict__ idx, uint32_t index_base,
                                                                const uint32_t *__restrict__ edge_ids, uint32_t edges,
                                                                const unsigned char *__restrict__ unsorted,
                                                                unsigned index_bits) {
  const uint32_t mask = static_cast<uint32_t>((1ull << index_bits) - 1);
  for (uint64_t k = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; k < edges;
       k += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const unsigned long long key = keys[k];
    sorted_idx[k] = unsorted[key >> index_bits] ? static_cast<uint32_t>(key) & mask : idx[edge_ids[k]] - index_base;
  }
}

int check_common(const float *in, float *out, const uint32_t *offsets, const uint32_t *indices, uint32_t rows,
                 uint32_t edges, uint32_t F, const char *who) {
  if (F == 0) return fail(NTS_ERR_INVALID, "spmm: feature width F is 0");
  if (rows == 0) return NTS_OK;
  if (!out || !offsets) return fail(NTS_ERR_INVALID, who);
  if (edges != 0 && (!in || !indices)) return fail(NTS_ERR_INVALID, who);
  return NTS_OK;
}

}  // namespace
}  // namespace nts

namespace {
// fn(first, last) over [0, n) on up to 16 host threads, in contiguous blocks.
template <typename Fn>
void parallel_blocks(uint32_t n, Fn fn) {
  unsigned t = std::thread::hardware_concurrency();
  if (t > 16) t = 16;
  if (t < 2 || n < 4096) {
    fn(0u, n);
    return;
  }
  std::vector<std::thread> pool;
  const uint32_t per = (n + t - 1) / t;
  for (uint32_t b = 0; b < n; b += per) pool.emplace_back(fn, b, std::min(n, b + per));
  for (std::thread &th : pool) th.join();
}

}  // namespace

namespace {
struct PlanMemory {
  using Error = hipError_t;
  using Block = nts::DeviceBlock;
  static constexpr hipError_t kSuccess = hipSuccess;
  static hipError_t retire(nts::DeviceBlock &block) { return nts::retire_blocks({&block}); }
  static bool out_of_memory(hipError_t err) { return err == hipErrorOutOfMemory; }
  static void clear_error() { (void)hipGetLastError(); }
};
}  // namespace

struct nts_spmm_plan {
  uint32_t rows = 0;
  uint32_t edges = 0;
  uint32_t chunk = 0;
  uint32_t n_items = 0;
  uint32_t n_splits = 0;
  uint32_t n_partials = 0;
  const uint32_t *offsets = nullptr;  // identity check only
  nts::DeviceBlock items_block, splits_block, sorted_block, ids_block;
  uint4 *items = nullptr;             // device
  uint4 *splits = nullptr;            // device
  // Scratch shared by every call on this plan: the partial sums of split rows and, for widths whose
  // rows do not start on 16-byte boundaries, a padded copy of the input.  `mu` serialises the host
  // side of the calls (growing the scratch, enqueueing); `done` is recorded after the last kernel of
  // each call, and a call on another stream waits for it before it touches the scratch.
  nts::PlanScratch<PlanMemory> scratch;
  uint32_t n_index = 0;               // rows of the gathered matrix (0 = not known: no padded copy)
  // At least 1 in 20 edges repeats the gather index of the edge before it: the wave kernel then loads
  // a row once per run of equal indices (and widths off 16-byte boundaries get the padded copy).
  bool dup_runs = false;
  bool ranged = false;                // built with source ranges
  uint64_t repeated_edges = 0;
  std::mutex mu;
  hipEvent_t done = nullptr;
  hipStream_t last_stream = nullptr;
  bool in_flight = false;
  // Only when rows had to be re-ordered for the source ranges: the schedule's own copy of the gather
  // indices (base already subtracted), and for each of its edges the position in the caller's order.
  uint32_t *sorted_idx = nullptr;     // device, [edges]
  uint32_t *edge_ids = nullptr;       // device, [edges]
  hipEvent_t ev_start = nullptr;      // optional profiling events around the main kernel
  hipEvent_t ev_stop = nullptr;
};

extern "C" {

int nts_spmm_gather(const float *in, float *out, const float *w, const uint32_t *offsets, const uint32_t *indices,
                    uint32_t index_base, uint32_t rows, uint32_t edges, uint32_t F, int accumulate,
                    nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_gather");
  if (int rc = nts::check_common(in, out, offsets, indices, rows, edges, F, "nts_spmm_gather: null pointer")) return rc;
  if (rows == 0) return NTS_OK;
  nts::LaunchArgs a{in, out, w, offsets, indices, index_base, rows, F, nullptr, nullptr, accumulate, stream};
  if (int rc = nts::launch_spmm_balanced(a, edges)) return rc;
  NTS_LAUNCH_CHECK("nts_spmm_gather");
  return NTS_OK;
}

int nts_spmm_gather_bounded(const float *in, float *out, const float *w, const uint32_t *offsets,
                            const uint32_t *indices, uint32_t index_base, uint32_t rows, uint32_t edges, uint32_t F,
                            int accumulate, uint32_t max_row_edges, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_gather_bounded");
  if (int rc = nts::check_common(in, out, offsets, indices, rows, edges, F, "nts_spmm_gather_bounded: null pointer"))
    return rc;
  if (rows == 0) return NTS_OK;
  nts::LaunchArgs a{in, out, w, offsets, indices, index_base, rows, F, nullptr, nullptr, accumulate, stream};
  if (max_row_edges != 0 && max_row_edges <= nts::kAutoChunk) {
    a.edges = edges;
    a.bounded = true;
    // No row can need cutting: one launch, a wavefront (or lane group) per row, no scratch.
    nts::launch_spmm(a);
  } else if (int rc = nts::launch_spmm_balanced(a, edges)) {
    return rc;
  }
  NTS_LAUNCH_CHECK("nts_spmm_gather_bounded");
  return NTS_OK;
}

int nts_spmm_gather_static_scratch(const float *in, float *out, const float *w, const uint32_t *offsets,
                                   const uint32_t *indices, uint32_t index_base, uint32_t rows, uint32_t edges,
                                   uint32_t F, int accumulate, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_gather_static_scratch");
  if (int rc = nts::check_common(in, out, offsets, indices, rows, edges, F,
                                 "nts_spmm_gather_static_scratch: null pointer"))
    return rc;
  if (rows == 0) return NTS_OK;
  unsigned char *fixed = nullptr;
  if (int rc = nts::static_scratch_address(&fixed)) return rc;
  nts::LaunchArgs a{in, out, w, offsets, indices, index_base, rows, F, nullptr, nullptr, accumulate, stream};
  if (int rc = nts::launch_spmm_balanced(a, edges, fixed, kStaticScratchBytes)) return rc;
  NTS_LAUNCH_CHECK("nts_spmm_gather_static_scratch");
  return NTS_OK;
}

namespace {

struct Piece {
  uint32_t slab, row, e0, e1, slot;
};

// Piece length of a schedule without source ranges when the caller names none.  A piece is one serial
// chain of row reads, so a launch lasts at least as long as its longest piece: with 4,096-edge pieces
// whatever the graph, the two widths of an Arxiv-shaped pass (2.48 M edges, F = 128) took 340 us, all of
// it the tail of a few hub rows.  The chip holds 8,192 wavefronts, so pieces of E / 8,192 edges keep the
// longest chain at the average share of a wavefront; shorter ones only add partial sums.  Measured, us
// per pass, 4,096-edge pieces -> the power of two below E / 8,192: 10,556 edges F = 1,433 163 -> 31, F = 16
// 44 -> 11; 200 K edges F = 128 206 -> 19; 2.48 M edges F = 128 340 -> 107, F = 16 809 -> 70, F = 602 1,187 -> 747;
// 6 M edges F = 128 326 -> 135.  From 33 M edges up it is 4,096, the better one there (50 M edges F = 128: 512
// 1,746, 4,096 1,406 us: long pieces of ascending rows keep neighbouring wavefronts on the same sources).
uint32_t default_chunk(uint32_t edges) {
  uint32_t chunk = 32;
  while (chunk < 4096u && 2u * chunk <= edges / 8192u) chunk *= 2;
  return chunk;
}

// Builds the work-item list.  Rows with more than `chunk` edges are split into pieces that write
// partial sums (slots numbered in ascending edge order inside a row, so the second-stage sum has
// a fixed order).  With n_slabs > 1 and a host copy of the gather indices, pieces of rows whose
// indices ascend are additionally cut at the boundaries of n_slabs equal ranges of the gather
// index space and the pieces are ordered slab by slab: wavefronts that run at the same time then
// gather from the same 1/n_slabs of the source rows, which is what lets each 4 MB L2 keep that
// range's hot rows resident.  Items: all pieces (slab-major, longest first inside a slab), then
// the unsplit rows by descending degree.
struct Schedule {
  std::vector<uint4> items;   // (row, first edge, end edge, partial slot or kNoSlot)
  std::vector<uint4> splits;  // (row, first slot, slot count, 0)
  uint32_t n_partials = 0;
  // Empty unless some row that is cut by source range did not have ascending indices: then a copy
  // of the index array in which those rows are sorted (stable), and the original position of each
  // of its edges.  Rows that are never cut keep their order.
  std::vector<uint32_t> sorted_idx;
  std::vector<uint32_t> edge_ids;
  // Edges whose gather index equals that of the edge before them in the same row (parallel edges of
  // a multigraph, adjacent when rows are sorted); counted in the index array the schedule gathers through.
  uint64_t repeated_edges = 0;
};

// The schedule without source ranges.  What it is made of follows from the lengths alone, so everything is placed
// by counting: one pass over the rows counts, the next writes each entry where it belongs (pieces by descending
// length, equal ones by slot; whole rows by descending length, equal ones by row; split rows by descending piece
// count).  No piece is written twice: with the short pieces of default_chunk there are often as many of them as rows,
// and making a list of them that was ordered afterwards took 275 us of a schedule (60 K vertices, 600 K edges) where
// the few 4,096-edge pieces of before had taken 212; placed at once it is 208 (30 K, 300 K: 152 -> 107; 5 K, 500 K,
// 19,000 items instead of 5,000: 102 -> 58).
void make_one_range_schedule(Schedule &out, const uint32_t *off, uint32_t rows, uint32_t chunk) {
  if (rows == 0) return;
  chunk = std::min(chunk, std::max(off[rows] - off[0], 1u));  // a longer piece cuts nothing
  std::vector<uint32_t> whole_at(static_cast<size_t>(chunk) + 2, 0u), rest_at(static_cast<size_t>(chunk) + 1, 0u);
  std::vector<uint32_t> long_rows;
  uint32_t n_full = 0, n_partials = 0, most = 0;
  for (uint32_t r = 0; r < rows; ++r) {
    const uint32_t deg = off[r + 1] - off[r];
    if (deg <= chunk) {
      ++whole_at[chunk - deg + 1];
      continue;
    }
    const uint32_t full = deg / chunk, rest = deg - full * chunk, n = full + (rest ? 1u : 0u);
    long_rows.push_back(r);
    n_full += full;
    n_partials += n;
    most = std::max(most, n);
    if (rest) ++rest_at[chunk - rest];
  }
  // rest_at[chunk - n] = position of the first piece of n < chunk edges; the full ones come before them
  uint32_t next = n_full;
  for (uint32_t &at : rest_at) {
    const uint32_t n = at;
    at = next;
    next += n;
  }
  whole_at[0] = n_partials;
  for (size_t i = 1; i < whole_at.size(); ++i) whole_at[i] += whole_at[i - 1];
  std::vector<uint32_t> split_at(static_cast<size_t>(most) + 2, 0u);
  for (uint32_t r : long_rows) ++split_at[most - (off[r + 1] - off[r] - 1) / chunk];
  for (size_t i = 1; i < split_at.size(); ++i) split_at[i] += split_at[i - 1];

  std::vector<uint4> &items = out.items;
  items.reserve(static_cast<size_t>(n_partials) + rows);  // (the split rows follow for the upload)
  items.resize(static_cast<size_t>(n_partials) + rows - long_rows.size());
  out.splits.resize(long_rows.size());
  uint32_t slot = 0, full_at = 0;
  for (uint32_t r : long_rows) {
    const uint32_t first = slot, end = off[r + 1];
    uint32_t k = off[r];
    for (; end - k >= chunk; k += chunk) items[full_at++] = make_uint4(r, k, k + chunk, slot++);
    if (k < end) items[rest_at[chunk - (end - k)]++] = make_uint4(r, k, end, slot++);
    out.splits[split_at[most - (slot - first)]++] = make_uint4(r, first, slot - first, 0u);
  }
  for (uint32_t r = 0; r < rows; ++r) {
    const uint32_t deg = off[r + 1] - off[r];
    if (deg <= chunk) items[whole_at[chunk - deg]++] = make_uint4(r, off[r], off[r + 1], nts::kNoSlot);
  }
  out.n_partials = n_partials;
}

// Host-only: needs nothing but the two index arrays.
void make_schedule(Schedule &out, const uint32_t *off, const uint32_t *idx_in, uint32_t rows, uint32_t chunk,
                   uint32_t n_slabs, uint32_t n_index) {
  const uint32_t *idx = idx_in;
  auto count_repeated = [&] {
    std::atomic<uint64_t> repeated(0);
    parallel_blocks(rows, [&](uint32_t r0, uint32_t r1) {
      uint64_t n = 0;
      for (uint32_t r = r0; r < r1; ++r)
        for (uint32_t k = off[r] + 1; k < off[r + 1]; ++k) n += idx[k] == idx[k - 1];
      repeated.fetch_add(n, std::memory_order_relaxed);
    });
    out.repeated_edges = repeated.load();
  };
  if (n_slabs <= 1 || idx == nullptr || n_index == 0) {
    make_one_range_schedule(out, off, rows, chunk);
    if (idx) count_repeated();
    return;
  }
  std::vector<Piece> pieces;
  std::vector<uint4> &splits = out.splits;
  uint32_t n_partials = 0;
  std::vector<uint32_t> bucket(static_cast<size_t>(chunk) + 2, 0u);
  // Source ranges come in three widths and a row is cut at the width that suits its length: every
  // piece costs one partial row (written, then read by the second stage), so shorter rows get
  // fewer, wider ranges.
  //   more than 4 * chunk edges    n_slabs ranges
  //   more than chunk edges        n_slabs / 2 ranges (2,048-edge rows at 32 ranges would be cut into 19-edge
  //                                pieces on average; 24.7 -> 24.2 ms per four-pass step on the 114.8 M-edge graph)
  //   more than chunk / 4 edges    n_slabs / 4 ranges; a row whose edges all fall into one of them stays whole
  // A piece is issued with the first narrow range it covers, so that wavefronts resident at the
  // same time gather from the same part of the source rows whatever the width of their ranges.
  // (Twice or four times as many, narrower ranges for rows above 2,048 .. 16,384 edges were
  // measured as well: no gain on the 114.8 M-edge power-law graph.)
  const uint32_t fine = n_slabs;
  const uint64_t fine_width = (static_cast<uint64_t>(n_index) + fine - 1) / fine;
  const uint32_t wide_ranges = n_slabs >= 8 ? n_slabs / 4 : 0;
  std::vector<uint8_t> was_cut(wide_ranges ? rows : 0, 0);
  // Rows long enough to be cut by source range must ascend.  Edge files are not always sorted
  // (the reference's loader leaves a CSR row in thread-arrival order), so such rows are sorted in
  // a copy of the index array that the schedule then gathers through; a stable sort, so equal
  // indices keep their edge order.  Sums of those rows are associated in source order.
  const uint32_t cut_above = wide_ranges ? chunk / 4 : chunk;
  std::vector<uint8_t> unsorted(rows, 0);
  std::atomic<bool> any(false);
  parallel_blocks(rows, [&](uint32_t r0, uint32_t r1) {
    for (uint32_t r = r0; r < r1; ++r) {
      const uint32_t b = off[r], e = off[r + 1];
      if (e - b <= cut_above) continue;
      for (uint32_t k = b + 1; k < e; ++k)
        if (idx_in[k - 1] > idx_in[k]) {
          unsorted[r] = 1;
          any.store(true, std::memory_order_relaxed);
          break;
        }
    }
  });
  if (any.load()) {
    const uint32_t edges = off[rows];
    out.sorted_idx.assign(idx_in, idx_in + edges);
    out.edge_ids.resize(edges);
    parallel_blocks(edges, [&](uint32_t e0, uint32_t e1) {
      for (uint32_t e = e0; e < e1; ++e) out.edge_ids[e] = e;
    });
    parallel_blocks(rows, [&](uint32_t r0, uint32_t r1) {
      for (uint32_t r = r0; r < r1; ++r) {
        if (!unsorted[r]) continue;
        uint32_t *ids = out.edge_ids.data() + off[r], *ids_end = out.edge_ids.data() + off[r + 1];
        std::stable_sort(ids, ids_end, [&](uint32_t a, uint32_t b) { return idx_in[a] < idx_in[b]; });
        for (uint32_t k = off[r]; k < off[r + 1]; ++k) out.sorted_idx[k] = idx_in[out.edge_ids[k]];
      }
    });
    idx = out.sorted_idx.data();
  }
  std::vector<uint32_t> stops;  // (narrow range id, end edge) of the non-empty ranges of one row
  // Cuts edges [b, e) of a row with ascending indices at `ranges` equal ranges; ranges divides fine.
  auto range_stops = [&](uint32_t b, uint32_t e, uint32_t ranges) {
    stops.clear();
    const uint32_t per = fine / ranges;
    uint32_t cut = b;
    for (uint32_t c = 0; c < ranges && cut < e; ++c) {
      const uint64_t hi = static_cast<uint64_t>(c + 1) * per * fine_width;  // first index of the next range
      const uint32_t stop =
          c + 1 == ranges ? e
                          : static_cast<uint32_t>(std::lower_bound(idx + cut, idx + e, hi,
                                                                   [](uint32_t v, uint64_t lim) { return v < lim; }) -
                                                  idx);
      if (stop > cut) {
        stops.push_back(c * per);
        stops.push_back(stop);
      }
      cut = stop;
    }
  };
  for (uint32_t r = 0; r < rows; ++r) {
    const uint32_t b = off[r], e = off[r + 1], deg = e - b;
    if (deg <= chunk) {
      if (wide_ranges && deg > chunk / 4) {
        range_stops(b, e, wide_ranges);
        if (stops.size() > 2) {
          const uint32_t first = n_partials;
          uint32_t from = b;
          for (size_t q = 0; q < stops.size(); q += 2) {
            pieces.push_back(Piece{stops[q], r, from, stops[q + 1], n_partials++});
            from = stops[q + 1];
          }
          splits.push_back(make_uint4(r, first, n_partials - first, 0u));
          was_cut[r] = 1;
          continue;
        }
      }
      ++bucket[chunk - deg + 1];  // descending degree
      continue;
    }
    const uint32_t first = n_partials;
    range_stops(b, e, (wide_ranges && deg <= 4 * static_cast<uint64_t>(chunk)) ? n_slabs / 2 : n_slabs);
    uint32_t from = b;
    for (size_t q = 0; q < stops.size(); q += 2) {
      for (uint32_t k = from; k < stops[q + 1]; k += chunk)
        pieces.push_back(Piece{stops[q], r, k, std::min(stops[q + 1], k + chunk), n_partials++});
      from = stops[q + 1];
    }
    splits.push_back(make_uint4(r, first, n_partials - first, 0u));
  }
  count_repeated();
  std::stable_sort(splits.begin(), splits.end(), [](const uint4 &a, const uint4 &b) { return a.z > b.z; });
  std::stable_sort(pieces.begin(), pieces.end(), [](const Piece &a, const Piece &b) {
    if (a.slab != b.slab) return a.slab < b.slab;
    return (a.e1 - a.e0) > (b.e1 - b.e0);
  });
  std::vector<uint4> &items = out.items;
  items.reserve(pieces.size() + rows + splits.size());  // (the split rows follow for the upload)
  for (const Piece &pc : pieces) items.push_back(make_uint4(pc.row, pc.e0, pc.e1, pc.slot));
  for (size_t i = 1; i < bucket.size(); ++i) bucket[i] += bucket[i - 1];
  const size_t base = items.size();
  items.resize(base + bucket.back());
  for (uint32_t r = 0; r < rows; ++r) {
    const uint32_t deg = off[r + 1] - off[r];
    if (deg <= chunk && !(wide_ranges && was_cut[r]))
      items[base + bucket[chunk - deg]++] = make_uint4(r, off[r], off[r + 1], nts::kNoSlot);
  }
  out.n_partials = n_partials;
}

int build_plan(nts_spmm_plan_t **plan_out, const uint32_t *offsets_dev, const std::vector<uint32_t> &off,
               const uint32_t *idx, uint32_t rows, uint32_t edges, uint32_t chunk, uint32_t n_slabs,
               uint32_t n_index) {
  Schedule sched;
  make_schedule(sched, off.data(), idx, rows, chunk, n_slabs, n_index);
  std::vector<uint4> &items = sched.items;
  const uint32_t n_partials = sched.n_partials;

  nts_spmm_plan *p = new (std::nothrow) nts_spmm_plan();
  if (!p) return nts::fail(NTS_ERR_NOMEM, "nts_spmm_plan_create: host allocation failed");
  p->rows = rows;
  p->edges = edges;
  p->chunk = chunk;
  p->offsets = offsets_dev;
  p->n_items = static_cast<uint32_t>(items.size());
  p->n_splits = static_cast<uint32_t>(sched.splits.size());
  p->n_partials = n_partials;
  p->n_index = n_index;
  p->repeated_edges = sched.repeated_edges;
  p->dup_runs = edges > 0 && sched.repeated_edges * 20 >= edges;
  p->ranged = n_slabs > 1;
  hipError_t err = hipEventCreateWithFlags(&p->done, hipEventDisableTiming);
  items.insert(items.end(), sched.splits.begin(), sched.splits.end());  // one block, one copy
  if (err == hipSuccess && !items.empty()) {
    err = p->items_block.take(items.size() * sizeof(uint4));
    p->items = p->items_block.as<uint4>();
    p->splits = p->items + p->n_items;
    if (err == hipSuccess)
      err = hipMemcpy(p->items, items.data(), items.size() * sizeof(uint4), hipMemcpyHostToDevice);
  }
  if (err == hipSuccess && !sched.sorted_idx.empty()) {
    const size_t bytes = sched.sorted_idx.size() * sizeof(uint32_t);
    err = p->sorted_block.take(bytes);
    p->sorted_idx = p->sorted_block.as<uint32_t>();
    if (err == hipSuccess) err = hipMemcpy(p->sorted_idx, sched.sorted_idx.data(), bytes, hipMemcpyHostToDevice);
    if (err == hipSuccess) err = p->ids_block.take(bytes);
    p->edge_ids = p->ids_block.as<uint32_t>();
    if (err == hipSuccess) err = hipMemcpy(p->edge_ids, sched.edge_ids.data(), bytes, hipMemcpyHostToDevice);
  }
  if (err != hipSuccess) {
    nts_spmm_plan_destroy(p);
    return nts::fail_hip(err, "nts_spmm_plan_create: device upload");
  }
  *plan_out = p;
  return NTS_OK;
}

// Builds the schedule of make_schedule on the device (kernels above).  *fell_back is set, and nothing built,
//  - where the first row does not start at edge 0: the edges before it belong to no row, while the kernels
//    give every edge to the row before it (row 0 would be ordered together with them);
//  - where rows have to be ordered and the sort's memory, some 25 bytes an edge with the ordered copies (36 with the
//    library's sort), is not to be had: the host orders them with the copies alone on the device, 8 bytes an edge.
int build_plan_device(nts_spmm_plan_t **plan_out, const uint32_t *offsets, const uint32_t *indices,
                      uint32_t index_base, uint32_t n_index, uint32_t rows, uint32_t edges, uint32_t chunk,
                      uint32_t n_slabs, hipStream_t stream, bool *fell_back) {
  using nts::Item;
  *fell_back = false;
  nts::PlanShape sh;
  sh.chunk = chunk;
  sh.n_slabs = n_slabs;
  sh.wide_ranges = n_slabs >= 8 ? n_slabs / 4 : 0;
  sh.fine_width = (static_cast<uint64_t>(n_index) + n_slabs - 1) / n_slabs;
  const size_t cells = static_cast<size_t>(rows) * n_slabs;
  unsigned key_bits = 1;
  while ((1ull << key_bits) < static_cast<uint64_t>(n_slabs) * (chunk + 1)) ++key_bits;
  unsigned whole_bits = 1;
  while ((1ull << whole_bits) < static_cast<uint64_t>(chunk) + 2) ++whole_bits;

  size_t scan_bytes = 0, sort_rows_bytes = 0;
  uint32_t *nul = nullptr;
  NTS_HIP_TRY(rocprim::exclusive_scan(nullptr, scan_bytes, nul, nul, 0u, cells + 1, rocprim::plus<uint32_t>(), stream,
                                      false));
  NTS_HIP_TRY(rocprim::radix_sort_pairs(nullptr, sort_rows_bytes, nul, nul, rocprim::counting_iterator<uint32_t>(0u), nul,
                                        rows, 0u, 32u, stream, false));
  const size_t tmp1_bytes = nts::up256(std::max(scan_bytes, sort_rows_bytes));
  const size_t cell_words = nts::up256((cells + 1) * sizeof(uint32_t));
  const size_t row_words = nts::up256((static_cast<size_t>(rows) + 1) * sizeof(uint32_t));
  // Every block is given back after the last wait for the stream, the error paths included; where that
  // wait fails the driver frees them.
  nts::DeviceBlock work, work2, sort_work, sorted_block, ids_block;
  struct GiveBack {
    hipStream_t s;
    std::array<nts::DeviceBlock *, 5> blocks;
    ~GiveBack() {
      const bool unused = hipStreamSynchronize(s) == hipSuccess;
      for (nts::DeviceBlock *b : blocks) (void)b->give(unused);
    }
  } give_back{stream, {&work, &work2, &sort_work, &sorted_block, &ids_block}};
  NTS_HIP_TRY(work.take(3 * cell_words + 6 * row_words + 256 + tmp1_bytes));
  unsigned char *cursor = work.as<unsigned char>();
  auto take = [&cursor](size_t bytes) {
    unsigned char *q = cursor;
    cursor += bytes;
    return q;
  };
  uint32_t *counts = reinterpret_cast<uint32_t *>(take(cell_words));
  uint32_t *stops = reinterpret_cast<uint32_t *>(take(cell_words));
  uint32_t *slot_base = reinterpret_cast<uint32_t *>(take(cell_words));
  uint32_t *whole_key = reinterpret_cast<uint32_t *>(take(row_words));
  uint32_t *split_key = reinterpret_cast<uint32_t *>(take(row_words));
  uint32_t *key_sorted = reinterpret_cast<uint32_t *>(take(row_words));
  uint32_t *whole_order = reinterpret_cast<uint32_t *>(take(row_words));
  uint32_t *split_order = reinterpret_cast<uint32_t *>(take(row_words));
  unsigned char *unsorted = take(row_words);  // a byte per row
  nts::PlanCounters *counters = reinterpret_cast<nts::PlanCounters *>(take(256));
  void *tmp1 = take(tmp1_bytes);

  NTS_HIP_TRY(hipMemsetAsync(counts, 0, (cells + 1) * sizeof(uint32_t), stream));
  NTS_HIP_TRY(hipMemsetAsync(counters, 0, sizeof(nts::PlanCounters), stream));
  NTS_HIP_TRY(hipMemsetAsync(unsorted, 0, rows, stream));
  const uint32_t row_blocks = nts::ceil_div(static_cast<uint64_t>(rows) + 1, 256);
  nts::PlanCounters host_counters;
  auto read_counters = [&]() -> hipError_t {
    hipError_t e = hipMemcpyAsync(&host_counters, counters, sizeof(host_counters), hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  };
  // Nothing follows the offsets before they are known to be in bounds.
  hipLaunchKernelGGL(nts::plan_check_offsets_kernel, dim3(std::min(row_blocks, nts::kCheckBlocks)), dim3(256), 0, stream,
                     offsets, rows, edges, counters);
  NTS_LAUNCH_CHECK("plan_check_offsets_kernel");
  NTS_HIP_TRY(read_counters());
  if (host_counters.bad_total) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create: offsets[rows] != edges");
  if (host_counters.bad_offsets) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create: offsets not ascending");
  if (host_counters.first_edge) {
    *fell_back = true;
    return NTS_OK;
  }
  const uint32_t edge_blocks = std::min(nts::ceil_div(edges, 1024), 2048u);
  auto scan_edges = [&](const uint32_t *idx) -> hipError_t {
    hipLaunchKernelGGL(nts::plan_scan_edges_kernel, dim3(edge_blocks), dim3(256), 0, stream, offsets, idx, rows, edges,
                       sh.wide_ranges ? chunk / 4 : chunk, unsorted, counters);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? read_counters() : e;
  };
  NTS_HIP_TRY(scan_edges(indices));
  if (host_counters.unsorted_long_row) {
    unsigned index_bits = 1, row_bits = 1;
    const uint64_t index_range = host_counters.largest_index - index_base;  // 32-bit difference: at most 32 bits
    while (index_range >> index_bits) ++index_bits;
    while (static_cast<uint64_t>(rows - 1) >> row_bits) ++row_bits;
    unsigned local_bits = 1;
    while (static_cast<uint64_t>(host_counters.longest_row - 1) >> local_bits) ++local_bits;
    // The sort of whole tiles where a row, an index and a place in the row fit an element.
    const bool tiled = edges >= nts::kTiledSortEdges && row_bits + index_bits + local_bits <= 64 && local_bits < 32;
    unsigned long long *nul64 = nullptr;
    size_t sort_edges_bytes = nts::sort_table_bytes(edges);
    rocprim::counting_iterator<uint32_t> ids_in(0u);
    if (!tiled)
      NTS_HIP_TRY(rocprim::radix_sort_pairs(nullptr, sort_edges_bytes, nul64, nul64, ids_in, nul, edges, 0u,
                                            index_bits + row_bits, stream, false));
    const size_t key_bytes = nts::up256(static_cast<size_t>(edges) * sizeof(unsigned long long));
    hipError_t taken = sorted_block.take(static_cast<size_t>(edges) * sizeof(uint32_t));
    if (taken == hipSuccess) taken = ids_block.take(static_cast<size_t>(edges) * sizeof(uint32_t));
    if (taken == hipSuccess) taken = sort_work.take(2 * key_bytes + nts::up256(sort_edges_bytes));
    if (taken == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      *fell_back = true;
      return NTS_OK;
    }
    NTS_HIP_TRY(taken);
    uint32_t *sorted_idx = sorted_block.as<uint32_t>(), *edge_ids = ids_block.as<uint32_t>();
    unsigned char *sort_bytes = sort_work.as<unsigned char>();
    unsigned long long *keys = reinterpret_cast<unsigned long long *>(sort_bytes);
    unsigned long long *keys_out = reinterpret_cast<unsigned long long *>(sort_bytes + key_bytes);
    hipLaunchKernelGGL(nts::plan_sort_keys_kernel, dim3(edge_blocks), dim3(256), 0, stream, keys, offsets, indices,
                       index_base, rows, edges, unsorted, index_bits, tiled ? local_bits : 0u);
    NTS_LAUNCH_CHECK("plan_sort_keys_kernel");
    if (tiled) {
      const nts::TakeSorted take{sorted_idx, edge_ids, offsets, indices, unsorted, index_base,
                                 static_cast<uint32_t>((1ull << index_bits) - 1), index_bits, local_bits};
      NTS_HIP_TRY(nts::sort_elements(keys, keys, keys_out, edges, local_bits, index_bits + row_bits,
                                     sort_bytes + 2 * key_bytes, stream, [&](nts::SortElement *) { return take; }));
    } else {
      NTS_HIP_TRY(rocprim::radix_sort_pairs(sort_bytes + 2 * key_bytes, sort_edges_bytes, keys, keys_out, ids_in, edge_ids,
                                            edges, 0u, index_bits + row_bits, stream, false));
      hipLaunchKernelGGL(nts::plan_take_indices_kernel, dim3(edge_blocks), dim3(256), 0, stream, sorted_idx, keys_out,
                         indices, index_base, edge_ids, edges, unsorted, index_bits);
      NTS_LAUNCH_CHECK("plan_take_indices_kernel");
    }
    indices = sorted_idx;
    index_base = 0;
    NTS_HIP_TRY(hipMemsetAsync(counters, 0, sizeof(nts::PlanCounters), stream));
    NTS_HIP_TRY(scan_edges(indices));  // counts the repeated edges of the copy
  }
  // (16 threads a row are more than a launch can have from 2^28 rows up)
  hipLaunchKernelGGL(nts::plan_cut_rows_kernel, dim3(std::min(nts::ceil_div(rows, 256 / nts::kCutLanes), 1u << 20)), dim3(256), 0, stream, counts,
                     stops, offsets, indices, index_base, rows, sh);
  NTS_LAUNCH_CHECK("plan_cut_rows_kernel");
  NTS_HIP_TRY(rocprim::exclusive_scan(tmp1, scan_bytes, counts, slot_base, 0u, cells + 1, rocprim::plus<uint32_t>(),
                                      stream, false));
  hipLaunchKernelGGL(nts::plan_row_keys_kernel, dim3(row_blocks), dim3(256), 0, stream, whole_key, split_key, slot_base,
                     offsets, rows, sh, counters);
  NTS_LAUNCH_CHECK("plan_row_keys_kernel");
  uint32_t n_pieces = 0;
  NTS_HIP_TRY(hipMemcpyAsync(&n_pieces, slot_base + cells, sizeof(n_pieces), hipMemcpyDeviceToHost, stream));
  NTS_HIP_TRY(read_counters());
  const uint32_t n_splits = host_counters.n_splits, n_whole = rows - n_splits;
  const uint64_t n_items64 = static_cast<uint64_t>(n_pieces) + n_whole;
  if (n_items64 > 0xFFFFFFF0ull) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create_slabs: too many work items");

  nts_spmm_plan *p = new (std::nothrow) nts_spmm_plan();
  if (!p) return nts::fail(NTS_ERR_NOMEM, "nts_spmm_plan_create_slabs: host allocation failed");
  p->rows = rows;
  p->edges = edges;
  p->chunk = chunk;
  p->offsets = offsets;
  p->n_items = static_cast<uint32_t>(n_items64);
  p->n_splits = n_splits;
  p->n_partials = n_pieces;
  p->n_index = n_index;
  p->repeated_edges = host_counters.repeated;
  p->dup_runs = edges > 0 && p->repeated_edges * 20 >= edges;
  p->ranged = true;
  auto bail = [&](hipError_t err, const char *what) {
    nts_spmm_plan_destroy(p);
    return nts::fail_hip(err, what);
  };
  hipError_t err = hipEventCreateWithFlags(&p->done, hipEventDisableTiming);
  if (err == hipSuccess) err = p->items_block.take(p->n_items * sizeof(uint4));
  if (err == hipSuccess) err = p->splits_block.take(n_splits * sizeof(uint4));
  p->items = p->items_block.as<uint4>();
  p->splits = p->splits_block.as<uint4>();
  if (err != hipSuccess) return bail(err, "nts_spmm_plan_create_slabs: device allocation");

  if (n_pieces) {
    size_t sort_pieces_bytes = 0;
    err = rocprim::radix_sort_pairs(nullptr, sort_pieces_bytes, nul, nul, rocprim::counting_iterator<uint32_t>(0u), nul,
                                    n_pieces, 0u, key_bits, stream, false);
    if (err != hipSuccess) return bail(err, "nts_spmm_plan_create_slabs: sort size");
    const size_t piece_items = nts::up256(static_cast<size_t>(n_pieces) * sizeof(Item));
    const size_t piece_words = nts::up256(static_cast<size_t>(n_pieces) * sizeof(uint32_t));
    err = work2.take(piece_items + 3 * piece_words + nts::up256(sort_pieces_bytes));
    if (err != hipSuccess) return bail(err, "nts_spmm_plan_create_slabs: device allocation");
    unsigned char *work2_bytes = work2.as<unsigned char>();
    Item *pieces = reinterpret_cast<Item *>(work2_bytes);
    uint32_t *keys = reinterpret_cast<uint32_t *>(work2_bytes + piece_items);
    uint32_t *keys_sorted = reinterpret_cast<uint32_t *>(work2_bytes + piece_items + piece_words);
    uint32_t *order = reinterpret_cast<uint32_t *>(work2_bytes + piece_items + 2 * piece_words);
    void *tmp2 = work2_bytes + piece_items + 3 * piece_words;
    hipLaunchKernelGGL(nts::plan_emit_pieces_kernel, dim3(nts::ceil_div(cells, 256)), dim3(256), 0, stream, pieces, keys,
                       counts, stops, slot_base, offsets, rows, sh);
    err = hipGetLastError();
    if (err == hipSuccess)
      err = rocprim::radix_sort_pairs(tmp2, sort_pieces_bytes, keys, keys_sorted, rocprim::counting_iterator<uint32_t>(0u),
                                      order, n_pieces, 0u, key_bits, stream, false);
    if (err != hipSuccess) return bail(err, "nts_spmm_plan_create_slabs: ordering of the pieces");
    hipLaunchKernelGGL(nts::auto_order_items_kernel, dim3(nts::ceil_div(n_pieces, 256)), dim3(256), 0, stream, p->items,
                       pieces, order, n_pieces);
  }
  err = rocprim::radix_sort_pairs(tmp1, sort_rows_bytes, whole_key, key_sorted, rocprim::counting_iterator<uint32_t>(0u),
                                  whole_order, rows, 0u, whole_bits, stream, false);
  if (err == hipSuccess)
    err = rocprim::radix_sort_pairs(tmp1, sort_rows_bytes, split_key, key_sorted, rocprim::counting_iterator<uint32_t>(0u),
                                    split_order, rows, 0u, 32u, stream, false);
  if (err != hipSuccess) return bail(err, "nts_spmm_plan_create_slabs: ordering of the rows");
  if (n_whole || n_splits)
    hipLaunchKernelGGL(nts::plan_finish_kernel, dim3(nts::ceil_div(std::max(n_whole, n_splits), 256)), dim3(256), 0, stream,
                       p->items, p->splits, whole_order, split_order, slot_base, offsets, n_pieces, n_whole, n_splits,
                       n_slabs);
  err = hipGetLastError();
  if (err == hipSuccess) err = hipStreamSynchronize(stream);
  if (err != hipSuccess) return bail(err, "nts_spmm_plan_create_slabs: device schedule");
  p->sorted_block.swap(sorted_block);
  p->ids_block.swap(ids_block);
  p->sorted_idx = p->sorted_block.as<uint32_t>();
  p->edge_ids = p->ids_block.as<uint32_t>();
  *plan_out = p;
  return NTS_OK;
}

int read_offsets(std::vector<uint32_t> &off, const uint32_t *offsets, uint32_t rows, uint32_t edges,
                 hipStream_t stream) {
  off.assign(static_cast<size_t>(rows) + 1, 0u);
  if (!rows) return NTS_OK;
  NTS_HIP_TRY(hipMemcpyAsync(off.data(), offsets, off.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
  NTS_HIP_TRY(hipStreamSynchronize(stream));
  if (off[rows] != edges) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create: offsets[rows] != edges");
  for (uint32_t r = 0; r < rows; ++r)
    if (off[r + 1] < off[r]) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create: offsets not ascending");
  return NTS_OK;
}

}  // namespace

int nts_spmm_plan_create(nts_spmm_plan_t **plan_out, const uint32_t *offsets, uint32_t rows, uint32_t edges,
                         uint32_t chunk_edges, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_plan_create");
  if (!plan_out) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create: null out-pointer");
  *plan_out = nullptr;
  if (rows != 0 && !offsets) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create: null offsets");
  std::vector<uint32_t> off;
  if (int rc = read_offsets(off, offsets, rows, edges, stream)) return rc;
  return build_plan(plan_out, offsets, off, nullptr, rows, edges, chunk_edges ? chunk_edges : default_chunk(edges), 1u, 0u);
}

int nts_spmm_plan_create_slabs(nts_spmm_plan_t **plan_out, const uint32_t *offsets, const uint32_t *indices,
                               uint32_t index_base, uint32_t n_index, uint32_t rows, uint32_t edges,
                               uint32_t chunk_edges, uint32_t n_slabs, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_plan_create_slabs");
  if (!plan_out) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create_slabs: null out-pointer");
  *plan_out = nullptr;
  if (rows != 0 && !offsets) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create_slabs: null offsets");
  if (edges != 0 && !indices) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_create_slabs: null indices");
  const uint32_t chunk = chunk_edges ? chunk_edges : 512u, slabs = n_slabs ? n_slabs : 32u;
  // The schedule is built on the device where that reproduces the host's (source ranges in use, sizes
  // within the 32-bit sort keys and the range table, rows from edge 0 on); NTS_SPMM_PLAN_HOST=1 forces the host path.
  static const bool force_host = [] {
    const char *e = getenv("NTS_SPMM_PLAN_HOST");
    return e && e[0] != '0';
  }();
  if (!force_host && slabs > 1 && n_index > 0 && rows > 0 && edges > 0 &&
      static_cast<uint64_t>(slabs) * (static_cast<uint64_t>(chunk) + 1) < (1ull << 32) && slabs <= 4096 &&
      static_cast<uint64_t>(rows) * slabs < (1ull << 31)) {
    bool fell_back = false;
    const int rc = build_plan_device(plan_out, offsets, indices, index_base, n_index, rows, edges, chunk, slabs, stream,
                                     &fell_back);
    if (rc || !fell_back) return rc;
  }
  std::vector<uint32_t> off;
  if (int rc = read_offsets(off, offsets, rows, edges, stream)) return rc;
  std::vector<uint32_t> idx(edges);
  if (edges) {
    NTS_HIP_TRY(hipMemcpyAsync(idx.data(), indices, idx.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    NTS_HIP_TRY(hipStreamSynchronize(stream));
    if (index_base)
      for (uint32_t &v : idx) v -= index_base;
  }
  return build_plan(plan_out, offsets, off, idx.data(), rows, edges, chunk, slabs, n_index);
}

int nts_spmm_plan_schedule_host(const uint32_t *offsets_host, const uint32_t *indices_host, uint32_t n_index,
                                uint32_t rows, uint32_t chunk_edges, uint32_t n_slabs, uint32_t *items_out,
                                uint64_t items_cap, uint32_t *n_items, uint32_t *n_split_rows, uint32_t *n_partials) {
  if (rows != 0 && !offsets_host) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_schedule_host: null offsets");
  for (uint32_t r = 0; r < rows; ++r)
    if (offsets_host[r + 1] < offsets_host[r])
      return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_schedule_host: offsets not ascending");
  if (rows && offsets_host[rows] != 0 && n_slabs > 1 && !indices_host)
    return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_schedule_host: null indices");
  Schedule sched;
  const bool with_ranges = indices_host != nullptr;
  const uint32_t edges = rows ? offsets_host[rows] : 0u;
  make_schedule(sched, offsets_host, indices_host, rows,
                chunk_edges ? chunk_edges : (with_ranges ? 512u : default_chunk(edges)),
                with_ranges ? (n_slabs ? n_slabs : 32u) : 1u, n_index);
  if (n_items) *n_items = static_cast<uint32_t>(sched.items.size());
  if (n_split_rows) *n_split_rows = static_cast<uint32_t>(sched.splits.size());
  if (n_partials) *n_partials = sched.n_partials;
  if (items_out) {
    if (items_cap < sched.items.size())
      return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_schedule_host: items_out too small");
    memcpy(items_out, sched.items.data(), sched.items.size() * sizeof(uint4));
  }
  return NTS_OK;
}

int nts_spmm_plan_destroy(nts_spmm_plan_t *plan) {
  NTS_TRACE_RANGE("nts_spmm_plan_destroy");
  if (!plan) return NTS_OK;
  { std::lock_guard<std::mutex> lock(plan->mu); }  // a call that is still enqueueing finishes first
  // Work queued on any stream of the plan's device may still read the arrays.
  const hipError_t given = nts::retire_blocks({&plan->items_block, &plan->splits_block, &plan->sorted_block,
                                               &plan->ids_block, plan->scratch.partial_block(), plan->scratch.copy_block()});
  const hipError_t event = plan->done ? hipEventDestroy(plan->done) : hipSuccess;
  delete plan;
  if (given != hipSuccess) return nts::fail_hip(given, "nts_spmm_plan_destroy");
  if (event != hipSuccess) return nts::fail_hip(event, "nts_spmm_plan_destroy");
  return NTS_OK;
}

int nts_spmm_plan_copy_schedule(const nts_spmm_plan_t *plan, uint32_t *items_out, uint64_t items_cap,
                                uint32_t *splits_out, uint64_t splits_cap) {
  NTS_TRACE_RANGE("nts_spmm_plan_copy_schedule");
  if (!plan) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_copy_schedule: null plan");
  if (items_out) {
    if (items_cap < plan->n_items) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_copy_schedule: items_out too small");
    if (plan->n_items)
      NTS_HIP_TRY(hipMemcpy(items_out, plan->items, plan->n_items * sizeof(uint4), hipMemcpyDeviceToHost));
  }
  if (splits_out) {
    if (splits_cap < plan->n_splits)
      return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_copy_schedule: splits_out too small");
    if (plan->n_splits)
      NTS_HIP_TRY(hipMemcpy(splits_out, plan->splits, plan->n_splits * sizeof(uint4), hipMemcpyDeviceToHost));
  }
  return NTS_OK;
}

int nts_spmm_plan_info(const nts_spmm_plan_t *plan, uint32_t *items, uint32_t *split_rows, uint32_t *partials) {
  NTS_TRACE_RANGE("nts_spmm_plan_info");
  if (!plan) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_info: null plan");
  if (items) *items = plan->n_items;
  if (split_rows) *split_rows = plan->n_splits;
  if (partials) *partials = plan->n_partials;
  return NTS_OK;
}

namespace {

// Row stride, in floats, of the padded input copy and of the partial sums for width F: rows of more
// than 128 floats that do not start on 16-byte boundaries can be gathered from a copy whose rows are
// padded to a multiple of 32 floats (whole 128-byte lines), so that the gather runs with 16-byte
// lanes -- three loads per neighbour row at F = 602 instead of ten.  0 = no copy (F itself is the
// stride).  Measured on the 114.8 M-edge R-MAT graph at F = 602: with one load per run of equal
// indices the copy pays (9.75 -> 9.21 ms per pass, the 0.25 ms copy not included; 25.7 -> 25.0 ms per
// four-pass step with it); without runs it does not (11.05 -> 11.7 ms, and 8.79 -> 8.93 ms on the same
// graph with its parallel edges removed), but column panels of whole lines do (panel_lanes, which has the figures), for rows
// of more than 256 floats: the copy costs two passes over the gathered matrix, the panels save a tenth of the gather, so
// there have to be 48 edges a gathered row, or 24 where rows are wider than 512 floats (300 floats 300 K rows, 10 M edges 1,082 ->
// 1,114 us, 1 M, 40 M 4,226 -> 4,275; 500 1 M, 24 M 5,213 -> 5,068, 450 4,664 -> 4,868; 602 2.45 M, 40 M 12,905 -> 14,108).
// NTS_SPMM_PAD=0 / 1 in the environment forces it off / on.
uint32_t padded_stride(const nts_spmm_plan *plan, uint32_t F) {
  static const int forced = [] {
    const char *e = getenv("NTS_SPMM_PAD");
    return e ? (e[0] != '0' ? 1 : 0) : -1;
  }();
  if (plan->n_index == 0 || F <= 128 || forced == 0) return 0;
  const uint32_t padded = (F + 31) / 32 * 32;
  if (forced == 1 || plan->dup_runs) return F % 4 ? padded : 0u;
  const uint64_t least = F > 512 ? 24 : 48;
  return plan->ranged && F > 256 && F < padded && padded <= 32 * nts::kMaxPanelLines && plan->edges >= least * plan->n_index ? padded : 0u;
}

// NTS_SPMM_RUNS=0 / 1 forces the one-load-per-run kernel off / on whatever the schedule found.
bool use_runs(const nts_spmm_plan *plan) {
  static const int forced = [] {
    const char *e = getenv("NTS_SPMM_RUNS");
    return e ? (e[0] != '0' ? 1 : 0) : -1;
  }();
  return forced < 0 ? plan->dup_runs : forced == 1;
}

nts::ScratchNeed scratch_need(const nts_spmm_plan *plan, uint32_t F) {
  return {plan->n_partials, F, padded_stride(plan, F), plan->n_index};
}

// Makes room in the plan's scratch for a call of width F and leaves the call's row stride (padded_stride) in *stride: 0 where it
// gathers from the rows as they are, with the same sums (PlanScratch::place).  Caller holds plan->mu.
int reserve_locked(nts_spmm_plan *plan, uint32_t F, bool heads, bool recorded, uint32_t *stride) {
  size_t ld = 0;
  NTS_HIP_TRY(plan->scratch.place(scratch_need(plan, F), !heads, recorded, &ld));
  *stride = static_cast<uint32_t>(ld);
  return NTS_OK;
}

// A call on `stream` is about to use the plan's scratch: if the previous call ran on another stream,
// `stream` first waits for it (in stream order, the host does not block).  Caller holds plan->mu.
// A stream that is being captured records its launches instead of running them: a call under capture
// neither waits for the plan's event (that would pull the other stream's work into the capture, or
// fail) nor records it, and leaves the plan's bookkeeping alone -- replays of the captured call are
// ordered against other uses of the plan by the caller.
bool stream_is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return status != hipStreamCaptureStatusNone;
}
int enter_stream(nts_spmm_plan *plan, hipStream_t stream) {
  if (stream_is_capturing(stream)) return NTS_OK;
  if (plan->in_flight && plan->last_stream != stream) NTS_HIP_TRY(hipStreamWaitEvent(stream, plan->done, 0));
  return NTS_OK;
}
int leave_stream(nts_spmm_plan *plan, hipStream_t stream) {
  if (stream_is_capturing(stream)) return NTS_OK;
  NTS_HIP_TRY(hipEventRecord(plan->done, stream));
  plan->last_stream = stream;
  plan->in_flight = true;
  return NTS_OK;
}

}  // namespace

int nts_spmm_plan_scratch_info(nts_spmm_plan_t *plan, uint32_t F, size_t *partial_bytes, size_t *padded_input_bytes,
                               uint64_t *repeated_edges, int *loads_once_per_run) {
  NTS_TRACE_RANGE("nts_spmm_plan_scratch_info");
  if (!plan) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_scratch_info: null plan");
  if (F == 0) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_scratch_info: F is 0");
  std::lock_guard<std::mutex> lock(plan->mu);
  const size_t ld = plan->scratch.stride_of(scratch_need(plan, F));
  if (partial_bytes) *partial_bytes = static_cast<size_t>(plan->n_partials) * (ld ? ld : F) * sizeof(float);
  if (padded_input_bytes) *padded_input_bytes = ld ? static_cast<size_t>(plan->n_index) * ld * sizeof(float) : 0;
  if (repeated_edges) *repeated_edges = plan->repeated_edges;
  if (loads_once_per_run) *loads_once_per_run = use_runs(plan) ? 1 : 0;
  return NTS_OK;
}

int nts_spmm_plan_reserve(nts_spmm_plan_t *plan, uint32_t F) {
  NTS_TRACE_RANGE("nts_spmm_plan_reserve");
  if (!plan) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_reserve: null plan");
  if (F == 0) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_reserve: F is 0");
  std::lock_guard<std::mutex> lock(plan->mu);
  plan->scratch.ask_again();
  uint32_t ld = 0;
  return reserve_locked(plan, F, false, false, &ld);
}

namespace {
int check_heads(const float *alpha, uint32_t H, uint32_t Fh, const char *who) {
  if (H == 0 || Fh == 0) return nts::fail(NTS_ERR_INVALID, who);
  if (static_cast<uint64_t>(H) * Fh > 0xFFFFFFFFull) return nts::fail(NTS_ERR_INVALID, who);
  if (!alpha) return nts::fail(NTS_ERR_INVALID, who);
  return NTS_OK;
}
}  // namespace

int nts_spmm_gather_heads(const float *in, float *out, const float *alpha, const uint32_t *perm,
                          const uint32_t *offsets, const uint32_t *indices, uint32_t rows, uint32_t edges, uint32_t H,
                          uint32_t Fh, int accumulate, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_gather_heads");
  if (int rc = check_heads(alpha, H, Fh, "nts_spmm_gather_heads: bad H / Fh / alpha")) return rc;
  if (rows == 0) return NTS_OK;
  if (!in || !out || !offsets || !indices) return nts::fail(NTS_ERR_INVALID, "nts_spmm_gather_heads: null pointer");
  nts::LaunchArgs a{in, out, alpha, offsets, indices, 0u, rows, H * Fh, nullptr, nullptr, accumulate, stream};
  a.heads = nts::HeadArgs{perm, H, Fh};
  if (int rc = nts::launch_spmm_balanced(a, edges)) return rc;
  NTS_LAUNCH_CHECK("nts_spmm_gather_heads");
  return NTS_OK;
}

int nts_spmm_gather_heads_bounded(const float *in, float *out, const float *alpha, const uint32_t *perm,
                                  const uint32_t *offsets, const uint32_t *indices, uint32_t rows, uint32_t edges,
                                  uint32_t H, uint32_t Fh, int accumulate, uint32_t max_row_edges, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_gather_heads_bounded");
  if (int rc = check_heads(alpha, H, Fh, "nts_spmm_gather_heads_bounded: bad H / Fh / alpha")) return rc;
  if (rows == 0) return NTS_OK;
  if (!in || !out || !offsets || !indices)
    return nts::fail(NTS_ERR_INVALID, "nts_spmm_gather_heads_bounded: null pointer");
  nts::LaunchArgs a{in, out, alpha, offsets, indices, 0u, rows, H * Fh, nullptr, nullptr, accumulate, stream};
  a.heads = nts::HeadArgs{perm, H, Fh};
  if (max_row_edges != 0 && max_row_edges <= nts::kAutoChunk) {
    a.edges = edges;
    a.bounded = true;
    nts::launch_spmm(a);
  } else if (int rc = nts::launch_spmm_balanced(a, edges)) {
    return rc;
  }
  NTS_LAUNCH_CHECK("nts_spmm_gather_heads_bounded");
  return NTS_OK;
}

int nts_gat_aggregate_bwd(float *gx, float *galpha, const float *x, const float *gout, const float *alpha,
                          const uint32_t *perm, const uint32_t *ro, const uint32_t *ci, const uint32_t *co,
                          const uint32_t *ri, uint32_t Vd, uint32_t Vs, uint32_t edges, uint32_t H, uint32_t Fh,
                          int accumulate, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_gat_aggregate_bwd");
  if (H == 0 || Fh == 0) return nts::fail(NTS_ERR_INVALID, "nts_gat_aggregate_bwd: H or Fh is 0");
  if (static_cast<uint64_t>(H) * Fh > 0xFFFFFFFFull) return nts::fail(NTS_ERR_INVALID, "nts_gat_aggregate_bwd: H*Fh overflows");
  if (Vs == 0) return NTS_OK;
  if (!gx || !ro || (edges && (!galpha || !x || !gout || !alpha || !ci)))
    return nts::fail(NTS_ERR_INVALID, "nts_gat_aggregate_bwd: null pointer");
  nts::LaunchArgs a{gout, gx, alpha, ro, ci, 0u, Vs, H * Fh, nullptr, nullptr, accumulate, stream};
  a.heads = nts::HeadArgs{perm, H, Fh};
  a.dot_rows = x;
  a.dot_out = galpha;
  if (!edges || !perm || !nts::attention_grad_takes(a) ||
      (co && ri && nts::separate_gradients_are_faster(a, edges))) {
    // Heads wider than the fused kernel's lanes, a structure without its edge permutation, or a size at which it is
    // faster: one pass per gradient.
    if (edges)
      if (int rc = nts_sddmm_heads(galpha, x, gout, co, ri, Vd, H, Fh, stream)) return rc;
    a.dot_rows = nullptr;
    a.dot_out = nullptr;
  }
  if (int rc = nts::launch_spmm_balanced(a, edges)) return rc;
  NTS_LAUNCH_CHECK("nts_gat_aggregate_bwd");
  return NTS_OK;
}

int nts_spmm_gather_heads_planned(nts_spmm_plan_t *plan, const float *in, float *out, const float *alpha,
                                  const uint32_t *perm, const uint32_t *offsets, const uint32_t *indices, uint32_t H,
                                  uint32_t Fh, int accumulate, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_gather_heads_planned");
  if (!plan) return nts::fail(NTS_ERR_INVALID, "nts_spmm_gather_heads_planned: null plan");
  if (offsets != plan->offsets)
    return nts::fail(NTS_ERR_INVALID,
                     "nts_spmm_gather_heads_planned: offsets differ from the array the plan was built from");
  if (int rc = check_heads(alpha, H, Fh, "nts_spmm_gather_heads_planned: bad H / Fh / alpha")) return rc;
  const uint32_t F = H * Fh;
  if (int rc = nts::check_common(in, out, offsets, indices, plan->rows, plan->edges, F,
                                 "nts_spmm_gather_heads_planned: null pointer"))
    return rc;
  if (plan->rows == 0) return NTS_OK;
  std::lock_guard<std::mutex> lock(plan->mu);
  uint32_t ld = 0;
  if (int rc = reserve_locked(plan, F, true, stream_is_capturing(stream), &ld)) return rc;
  if (int rc = enter_stream(plan, stream)) return rc;
  nts::LaunchArgs a{in,  out,         alpha,         offsets,    indices, 0u, plan->n_items,
                    F,   plan->items, plan->scratch.partial(), accumulate, stream};
  a.heads = nts::HeadArgs{perm, H, Fh};
  a.scheduled_rows = plan->rows;
  a.ranged = plan->ranged;
  a.edges = plan->edges;
  if (plan->sorted_idx) {
    a.indices = plan->sorted_idx;
    a.edge_ids = plan->edge_ids;
  }
  nts::launch_spmm(a);
  NTS_LAUNCH_CHECK("nts_spmm_gather_heads_planned");
  if (plan->n_splits) {
    nts::launch_reduce_partials(out, plan->scratch.partial(), plan->splits, plan->n_splits, F, accumulate, stream);
    NTS_LAUNCH_CHECK("spmm_reduce_partials_kernel");
  }
  return leave_stream(plan, stream);
}

int nts_spmm_plan_set_events(nts_spmm_plan_t *plan, nts_event_t start, nts_event_t stop) {
  NTS_TRACE_RANGE("nts_spmm_plan_set_events");
  if (!plan) return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_set_events: null plan");
  if ((start == nullptr) != (stop == nullptr))
    return nts::fail(NTS_ERR_INVALID, "nts_spmm_plan_set_events: pass both events or neither");
  plan->ev_start = start;
  plan->ev_stop = stop;
  return NTS_OK;
}

int nts_spmm_gather_planned(nts_spmm_plan_t *plan, const float *in, float *out, const float *w,
                            const uint32_t *offsets, const uint32_t *indices, uint32_t index_base, uint32_t F,
                            int accumulate, nts_stream_t stream) {
  NTS_TRACE_RANGE("nts_spmm_gather_planned");
  if (!plan) return nts::fail(NTS_ERR_INVALID, "nts_spmm_gather_planned: null plan");
  if (offsets != plan->offsets)
    return nts::fail(NTS_ERR_INVALID, "nts_spmm_gather_planned: offsets differ from the array the plan was built from");
  if (int rc = nts::check_common(in, out, offsets, indices, plan->rows, plan->edges, F,
                                 "nts_spmm_gather_planned: null pointer"))
    return rc;
  if (plan->rows == 0) return NTS_OK;
  std::lock_guard<std::mutex> lock(plan->mu);
  uint32_t ld = 0;
  if (int rc = reserve_locked(plan, F, false, stream_is_capturing(stream), &ld)) return rc;
  if (int rc = enter_stream(plan, stream)) return rc;
  nts::LaunchArgs a{in,  out,         w,           offsets,       indices,   index_base, plan->n_items,
                    F,   plan->items, plan->scratch.partial(), accumulate, stream};
  if (plan->sorted_idx) {  // the schedule's own copy of the indices, base already subtracted
    a.indices = plan->sorted_idx;
    a.index_base = 0;
    a.edge_ids = plan->edge_ids;
  }
  a.dup_runs = use_runs(plan);
  a.scheduled_rows = plan->rows;
  a.ranged = plan->ranged;
  a.edges = plan->edges;
  if (ld) {
    // Rows off whole lines: gather from a padded copy.
    const uint64_t vecs = static_cast<uint64_t>(plan->n_index) * (ld / 4);
    const uint32_t blocks = static_cast<uint32_t>(std::min<uint64_t>((vecs + 255) / 256, 1u << 16));
    hipLaunchKernelGGL(nts::pad_rows_kernel, dim3(blocks), dim3(256), 0, stream,
                       reinterpret_cast<float4 *>(plan->scratch.copy()), in, plan->n_index, F, ld);
    NTS_LAUNCH_CHECK("pad_rows_kernel");
    a.in = plan->scratch.copy();
    a.in_ld = ld;
    a.partial_ld = ld;
  }
  if (plan->ev_start && plan->ev_stop) NTS_HIP_TRY(hipEventRecord(plan->ev_start, stream));
  nts::launch_spmm(a);
  NTS_LAUNCH_CHECK("nts_spmm_gather_planned");
  if (plan->ev_start && plan->ev_stop) NTS_HIP_TRY(hipEventRecord(plan->ev_stop, stream));
  if (plan->n_splits) {
    nts::launch_reduce_partials(out, plan->scratch.partial(), plan->splits, plan->n_splits, F, accumulate, stream, a.partial_ld);
    NTS_LAUNCH_CHECK("spmm_reduce_partials_kernel");
  }
  return leave_stream(plan, stream);
}

}  // extern "C"
