// Gather (Arrow `take`) for CDNA4: out[i] = values[indices[i]].
//
// Semantics follow the reference (Sources/ArrowMetal/Kernels/Take.swift:41-80,
// KernelSource.swift:209-227): a null index gives a null output, a null source element gives a null,
// and an index outside [0, length) makes the call fail with "take: index out of range (array length
// N)" once the kernel has run. Each wave handles 64 consecutive outputs, so the output validity is one
// 64-bit ballot per wave, written as one word; nulls are counted per workgroup, without atomics. Large random
// gathers run in three passes by source slice, and whole tables are gathered as rows (both below).
#include "am_internal.hpp"

#include <algorithm>

namespace am {
namespace {

// In pinned host memory: the kernel stores the flag only when an index is out of range, and the null
// count is written by take_nulls, so a take without nulls is one launch.
struct TakeStatus {
  unsigned int out_of_range;
  unsigned int pad;
  unsigned long long nulls;
};

__device__ const uint8_t kTakeAllValid = 0xFFu;

// Four 64-row groups per wave per step, whose index loads and then gathers are issued together: each
// gather is a line of its own, so the step waits for one memory latency, not four.
constexpr int TAKE_GROUPS = 4;

// Bit `bit` (0 for a column without a bitmap, which reads the all-valid byte) of a validity byte.
__device__ __forceinline__ uint32_t take_vbyte(const uint8_t* valid, int64_t b) {
  return load_global(valid ? valid + (b >> 3) : &kTakeAllValid) >> uint32_t(b & 7);
}

// NULLS: the indices or the values have nulls; the null count of each workgroup goes to block_nulls. (A
// counter that every wave bumps is one memory-side atomic per 64 rows on one address: it took 150 us of
// 4M rows' 160.)
template <typename V, typename I, bool NULLS>
__device__ __forceinline__ void take_rows(const V* __restrict__ vals, const uint8_t* __restrict__ vvalid, int64_t voff,
                                          int64_t len, const I* __restrict__ idx, const uint8_t* __restrict__ ivalid,
                                          int64_t ioff, int64_t n, V* __restrict__ out,
                                          unsigned long long* __restrict__ out_valid,
                                          uint32_t* __restrict__ block_nulls, TakeStatus* st) {
  __shared__ uint32_t s_nulls[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t step = int64_t(gridDim.x) * 256 * TAKE_GROUPS;
  uint32_t nulls = 0;
  bool bad = false;
  for (int64_t base = (int64_t(blockIdx.x) * 4 + w) * 64 * TAKE_GROUPS; base < n; base += step) {
    int64_t j[TAKE_GROUPS];
    uint32_t ok[TAKE_GROUPS], vb[TAKE_GROUPS];
    V v[TAKE_GROUPS];
#pragma unroll
    for (int g = 0; g < TAKE_GROUPS; g++) {   // rows past the end read the last index
      const int64_t i = std::min<int64_t>(base + g * 64 + lane, n - 1);
      j[g] = int64_t(idx[i]);
      ok[g] = NULLS ? take_vbyte(ivalid, ioff + i) & 1u : 1u;
    }
#pragma unroll
    for (int g = 0; g < TAKE_GROUPS; g++) {
      const bool in = j[g] >= 0 && j[g] < len;
      bad = bad || (ok[g] && !in);
      ok[g] &= in ? 1u : 0u;
      if (!ok[g]) j[g] = 0;   // len >= 1 whenever a gather is launched
      v[g] = vals[j[g]];
      vb[g] = NULLS ? take_vbyte(vvalid, voff + j[g]) : 1u;
    }
#pragma unroll
    for (int g = 0; g < TAKE_GROUPS; g++) {
      const int64_t i = base + g * 64 + lane;
      if (i < n) out[i] = ok[g] ? v[g] : V(0);
      if (NULLS) {
        const unsigned long long bal = __ballot(i < n && (ok[g] & vb[g] & 1u));
        const int64_t rows = std::min<int64_t>(64, n - (base + g * 64));
        if (rows > 0) {
          if (lane == 0) out_valid[(base >> 6) + g] = bal;
          nulls += uint32_t(rows) - uint32_t(__popcll(bal));
        }
      }
    }
  }
  if (bad) st->out_of_range = 1u;
  if (NULLS) {
    if (lane == 0) s_nulls[w] = nulls;
    __syncthreads();
    if (threadIdx.x == 0) block_nulls[blockIdx.x] = s_nulls[0] + s_nulls[1] + s_nulls[2] + s_nulls[3];
  }
}

template <typename V, typename I, bool NULLS>
__global__ __launch_bounds__(256) void take_kernel(const V* __restrict__ vals, const uint8_t* __restrict__ vvalid,
                                                   int64_t voff, int64_t len, const I* __restrict__ idx,
                                                   const uint8_t* __restrict__ ivalid, int64_t ioff, int64_t n,
                                                   V* __restrict__ out, unsigned long long* __restrict__ out_valid,
                                                   uint32_t* __restrict__ block_nulls, TakeStatus* st) {
  take_rows<V, I, NULLS>(vals, vvalid, voff, len, idx, ivalid, ioff, n, out, out_valid, block_nulls, st);
}

// A gather from an empty array: every non-null index is out of range.
template <typename I>
__global__ __launch_bounds__(256) void take_empty(const I* idx, const uint8_t* ivalid, int64_t ioff, int64_t n, char* out,
                                                  int width, unsigned long long* out_valid, uint32_t* block_nulls,
                                                  TakeStatus* st) {
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
    if (take_vbyte(ivalid, ioff + i) & 1u) st->out_of_range = 1u;
    for (int b = 0; b < width; b++) out[i * width + b] = 0;
    if (out_valid && (i & 63) == 0) out_valid[i >> 6] = 0ull;
  }
  if (block_nulls && threadIdx.x == 0) block_nulls[blockIdx.x] = blockIdx.x == 0 ? uint32_t(n) : 0u;
  (void)idx;
}

// One workgroup: the null count of the whole result, into pinned host memory.
__global__ __launch_bounds__(1024) void take_nulls(const uint32_t* block_nulls, uint32_t blocks, TakeStatus* st) {
  __shared__ unsigned long long s[16];
  unsigned long long z = 0;
  for (uint32_t b = threadIdx.x; b < blocks; b += 1024) z += block_nulls[b];
  for (int off = 32; off > 0; off >>= 1) z += __shfl_down(z, off, 64);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = z;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; w++) z += s[w];
    st->nulls = z;
  }
}

// ---------------------------------------------------------------- large random gathers
//
// A gather of random rows from a large column is bound by the 128-byte line it fetches per row, whichever
// memory that comes from: 50M float64 values took 1006 us, 6.9 GB of lines for 1 GB of data. Such a gather
// runs in three passes instead:
//   tk_split   each tile of TK_TILE outputs groups its indices by source slice (a 256th of the column), in
//              LDS: the grouped indices, each one's place in the tile, and the tile's slice offsets
//   tk_fetch   slice by slice, every tile's run of indices into it -> the values, in the grouped order. An
//              XCD's workgroups all work on one slice at a time, so a line comes from its L2, and several
//              rows of a wave may share one
//   tk_place   each tile's values to their places, through LDS
// 50M float64: 113 + 534 + 152 us, 811 us a call (1010 before); 50M float32: 117 + 453 + 88, 656 us (972). The
// fetch is still bound by L1 filling a line per row: the same loop reads neighbours in 271 us.
//
// Values and indices without nulls only: the passes carry no validity. Which way a call goes is decided on the
// device from a sample of the indices: runs of neighbours are
// cheaper read directly, and tk_fetch then is the plain gather: neighbours cost such a call
// 5 us for the two kernels that return (50M float64 187 and 196, 24M float32 65 and 68).
constexpr uint32_t TK_TILE = 16384;
constexpr uint32_t TK_SLICES = 256;
constexpr uint32_t TK_THREADS = 1024;
constexpr int TK_PER = int(TK_TILE / TK_THREADS);
constexpr uint32_t TK_FETCH_TILES = 16;   // tiles per work item of tk_fetch, four per wave
// Where the passes win over the plain gather, calls of random indices, in us (plain / three passes):
//   float32, as many rows as the source: 6M 107/115, 8M 145/131, 12M 227/177, 24M 460/335, 50M 972/656
//   float64:                             6M 125/128, 8M 165/156, 12M 249/231, 24M 487/414, 50M 1010/811
//   smaller sources, 16M rows:           float32 of 2M 167/200, of 4M 236/209; float64 of 2M 250/253, of 4M 292/261
//   larger ones:                         float32 16M of 64M 322/273, 8M of 64M 170/173; float64 333/351, 175/224
// So from 3 * 2^22 rows (below, the gain is near the 5 us that a call of neighbours loses), of a
// source of at most twice as many rows (a tile's run in a slice is short otherwise) and of 16 MiB (the
// eight L2s hold a smaller one).
template <typename V>
bool take_by_slices(int64_t n, int64_t len) {
  return n >= int64_t(3) << 22 && n <= int64_t(UINT32_MAX) - TK_TILE && len <= 2 * n && len <= int64_t(UINT32_MAX) &&
         len * int64_t(sizeof(V)) >= int64_t(1) << 24;
}

struct TkCtl {
  uint32_t scattered, pad[31];
  struct { uint32_t next, pad[31]; } item[NXCD];   // the next work item of each XCD, a line each
};

// 64 groups of 64 consecutive outputs, evenly spread, four per wave: true, for the whole workgroup, if in most
// of them at least half of the neighbours lie on different lines and half of the rows 1 MiB or more from
// the group's first. Every workgroup reads the same sample.
template <typename I>
__device__ __forceinline__ bool tk_scattered(const I* idx, int64_t n, int width, uint32_t* s_cnt) {
  const int lane = threadIdx.x & 63;
  if (threadIdx.x == 0) *s_cnt = 0u;
  __syncthreads();
  I j[4];
#pragma unroll
  for (int k = 0; k < 4; k++) j[k] = idx[(n - 64) / 63 * (int64_t(k) * 16 + (threadIdx.x >> 6)) + lane];
  uint32_t mine = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int64_t at = int64_t(uint64_t(j[k]) * uint64_t(width));   // any index, also one out of range
    const uint64_t line = uint64_t(at) >> 7, prev = __shfl_up(line, 1, 64), first = __shfl(line, 0, 64);
    const uint64_t far = uint64_t(int64_t(line - first) + 8191);    // within 8191 lines either way: at most 16382
    const uint32_t moved = uint32_t(__popcll(__ballot(line != prev))), apart = uint32_t(__popcll(__ballot(far > 16382u)));
    mine += moved >= 32u && apart >= 32u ? 1u : 0u;
  }
  if (lane == 0) atomicAdd(s_cnt, mine);
  __syncthreads();
  return *s_cnt >= 48u;
}

// Tile by tile, if the indices are scattered: off[s][tile] = where slice s starts in the tile (off[TK_SLICES][tile]: the tile's rows).
template <typename I>
__global__ __launch_bounds__(TK_THREADS) void tk_split(const I* idx, uint32_t n, int64_t len, uint32_t shift,
                                                       int width, TkCtl* ctl, uint32_t tiles, uint32_t* part_idx,
                                                       uint16_t* part_pos, uint32_t* off, TakeStatus* st) {
  __shared__ uint32_t s_cnt[TK_SLICES], s_start[TK_SLICES];
  __shared__ uint32_t s_idx[TK_TILE];
  __shared__ uint16_t s_pos[TK_TILE];
  __shared__ uint32_t s_sample;
  const bool scattered = tk_scattered(idx, int64_t(n), width, &s_sample);
  if (blockIdx.x == 0) {   // for the kernels that follow
    if (threadIdx.x == 0) ctl->scattered = scattered ? 1u : 0u;
    if (threadIdx.x < uint32_t(NXCD)) ctl->item[threadIdx.x].next = 0u;
  }
  if (!scattered) return;   // uniform over the grid
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t t0 = tile * TK_TILE, rows = min(TK_TILE, n - t0);
    if (threadIdx.x < TK_SLICES) s_cnt[threadIdx.x] = 0u;
    __syncthreads();   // also: the tile before has been written out
    uint32_t j[TK_PER], rank[TK_PER];
    bool bad = false;
#pragma unroll
    for (int k = 0; k < TK_PER; k++) {   // every load first; rows past the end read the last index
      const int64_t v = int64_t(idx[t0 + min(uint32_t(k) * TK_THREADS + threadIdx.x, rows - 1u)]);
      const bool in = v >= 0 && v < len;
      bad = bad || !in;
      j[k] = in ? uint32_t(v) : 0u;
    }
#pragma unroll
    for (int k = 0; k < TK_PER; k++)
      rank[k] = uint32_t(k) * TK_THREADS + threadIdx.x < rows ? atomicAdd(&s_cnt[j[k] >> shift], 1u) : 0u;
    __syncthreads();
    if (threadIdx.x < 64) {   // the exclusive scan of the counts, PER consecutive ones per lane of the first wave
      constexpr uint32_t PER = TK_SLICES / 64;
      uint32_t c[PER], sum = 0;
#pragma unroll
      for (uint32_t q = 0; q < PER; q++) {
        c[q] = s_cnt[PER * threadIdx.x + q];
        sum += c[q];
      }
      uint32_t x = sum;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d, 64);
        if (int(threadIdx.x) >= d) x += y;
      }
      uint32_t run = x - sum;
#pragma unroll
      for (uint32_t q = 0; q < PER; q++) {
        s_start[PER * threadIdx.x + q] = run;
        run += c[q];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TK_PER; k++) {
      const uint32_t r = uint32_t(k) * TK_THREADS + threadIdx.x;
      if (r < rows) {
        const uint32_t p = s_start[j[k] >> shift] + rank[k];
        s_idx[p] = j[k];
        s_pos[p] = uint16_t(r);
      }
    }
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < rows; p += TK_THREADS) {
      part_idx[t0 + p] = s_idx[p];
      part_pos[t0 + p] = s_pos[p];
    }
    if (threadIdx.x <= TK_SLICES)
      off[size_t(threadIdx.x) * tiles + tile] = threadIdx.x < TK_SLICES ? s_start[threadIdx.x] : rows;
    if (bad) st->out_of_range = 1u;
  }
}

// Slices x, x + 8, x + 16, ... belong to XCD x, in that order; a work item is one slice of TK_FETCH_TILES
// tiles. A workgroup whose XCD has no item left takes the others'. Without scattered indices: the plain
// gather.
template <typename V, typename I>
__global__ __launch_bounds__(256) void tk_fetch(const V* vals, uint32_t tiles, TkCtl* ctl, const uint32_t* part_idx,
                                                const uint32_t* off, V* part_val, int64_t len, const I* idx, int64_t n,
                                                V* out, TakeStatus* st) {
  __shared__ uint32_t s_item;
  if (!ctl->scattered) {   // uniform over the grid
    take_rows<V, I, false>(vals, nullptr, 0, len, idx, nullptr, 0, n, out, nullptr, nullptr, st);
    return;
  }
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const uint32_t per_slice = (tiles + TK_FETCH_TILES - 1) / TK_FETCH_TILES, items = per_slice * (TK_SLICES / NXCD);
  const uint32_t home = xcd_id();
  for (uint32_t h = 0; h < uint32_t(NXCD); h++) {
    const uint32_t x = (home + h) & uint32_t(NXCD - 1);
    while (true) {
      if (threadIdx.x == 0) s_item = atomicAdd(&ctl->item[x].next, 1u);
      __syncthreads();
      const uint32_t item = s_item;
      __syncthreads();
      if (item >= items) break;   // uniform: this XCD's items are all taken
      const uint32_t slice = (item / per_slice) * NXCD + x;
      const uint32_t tile0 = (item % per_slice) * TK_FETCH_TILES + w * 4u;
      uint32_t begin[4], len[4], most = 0;
#pragma unroll
      for (uint32_t u = 0; u < 4; u++) {   // the same for the wave
        const uint32_t t = min(tile0 + u, tiles - 1u);
        const uint32_t a = off[size_t(slice) * tiles + t], b = off[size_t(slice + 1u) * tiles + t];
        begin[u] = t * TK_TILE + a;
        len[u] = tile0 + u < tiles ? b - a : 0u;
        most = max(most, len[u]);
      }
      for (uint32_t p = lane; p - lane < most; p += 64u) {
        uint32_t j[4];
        V v[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) j[u] = p < len[u] ? __builtin_nontemporal_load(part_idx + begin[u] + p) : 0u;
#pragma unroll
        for (uint32_t u = 0; u < 4; u++)
          if (p < len[u]) v[u] = vals[j[u]];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++)
          if (p < len[u]) __builtin_nontemporal_store(v[u], part_val + begin[u] + p);
      }
    }
  }
}

template <typename V>
__global__ __launch_bounds__(TK_THREADS) void tk_place(uint32_t n, uint32_t tiles, const TkCtl* ctl, const V* part_val,
                                                       const uint16_t* part_pos, V* out) {
  __shared__ V s_val[TK_TILE];
  if (!ctl->scattered) return;   // uniform over the grid
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t t0 = tile * TK_TILE, rows = min(TK_TILE, n - t0);
    V v[TK_PER];
    uint32_t p[TK_PER];
#pragma unroll
    for (int k = 0; k < TK_PER; k++) {
      const uint32_t r = t0 + min(uint32_t(k) * TK_THREADS + threadIdx.x, rows - 1u);   // the last row more than once: the same value
      v[k] = part_val[r];
      p[k] = part_pos[r];
    }
    __syncthreads();   // the tile before has been written out
#pragma unroll
    for (int k = 0; k < TK_PER; k++) s_val[p[k]] = v[k];
    __syncthreads();
    for (uint32_t r = threadIdx.x; r < rows; r += TK_THREADS) out[t0 + r] = s_val[r];
  }
}

// Queues the passes. False, and nothing queued, if their scratch (14 or 10 bytes a row) cannot be had: the
// plain gather needs none.
template <typename V, typename I>
bool launch_take_slices(const Array& a, const Array& ix, Array* out, TakeStatus* st, hipStream_t s) {
  const uint32_t n = uint32_t(ix.length), tiles = (n + TK_TILE - 1) / TK_TILE, cus = uint32_t(device().cu_count);
  uint32_t shift = 0;
  while (((uint64_t(a.length) - 1u) >> shift) >= TK_SLICES) shift++;
  DevBuf cb, pi, pp, pv, ob;
  try {
    cb = device_alloc(sizeof(TkCtl));
    pi = device_alloc(size_t(n) * 4);
    pp = device_alloc(size_t(n) * 2);
    pv = device_alloc(size_t(n) * sizeof(V));
    ob = device_alloc(size_t(TK_SLICES + 1) * tiles * 4);
  } catch (const OutOfMemory&) {
    return false;
  }
  auto* ctl = static_cast<TkCtl*>(cb->ptr);
  const I* idx = static_cast<const I*>(ix.data());
  const V* vals = static_cast<const V*>(a.data());
  V* o = static_cast<V*>(out->values->ptr);
  auto* part_idx = static_cast<uint32_t*>(pi->ptr);
  auto* part_pos = static_cast<uint16_t*>(pp->ptr);
  auto* part_val = static_cast<V*>(pv->ptr);
  auto* off = static_cast<uint32_t*>(ob->ptr);
  {
    ProfScope ps("take_split");
    hipLaunchKernelGGL(tk_split<I>, dim3(std::min(tiles, cus)), dim3(TK_THREADS), 0, s, idx, n, a.length, shift, int(sizeof(V)),
                       ctl, tiles, part_idx, part_pos, off, st);
  }
  {
    ProfScope ps("take");
    hipLaunchKernelGGL((tk_fetch<V, I>), dim3(cus * 8u), dim3(256), 0, s, vals, tiles, ctl, part_idx, off, part_val, a.length,
                       idx, ix.length, o, st);
  }
  {
    ProfScope ps("take_place");
    hipLaunchKernelGGL(tk_place<V>, dim3(std::min(tiles, cus * (sizeof(V) == 4 ? 2u : 1u))), dim3(TK_THREADS), 0, s, n, tiles,
                       ctl, part_val, part_pos, o);
  }
  AM_HIP(hipGetLastError());
  return true;
}

template <typename V, typename I>
void launch_take(const Array& a, const Array& ix, Array* out, uint32_t blocks, uint32_t* block_nulls, TakeStatus* st,
                 hipStream_t s) {
  const V* vals = static_cast<const V*>(a.data());
  const I* idx = static_cast<const I*>(ix.data());
  const uint8_t* vv = a.has_nulls() ? a.valid_bits() : nullptr;
  const uint8_t* iv = ix.has_nulls() ? ix.valid_bits() : nullptr;
  unsigned long long* ov = out->validity ? static_cast<unsigned long long*>(out->validity->ptr) : nullptr;
  V* o = static_cast<V*>(out->values->ptr);
  if (a.length == 0)
    hipLaunchKernelGGL((take_empty<I>), dim3(blocks), dim3(256), 0, s, idx, iv, ix.offset, ix.length,
                       reinterpret_cast<char*>(o), int(sizeof(V)), ov, block_nulls, st);
  else if (ov) {
    ProfScope ps("take");
    hipLaunchKernelGGL((take_kernel<V, I, true>), dim3(blocks), dim3(256), 0, s, vals, vv, a.offset, a.length, idx, iv,
                       ix.offset, ix.length, o, ov, block_nulls, st);
  } else {
    if constexpr (sizeof(V) >= 4) {   // not in a batch, which would hold the scratch to its end
      if (!in_batch() && take_by_slices<V>(ix.length, a.length) && launch_take_slices<V, I>(a, ix, out, st, s)) return;
    }
    ProfScope ps("take");
    hipLaunchKernelGGL((take_kernel<V, I, false>), dim3(blocks), dim3(256), 0, s, vals, vv, a.offset, a.length, idx, iv,
                       ix.offset, ix.length, o, ov, block_nulls, st);
  }
  AM_HIP(hipGetLastError());
}

template <typename V>
void launch_take(const Array& a, const Array& ix, Array* out, uint32_t blocks, uint32_t* block_nulls, TakeStatus* st,
                 hipStream_t s) {
  switch (ix.type) {
    case T_I32: launch_take<V, int32_t>(a, ix, out, blocks, block_nulls, st, s); break;
    case T_U32: launch_take<V, uint32_t>(a, ix, out, blocks, block_nulls, st, s); break;
    default: launch_take<V, int64_t>(a, ix, out, blocks, block_nulls, st, s); break;
  }
}

// ---------------------------------------------------------------- the rows of a table
//
// A gather of random rows costs a 128-byte line per row and column. permute_columns lays up to PK_COLS columns
// out row by row (pk_pack: the values, widest first, and one byte of validity bits) and fetches each output's
// row once, writing the columns from LDS (pk_unpack). A null count is the column's own and nothing can be out
// of range, so the two launches are all there is. 4M rows of i32 and f64 with nulls, i64 and i32 (32-byte
// rows): 50 + 93 us; one gather per column took 280. The fetch moves 4M 128-byte lines in that time, the pack
// streams 60 B a row.
constexpr int PK_COLS = 8;
constexpr uint32_t PK_BYTES = 64;   // of a row at most: 8 words

struct PackCols {
  struct Col {
    const void* src;
    const uint8_t* valid;            // nullptr without nulls
    int64_t voff;
    void* dst;
    unsigned long long* dst_valid;   // nullptr without nulls
    uint32_t width, at;              // bytes, and where in the row
  } c[PK_COLS];
  uint32_t cols, words, bits_at, has_bits;
};

struct PackRow {
  unsigned long long v[PK_COLS];
  uint32_t vb[PK_COLS];
};

__device__ __forceinline__ unsigned long long pk_value(const void* at, uint32_t width, uint32_t r) {
  if (width == 8) return static_cast<const unsigned long long*>(at)[r];
  if (width == 4) return static_cast<const uint32_t*>(at)[r];
  if (width == 2) return static_cast<const uint16_t*>(at)[r];
  return static_cast<const uint8_t*>(at)[r];
}

__device__ __forceinline__ void pk_set(void* at, uint32_t width, uint32_t r, unsigned long long v) {
  if (width == 8) static_cast<unsigned long long*>(at)[r] = v;
  else if (width == 4) static_cast<uint32_t*>(at)[r] = uint32_t(v);
  else if (width == 2) static_cast<uint16_t*>(at)[r] = uint16_t(v);
  else static_cast<uint8_t*>(at)[r] = uint8_t(v);
}

// Row r of the columns: every load before the first use.
__device__ __forceinline__ void pk_load(const PackCols& p, uint32_t r, PackRow& x) {
#pragma unroll
  for (int c = 0; c < PK_COLS; c++) {
    x.v[c] = 0;
    x.vb[c] = 1u;
    if (c >= int(p.cols)) continue;   // uniform
    x.v[c] = pk_value(p.c[c].src, p.c[c].width, r);
    if (p.c[c].valid) x.vb[c] = p.c[c].valid[(p.c[c].voff + r) >> 3];
  }
}

// The row as it is laid out, at `row` (8-byte aligned).
__device__ __forceinline__ void pk_put(const PackCols& p, uint32_t r, const PackRow& x, char* row) {
  uint32_t bits = 0;
#pragma unroll
  for (int c = 0; c < PK_COLS; c++) {
    if (c >= int(p.cols)) continue;
    pk_set(row + p.c[c].at, p.c[c].width, 0u, x.v[c]);
    bits |= (p.c[c].valid ? (x.vb[c] >> uint32_t((p.c[c].voff + r) & 7)) & 1u : 1u) << c;
  }
  if (p.has_bits) *reinterpret_cast<uint8_t*>(row + p.bits_at) = uint8_t(bits);
}

// Output i of every column from the row at `row`, for a whole wave of consecutive outputs that begins at a
// multiple of 64.
__device__ __forceinline__ void pk_get(const PackCols& p, const char* row, uint32_t i, uint32_t n) {
  const uint32_t bits = p.has_bits ? *reinterpret_cast<const uint8_t*>(row + p.bits_at) : 0xFFu;
  for (uint32_t c = 0; c < p.cols; c++) {
    if (i < n) pk_set(p.c[c].dst, p.c[c].width, i, pk_value(row + p.c[c].at, p.c[c].width, 0u));
    if (p.c[c].dst_valid) {
      const unsigned long long bal = __ballot(i < n && ((bits >> c) & 1u));
      if ((threadIdx.x & 63) == 0 && i < n) p.c[c].dst_valid[i >> 6] = bal;
    }
  }
}

// The next group of columns from position k of `order` on (widest first, so that every value lies at a
// multiple of its width); k moves past it. The outputs' null counts and buffers are set.
PackCols pack_group(const std::vector<const Array*>& cols, const std::vector<Array*>& out,
                           const std::vector<size_t>& order, size_t& k) {
  PackCols p{};
  uint32_t bytes = 0;
  for (; k < order.size() && p.cols < uint32_t(PK_COLS); k++) {
    const Array& c = *cols[order[k]];
    const Array* o = out[order[k]];
    const uint32_t bits = p.has_bits || o->null_count > 0 ? 1u : 0u;
    if (bytes + uint32_t(c.width()) + bits > PK_BYTES) break;
    PackCols::Col& d = p.c[p.cols++];
    d.src = c.data();
    d.valid = o->null_count > 0 ? c.valid_bits() : nullptr;
    d.voff = c.offset;
    d.dst = o->values->ptr;
    d.dst_valid = o->null_count > 0 ? static_cast<unsigned long long*>(o->validity->ptr) : nullptr;
    d.width = uint32_t(c.width());
    d.at = bytes;
    bytes += d.width;
    p.has_bits = bits;
  }
  p.bits_at = bytes;
  p.words = (bytes + p.has_bits + 7u) / 8u;
  return p;
}

std::vector<size_t> widest_first(const std::vector<const Array*>& cols) {
  std::vector<size_t> order(cols.size());
  for (size_t c = 0; c < cols.size(); c++) order[c] = c;
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return cols[a]->width() > cols[b]->width(); });
  return order;
}

// f(std::integral_constant<int, words>) for 1 to 8 words.
template <typename F>
void with_words(uint32_t words, F&& f) {
  switch (words) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    default: f(std::integral_constant<int, 8>{}); break;
  }
}

// Tiles of 256 rows, one per thread: coalesced loads column by column, coalesced stores of whole rows. The
// rows of a tile are a word apart in LDS beyond their WORDS, so a wave's accesses spread over the banks.
template <int WORDS>
__global__ __launch_bounds__(256) void pk_pack(PackCols p, uint32_t n, unsigned long long* rows_out) {
  __shared__ unsigned long long s_row[256 * (WORDS + 1)];
  const uint32_t t0 = blockIdx.x * 256u, r = min(t0 + threadIdx.x, n - 1u), rows = min(256u, n - t0);
  PackRow x;
  pk_load(p, r, x);
  pk_put(p, r, x, reinterpret_cast<char*>(s_row + threadIdx.x * (WORDS + 1)));
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < rows * WORDS; k += 256u)
    rows_out[size_t(t0) * WORDS + k] = s_row[(k / WORDS) * (WORDS + 1) + k % WORDS];
}

// Tiles of 256 outputs. WORDS / VEC neighbouring lanes fetch one row, VEC words each.
template <int WORDS>
__global__ __launch_bounds__(256) void pk_unpack(PackCols p, uint32_t n, const uint32_t* __restrict__ idx,
                                                 const unsigned long long* __restrict__ rows_in) {
  constexpr int VEC = WORDS % 2 == 0 ? 2 : 1, LANES = WORDS / VEC;
  struct alignas(8 * VEC) Part {
    unsigned long long w[VEC];
  };
  __shared__ unsigned long long s_row[256 * (WORDS + 1)];
  __shared__ uint32_t s_idx[256];
  const uint32_t t0 = blockIdx.x * 256u, i = t0 + threadIdx.x;
  s_idx[threadIdx.x] = min(idx[min(i, n - 1u)], n - 1u);   // a permutation: the bound only keeps reads in range
  __syncthreads();
  Part v[LANES];
#pragma unroll
  for (int u = 0; u < LANES; u++) {
    const uint32_t k = uint32_t(u) * 256u + threadIdx.x;
    v[u] = reinterpret_cast<const Part*>(rows_in)[size_t(s_idx[k / LANES]) * LANES + k % LANES];
  }
#pragma unroll
  for (int u = 0; u < LANES; u++) {
    const uint32_t k = uint32_t(u) * 256u + threadIdx.x;
#pragma unroll
    for (int q = 0; q < VEC; q++) s_row[(k / LANES) * (WORDS + 1) + (k % LANES) * VEC + q] = v[u].w[q];
  }
  __syncthreads();
  pk_get(p, reinterpret_cast<const char*>(s_row + threadIdx.x * (WORDS + 1)), i, n);
}

}  // namespace

bool permute_columns(const std::vector<const Array*>& cols, const Array& idx, std::vector<Array*>& out) {
  out.clear();
  const int64_t n = idx.length;
  if (cols.size() < 2 || idx.type != T_U32 || idx.has_nulls() || n <= 0 || n > int64_t(UINT32_MAX)) return false;
  for (const Array* c : cols)
    if (c->length != n || !type_is_primitive(c->type) || c->width() == 0) return false;
  hipStream_t s = stream();
  const std::vector<size_t> order = widest_first(cols);
  try {
    for (const Array* c : cols) {
      Array* o = new_array(c->format, c->type, n);
      out.push_back(o);
      o->null_count = c->validity ? (c->null_count < 0 ? count_nulls(*c) : c->null_count) : 0;
      o->values = device_alloc(size_t(n) * c->width());
      if (o->null_count > 0) o->validity = device_alloc(size_t((n + 63) / 64) * 8);
    }
    const dim3 grid(uint32_t((n + 255) / 256)), block(256);
    for (size_t k = 0; k < order.size();) {
      const PackCols p = pack_group(cols, out, order, k);
      DevBuf rows;
      try {
        rows = device_alloc(size_t(n) * p.words * 8u);
      } catch (const OutOfMemory&) {   // no room: column by column, which needs none
        for (Array* a : out) release_array(a);
        out.clear();
        return false;
      }
      auto* r = static_cast<unsigned long long*>(rows->ptr);
      with_words(p.words, [&](auto words) {
        constexpr int W = decltype(words)::value;
        {
          ProfScope ps("take_pack");
          hipLaunchKernelGGL(pk_pack<W>, grid, block, 0, s, p, uint32_t(n), r);
        }
        ProfScope ps("take_unpack");
        hipLaunchKernelGGL(pk_unpack<W>, grid, block, 0, s, p, uint32_t(n), static_cast<const uint32_t*>(idx.data()),
                           static_cast<const unsigned long long*>(r));
      });
      AM_HIP(hipGetLastError());
    }
    if (!in_batch()) sync();
  } catch (...) {
    for (Array* a : out) release_array(a);
    out.clear();
    throw;
  }
  return true;
}

Array* take(const Array& a, const Array& ix) {
  check_length(a.length);
  check_length(ix.length);
  if (ix.type != T_I32 && ix.type != T_I64 && ix.type != T_U32)
    fail_unsupported("take indices must be int32, int64 or uint32");
  int w = a.width();
  if (w == 0) fail_unsupported("take of " + a.format + " is not supported by this build");
  int64_t n = ix.length;
  Array* out = new_array(a.format, a.type, n);
  try {
    hipStream_t s = stream();
    out->values = device_alloc(size_t(std::max<int64_t>(n, 1)) * w);
    bool need_validity = a.has_nulls() || ix.has_nulls();
    if (need_validity) out->validity = device_alloc(size_t((std::max<int64_t>(n, 1) + 63) / 64) * 8);
    std::shared_ptr<void> slot = pinned_slot();
    auto* st = static_cast<TakeStatus*>(slot.get());
    *st = TakeStatus{0, 0, 0};
    if (n > 0) {
      const uint32_t blocks = uint32_t(std::min<int64_t>((n + 256 * TAKE_GROUPS - 1) / (256 * TAKE_GROUPS), int64_t(device().cu_count) * 16));
      DevBuf bn;
      if (need_validity) bn = device_alloc(size_t(blocks) * 4);
      uint32_t* block_nulls = bn ? static_cast<uint32_t*>(bn->ptr) : nullptr;
      switch (w) {
        case 1: launch_take<uint8_t>(a, ix, out, blocks, block_nulls, st, s); break;
        case 2: launch_take<uint16_t>(a, ix, out, blocks, block_nulls, st, s); break;
        case 4: launch_take<uint32_t>(a, ix, out, blocks, block_nulls, st, s); break;
        default: launch_take<unsigned long long>(a, ix, out, blocks, block_nulls, st, s); break;
      }
      if (need_validity) {
        hipLaunchKernelGGL(take_nulls, dim3(1), dim3(1024), 0, s, static_cast<const uint32_t*>(block_nulls), blocks, st);
        AM_HIP(hipGetLastError());
      }
    }
    int64_t len = a.length;
    Array* res = out;
    retain_array(res);   // the check below may run at the end of a batch
    after_sync([slot, len, res, need_validity] {
      struct Drop {
        Array* a;
        ~Drop() { release_array(a); }
      } drop{res};
      const TakeStatus* host = static_cast<const TakeStatus*>(slot.get());
      if (host->out_of_range) fail_invalid("take: index out of range (array length " + std::to_string(len) + ")");
      res->null_count = need_validity ? int64_t(host->nulls) : 0;
      if (res->null_count == 0) res->validity.reset();
    });
    if (!in_batch()) {
      sync();
    } else {
      // Inside a batch the null count is not known until the batch ends; the validity is kept.
      out->null_count = need_validity ? -1 : 0;
    }
  } catch (...) {
    release_array(out);
    throw;
  }
  return out;
}

}  // namespace am
