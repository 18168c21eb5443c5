// Stable LSD radix argsort for CDNA4 (gfx950, wave64).
//
// Semantics follow the reference's radix sort (Sources/ArrowMetal/Kernels/Sort.swift:190-504 and
// SortSource.swift:131-330): an order-preserving unsigned key per value, a stable three-way split of
// the rows into [values][NaN][nulls] (or [nulls][NaN][values] for nulls first), 8-bit digits, and a
// pass skipped when its digit is the same in every value key. The way it runs on the GPU is this
// build's own:
//
//   sort_init      clears the per-call control block (a fill kernel, no hipMemset, so that the
//                  sequence can be captured in a graph)
//   sort_upsweep   one read of the column: maps every key, counts values / NaN / nulls, and builds
//                  the digit histograms of all (varying) digits at once plus the OR / AND of the keys
//                  The last workgroup done makes the plan: active-pass mask, block bases of the three
//                  buckets, and the exclusive digit prefix of every pass
//   sort_first     the first active pass reads the raw column again, maps keys on the fly, and
//                  scatters values by digit while NaN and null rows go straight to their final slots
//   sort_mid       one launch per further active digit; the last active pass writes only the row
//                  numbers, into the output. Inputs of 2^16 rows and more read the plan back once and
//                  launch only the active passes; smaller ones (and graph captures) launch one kernel
//                  per digit that exits at once when its digit is inactive
//
// Inputs of at most 16,384 rows take none of these: sort_rank sorts them in one launch. Larger ones of 32 or
// 64 bits take the MSD sort of msd_levels.hpp from the row counts at hybrid_min, below.
//
// Each scatter pass is "onesweep": tiles of 256 threads x ITEMS keys take dynamic tile ids, rank
// their keys inside the tile with wave64 ballots (a 9-bit match per 64-lane row), publish their
// per-bin counts and look back over earlier tiles for the exclusive prefix (decoupled look-back with
// epoch-tagged 64-bit status words, so the status table is never cleared between passes), then stage
// the tile in LDS in digit order so that the global writes are runs of consecutive addresses.
#include "msd_levels.hpp"

namespace am {
namespace {

struct SortCtl {
  uint32_t m;                       // value rows
  // Bumped by every workgroup of a pass, so on cache lines of their own: a line that also holds
  // words the same workgroups read slows the pass down.
  alignas(128) uint32_t tile_counter[16];   // [0] first pass, [1 + p] pass p, [11] units
  alignas(128) uint32_t digit_base[8][RADIX];   // exclusive digit prefix inside the value block, per pass
  uint32_t bin_total[NBINS_FIRST], first_base[NBINS_FIRST];   // the hybrid sort's analysis
  uint32_t active_mask, first_active, last_active;
  uint32_t lsd;                     // the hybrid sort's analysis has counted for the LSD passes instead
  uint32_t value_base, nan_base, null_base, pad2;
  // Per-XCD partials of the upsweep, folded into the fields above by sort_plan.
  uint32_t xhist[NXCD][8][RADIX];
  uint32_t xm[NXCD], xq[NXCD], xz[NXCD], pad3[NXCD];
  unsigned long long xor_[NXCD], xand[NXCD];
};

// ---------------------------------------------------------------- kernels

// A cleared control block (by one workgroup).
__device__ __forceinline__ void clear_ctl(SortCtl* ctl) {
  for (uint32_t i = threadIdx.x; i < uint32_t(NXCD * 8 * RADIX); i += blockDim.x) (&ctl->xhist[0][0][0])[i] = 0u;
  if (threadIdx.x < NXCD) {
    ctl->xm[threadIdx.x] = ctl->xq[threadIdx.x] = ctl->xz[threadIdx.x] = 0u;
    ctl->xor_[threadIdx.x] = 0ull;
    ctl->xand[threadIdx.x] = ~0ull;
  }
  if (threadIdx.x < 16) ctl->tile_counter[threadIdx.x] = 0u;
}

__global__ void sort_init(SortCtl* ctl) { clear_ctl(ctl); }

// Copies the plan (active mask, first and last active pass, value rows) to pinned host memory.
__global__ void sort_read_plan(const SortCtl* ctl, uint32_t* out) {
  out[0] = ctl->active_mask;
  out[1] = ctl->first_active;
  out[2] = ctl->last_active;
  out[3] = ctl->m;
}


// Waits for an atomic by its result: it has been carried out at the memory side, where every XCD's
// atomics meet. (A device-scope fence would write back the XCD's whole L2 instead.)
template <typename T>
__device__ __forceinline__ void atomic_done(T result) {
  asm volatile("" ::"v"(result) : "memory");
}

// True in the last workgroup of the grid to ask (one thread each); the counter is 0 again after it.
__device__ __forceinline__ bool last_block(uint32_t* ticket) {
  const bool mine = atomicInc(ticket, gridDim.x - 1u) == gridDim.x - 1u;
  asm volatile("" ::: "memory");
  return mine;
}

// One LDS count of bin b (b < 2^31; lanes that count nothing pass b = ~0u). The lanes of the wave on the
// first counting lane's bin take one atomic together: a digit that is the same on most rows (the high
// digits of small integers, a skewed column) would otherwise serialize its 64 lanes on one address.
__device__ __forceinline__ void count_bin(uint32_t* h, uint32_t b) {
  const uint32_t lead = __builtin_amdgcn_readfirstlane(b);
  const unsigned long long m = __ballot(b == lead);
  if (b == lead) {
    if (lead != ~0u && int(threadIdx.x & 63u) == __builtin_ctzll(m)) atomicAdd(&h[lead], uint32_t(__popcll(m)));
  } else if (b != ~0u) {
    atomicAdd(&h[b], 1u);
  }
}

// The same with a check for a digit that is one on the whole wave only: cheaper, for the LSD passes' analysis
// of every digit (10M uniform float32 keys: 32 us less than with count_bin). In a column with nulls, one on all
// lanes that count.
template <bool NULLS>
__device__ __forceinline__ void count_digit(uint32_t* h, uint32_t b) {
  if constexpr (!NULLS) {
    const uint32_t lead = __builtin_amdgcn_readfirstlane(b);
    if (__all(b == lead)) {   // uniform
      if (lead != ~0u && (threadIdx.x & 63u) == 0u) atomicAdd(&h[lead], 64u);
      return;
    }
  } else {
    const unsigned long long m = __ballot(b != ~0u);
    if (m == 0ull) return;
    const int first = __builtin_ctzll(m);
    const uint32_t lead = __builtin_amdgcn_readlane(b, first);
    if (__ballot(b == lead) == m) {   // uniform
      if (int(threadIdx.x & 63u) == first) atomicAdd(&h[lead], uint32_t(__popcll(m)));
      return;
    }
  }
  if (b != ~0u) atomicAdd(&h[b], 1u);
}

// f(std::true_type) for a column with a validity bitmap, f(std::false_type) for one without.
template <class F>
__device__ __forceinline__ void with_nulls(const uint8_t* valid, F&& f) {
  if (valid) f(std::true_type{});
  else f(std::false_type{});
}

// Runs count(base, raw, vb) over the rows [begin, end) of a workgroup, UP_ITEMS rows per thread per step,
// loaded before any is counted; two steps' rows take turns, so that the next step's loads are in flight
// while this step is counted, and every loaded register is taken at the top of a step (a load the compiler
// moved into one of the classification's branches would be waited for there alone). The step count is the
// same for every thread of the block.
constexpr int UP_ITEMS = 8;
constexpr uint32_t UP_STEP = BLOCK * UP_ITEMS;

template <int W, class F>
__device__ __forceinline__ void up_steps(const void* vals, const uint8_t* valid, int64_t voff, uint32_t begin,
                                         uint32_t end, F&& count) {
  const int steps = end > begin ? int((end - begin + UP_STEP - 1) / UP_STEP) : 0;
  if (steps == 0) return;
  uint64_t raw_a[UP_ITEMS], raw_b[UP_ITEMS];
  uint32_t vb_a[UP_ITEMS], vb_b[UP_ITEMS];
  auto load_step = [&](uint64_t base, uint64_t (&raw)[UP_ITEMS], uint32_t (&vb)[UP_ITEMS]) {
#pragma unroll
    for (int u = 0; u < UP_ITEMS; u++) {   // rows past the end read the last row
      const uint32_t i = uint32_t(std::min<uint64_t>(base + uint64_t(u) * BLOCK + threadIdx.x, uint64_t(end) - 1u));
      uint32_t bit;
      raw[u] = load_raw<W>(vals, i);
      vb[u] = load_valid_byte(valid, voff, i, bit);
    }
  };
  auto count_step = [&](uint64_t base, const uint64_t (&raw)[UP_ITEMS], const uint32_t (&vb)[UP_ITEMS]) {
#pragma unroll
    for (int u = 0; u < UP_ITEMS; u++) asm volatile("" ::"v"(raw[u]), "v"(vb[u]));
    count(base, raw, vb);
  };
  load_step(begin, raw_a, vb_a);
  for (int t = 0; t < steps; t += 2) {
    const uint64_t base = uint64_t(begin) + uint64_t(t) * UP_STEP;
    load_step(base + UP_STEP, raw_b, vb_b);
    count_step(base, raw_a, vb_a);
    if (t + 1 >= steps) break;
    load_step(base + 2 * UP_STEP, raw_a, vb_a);
    count_step(base + UP_STEP, raw_b, vb_b);
  }
}

// What the rows of a workgroup have in common: OR / AND of the value keys, and how many rows are values,
// NaN and null.
struct UpStat {
  unsigned long long key_or, key_and;
  uint32_t m, q, z, pad;
};

// The classes and keys of one step's rows (3: past the end), counted into this thread's statistics.
template <typename K>
__device__ __forceinline__ void up_classify(uint64_t base, uint32_t end, const uint64_t (&raw)[UP_ITEMS],
                                            const uint32_t (&vb)[UP_ITEMS], bool has_valid, int64_t voff, int type,
                                            int forder, int desc, K (&kk)[UP_ITEMS], int (&cc)[UP_ITEMS], UpStat& st) {
#pragma unroll
  for (int u = 0; u < UP_ITEMS; u++) {
    const uint64_t i = base + uint64_t(u) * BLOCK + threadIdx.x;
    const uint32_t ic = uint32_t(std::min<uint64_t>(i, uint64_t(end) - 1u));
    const uint32_t bit = has_valid ? uint32_t((voff + int64_t(ic)) & 7) : 0u;
    kk[u] = 0;
    cc[u] = i < end ? classify_raw<K>(raw[u], (vb[u] >> bit) & 1u, type, forder, desc, kk[u]) : 3;
    st.m += cc[u] == 0 ? 1u : 0u;
    st.q += cc[u] == 1 ? 1u : 0u;
    st.z += cc[u] == 2 ? 1u : 0u;
    if (cc[u] == 0) {
      st.key_or |= (unsigned long long)kk[u];
      st.key_and &= (unsigned long long)kk[u] | (sizeof(K) == 4 ? 0xFFFFFFFF00000000ull : 0ull);
    }
  }
}

// The workgroup's statistics in thread 0 (s: WAVES entries of LDS).
__device__ __forceinline__ void up_reduce(UpStat& st, UpStat* s) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    st.m += __shfl_down(st.m, off, 64);
    st.q += __shfl_down(st.q, off, 64);
    st.z += __shfl_down(st.z, off, 64);
    st.key_or |= __shfl_down(st.key_or, off, 64);
    st.key_and &= __shfl_down(st.key_and, off, 64);
  }
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = st;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < WAVES; w++) {
      st.m += s[w].m;
      st.q += s[w].q;
      st.z += s[w].z;
      st.key_or |= s[w].key_or;
      st.key_and &= s[w].key_and;
    }
  }
}

// The digits that the LSD passes sort, and the bases of the three blocks, for m values, q NaN and z null rows.
__device__ __forceinline__ void set_lsd_plan(SortCtl* ctl, uint32_t varying, uint32_t m, uint32_t q, uint32_t z,
                                             int nulls_first) {
  // No varying digit (a single value, or one repeated key): one pass over digit 0 is then a
  // stable compaction of the value rows, which is exactly the answer.
  const uint32_t mask = varying == 0u || m <= 1u ? 1u : varying;
  ctl->m = m;
  ctl->active_mask = mask;
  ctl->first_active = uint32_t(__builtin_ctz(mask));
  ctl->last_active = 31u - uint32_t(__builtin_clz(mask));
  ctl->null_base = nulls_first ? 0u : m + q;
  ctl->nan_base = nulls_first ? z : m;
  ctl->value_base = nulls_first ? z + q : 0u;
}

// The LSD passes' plan, by the analysis' last workgroup: the XCDs' partial counts folded, the active digits,
// the bases of the three blocks, and the exclusive digit prefix of every active pass.
template <int P>
__device__ __forceinline__ void sort_plan(SortCtl* ctl, int nulls_first, uint32_t digits) {
  __shared__ uint32_t tmp[WAVES];
  auto fold = [](const uint32_t* p, size_t stride) {
    uint32_t v = 0;
#pragma unroll
    for (int x = 0; x < NXCD; x++) v += __hip_atomic_load(p + x * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return v;
  };
  uint32_t v[P];
#pragma unroll
  for (int p = 0; p < P; p++) v[p] = fold(&ctl->xhist[0][p][threadIdx.x], 8 * RADIX);   // every load first
#pragma unroll
  for (int p = 0; p < P; p++) {
    if (!((digits >> p) & 1u)) continue;   // uniform
    uint32_t total;
    ctl->digit_base[p][threadIdx.x] = block_excl_scan(v[p], tmp, total);
  }
  if (threadIdx.x == 0) {
    const uint32_t m = fold(ctl->xm, 1), q = fold(ctl->xq, 1), z = fold(ctl->xz, 1);
    unsigned long long o = 0ull, a = ~0ull;
    for (int x = 0; x < NXCD; x++) {
      o |= __hip_atomic_load(&ctl->xor_[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      a &= __hip_atomic_load(&ctl->xand[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const unsigned long long diff = o ^ a;
    uint32_t mask = 0;
    for (int p = 0; p < P; p++)
      if ((diff >> (8 * p)) & 0xFFull) mask |= 1u << p;
    set_lsd_plan(ctl, mask, m, q, z, nulls_first);
  }
}

// The LSD passes' analysis: the histograms of the digits in `digits` (a bit per digit; a digit known not to
// vary needs none), the row counts and the OR / AND; the last workgroup done makes the plan.
template <typename K, int W>
__global__ __launch_bounds__(BLOCK) void sort_upsweep(const void* vals, const uint8_t* valid, int64_t voff,
                                                      uint32_t n, int type, int forder, int desc,
                                                      uint32_t rows_per_block, SortCtl* ctl, uint32_t digits,
                                                      int nulls_first, uint32_t* ticket) {
  constexpr int P = int(sizeof(K));
  __shared__ uint32_t h[P][RADIX];
  __shared__ UpStat s_st[WAVES];
  __shared__ uint32_t s_last;
  for (int i = threadIdx.x; i < P * RADIX; i += BLOCK) (&h[0][0])[i] = 0u;
  __syncthreads();
  const uint32_t begin = blockIdx.x * rows_per_block;
  const uint32_t end = begin + min(n - begin, rows_per_block);   // (begin + rows_per_block may pass 2^32)
  UpStat st{0ull, ~0ull, 0u, 0u, 0u, 0u};
  with_nulls(valid, [&](auto nulls) {
    constexpr bool NULLS = decltype(nulls)::value;
    up_steps<W>(vals, valid, voff, begin, end, [&](uint64_t base, const uint64_t (&raw)[UP_ITEMS], const uint32_t (&vb)[UP_ITEMS]) {
      K kk[UP_ITEMS];
      int cc[UP_ITEMS];
      up_classify<K>(base, end, raw, vb, NULLS, voff, type, forder, desc, kk, cc, st);
#pragma unroll
      for (int p = 0; p < P; p++) {
        if (!((digits >> p) & 1u)) continue;   // uniform
#pragma unroll
        for (int u = 0; u < UP_ITEMS; u++) count_digit<NULLS>(h[p], cc[u] == 0 ? uint32_t(kk[u] >> (8 * p)) & 0xFFu : ~0u);
      }
    });
  });
  up_reduce(st, s_st);
  __syncthreads();
  const uint32_t x = xcd_id();
  uint32_t* xh = &ctl->xhist[x][0][0];
  uint32_t done = 0;
  for (int i = threadIdx.x; i < P * RADIX; i += BLOCK) {
    const uint32_t v = (&h[0][0])[i];
    if (v) done |= atomicAdd(xh + i, v);
  }
  atomic_done(done);
  if (threadIdx.x == 0) {
    if (st.m) {
      atomic_done(atomicAdd(&ctl->xm[x], st.m));
      atomic_done(atomicOr(&ctl->xor_[x], st.key_or));
      atomic_done(atomicAnd(&ctl->xand[x], st.key_and));
    }
    if (st.q) atomic_done(atomicAdd(&ctl->xq[x], st.q));
    if (st.z) atomic_done(atomicAdd(&ctl->xz[x], st.z));
  }
  __syncthreads();   // every thread's counts are in memory
  if (threadIdx.x == 0) s_last = last_block(ticket) ? 1u : 0u;
  __syncthreads();
  if (s_last) sort_plan<P>(ctl, nulls_first, digits);   // uniform
}

// ---------------------------------------------------------------- the hybrid sort's analysis
//
// Rows per unit of the top-digit partition (a power of two): the analysis counts the top digit, NaN and
// null rows of every unit, so that the partition knows every unit's destinations before it starts.
// Units are 2^unit_shift rows: 16K for 4M rows and more, 4K (one tile of the partition) below, so that a
// 1M-row input still has ~250 units to spread over the CUs.
constexpr uint32_t UNIT_SHIFT_LARGE = 14, UNIT_SHIFT_SMALL = 12;
constexpr uint32_t UNITS_PER_BLOCK = 8;   // most units one workgroup counts
// Most rows of the hybrid sort: a workgroup's, a unit's and a tile's first row past the end are 32-bit numbers.
constexpr uint32_t HYBRID_MAX_ROWS = UINT32_MAX - (UNITS_PER_BLOCK << UNIT_SHIFT_LARGE);

// 32-bit keys have four LSD passes only, so the hybrid sort must come out with about one level (every
// top-digit bucket at most 2^18 rows, which a second digit brings to bucket-sort size), or save whole passes
// over a large column. 10M float32 values over 10,000 distinct: LSD 481 us, hybrid 660; 40M uniform float32:
// 1.71 against 1.33 ms; 3M full-range int32: 237 against 167 us.
constexpr uint32_t MSD32_TOP_MAX = 1u << 18, MSD32_SAVES = 1u << 24;

// Whether the LSD passes sort a 32-bit column, from 4 neighbours at each of 16 places over its length, which every
// wave reads: one top digit on all of them, or one on so many that its bucket is too large. (Only a guess at the
// faster way: either sorts any column. A column that is counted for the one and sorted by the other is read once
// more: 1M int32 values of 0 to 2^20 154 us so, 140 when guessed; of 6M full-range
// ones 261 and 264.)
template <typename K, int W>
__device__ __forceinline__ bool sampled_lsd(const void* vals, const uint8_t* valid, int64_t voff, uint32_t n, int type,
                                            int forder, int desc) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t i = uint32_t(uint64_t(n - 4u) * (lane >> 2) / 15u) + (lane & 3u);
  const uint64_t raw = load_raw<W>(vals, i);
  uint32_t bit;
  const uint32_t vb = load_valid_byte(valid, voff, i, bit);
  K key = 0;
  const int cat = classify_raw<K>(raw, (vb >> bit) & 1u, type, forder, desc, key);
  const uint32_t b = cat == 0 ? uint32_t(key >> (8 * (sizeof(K) - 1))) & 0xFFu : ~0u;
  const unsigned long long counting = __ballot(b != ~0u);
  if (counting == 0ull) return true;
  if (__ballot(b == uint32_t(__builtin_amdgcn_readlane(b, __builtin_ctzll(counting)))) == counting) return true;
  if (n >= MSD32_SAVES) return false;
  // The digits of eight lanes: a digit on many rows is one of them. Well over the share that makes a bucket too
  // large, and over what chance gives one of 256 evenly spread digits.
  uint32_t most = 0;
#pragma unroll
  for (int k = 0; k < 64; k += 8) {
    const uint32_t d = __builtin_amdgcn_readlane(b, k);
    if (d != ~0u) most = max(most, uint32_t(__popcll(__ballot(b == d))));
  }
  const uint32_t share = uint32_t(uint64_t(MSD32_TOP_MAX) * 64u / n);
  return most > max(8u, share + share / 2u + 4u);
}

// Every unit's counts, bin-major (unit_hist[b][unit]), and every workgroup's statistics. With guess (32-bit keys),
// for a column that the LSD passes will sort: every digit's counts of every workgroup (unit_hist[256 p + b][workgroup]).
template <typename K, int W>
__global__ __launch_bounds__(BLOCK) void msd_upsweep(const void* vals, const uint8_t* valid, int64_t voff, uint32_t n,
                                                     int type, int forder, int desc, uint32_t rows_per_block,
                                                     UpStat* stats, uint32_t* unit_hist, uint32_t nunits,
                                                     uint32_t unit_shift, int guess, SortCtl* ctl) {
  constexpr int P = int(sizeof(K));
  __shared__ uint32_t hu[UNITS_PER_BLOCK * NBINS_FIRST];
  __shared__ UpStat s_st[WAVES];
  bool lsd = false;
  if constexpr (P == 4) lsd = guess && sampled_lsd<K, W>(vals, valid, voff, n, type, forder, desc);
  if (blockIdx.x == 0 && threadIdx.x == 0) ctl->lsd = lsd ? 1u : 0u;
  const uint32_t begin = blockIdx.x * rows_per_block;
  const uint32_t end = min(n, begin + rows_per_block);
  const uint32_t nu = (end - begin + (1u << unit_shift) - 1u) >> unit_shift;
  for (uint32_t i = threadIdx.x; i < (lsd ? 4u * RADIX : nu * NBINS_FIRST); i += BLOCK) hu[i] = 0u;
  __syncthreads();
  UpStat st{0ull, ~0ull, 0u, 0u, 0u, 0u};
  if (lsd) {   // uniform over the grid
    static_assert(UNITS_PER_BLOCK * NBINS_FIRST >= 4 * RADIX, "the digits' counts fit where the units' are");
    with_nulls(valid, [&](auto nulls) {
      constexpr bool NULLS = decltype(nulls)::value;
      up_steps<W>(vals, valid, voff, begin, end, [&](uint64_t base, const uint64_t (&raw)[UP_ITEMS], const uint32_t (&vb)[UP_ITEMS]) {
        K kk[UP_ITEMS];
        int cc[UP_ITEMS];
        up_classify<K>(base, end, raw, vb, NULLS, voff, type, forder, desc, kk, cc, st);
#pragma unroll
        for (uint32_t p = 0; p < 4; p++)
#pragma unroll
          for (int u = 0; u < UP_ITEMS; u++)
            count_digit<NULLS>(hu + p * RADIX, cc[u] == 0 ? uint32_t(kk[u] >> (8 * p)) & 0xFFu : ~0u);
      });
    });
    up_reduce(st, s_st);
    if (threadIdx.x == 0) stats[blockIdx.x] = st;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 4u * RADIX; i += BLOCK) unit_hist[size_t(i) * gridDim.x + blockIdx.x] = hu[i];
    return;
  }
  up_steps<W>(vals, valid, voff, begin, end, [&](uint64_t base, const uint64_t (&raw)[UP_ITEMS], const uint32_t (&vb)[UP_ITEMS]) {
    K kk[UP_ITEMS];
    int cc[UP_ITEMS];
    up_classify<K>(base, end, raw, vb, valid != nullptr, voff, type, forder, desc, kk, cc, st);
#pragma unroll
    for (int u = 0; u < UP_ITEMS; u++) {
      const uint32_t ui = uint32_t(base + uint64_t(u) * BLOCK + threadIdx.x - begin) >> unit_shift;
      const uint32_t bin = cc[u] == 0 ? uint32_t(kk[u] >> (8 * (P - 1))) & 0xFFu : cc[u] == 1 ? uint32_t(BIN_NAN) : uint32_t(BIN_NULL);
      count_bin(hu, cc[u] < 3 ? ui * NBINS_FIRST + bin : ~0u);
    }
  });
  up_reduce(st, s_st);
  if (threadIdx.x == 0) stats[blockIdx.x] = st;
  __syncthreads();
  const uint32_t u0 = begin >> unit_shift;
  for (uint32_t b = threadIdx.x; b < uint32_t(NBINS_FIRST); b += BLOCK)
    for (uint32_t ui = 0; ui < nu; ui++) unit_hist[size_t(b) * nunits + u0 + ui] = hu[ui * NBINS_FIRST + b];
}

template <typename K, int W, int ITEMS>
__global__ __launch_bounds__(BLOCK, 3) void sort_first(const void* vals, const uint8_t* valid, int64_t voff,
                                                    uint32_t n, int type, int forder, int desc,
                                                    SortCtl* ctl, unsigned long long* status, uint32_t epoch,
                                                    K* out_keys, uint32_t* out_rows, uint32_t* out_idx) {
  constexpr int TILE = BLOCK * ITEMS;
  __shared__ uint32_t wc[WAVES][WC_STRIDE];
  __shared__ uint32_t tile_total[WC_STRIDE];
  __shared__ uint32_t bin_start[RADIX];
  __shared__ uint32_t bin_base[WC_STRIDE];
  __shared__ uint32_t tmp[WAVES];
  __shared__ uint32_t s_tile;
  __shared__ uint8_t s_digit[TILE];
  __shared__ K s_stage[TILE];

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < WAVES * WC_STRIDE; i += BLOCK) (&wc[0][0])[i] = 0u;
  if (threadIdx.x == 0) s_tile = atomicAdd(&ctl->tile_counter[0], 1u);
  __syncthreads();
  const uint32_t tile = s_tile;
  const uint32_t first = ctl->first_active;
  const bool last = first == ctl->last_active;
  const int shift = int(8 * first);

  K keys[ITEMS];
  uint32_t bins[ITEMS];
  const uint32_t rows[1] = {0};   // rows are base_e + 64 * j (ROWS_IOTA)
  const uint32_t base_e = tile * uint32_t(TILE) + uint32_t(w) * 64u * ITEMS + uint32_t(lane);
  // Every load first (lanes past the end read the last row), then the mapping on registers.
  uint32_t vbit[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const uint32_t e = min(base_e + uint32_t(j) * 64u, n - 1u);
    uint32_t bit;
    const uint32_t vb = load_valid_byte(valid, voff, e, bit);
    vbit[j] = (vb >> bit) & 1u;
    keys[j] = K(load_raw<W>(vals, e));
  }
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    uint32_t e = base_e + uint32_t(j) * 64u;
    uint32_t b = BIN_NONE;
    const uint64_t raw = uint64_t(keys[j]);
    keys[j] = 0;
    if (e < n) {
      K k;
      int c = classify_raw<K>(raw, vbit[j] != 0u, type, forder, desc, k);
      if (c == 0) {
        keys[j] = k;
        b = uint32_t(k >> shift) & 0xFFu;
      } else {
        b = c == 1 ? BIN_NAN : BIN_NULL;
      }
    }
    bins[j] = b;
  }
  rank_tile<ITEMS, 9>(bins, wc[w], lane);
  __syncthreads();
  uint32_t vcount = tile_bin_layout<NBINS_FIRST>(wc, tile_total, bin_start, tmp);
  look_back<NBINS_FIRST>(status, tile, epoch, tile_total, bin_base);
  __syncthreads();
  // Turn the exclusive prefixes into absolute destinations.
  for (int b = threadIdx.x; b < NBINS_FIRST; b += BLOCK) {
    uint32_t base;
    if (b < RADIX) base = ctl->digit_base[first][b] + (last ? ctl->value_base : 0u);
    else base = b == BIN_NAN ? ctl->nan_base : ctl->null_base;
    bin_base[b] += base;
  }
  __syncthreads();
  // NaN and null rows go straight to their final slots, in input order.
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    uint32_t b = bin_of(bins[j]);
    if (b == BIN_NAN || b == BIN_NULL) out_idx[bin_base[b] + wc[w][b] + rank_of(bins[j])] = base_e + uint32_t(j) * 64u;
  }
  if (last) {
    scatter_values<K, ITEMS, false, true>(keys, rows, bins, wc[w], bin_start, bin_base, s_digit, s_stage, vcount,
                                          nullptr, out_idx, base_e);
  } else {
    scatter_values<K, ITEMS, true, true>(keys, rows, bins, wc[w], bin_start, bin_base, s_digit, s_stage, vcount,
                                         out_keys, out_rows, base_e);
  }
}

// MODE: PASS_MID and PASS_LAST are launched by a host that read the plan back (only active passes,
// the last one known); PASS_DEVICE is launched for every digit and decides everything on the GPU.
constexpr int PASS_MID = 0, PASS_LAST = 1, PASS_DEVICE = 2;

template <typename K, int ITEMS, int MODE>
__global__ __launch_bounds__(BLOCK) void sort_mid(int pass, SortCtl* ctl, unsigned long long* status,
                                                  uint32_t epoch, K* keys0, uint32_t* rows0, K* keys1,
                                                  uint32_t* rows1, uint32_t* out_idx) {
  constexpr int TILE = BLOCK * ITEMS;
  __shared__ uint32_t wc[WAVES][WC_STRIDE];
  __shared__ uint32_t tile_total[WC_STRIDE];
  __shared__ uint32_t bin_start[RADIX];
  __shared__ uint32_t bin_base[WC_STRIDE];
  __shared__ uint32_t tmp[WAVES];
  __shared__ uint32_t s_tile;
  __shared__ uint8_t s_digit[TILE];
  __shared__ K s_stage[TILE];

  const uint32_t mask = ctl->active_mask;
  const uint32_t first = ctl->first_active;
  if (!((mask >> pass) & 1u) || uint32_t(pass) == first) return;   // uniform over the grid
  const uint32_t m = ctl->m;
  const uint32_t ntiles = (m + TILE - 1) / TILE;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < WAVES * WC_STRIDE; i += BLOCK) (&wc[0][0])[i] = 0u;
  if (threadIdx.x == 0) s_tile = atomicAdd(&ctl->tile_counter[1 + pass], 1u);
  __syncthreads();
  const uint32_t tile = s_tile;
  if (tile >= ntiles) return;   // surplus block: the grid is sized for every row, the pass for values
  const uint32_t rank = uint32_t(__builtin_popcount(mask & ((1u << pass) - 1u)));
  const bool last = MODE == PASS_DEVICE ? uint32_t(pass) == ctl->last_active : MODE == PASS_LAST;
  const K* in_keys = (rank & 1u) ? keys0 : keys1;
  const uint32_t* in_rows = (rank & 1u) ? rows0 : rows1;
  K* out_keys = (rank & 1u) ? keys1 : keys0;
  uint32_t* out_rows = (rank & 1u) ? rows1 : rows0;
  const int shift = 8 * pass;

  K keys[ITEMS];
  uint32_t rows[ITEMS], bins[ITEMS];
  const uint32_t base_e = tile * uint32_t(TILE) + uint32_t(w) * 64u * ITEMS + uint32_t(lane);
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    uint32_t e = base_e + uint32_t(j) * 64u;
    if (e < m) {
      keys[j] = in_keys[e];
      rows[j] = in_rows[e];
      bins[j] = uint32_t(keys[j] >> shift) & 0xFFu;
    } else {
      keys[j] = 0;
      rows[j] = 0;
      bins[j] = BIN_NONE;
    }
  }
  // A full tile has no lanes past the end, so its bins need 8 bits; the last tile needs the 9th.
  if ((tile + 1u) * uint32_t(TILE) <= m) rank_tile<ITEMS, 8>(bins, wc[w], lane);
  else rank_tile<ITEMS, 9>(bins, wc[w], lane);
  __syncthreads();
  uint32_t vcount = tile_bin_layout<RADIX>(wc, tile_total, bin_start, tmp);
  look_back<RADIX>(status, tile, epoch, tile_total, bin_base);
  __syncthreads();
  const uint32_t vb = last ? ctl->value_base : 0u;
  bin_base[threadIdx.x] += ctl->digit_base[pass][threadIdx.x] + vb;
  __syncthreads();
  if (last) {
    scatter_values<K, ITEMS, false>(keys, rows, bins, wc[w], bin_start, bin_base, s_digit, s_stage, vcount,
                                    nullptr, out_idx);
  } else {
    scatter_values<K, ITEMS, true>(keys, rows, bins, wc[w], bin_start, bin_base, s_digit, s_stage, vcount,
                                   out_keys, out_rows);
  }
}

// ---------------------------------------------------------------- small inputs: rank by counting
//
// Up to RANK_MAX rows an argsort is one launch: every workgroup maps all n keys into its LDS and finds
// the places of its own 64 rows, each the number of keys before it in the stable order. No workgroup
// waits for another, and nothing is read back; the work is n^2 compares spread over n / 64 workgroups.
// The LSD passes need a launch per digit, each bound by its launch and one tile's latency. Measured, the
// whole call, int64 (int32) keys with nulls: 1,000 rows 75 -> 18 us (55 -> 18), 8,000 rows 102 -> 30
// (67 -> 30), 16,000 rows 109 -> 46 (71 -> 44). Beyond 16,384 rows the keys no longer fit in LDS and the
// compares of every CU grow with n^2: the passes take over.
constexpr uint32_t RANK_THREADS = 1024;
constexpr uint32_t RANK_WAVES = RANK_THREADS / 64;
constexpr uint32_t RANK_MAX = 16384;   // 128 KiB of 64-bit keys in LDS
constexpr uint32_t RANK_PAD = 256;     // the padded key count is a multiple of it: 16 keys per wave

template <typename K, int W>
__global__ __launch_bounds__(RANK_THREADS) void sort_rank(const void* vals, const uint8_t* valid, int64_t voff,
                                                          uint32_t n, int type, int forder, int desc,
                                                          int nulls_first, uint32_t padded, uint32_t* out_idx) {
  // The keys of all rows (all ones for NaN and null rows and for the padding), which rows are values and
  // which are null, one bit each.
  extern __shared__ __align__(16) unsigned char rank_lds[];
  K* s_key = reinterpret_cast<K*>(rank_lds);
  unsigned long long* s_val = reinterpret_cast<unsigned long long*>(s_key + padded);
  unsigned long long* s_null = s_val + padded / 64;
  __shared__ uint32_t s_cnt[RANK_WAVES][64];
  __shared__ uint32_t s_m, s_z;
  const int lane = threadIdx.x & 63;
  const uint32_t w = threadIdx.x >> 6;
  if (threadIdx.x == 0) s_m = s_z = 0u;
  __syncthreads();
  uint32_t m_here = 0, z_here = 0;
  constexpr int U = 4;   // rows per thread whose loads are issued together
  for (uint32_t base = threadIdx.x; base - threadIdx.x < padded; base += RANK_THREADS * U) {
    uint64_t raw[U];
    uint32_t vb[U], bit[U];
#pragma unroll
    for (int u = 0; u < U; u++) {   // rows past the end read the last row
      const uint32_t j = min(base + uint32_t(u) * RANK_THREADS, n - 1u);
      raw[u] = load_raw<W>(vals, j);
      vb[u] = load_valid_byte(valid, voff, j, bit[u]);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t j = base + uint32_t(u) * RANK_THREADS;
      K key = 0;
      const int cat = j < n ? classify_raw<K>(raw[u], (vb[u] >> bit[u]) & 1u, type, forder, desc, key) : 3;
      const unsigned long long vbal = __ballot(cat == 0), zbal = __ballot(cat == 2);
      if (j < padded) {   // the same for the wave's 64 rows
        s_key[j] = cat == 0 ? key : K(~K(0));
        if (lane == 0) {
          s_val[j >> 6] = vbal;
          s_null[j >> 6] = zbal;
        }
      }
      m_here += uint32_t(__popcll(vbal));
      z_here += uint32_t(__popcll(zbal));
    }
  }
  if (lane == 0 && m_here) atomicAdd(&s_m, m_here);
  if (lane == 0 && z_here) atomicAdd(&s_z, z_here);
  __syncthreads();
  // A wave holds the 64 rows four times over, four rows per lane, and each quarter of its lanes counts
  // every fourth group of four keys of the wave's share: one LDS read serves four rows (with one row per
  // lane the reads bound the kernel). A key of an earlier row counts when it is not above the row's own,
  // one of a later row when it is below.
  const uint32_t r0 = blockIdx.x * 64u, rl = uint32_t(lane) & 15u, part = uint32_t(lane) >> 4;
  K mine[4];
  uint32_t cnt[4];
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) {
    mine[q] = s_key[r0 + rl + 16u * q];
    cnt[q] = 0u;
  }
  // [j0, a1): earlier rows; [a1, b0): this workgroup's; [b0, j1): later rows (all multiples of 16).
  const uint32_t share = padded / RANK_WAVES;
  const uint32_t j0 = w * share, j1 = j0 + share;
  const uint32_t a1 = min(max(r0, j0), j1), b0 = min(max(r0 + 64u, j0), j1);
  for (uint32_t j = j0 + 4u * part; j < a1; j += 16) {
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
      const K k = s_key[j + u];
#pragma unroll
      for (uint32_t q = 0; q < 4; q++) cnt[q] += k <= mine[q] ? 1u : 0u;
    }
  }
  for (uint32_t j = a1 + 4u * part; j < b0; j += 16) {
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
      const K k = s_key[j + u];
#pragma unroll
      for (uint32_t q = 0; q < 4; q++)
        cnt[q] += (k < mine[q] || (k == mine[q] && j + u < r0 + rl + 16u * q)) ? 1u : 0u;
    }
  }
  for (uint32_t j = b0 + 4u * part; j < j1; j += 16) {
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
      const K k = s_key[j + u];
#pragma unroll
      for (uint32_t q = 0; q < 4; q++) cnt[q] += k < mine[q] ? 1u : 0u;
    }
  }
#pragma unroll
  for (uint32_t q = 0; q < 4; q++) {
    cnt[q] += __shfl_xor(cnt[q], 16, 64);
    cnt[q] += __shfl_xor(cnt[q], 32, 64);
    if (part == q) s_cnt[w][16u * q + rl] = cnt[q];
  }
  __syncthreads();
  const uint32_t i = r0 + uint32_t(lane);
  if (w != 0 || i >= n) return;
  uint32_t before = 0;   // keys before this row's
  for (uint32_t v = 0; v < RANK_WAVES; v++) before += s_cnt[v][lane];
  const bool is_val = (s_val[blockIdx.x] >> lane) & 1ull, is_null = (s_null[blockIdx.x] >> lane) & 1ull;
  const uint32_t m = s_m, z = s_z, q = n - m - z;
  const unsigned long long below = (1ull << lane) - 1ull;
  uint32_t dest;
  if (is_val && s_key[i] != K(~K(0))) {
    dest = (nulls_first ? z + q : 0u) + before;
  } else {
    // Rows before this one that are values, and that are null. (A value whose key is all ones was also
    // counted past the NaN and null rows before it, which hold all ones too.)
    uint32_t vals_before = uint32_t(__popcll(s_val[blockIdx.x] & below)), nulls_before = uint32_t(__popcll(s_null[blockIdx.x] & below));
    for (uint32_t b = 0; b < blockIdx.x; b++) {
      vals_before += uint32_t(__popcll(s_val[b]));
      nulls_before += uint32_t(__popcll(s_null[b]));
    }
    if (is_val) dest = (nulls_first ? z + q : 0u) + before - (i - vals_before);
    else if (is_null) dest = (nulls_first ? 0u : m + q) + nulls_before;
    else dest = (nulls_first ? z : m) + (i - vals_before - nulls_before);
  }
  out_idx[dest] = i;
}

template <typename K, int W>
void run_rank(const void* vals, int type, const uint8_t* valid, int64_t voff, uint32_t n, bool desc, int placement,
              int forder, uint32_t* out_idx, hipStream_t s) {
  const uint32_t padded = (n + RANK_PAD - 1) / RANK_PAD * RANK_PAD;
  const size_t lds = size_t(padded) * sizeof(K) + padded / 64 * 16;
  if (lds > 32768)
    AM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(sort_rank<K, W>), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
  ProfScope ps("sort_rank");
  hipLaunchKernelGGL((sort_rank<K, W>), dim3((n + 63u) / 64u), dim3(RANK_THREADS), lds, s, vals, valid, voff, n, type, forder,
                     desc ? 1 : 0, placement == 1 ? 1 : 0, padded, out_idx);
  AM_HIP(hipGetLastError());
}

// ---------------------------------------------------------------- top-digit partition by units
//
// The hybrid sort's first pass, without look-back: the analysis counted every unit's top digits, NaN and
// null rows, so one workgroup per bin scans those counts into every unit's destinations and the last of
// them makes the plan (msd_unit_scan), and persistent workgroups then partition whole units, tile after
// tile, keeping a running destination per bin in LDS (msd_part). Units are taken from a counter, in any
// order. The plan tells the host which digits vary, and whether any bucket needs a level at all: a sort whose
// buckets all fit the bucket sort is five launches and one read-back (it was twelve and two: 17,000 int64
// keys 105 -> 62 us, 300,000 108 -> 71 us; with the 32-bit keys' hybrid sort, full-range int32: 300,000 keys
// 115 -> 65 us, 1M 165 -> 80, 10M 472 -> 298, 40M 1604 -> 914).

// What the host reads of the analysis, in pinned memory.
struct MsdPlan {
  uint32_t mask;             // active digits
  uint32_t m;                // value rows
  uint32_t large, biggest;   // top-digit buckets that need a level, the largest of the others (not of equal keys)
  uint32_t local, top;       // entries of the bucket sort's list; the largest top-digit bucket
  uint32_t lsd;              // the control block holds the LSD passes' plan instead (of the rest, mask and m are set)
};

// The statistics of all workgroups of an analysis, in thread 0.
__device__ __forceinline__ UpStat fold_stats(const UpStat* stats, uint32_t blocks, UpStat* s) {
  UpStat st{0ull, ~0ull, 0u, 0u, 0u, 0u};
  for (uint32_t k = threadIdx.x; k < blocks; k += BLOCK) {
    const UpStat x = stats[k];
    st.m += x.m;
    st.q += x.q;
    st.z += x.z;
    st.key_or |= x.key_or;
    st.key_and &= x.key_and;
  }
  up_reduce(st, s);
  return st;
}

template <int P>
__device__ __forceinline__ uint32_t varying_digits(const UpStat& st) {
  const unsigned long long diff = st.m ? st.key_or ^ st.key_and : 0ull;
  uint32_t mask = 0;
  for (int p = 0; p < P; p++)
    if ((diff >> (8 * p)) & 0xFFull) mask |= 1u << p;
  return mask;
}

// The LSD passes' plan from the counts of their digits, workgroup b totalling value b of each of the four; the
// last one done makes the plan.
__device__ __forceinline__ void lsd_scan(SortCtl* ctl, const uint32_t* counts, const UpStat* stats, uint32_t blocks,
                                         int nulls_first, uint32_t* ticket, MsdPlan* plan) {
  __shared__ uint32_t tmp[WAVES], s_sum[WAVES][4];
  __shared__ UpStat s_st[WAVES];
  __shared__ uint32_t s_last;
  const uint32_t b = blockIdx.x;
  uint32_t sum[4] = {0u, 0u, 0u, 0u};
  if (b < uint32_t(RADIX))
    for (uint32_t k = threadIdx.x; k < blocks; k += BLOCK)
#pragma unroll
      for (uint32_t p = 0; p < 4; p++) sum[p] += counts[(size_t(p) * RADIX + b) * blocks + k];
#pragma unroll
  for (uint32_t p = 0; p < 4; p++) {
    for (int off = 32; off > 0; off >>= 1) sum[p] += __shfl_xor(sum[p], off, 64);
    if ((threadIdx.x & 63u) == 0u) s_sum[threadIdx.x >> 6][p] = sum[p];
  }
  __syncthreads();
  if (threadIdx.x < 4u && b < uint32_t(RADIX)) {
    uint32_t t = 0;
    for (int w = 0; w < WAVES; w++) t += s_sum[w][threadIdx.x];
    atomic_done(atomicExch(&ctl->digit_base[threadIdx.x][b], t));
  }
  __syncthreads();
  if (threadIdx.x == 0) s_last = last_block(ticket) ? 1u : 0u;
  __syncthreads();
  if (!s_last) return;   // uniform
  const UpStat st = fold_stats(stats, blocks, s_st);
  uint32_t v[4];
#pragma unroll
  for (uint32_t p = 0; p < 4; p++)   // every load first
    v[p] = __hip_atomic_load(&ctl->digit_base[p][threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (uint32_t p = 0; p < 4; p++) {
    uint32_t total;
    ctl->digit_base[p][threadIdx.x] = block_excl_scan(v[p], tmp, total);
  }
  if (threadIdx.x < 16) ctl->tile_counter[threadIdx.x] = 0u;
  if (threadIdx.x == 0) {
    const uint32_t varying = varying_digits<4>(st);
    set_lsd_plan(ctl, varying, st.m, st.q, st.z, nulls_first);
    plan->mask = varying;
    plan->m = st.m;
    plan->lsd = 1u;
  }
}

// Workgroup b: the exclusive scan of bin b's unit counts in place, and its total. The last workgroup done
// makes the plan: the active digits, where each bin's rows start (first_base), the level kernels' control
// words, and the top-digit buckets, into the first large-bucket list or the bucket sort's list.
template <int P>
__global__ __launch_bounds__(BLOCK) void msd_unit_scan(SortCtl* ctl, uint32_t* unit_hist, uint32_t nunits,
                                                       const UpStat* stats, uint32_t blocks, int nulls_first,
                                                       MsdCtl* mc, uint32_t epoch, Bucket* large, Bucket* local,
                                                       uint32_t local_cap, uint32_t* lc, void* key_out,
                                                       unsigned long long key_xor, uint32_t* bucket_base, uint32_t* ticket,
                                                       MsdPlan* plan) {
  __shared__ uint32_t tmp[WAVES];
  __shared__ uint32_t s_last, s_mask, s_first[NBINS_FIRST];
  __shared__ UpStat s_st[WAVES];
  __shared__ LongCopies s_long;
  if constexpr (P == 4) {
    if (ctl->lsd) {   // uniform over the grid
      lsd_scan(ctl, unit_hist, stats, blocks, nulls_first, ticket, plan);
      return;
    }
  }
  const uint32_t b = blockIdx.x;
  uint32_t* h = unit_hist + size_t(b) * nunits;
  uint32_t carry = 0;
  for (uint32_t u0 = 0; u0 < nunits; u0 += BLOCK) {
    const uint32_t u = u0 + threadIdx.x;
    const uint32_t v = u < nunits ? h[u] : 0u;
    uint32_t total;
    const uint32_t ex = block_excl_scan(v, tmp, total);
    if (u < nunits) h[u] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) {
    atomic_done(atomicExch(&ctl->bin_total[b], carry));
    s_last = last_block(ticket) ? 1u : 0u;
  }
  __syncthreads();
  if (!s_last) return;   // uniform
  const UpStat st = fold_stats(stats, blocks, s_st);
  uint32_t total;
  const uint32_t size = __hip_atomic_load(&ctl->bin_total[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint32_t start = block_excl_scan(size, tmp, total);
  if (threadIdx.x < LC_WORDS) lc[threadIdx.x] = 0u;
  if (threadIdx.x == 0) {
    const uint32_t mask = varying_digits<P>(st);
    s_mask = mask;
    s_long.count = 0u;
    const uint32_t value_base = nulls_first ? st.z + st.q : 0u;
    s_first[BIN_NAN] = nulls_first ? st.z : st.m;
    s_first[BIN_NULL] = nulls_first ? 0u : st.m + st.q;
    *mc = {mask, value_base, epoch, 0u, key_out, key_xor};
    plan->mask = mask;
    plan->m = st.m;
    plan->lsd = 0u;
  }
  clear_ctl(ctl);   // the partition's unit counter, and the rest in case the LSD passes run
  s_first[threadIdx.x] = start;
  if (bucket_base) bucket_base[threadIdx.x] = start;
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < uint32_t(NBINS_FIRST); k += BLOCK) ctl->first_base[k] = s_first[k];
  const uint32_t low = s_mask & ((1u << (P - 1)) - 1u);
  const bool is_large = size > LOCAL_MAX && low != 0u, is_local = size != 0u && !is_large;
  const Bucket bk{start, size, 0u, uint32_t(P - 1)};
  const uint32_t pieces = !is_local ? 0u : low == 0u ? copy_pieces(size, 0u) : 1u;   // without a lower digit: copies
  uint32_t n_large, n_local;
  const uint32_t at_large = block_excl_scan(is_large ? 1u : 0u, tmp, n_large);
  const uint32_t at_local = block_excl_scan(pieces, tmp, n_local);
  const uint32_t biggest = block_incl_max(is_local && low != 0u ? size : 0u, tmp);
  const uint32_t top = block_incl_max(size, tmp);
  if (is_large) large[at_large] = bk;
  if (pieces == 1u && at_local < local_cap) local[at_local] = bk;
  if (pieces > 1u) s_long.add(start, size, at_local);
  __syncthreads();
  s_long.write(local, local_cap, 0u, 0u, uint32_t(P - 1));
  if (threadIdx.x == BLOCK - 1) {
    lc[LC_LIST] = n_large;
    lc[LC_LOCAL] = n_local;
    lc[LC_MAXLOCAL] = biggest;
    lc[LC_OVERFLOW] = n_local > local_cap ? 1u : 0u;
    plan->large = n_large;
    plan->biggest = biggest;
    plan->local = n_local;
    plan->top = top;
  }
}

// POS_ROWS: the rows written beside the keys are their own positions in this pass's output, and
// pos_of_row[row] gets that position (all ones for NaN and null rows), for the ORDER BY of whole
// tables (order_by_columns).
template <typename K, int W, int ITEMS, bool POS_ROWS = false>
__global__ __launch_bounds__(BLOCK, 3) void msd_part(const void* vals, const uint8_t* valid, int64_t voff,
                                                     uint32_t n, int type, int forder, int desc, SortCtl* ctl,
                                                     const uint32_t* unit_off, uint32_t nunits,
                                                     uint32_t unit_shift, K* out_keys, uint32_t* out_rows,
                                                     uint32_t* out_idx, uint32_t* pos_of_row = nullptr) {
  constexpr int P = int(sizeof(K));
  constexpr int TILE = BLOCK * ITEMS;
  static_assert((1u << UNIT_SHIFT_SMALL) % TILE == 0, "units hold whole tiles");
  __shared__ uint32_t wc[WAVES][WC_STRIDE];
  __shared__ uint32_t tile_total[WC_STRIDE];
  __shared__ uint32_t bin_start[RADIX];
  __shared__ uint32_t bin_base[WC_STRIDE];
  __shared__ uint32_t running[WC_STRIDE];
  __shared__ uint32_t tmp[WAVES];
  __shared__ uint32_t s_unit;
  __shared__ uint8_t s_digit[TILE];
  __shared__ K s_stage[TILE];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int shift = 8 * (P - 1);
  const uint32_t rows[1] = {0};   // rows are base_e + 64 * j (ROWS_IOTA)
  while (true) {
    if (threadIdx.x == 0) s_unit = atomicAdd(&ctl->tile_counter[11], 1u);
    __syncthreads();
    const uint32_t unit = s_unit;
    if (unit >= nunits) return;   // uniform: every workgroup ends here once the units run out
    for (int b = threadIdx.x; b < NBINS_FIRST; b += BLOCK) running[b] = ctl->first_base[b] + unit_off[size_t(b) * nunits + unit];
    const uint32_t begin = unit << unit_shift;
    const uint32_t end = min(n, begin + (1u << unit_shift));
    for (uint32_t t0 = begin; t0 < end; t0 += TILE) {
      for (int i = threadIdx.x; i < WAVES * WC_STRIDE; i += BLOCK) (&wc[0][0])[i] = 0u;
      __syncthreads();
      K keys[ITEMS];
      uint32_t bins[ITEMS], vbit[ITEMS];
      const uint32_t base_e = t0 + uint32_t(w) * 64u * ITEMS + uint32_t(lane);
#pragma unroll
      for (int j = 0; j < ITEMS; j++) {   // every load first (lanes past the unit read its last row)
        const uint32_t e = min(base_e + uint32_t(j) * 64u, end - 1u);
        uint32_t bit;
        const uint32_t vb = load_valid_byte(valid, voff, e, bit);
        vbit[j] = (vb >> bit) & 1u;
        keys[j] = K(load_raw<W>(vals, e));
      }
#pragma unroll
      for (int j = 0; j < ITEMS; j++) {
        const uint32_t e = base_e + uint32_t(j) * 64u;
        uint32_t b = BIN_NONE;
        const uint64_t raw = uint64_t(keys[j]);
        keys[j] = 0;
        if (e < end) {
          K k;
          const int c = classify_raw<K>(raw, vbit[j] != 0u, type, forder, desc, k);
          if (c == 0) {
            keys[j] = k;
            b = uint32_t(k >> shift) & 0xFFu;
          } else {
            b = c == 1 ? BIN_NAN : BIN_NULL;
          }
        }
        bins[j] = b;
      }
      rank_tile<ITEMS, 9>(bins, wc[w], lane);
      __syncthreads();
      const uint32_t vcount = tile_bin_layout<NBINS_FIRST>(wc, tile_total, bin_start, tmp);
      for (int b = threadIdx.x; b < NBINS_FIRST; b += BLOCK) {
        bin_base[b] = running[b];
        running[b] += tile_total[b];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < ITEMS; j++) {   // NaN and null rows go straight to their final slots
        const uint32_t b = bin_of(bins[j]);
        if (b == BIN_NAN || b == BIN_NULL) {
          out_idx[bin_base[b] + wc[w][b] + rank_of(bins[j])] = base_e + uint32_t(j) * 64u;
          if constexpr (POS_ROWS) pos_of_row[base_e + uint32_t(j) * 64u] = 0xFFFFFFFFu;
        }
      }
      scatter_values<K, ITEMS, true, true, POS_ROWS>(keys, rows, bins, wc[w], bin_start, bin_base, s_digit, s_stage,
                                                     vcount, out_keys, out_rows, base_e, pos_of_row);
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------- hybrid MSD sort (64- and 32-bit keys)
//
// For large inputs of 64- and 32-bit keys whose top digit varies: the first pass partitions the value rows
// stably by the top digit (msd_part, above). Then, level by level down the active digits, every
// bucket still larger than LOCAL_MAX rows is partitioned stably by the next digit (onesweep tiles
// whose look-back stops at their bucket's first tile), into the other key / row buffer at the same
// positions; a bucket whose digit is the same on all its rows is carried to the next level without
// moving. Buckets of at most LOCAL_MAX rows leave for the bucket sort, which sorts each in LDS by its
// remaining digits and writes its rows to their final slots. After the lowest active digit every
// bucket holds equal keys, in input order, and is copied. Uniform keys take three passes over the
// rows (top digit, second digit, bucket sort) instead of eight.

#ifndef AM_MSD_FITEMS
#define AM_MSD_FITEMS 16   // keys per thread of the top-digit partition
#endif
// ---------------------------------------------------------------- host side

// The counter that the last workgroup of an analysis finds itself by: one per thread, zero between kernels.
uint32_t* scan_ticket(hipStream_t s) {
  thread_local DevBuf buf;
  if (!buf) {
    buf = device_alloc_thread(128);
    hipLaunchKernelGGL(fill_u64, dim3(1), dim3(64), 0, s, static_cast<unsigned long long*>(buf->ptr), size_t(16), 0ull);
    AM_HIP(hipGetLastError());
  }
  retain(buf);
  return static_cast<uint32_t*>(buf->ptr);
}

// With pos_of_row (the ORDER BY of whole tables): only the hybrid sort runs, with positions for rows
// (msd_part's POS_ROWS form); when it cannot (too few rows, a constant top digit, a full bucket list)
// the call returns false and out_idx holds nothing to use. *value_rows receives m. With key_out (an
// integer key) the bucket sorts also write the value block of the sorted key column there; *keys_written
// says whether they did (the LSD passes do not).
// Rows from which the LSD passes' plan is read back.
constexpr uint32_t PLAN_READ_MIN = 1u << 16;
// Rows from which a key type's columns are analysed for the hybrid sort. Integers spread over the top digit's
// values, so from the counting sort's limit (64-bit) and from where the LSD passes read their plan back too
// (32-bit; int32 values below 5,000, which the LSD passes then take, would lose 10 us before). The top digit
// of floats holds their sign and exponent: a few buckets hold most rows and take a level or two, which pays
// from 2^16 rows for eight digits (40,000 rows: 123 us LSD, 148 hybrid; 100,000: 134 against 118) and from
// 2^24 for four.
uint32_t hybrid_min(int type) {
  switch (type) {
    case T_I64: case T_U64: return RANK_MAX + 1u;
    case T_F64: case T_I32: case T_U32: return 1u << 16;
    case T_F32: return 1u << 24;
    default: return ~0u;   // narrower keys: at most two digits vary
  }
}

// The analysis of the hybrid sort: units counted and scanned, the plan on its way to host_plan_words().
struct Units {
  DevBuf buf;
  uint32_t* hist = nullptr;   // [NBINS_FIRST][count], each bin's running offsets
  uint32_t count = 0, shift = 0;
};

template <typename K, int W>
Units msd_analyse(const void* vals, int type, const uint8_t* valid, int64_t voff, uint32_t n, int desc, int placement,
                  int forder, SortCtl* ctl, const MsdWork& w, uint32_t epoch, void* key_out,
                  unsigned long long key_xor, uint32_t* bucket_base, hipStream_t s, bool guess = false) {
  Units un;
  un.shift = n >= (1u << 22) ? UNIT_SHIFT_LARGE : UNIT_SHIFT_SMALL;
  const uint32_t unit_rows = 1u << un.shift, cus = uint32_t(device().cu_count);
  un.count = (n + unit_rows - 1) / unit_rows;
  // Workgroups of whole units, at most UNITS_PER_BLOCK: one each until every CU has four.
  const uint32_t per = std::min(UNITS_PER_BLOCK, std::max(1u, (un.count + cus * 4u - 1u) / (cus * 4u)));
  const uint32_t rpb = per * unit_rows, blocks = (n + rpb - 1) / rpb;
  size_t words = size_t(un.count) * NBINS_FIRST;
  if (guess) words = std::max(words, size_t(blocks) * 4 * RADIX);
  un.buf = device_alloc(words * 4 + size_t(blocks) * sizeof(UpStat) + 16);
  UpStat* stats = static_cast<UpStat*>(un.buf->ptr);
  un.hist = reinterpret_cast<uint32_t*>(stats + blocks);
  {
    ProfScope ps("sort_upsweep");
    hipLaunchKernelGGL((msd_upsweep<K, W>), dim3(blocks), dim3(BLOCK), 0, s, vals, valid, voff, n, type, forder, desc, rpb,
                       stats, un.hist, un.count, un.shift, guess ? 1 : 0, ctl);
    AM_HIP(hipGetLastError());
  }
  ProfScope ps("sort_msd_unit_scan");
  hipLaunchKernelGGL(msd_unit_scan<int(sizeof(K))>, dim3(NBINS_FIRST), dim3(BLOCK), 0, s, ctl, un.hist, un.count,
                     static_cast<const UpStat*>(stats), blocks, placement == 1 ? 1 : 0, w.mc, epoch, w.large[0], w.local,
                     w.local_cap, w.lc, key_out, key_xor, bucket_base, scan_ticket(s),
                     reinterpret_cast<MsdPlan*>(host_plan_words()));
  AM_HIP(hipGetLastError());
  return un;
}

template <typename K, int W, int ITEMS>
bool run_sort(const void* vals, int type, const uint8_t* valid, int64_t voff, uint32_t n, bool desc,
              int placement, int forder, uint32_t* out_idx, hipStream_t s, uint32_t* pos_of_row = nullptr,
              uint32_t* value_rows = nullptr, uint32_t* bucket_base = nullptr, void* key_out = nullptr,
              unsigned long long key_xor = 0, bool* keys_written = nullptr) {
  constexpr int P = int(sizeof(K));
  const bool hybrid_ok = n >= hybrid_min(type) && n <= HYBRID_MAX_ROWS && !capturing(s);
  if (pos_of_row && !hybrid_ok) return false;
  constexpr int TILE = BLOCK * ITEMS;
  // The first pass keeps at most 16 keys per thread: its raw-column loads and 258-bin classification
  // need more registers, and 16 keeps it at three workgroups per CU.
  constexpr int FITEMS = ITEMS > 16 ? 16 : ITEMS;
  constexpr int FTILE = BLOCK * FITEMS;
  const uint32_t tiles = (n + TILE - 1) / TILE;
  const uint32_t ftiles = (n + FTILE - 1) / FTILE;
  DevBuf ctl_buf = device_alloc(sizeof(SortCtl));
  SortCtl* ctl = static_cast<SortCtl*>(ctl_buf->ptr);
  // Status rows for every tile of a pass; a level of the hybrid sort has up to one more tile per large
  // bucket (fewer than the levels' bucket capacity, m / 2048 + 4096).
  const uint32_t hyb_tiles = tiles + n / 2048u + 4096u + 2u;
  uint32_t epoch = reserve_status(size_t(std::max(hyb_tiles, ftiles)) * STATUS_STRIDE, s);
  unsigned long long* status = static_cast<unsigned long long*>(t_ws.status->ptr);
  retain(t_ws.status);
  DevBuf k0 = device_alloc(size_t(n) * sizeof(K)), k1 = device_alloc(size_t(n) * sizeof(K));
  DevBuf r0 = device_alloc(size_t(n) * 4), r1 = device_alloc(size_t(n) * 4);
  const int dsc = desc ? 1 : 0;
  K* kp0 = static_cast<K*>(k0->ptr);
  K* kp1 = static_cast<K*>(k1->ptr);
  uint32_t* rp0 = static_cast<uint32_t*>(r0->ptr);
  uint32_t* rp1 = static_cast<uint32_t*>(r1->ptr);
  // Large inputs of 32- and 64-bit keys may take the hybrid sort: its analysis is read back once.
  uint32_t digits = (1u << P) - 1u;
  bool planned = false, tried = false;   // analysed; partitioned (the control block is used up)
  MsdPlan plan{};
  MsdWork w;
  Units un;
  bool hybrid = hybrid_ok;
  if (hybrid) {
    try {   // some 3 bytes a row beside the buffers above, without which the LSD passes sort
      w = msd_work(n, ITEMS, device_alloc);
      un = msd_analyse<K, W>(vals, type, valid, voff, n, dsc, placement, forder, ctl, w, epoch, key_out, key_xor,
                             bucket_base, s, P == 4);
    } catch (const OutOfMemory&) {
      hybrid = false;
    }
  }
  if (hybrid) {
    const uint32_t nunits = un.count, unit_shift = un.shift;
    uint32_t* unit_hist = un.hist;
    MsdPlan* hp = reinterpret_cast<MsdPlan*>(host_plan_words());
    AM_HIP(hipStreamSynchronize(s));
    plan = *hp;
    planned = true;
    digits = plan.mask ? plan.mask : 1u;
    if (value_rows) *value_rows = plan.m;
    const bool take = !plan.lsd && ((plan.mask >> (P - 1)) & 1u) && (P == 8 || plan.top <= MSD32_TOP_MAX || n >= MSD32_SAVES);
    if (pos_of_row && !take) return false;
    if (take) {
      tried = true;
      {
        ProfScope ps("sort_msd_first");
        const uint32_t workers = std::min(nunits, uint32_t(device().cu_count) * 3u);
        if (pos_of_row)
          hipLaunchKernelGGL((msd_part<K, W, AM_MSD_FITEMS, true>), dim3(workers), dim3(BLOCK), 0, s, vals, valid, voff, n,
                             type, forder, dsc, ctl, unit_hist, nunits, unit_shift, kp0, rp0, out_idx, pos_of_row);
        else
          hipLaunchKernelGGL((msd_part<K, W, AM_MSD_FITEMS>), dim3(workers), dim3(BLOCK), 0, s, vals, valid, voff, n, type,
                             forder, dsc, ctl, unit_hist, nunits, unit_shift, kp0, rp0, out_idx, nullptr);
        AM_HIP(hipGetLastError());
      }
      if (msd_levels<K, ITEMS>(w, plan.m, P - 1, plan.mask, false, LOCAL_MAX, status, kp0, rp0, kp1, rp1, out_idx, s,
                               key_out != nullptr, &plan.large, &plan.biggest, &plan.local)) {
        if (keys_written) *keys_written = true;
        return true;
      }
      // The bucket sort's list ran out of room: the LSD passes below.
    }
  }
  if (pos_of_row) return false;
  if (!planned || tried) {
    ProfScope ps("sort_init");
    hipLaunchKernelGGL(sort_init, dim3(1), dim3(1024), 0, s, ctl);
    AM_HIP(hipGetLastError());
  }
  if (!plan.lsd) {
    // Two workgroups per CU, and four from 2^23 rows: each adds up to 256 counts per digit to shared ones, which a
    // long share of rows repays (int64 below 5,000, 50M rows 1294 -> 1244 us; 1M float32 170 either way).
    const uint64_t rows = n, max_blocks = uint64_t(device().cu_count) * (n >= (1u << 23) ? 4u : 2u);   // 64 bits: the sums may pass 2^32
    const uint64_t wanted = std::max<uint64_t>(1, std::min(max_blocks, (rows + 2u * UP_STEP - 1u) / (2u * UP_STEP)));
    const uint32_t rpb = uint32_t(std::min<uint64_t>(((rows + wanted - 1) / wanted + UP_STEP - 1) / UP_STEP * UP_STEP, UINT32_MAX));
    const uint32_t blocks = uint32_t((rows + rpb - 1) / rpb);
    {
      ProfScope ps("sort_upsweep");
      hipLaunchKernelGGL((sort_upsweep<K, W>), dim3(blocks), dim3(BLOCK), 0, s, vals, valid, voff, n, type, forder, dsc, rpb,
                         ctl, digits, placement == 1 ? 1 : 0, scan_ticket(s));
      AM_HIP(hipGetLastError());
    }
  }
  // Large inputs read the plan back once (one sync, as the reference's analysis readback does), so
  // that only active passes are launched, over the value rows only; the hybrid sort's analysis has it.
  const bool analyse = planned || (n >= PLAN_READ_MIN && !capturing(s));
  struct Plan { uint32_t mask, first, last, m; } lsd{0xFFu, 0, uint32_t(P - 1), n};
  if (planned) {
    const uint32_t mask = plan.m <= 1u ? 1u : digits;   // as sort_plan has it
    lsd = Plan{mask, uint32_t(__builtin_ctz(mask)), 31u - uint32_t(__builtin_clz(mask)), plan.m};
  } else if (analyse) {
    Plan* hp = reinterpret_cast<Plan*>(host_plan_words());
    hipLaunchKernelGGL(sort_read_plan, dim3(1), dim3(1), 0, s, ctl, reinterpret_cast<uint32_t*>(hp));
    AM_HIP(hipGetLastError());
    AM_HIP(hipStreamSynchronize(s));
    lsd = *hp;
  }
  {
    ProfScope ps("sort_first");
    hipLaunchKernelGGL((sort_first<K, W, FITEMS>), dim3(ftiles), dim3(BLOCK), 0, s, vals, valid, voff, n, type, forder,
                       dsc, ctl, status, epoch, kp0, rp0, out_idx);
    AM_HIP(hipGetLastError());
  }
  if (analyse) {
    // The host read the plan back: launch only the active passes, each over the value rows, with
    // the last one's kernel known (no key writes).
    const uint32_t mtiles = std::max<uint32_t>(1, (lsd.m + TILE - 1) / TILE);
    for (int p = 0; p < P; p++) {
      if (!((lsd.mask >> p) & 1u) || uint32_t(p) == lsd.first) continue;
      if (uint32_t(p) == lsd.last) {
        ProfScope ps("sort_scatter_last");
        hipLaunchKernelGGL((sort_mid<K, ITEMS, PASS_LAST>), dim3(mtiles), dim3(BLOCK), 0, s, p, ctl, status,
                           epoch + 1u + uint32_t(p), kp0, rp0, kp1, rp1, out_idx);
      } else {
        ProfScope ps("sort_scatter");
        hipLaunchKernelGGL((sort_mid<K, ITEMS, PASS_MID>), dim3(mtiles), dim3(BLOCK), 0, s, p, ctl, status,
                           epoch + 1u + uint32_t(p), kp0, rp0, kp1, rp1, out_idx);
      }
      AM_HIP(hipGetLastError());
    }
  } else {
    for (int p = 0; p < P; p++) {
      ProfScope ps("sort_pass_dev");
      hipLaunchKernelGGL((sort_mid<K, ITEMS, PASS_DEVICE>), dim3(tiles), dim3(BLOCK), 0, s, p, ctl, status,
                         epoch + 1u + uint32_t(p), kp0, rp0, kp1, rp1, out_idx);
      AM_HIP(hipGetLastError());
    }
  }
  return true;
}

template <typename K, int W>
void dispatch_items(int items, const void* vals, int type, const uint8_t* valid, int64_t voff, uint32_t n,
                    bool desc, int placement, int forder, uint32_t* out_idx, hipStream_t s) {
  switch (items) {
    case 4: run_sort<K, W, 4>(vals, type, valid, voff, n, desc, placement, forder, out_idx, s); break;
    case 8: run_sort<K, W, 8>(vals, type, valid, voff, n, desc, placement, forder, out_idx, s); break;
    case 12: run_sort<K, W, 12>(vals, type, valid, voff, n, desc, placement, forder, out_idx, s); break;
    case 20: run_sort<K, W, 20>(vals, type, valid, voff, n, desc, placement, forder, out_idx, s); break;
    default: run_sort<K, W, 16>(vals, type, valid, voff, n, desc, placement, forder, out_idx, s); break;
  }
}

// ---------------------------------------------------------------- keep-first distinct rows
//
// The rows of distinct mixed keys (a bijection of the original keys, so that the digits are spread whatever
// the keys are): partitioned by the hybrid sort's passes until a bucket fits in LDS, deduplicated there
// (hyb_dedupe marks every row whose key an earlier one holds), and the unmarked rows compacted in row
// order. No table in global memory is probed (an insert of a new key is an atomic at the memory side), and
// nothing is sorted beyond the buckets. 10M rows over two int64 columns (9.95M distinct), unique rows and both
// columns taken: 3.26 ms by the hash mapping, its two sorts and lowest rows, 0.58 ms so; the passes run at 1.5
// to 3 TB/s, the marks' random bytes at 1.5.
constexpr uint32_t KEEP_TILE = 4096;   // rows per workgroup of the compaction, 16 consecutive ones per thread

__device__ __forceinline__ uint32_t keep_flags(const uint8_t* dup, uint32_t n, uint32_t row0) {
  // Sixteen consecutive marks (dup is padded to whole tiles) -> a bit per kept row.
  const uint4 v = *reinterpret_cast<const uint4*>(dup + row0);
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t keep = 0;
#pragma unroll
  for (int k = 0; k < 16; k++) keep |= (((w[k >> 2] >> (8 * (k & 3))) & 1u) ^ 1u) << k;
  const uint32_t left = row0 < n ? min(n - row0, 16u) : 0u;
  return keep & ((1u << left) - 1u);
}

// Each tile's kept rows; the last workgroup scans them into bases and reports the total.
__global__ __launch_bounds__(BLOCK) void keep_count(const uint8_t* dup, uint32_t n, uint32_t* base, uint32_t* ticket,
                                                    uint32_t* total) {
  __shared__ uint32_t tmp[WAVES];
  __shared__ uint32_t s_last;
  const uint32_t c = uint32_t(__popc(keep_flags(dup, n, blockIdx.x * KEEP_TILE + threadIdx.x * 16u)));
  uint32_t sum;
  block_excl_scan(c, tmp, sum);
  if (threadIdx.x == 0) {
    atomic_done(atomicExch(&base[blockIdx.x], sum));
    s_last = last_block(ticket) ? 1u : 0u;
  }
  __syncthreads();
  if (!s_last) return;   // uniform
  uint32_t carry = 0;
  for (uint32_t t0 = 0; t0 < gridDim.x; t0 += BLOCK * 4u) {
    uint32_t v[4], x = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
      const uint32_t t = t0 + threadIdx.x * 4u + k;
      v[k] = t < gridDim.x ? __hip_atomic_load(&base[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
      x += v[k];
    }
    uint32_t step;
    uint32_t run = carry + block_excl_scan(x, tmp, step);
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
      const uint32_t t = t0 + threadIdx.x * 4u + k;
      if (t < gridDim.x) base[t] = run;
      run += v[k];
    }
    carry += step;
  }
  if (threadIdx.x == 0) *total = carry;
}

__global__ __launch_bounds__(BLOCK) void keep_write(const uint8_t* dup, uint32_t n, const uint32_t* base, uint32_t* out) {
  __shared__ uint32_t tmp[WAVES];
  __shared__ uint32_t s_row[KEEP_TILE];
  const uint32_t row0 = blockIdx.x * KEEP_TILE + threadIdx.x * 16u;
  uint32_t keep = keep_flags(dup, n, row0), total;
  uint32_t at = block_excl_scan(uint32_t(__popc(keep)), tmp, total);
  while (keep) {
    const uint32_t b = uint32_t(__ffs(int(keep))) - 1u;
    keep &= keep - 1u;
    s_row[at++] = row0 + b;
  }
  __syncthreads();
  uint32_t* o = out + base[blockIdx.x];
  for (uint32_t j = threadIdx.x; j < total; j += BLOCK) o[j] = s_row[j];
}

template <typename K>
bool distinct_rows_t(const void* keys, uint32_t n, DevBuf& rows, uint32_t& kept, hipStream_t s) {
  constexpr int ITEMS = 16, W = int(sizeof(K));
  constexpr int TYPE = W == 8 ? T_U64 : T_U32;
  DevBuf ctl_buf = device_alloc(sizeof(SortCtl));
  SortCtl* ctl = static_cast<SortCtl*>(ctl_buf->ptr);
  const uint32_t epoch = reserve_status(size_t(n / (BLOCK * ITEMS) + n / 2048u + 4100u) * STATUS_STRIDE, s);
  unsigned long long* status = static_cast<unsigned long long*>(t_ws.status->ptr);
  retain(t_ws.status);
  const MsdWork w = msd_work(n, ITEMS, device_alloc);
  const Units un = msd_analyse<K, W>(keys, TYPE, nullptr, 0, n, 0, 0, 0, ctl, w, epoch, nullptr, 0, nullptr, s);
  const uint32_t tiles = (n + KEEP_TILE - 1) / KEEP_TILE;
  DevBuf dup_buf = device_alloc(size_t(tiles) * KEEP_TILE);
  auto* dup = static_cast<uint8_t*>(dup_buf->ptr);
  hipLaunchKernelGGL(fill_u64, dim3(std::min(tiles, 2048u)), dim3(256), 0, s, reinterpret_cast<unsigned long long*>(dup),
                     size_t(tiles) * KEEP_TILE / 8, 0ull);
  AM_HIP(hipGetLastError());
  DevBuf k0 = device_alloc(size_t(n) * W), k1 = device_alloc(size_t(n) * W);
  DevBuf r0 = device_alloc(size_t(n) * 4), r1 = device_alloc(size_t(n) * 4);
  K *kp0 = static_cast<K*>(k0->ptr), *kp1 = static_cast<K*>(k1->ptr);
  auto *rp0 = static_cast<uint32_t*>(r0->ptr), *rp1 = static_cast<uint32_t*>(r1->ptr);
  AM_HIP(hipStreamSynchronize(s));
  const MsdPlan plan = *reinterpret_cast<MsdPlan*>(host_plan_words());
  if (!((plan.mask >> (W - 1)) & 1u)) return false;   // a key or two: any other way is as good
  {
    ProfScope ps("sort_msd_first");
    hipLaunchKernelGGL((msd_part<K, W, AM_MSD_FITEMS>), dim3(std::min(un.count, uint32_t(device().cu_count) * 3u)), dim3(BLOCK),
                       0, s, keys, static_cast<const uint8_t*>(nullptr), int64_t(0), n, TYPE, 0, 0, ctl, un.hist, un.count,
                       un.shift, kp0, rp0, static_cast<uint32_t*>(nullptr), nullptr);
    AM_HIP(hipGetLastError());
  }
  if (!msd_levels<K, ITEMS>(w, plan.m, W - 1, plan.mask, false, LOCAL_MAX, status, kp0, rp0, kp1, rp1, nullptr, s, false,
                            &plan.large, &plan.biggest, &plan.local, dup))
    return false;
  DevBuf all = device_alloc(size_t(n) * 4), base = device_alloc(size_t(tiles) * 4);
  std::shared_ptr<void> slot = pinned_slot();
  auto* total = static_cast<uint32_t*>(slot.get());
  {
    ProfScope ps("keep_rows");
    hipLaunchKernelGGL(keep_count, dim3(tiles), dim3(BLOCK), 0, s, static_cast<const uint8_t*>(dup), n,
                       static_cast<uint32_t*>(base->ptr), scan_ticket(s), total);
    hipLaunchKernelGGL(keep_write, dim3(tiles), dim3(BLOCK), 0, s, static_cast<const uint8_t*>(dup), n,
                       static_cast<const uint32_t*>(base->ptr), static_cast<uint32_t*>(all->ptr));
    AM_HIP(hipGetLastError());
  }
  AM_HIP(hipStreamSynchronize(s));
  kept = *total;
  rows = all;
  if (n >= (1u << 20) && kept < n / 8) {   // the result outlives the call: in a block of its own size
    rows = device_alloc(size_t(kept) * 4);
    AM_HIP(hipMemcpyAsync(rows->ptr, all->ptr, size_t(kept) * 4, hipMemcpyDeviceToDevice, s));
    sync();
  }
  return true;
}

// ---------------------------------------------------------------- ORDER BY of whole tables
//
// order_by_columns sorts by one 64-bit integer key with the hybrid sort in its POS_ROWS form: rows carried
// through the levels are positions p in the top-digit partition's output (the value block), and
// pos_of_row[r] = p for every value row r. A column then moves in two row passes:
//   ob_partition  part[pos_of_row[r]] = col[r]: the column laid out as the partition laid out its keys
//                 (reads in row order; writes in runs, as the partition's own)
//   ob_gather     out[i] = part[out_idx[i]] in the value block, col[out_idx[i]] in the null block
//                 (whose rows keep input order)
// Output i of the value block and its position p lie in the same top-digit bucket, so the gather of an
// output range reads one bucket's part of the column. Each XCD takes its own eighth of the outputs
// (XCD-private chunk counters; a workgroup that finds its eighth done takes chunks of the others), so a
// bucket's lines are fetched into one L2, not eight.

#ifndef AM_OB_CHUNK
#define AM_OB_CHUNK 4096
#endif
#ifndef AM_OB_GATHER_WG
#define AM_OB_GATHER_WG 4
#endif
constexpr uint32_t OB_CHUNK = AM_OB_CHUNK;   // outputs per chunk of the gather (64-row words)
constexpr uint32_t OB_GROUPS = OB_CHUNK / 64 / WAVES;   // 64-row groups per wave per chunk

// Each workgroup takes one contiguous range of rows, tile by tile. The partition is stable, so the
// rows of one tile that belong to one top-digit bucket have consecutive positions p: the tile is
// staged in LDS in position order (bucket by bucket, found by a binary search of p in the buckets'
// starts) and written out as runs of consecutive addresses, from this XCD's L2 only.
constexpr uint32_t OBP_ITEMS = 8;
constexpr uint32_t OBP_TILE = BLOCK * OBP_ITEMS;
template <int W>
__global__ __launch_bounds__(BLOCK) void ob_partition(const void* col, const uint8_t* valid, int64_t voff,
                                                      uint32_t n, uint32_t rows_per_block, const uint32_t* pos_of_row,
                                                      const uint32_t* bucket_base, void* part, uint8_t* vpart) {
  __shared__ uint32_t s_base[RADIX];
  __shared__ uint32_t s_minp[RADIX], s_cnt[RADIX], s_off[RADIX];
  __shared__ uint32_t tmp[WAVES];
  __shared__ uint64_t s_val[OBP_TILE];
  __shared__ uint8_t s_bkt[OBP_TILE];
  __shared__ uint8_t s_vb[OBP_TILE];
  s_base[threadIdx.x] = bucket_base[threadIdx.x];
  s_minp[threadIdx.x] = 0xFFFFFFFFu;
  s_cnt[threadIdx.x] = 0u;
  __syncthreads();
  const uint32_t first = blockIdx.x * rows_per_block;
  const uint32_t last = min(n, first + rows_per_block);
  for (uint32_t t0 = first; t0 < last; t0 += OBP_TILE) {
    uint32_t p[OBP_ITEMS], bk[OBP_ITEMS], vb[OBP_ITEMS], bit[OBP_ITEMS];
    uint64_t v[OBP_ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < OBP_ITEMS; j++) {   // every load first (rows past the range read its last row)
      const uint32_t r = min(t0 + j * BLOCK + threadIdx.x, last - 1u);
      p[j] = pos_of_row[r];
      v[j] = load_raw<W>(col, r);
      vb[j] = load_valid_byte(valid, voff, r, bit[j]);
    }
#pragma unroll
    for (uint32_t j = 0; j < OBP_ITEMS; j++) {
      bk[j] = 0xFFFFFFFFu;
      if (t0 + j * BLOCK + threadIdx.x >= last || p[j] == 0xFFFFFFFFu) continue;
      uint32_t lo = 0, hi = RADIX;   // the last bucket whose start is <= p
      while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_base[mid] <= p[j]) lo = mid;
        else hi = mid;
      }
      bk[j] = lo;
      atomicMin(&s_minp[lo], p[j]);
      atomicAdd(&s_cnt[lo], 1u);
    }
    __syncthreads();
    uint32_t total;
    s_off[threadIdx.x] = block_excl_scan(s_cnt[threadIdx.x], tmp, total);
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < OBP_ITEMS; j++) {
      if (bk[j] == 0xFFFFFFFFu) continue;
      const uint32_t k = s_off[bk[j]] + (p[j] - s_minp[bk[j]]);
      if (k >= OBP_TILE) continue;   // cannot happen for a stable partition; keeps LDS writes in bounds
      s_val[k] = v[j];
      s_bkt[k] = uint8_t(bk[j]);
      s_vb[k] = uint8_t((vb[j] >> bit[j]) & 1u);
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < total; k += BLOCK) {
      const uint32_t b = s_bkt[k];
      const uint32_t dest = s_minp[b] + (k - s_off[b]);
      if constexpr (W == 8) static_cast<uint64_t*>(part)[dest] = s_val[k];
      else if constexpr (W == 4) static_cast<uint32_t*>(part)[dest] = uint32_t(s_val[k]);
      else if constexpr (W == 2) static_cast<uint16_t*>(part)[dest] = uint16_t(s_val[k]);
      else static_cast<uint8_t*>(part)[dest] = uint8_t(s_val[k]);
      if (vpart) vpart[dest] = s_vb[k];
    }
    __syncthreads();
    s_minp[threadIdx.x] = 0xFFFFFFFFu;
    s_cnt[threadIdx.x] = 0u;
    __syncthreads();
  }
}

// Counters of the gather: [x * 32] the next chunk of XCD x's eighth (each on its own 128-byte line).
constexpr uint32_t OB_CTR_STRIDE = 32;

template <int W>
__global__ __launch_bounds__(BLOCK) void ob_gather(const uint32_t* out_idx, uint32_t n, uint32_t vbase, uint32_t m,
                                                   const void* part, const uint8_t* vpart, const void* col,
                                                   const uint8_t* valid, int64_t voff, void* out,
                                                   unsigned long long* out_valid, uint32_t* ctr) {
  __shared__ uint32_t s_chunk;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t words = (n + 63u) / 64u;
  // Eighth x of the outputs: 64-row words [x * words / 8, (x + 1) * words / 8).
  const uint32_t home = xcd_id();
  for (uint32_t k = 0; k < uint32_t(NXCD); k++) {
    const uint32_t x = (home + k) & uint32_t(NXCD - 1);
    const uint32_t w0 = uint32_t(uint64_t(words) * x / NXCD), w1 = uint32_t(uint64_t(words) * (x + 1) / NXCD);
    const uint32_t chunks = (w1 - w0 + OB_CHUNK / 64 - 1) / (OB_CHUNK / 64);
    while (true) {
      if (threadIdx.x == 0) s_chunk = atomicAdd(&ctr[x * OB_CTR_STRIDE], 1u);
      __syncthreads();
      const uint32_t c = s_chunk;
      __syncthreads();
      if (c >= chunks) break;   // uniform: this eighth has no chunk left
      uint32_t idx[OB_GROUPS];
      bool in_val[OB_GROUPS];
#pragma unroll
      for (uint32_t g = 0; g < OB_GROUPS; g++) {
        const uint32_t word = w0 + c * (OB_CHUNK / 64) + uint32_t(w) * OB_GROUPS + g;
        const uint32_t i = min(word * 64u + uint32_t(lane), n - 1u);
        in_val[g] = i - vbase < m;
        // Positions index the m-row partition, rows the n-row column (clamped: reads stay in bounds).
        idx[g] = min(out_idx[i], (in_val[g] ? m : n) - 1u);
      }
      uint64_t v[OB_GROUPS];
      uint32_t vb[OB_GROUPS], bit[OB_GROUPS];
#pragma unroll
      for (uint32_t g = 0; g < OB_GROUPS; g++) {
        // A value-block output reads the partitioned column at its position, any other the column at
        // its row.
        const void* src = in_val[g] ? part : col;
        v[g] = load_raw<W>(src, idx[g]);
        if (in_val[g]) {
          vb[g] = vpart ? load_global(vpart + idx[g]) : 1u;
          bit[g] = 0u;
        } else {
          vb[g] = load_valid_byte(valid, voff, idx[g], bit[g]);
        }
      }
#pragma unroll
      for (uint32_t g = 0; g < OB_GROUPS; g++) {
        const uint32_t word = w0 + c * (OB_CHUNK / 64) + uint32_t(w) * OB_GROUPS + g;
        const uint32_t i = word * 64u + uint32_t(lane);
        const bool live = word < w1 && i < n;
        if (live) {
          if constexpr (W == 8) static_cast<uint64_t*>(out)[i] = v[g];
          else if constexpr (W == 4) static_cast<uint32_t*>(out)[i] = uint32_t(v[g]);
          else if constexpr (W == 2) static_cast<uint16_t*>(out)[i] = uint16_t(v[g]);
          else static_cast<uint8_t*>(out)[i] = uint8_t(v[g]);
        }
        if (out_valid) {
          const unsigned long long bits = __ballot(live && ((vb[g] >> bit[g]) & 1u));
          if (lane == 0 && word < w1) out_valid[word] = bits;
        }
      }
    }
  }
}

__global__ void ob_clear(uint32_t* ctr) {
  if (threadIdx.x < uint32_t(NXCD * OB_CTR_STRIDE)) ctr[threadIdx.x] = 0u;
}

template <int W>
void ob_move_column(const Array& c, bool nulls, const uint32_t* pos_of_row, const uint32_t* bucket_base,
                    const uint32_t* out_idx, uint32_t n, uint32_t vbase, uint32_t m, Array* out, uint32_t* ctr,
                    hipStream_t s) {
  DevBuf part = device_alloc(size_t(std::max<uint32_t>(m, 1)) * W);
  DevBuf vpart;
  if (nulls) vpart = device_alloc(std::max<uint32_t>(m, 1));
  retain(part);
  if (vpart) retain(vpart);
  const uint8_t* valid = nulls ? c.valid_bits() : nullptr;
  {
    ProfScope ps("order_by_partition");
    const uint32_t tiles = (n + OBP_TILE - 1) / OBP_TILE;
    const uint32_t blocks = std::max(1u, std::min(uint32_t(device().cu_count) * 4u, tiles));
    const uint32_t rpb = (tiles + blocks - 1) / blocks * OBP_TILE;   // whole tiles per workgroup
    hipLaunchKernelGGL((ob_partition<W>), dim3(blocks), dim3(BLOCK), 0, s, c.data(), valid, c.offset, n, rpb,
                       pos_of_row, bucket_base, part->ptr, nulls ? static_cast<uint8_t*>(vpart->ptr) : nullptr);
    AM_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(ob_clear, dim3(1), dim3(BLOCK), 0, s, ctr);
  AM_HIP(hipGetLastError());
  {
    ProfScope ps("order_by_gather");
    const uint32_t blocks = uint32_t(device().cu_count) * AM_OB_GATHER_WG;   // workgroups per CU
    hipLaunchKernelGGL((ob_gather<W>), dim3(blocks), dim3(BLOCK), 0, s, out_idx, n, vbase, m, part->ptr,
                       nulls ? static_cast<const uint8_t*>(vpart->ptr) : nullptr, c.data(), valid, c.offset,
                       out->values->ptr, nulls ? static_cast<unsigned long long*>(out->validity->ptr) : nullptr, ctr);
    AM_HIP(hipGetLastError());
  }
}

template <int ITEMS>
bool ob_sort(const Array& key, bool desc, int placement, uint32_t* out_idx, uint32_t* pos_of_row,
             uint32_t* m, uint32_t* bucket_base, hipStream_t s, unsigned long long* key_out,
             unsigned long long key_xor) {
  return run_sort<unsigned long long, 8, ITEMS>(key.data(), key.type, key.has_nulls() ? key.valid_bits() : nullptr,
                                                key.offset, uint32_t(key.length), desc, placement, 0, out_idx,
                                                s, pos_of_row, m, bucket_base, key_out, key_xor);
}

// The rest of a sorted integer key column whose value block the bucket sorts wrote: zeros outside the
// value block [vbase, vbase + m), and the validity bitmap (the value block valid, the rest null).
template <typename V>
__global__ void ob_key_rest(V* out, uint32_t n, uint32_t vbase, uint32_t m, unsigned long long* out_valid) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool in_val = i - vbase < m;
  if (i < n && !in_val) out[i] = V(0);
  if (out_valid) {
    const unsigned long long bits = __ballot(i < n && in_val);
    if ((threadIdx.x & 63) == 0 && i < n) out_valid[i / 64u] = bits;
  }
}

// A sorted integer column: the bucket sorts write its values beside the rows, so nothing is gathered. 6M
// full-range int32 259 us a call, 355 with an argsort and a gather of random rows; 50M int64 1.49 ms, where the
// argsort and gather of an ORDER BY take 2.0.
template <typename K, int ITEMS>
Array* sorted_ints_t(const Array& a, bool desc, int placement, Array* idx, hipStream_t s) {
  constexpr int W = int(sizeof(K));
  const uint32_t n = uint32_t(a.length);
  DevBuf values = device_alloc(size_t(n) * W);
  const bool is_signed = a.type == T_I64 || a.type == T_I32;
  const K flip = (is_signed ? K(1) << (8 * W - 1) : K(0)) ^ (desc ? ~K(0) : K(0));
  uint32_t m = 0;
  bool written = false;
  run_sort<K, W, ITEMS>(a.data(), a.type, a.has_nulls() ? a.valid_bits() : nullptr, a.offset, n, desc, placement, 0,
                        static_cast<uint32_t*>(idx->values->ptr), s, nullptr, &m, nullptr, values->ptr,
                        (unsigned long long)(flip), &written);
  if (!written) {   // the LSD passes sorted the rows only
    values.reset();
    return take(a, *idx);
  }
  Array* out = new_array(a.format, a.type, a.length);
  try {
    out->values = values;
    out->null_count = int64_t(n - m);
    if (m < n) {
      out->validity = device_alloc(size_t((n + 63) / 64) * 8);
      hipLaunchKernelGGL(ob_key_rest<K>, dim3((n + 255u) / 256u), dim3(256), 0, s, static_cast<K*>(values->ptr), n,
                         placement == 1 ? n - m : 0u, m, static_cast<unsigned long long*>(out->validity->ptr));
      AM_HIP(hipGetLastError());
    }
    sync();
  } catch (...) {
    release_array(out);
    throw;
  }
  return out;
}

template <typename K>
Array* sorted_ints_t(const Array& a, bool desc, int placement, Array* idx, hipStream_t s) {
  switch (sort_tune(a.length, int(sizeof(K))).items) {
    case 4: return sorted_ints_t<K, 4>(a, desc, placement, idx, s);
    case 8: return sorted_ints_t<K, 8>(a, desc, placement, idx, s);
    case 12: return sorted_ints_t<K, 12>(a, desc, placement, idx, s);
    case 20: return sorted_ints_t<K, 20>(a, desc, placement, idx, s);
    default: return sorted_ints_t<K, 16>(a, desc, placement, idx, s);
  }
}

}  // namespace

bool distinct_rows(const void* keys, int width, uint32_t n, DevBuf& rows, uint32_t& kept) {
  if (n > HYBRID_MAX_ROWS || capturing(stream())) return false;
  return width == 8 ? distinct_rows_t<unsigned long long>(keys, n, rows, kept, stream())
                    : distinct_rows_t<uint32_t>(keys, n, rows, kept, stream());
}

void argsort_device(const void* vals, int type, const uint8_t* validity, int64_t vbit_off, int64_t n,
                    bool descending, int null_placement, int float_order, uint32_t* out_idx, hipStream_t s) {
  if (n <= 0) return;
  if (n > int64_t(UINT32_MAX)) fail("arrays above 2^32 elements are not supported yet");
  int w = type_width(type);
  if (w == 0) fail("argsort: unsupported element type");
  int kb = w == 8 ? 8 : 4;
  if (n <= int64_t(RANK_MAX)) {
    auto rank = [&](auto k, auto wc) {
      run_rank<decltype(k), decltype(wc)::value>(vals, type, validity, vbit_off, uint32_t(n), descending, null_placement,
                                                 float_order, out_idx, s);
    };
    switch (w) {
      case 8: rank(0ull, std::integral_constant<int, 8>{}); break;
      case 4: rank(uint32_t(0), std::integral_constant<int, 4>{}); break;
      case 2: rank(uint32_t(0), std::integral_constant<int, 2>{}); break;
      default: rank(uint32_t(0), std::integral_constant<int, 1>{}); break;
    }
    return;
  }
  SortTune t = sort_tune(n, kb);
  switch (w) {
    case 8:
      dispatch_items<unsigned long long, 8>(t.items, vals, type, validity, vbit_off, uint32_t(n), descending,
                                            null_placement, float_order, out_idx, s);
      break;
    case 4:
      dispatch_items<uint32_t, 4>(t.items, vals, type, validity, vbit_off, uint32_t(n), descending, null_placement,
                                  float_order, out_idx, s);
      break;
    case 2:
      dispatch_items<uint32_t, 2>(t.items, vals, type, validity, vbit_off, uint32_t(n), descending, null_placement,
                                  float_order, out_idx, s);
      break;
    default:
      dispatch_items<uint32_t, 1>(t.items, vals, type, validity, vbit_off, uint32_t(n), descending, null_placement,
                                  float_order, out_idx, s);
      break;
  }
}

Array* argsort(const Array& a, bool descending, int null_placement, int float_order) {
  check_length(a.length);
  check_index_rows(a.length, "argsort");
  if (!type_is_primitive(a.type)) fail_unsupported("sort by " + a.format + " is not implemented");
  Array* out = new_array("I", T_U32, a.length);
  try {
    out->values = device_alloc(size_t(std::max<int64_t>(a.length, 1)) * 4);
    out->null_count = 0;
    if (a.length > 0) {
      argsort_device(a.data(), a.type, a.has_nulls() ? a.valid_bits() : nullptr, a.offset, a.length, descending,
                     null_placement, float_order, static_cast<uint32_t*>(out->values->ptr), stream());
    }
    sync();
  } catch (...) {
    release_array(out);
    throw;
  }
  return out;
}

Array* sorted_ints(const Array& a, bool descending, int null_placement) {
  check_length(a.length);
  check_index_rows(a.length, "argsort");
  if ((a.type != T_I64 && a.type != T_U64 && a.type != T_I32 && a.type != T_U32) || a.length < int64_t(hybrid_min(a.type)) ||
      a.length > int64_t(HYBRID_MAX_ROWS) || capturing(stream()))
    return nullptr;
  Array* idx = new_array("I", T_U32, a.length);
  struct Drop {
    Array* a;
    ~Drop() { release_array(a); }
  } drop{idx};
  try {
    idx->values = device_alloc(size_t(a.length) * 4);
    idx->null_count = 0;
    return a.width() == 8 ? sorted_ints_t<unsigned long long>(a, descending, null_placement, idx, stream())
                          : sorted_ints_t<uint32_t>(a, descending, null_placement, idx, stream());
  } catch (const OutOfMemory&) {   // the values beside the sort's scratch; an argsort and a take hold them apart
    return nullptr;
  }
}

bool order_by_columns(const Array& key, bool descending, int null_placement, const std::vector<const Array*>& cols,
                      std::vector<Array*>& out) {
  out.clear();
  const int64_t n = key.length;
  if (n < (int64_t(1) << 18) || n > int64_t(UINT32_MAX) || capturing(stream())) return false;
  // Only with an integer key among the columns, which comes out of the bucket sorts, and at most one column
  // beside it. In us, this way / an argsort and permute_columns: an int64 key alone, 270K rows 77/88, 1M 139/158,
  // 4M 223/291, 50M 1542/2079; with one float64, 270K 107/100, 1M 175/172, 4M 292/328, 50M 2301/2719; with two,
  // 270K 146/105, 1M 216/181, 4M 361/361; with three, 4M 436/365, 50M 3834/3347. (A float64 key's column had to be
  // moved by the two passes as well: alone, 270K 171/155, 4M 424/399, 50M 3957/3266.)
  if ((key.type != T_I64 && key.type != T_U64) || cols.size() > 2 || std::find(cols.begin(), cols.end(), &key) == cols.end())
    return false;
  for (const Array* c : cols)
    if (c->length != n || !type_is_primitive(c->type)) return false;
  check_index_rows(n, "argsort");
  hipStream_t s = stream();
  DevBuf idx = device_alloc(size_t(n) * 4), pos = device_alloc(size_t(n) * 4), ctr = device_alloc(NXCD * OB_CTR_STRIDE * 4);
  DevBuf bb = device_alloc(RADIX * 4);
  retain(idx);
  retain(pos);
  retain(ctr);
  retain(bb);
  auto* out_idx = static_cast<uint32_t*>(idx->ptr);
  auto* pos_of_row = static_cast<uint32_t*>(pos->ptr);
  auto* bbase = static_cast<uint32_t*>(bb->ptr);
  uint32_t m = 0;
  const int place = null_placement == 1 ? 1 : 0;
  // The key column comes out of the bucket sorts themselves: the mapped keys are a bijection of its values
  // (x ^ 2^63 for int64, then ~ when descending).
  DevBuf key_vals = device_alloc(size_t(n) * 8);
  const unsigned long long key_xor = (key.type == T_I64 ? 0x8000000000000000ull : 0ull) ^ (descending ? ~0ull : 0ull);
  auto* kout = static_cast<unsigned long long*>(key_vals->ptr);
  bool ok;
  switch (sort_tune(n, 8).items) {
    case 4: ok = ob_sort<4>(key, descending, place, out_idx, pos_of_row, &m, bbase, s, kout, key_xor); break;
    case 8: ok = ob_sort<8>(key, descending, place, out_idx, pos_of_row, &m, bbase, s, kout, key_xor); break;
    case 12: ok = ob_sort<12>(key, descending, place, out_idx, pos_of_row, &m, bbase, s, kout, key_xor); break;
    case 20: ok = ob_sort<20>(key, descending, place, out_idx, pos_of_row, &m, bbase, s, kout, key_xor); break;
    default: ok = ob_sort<16>(key, descending, place, out_idx, pos_of_row, &m, bbase, s, kout, key_xor); break;
  }
  if (!ok) return false;
  // The value block: [0, m) with nulls last, [n - m, n) with nulls first.
  const uint32_t vbase = place == 1 ? uint32_t(n) - m : 0u;
  try {
    for (const Array* c : cols) {
      Array* o = new_array(c->format, c->type, n);
      out.push_back(o);
      int64_t nulls = c->validity ? c->null_count : 0;
      if (nulls < 0) nulls = count_nulls(*c);
      o->null_count = nulls;   // a permutation keeps the null count
      if (nulls > 0) o->validity = device_alloc(size_t((n + 63) / 64) * 8);
      if (c == &key) {
        o->values = key_vals;
        hipLaunchKernelGGL(ob_key_rest<unsigned long long>, dim3((uint32_t(n) + 255u) / 256u), dim3(256), 0, s,
                           static_cast<unsigned long long*>(key_vals->ptr), uint32_t(n), vbase, m,
                           nulls > 0 ? static_cast<unsigned long long*>(o->validity->ptr) : nullptr);
        AM_HIP(hipGetLastError());
        continue;
      }
      o->values = device_alloc(size_t(n) * c->width());
      auto* ctrp = static_cast<uint32_t*>(ctr->ptr);
      switch (c->width()) {
        case 8: ob_move_column<8>(*c, nulls > 0, pos_of_row, bbase, out_idx, uint32_t(n), vbase, m, o, ctrp, s); break;
        case 4: ob_move_column<4>(*c, nulls > 0, pos_of_row, bbase, out_idx, uint32_t(n), vbase, m, o, ctrp, s); break;
        case 2: ob_move_column<2>(*c, nulls > 0, pos_of_row, bbase, out_idx, uint32_t(n), vbase, m, o, ctrp, s); break;
        default: ob_move_column<1>(*c, nulls > 0, pos_of_row, bbase, out_idx, uint32_t(n), vbase, m, o, ctrp, s); break;
      }
    }
    sync();
  } catch (...) {
    for (Array* a : out) release_array(a);
    out.clear();
    throw;
  }
  return true;
}

}  // namespace am
