// Gather (Arrow `take`) for CDNA4: out[i] = values[indices[i]].
//
// Semantics follow the reference (Sources/ArrowMetal/Kernels/Take.swift:41-80,
// KernelSource.swift:209-227): a null index gives a null output, a null source element gives a null,
// and an index outside [0, length) makes the call fail with "take: index out of range (array length
// N)" once the kernel has run. Each wave handles 64 consecutive outputs, so the output validity is one
// 64-bit ballot per wave, written as one word; nulls are counted per workgroup, without atomics.
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
__global__ __launch_bounds__(256) void take_kernel(const V* __restrict__ vals, const uint8_t* __restrict__ vvalid,
                                                   int64_t voff, int64_t len, const I* __restrict__ idx,
                                                   const uint8_t* __restrict__ ivalid, int64_t ioff, int64_t n,
                                                   V* __restrict__ out, unsigned long long* __restrict__ out_valid,
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
  else if (ov)
    hipLaunchKernelGGL((take_kernel<V, I, true>), dim3(blocks), dim3(256), 0, s, vals, vv, a.offset, a.length, idx, iv,
                       ix.offset, ix.length, o, ov, block_nulls, st);
  else
    hipLaunchKernelGGL((take_kernel<V, I, false>), dim3(blocks), dim3(256), 0, s, vals, vv, a.offset, a.length, idx, iv,
                       ix.offset, ix.length, o, ov, block_nulls, st);
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

}  // namespace

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
      ProfScope ps("take");
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
