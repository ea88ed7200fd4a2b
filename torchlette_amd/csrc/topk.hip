// Top-k of one logits row on the device, so that the 256 000 logits the LM-head
// GEMV produces are never read back (the reference's sampling prefilter,
// src/backend/webgpu/topk-kernel.ts:1-30; readTopK / deviceTopK,
// src/backend/types.ts:632-634, 669-678).  Result: the k largest values in
// descending order, ties broken towards the smaller index (what a linear scan that
// keeps the first maximum gives), as (value, index) pairs.
//
// Every element becomes a 64-bit key, (order-preserving bits of the value) << 32 |
// (0xffffffff - index), so that "larger key" is exactly "larger value, then smaller
// index"; NaN maps below every number.  A workgroup reduces up to 4096 keys to their k
// largest; levels repeat (chunk -> k per workgroup) until one workgroup holds the answer.
//
// What bounds it: latency.  A row is 1 MB (0.2 us of HBM), the rest is dependent steps and
// launches.  Up to k = 256 a workgroup therefore selects instead of sorting
// (topk_select_kernel), and up to 8192 surviving keys the workgroup that arrives last does
// the last level in the same launch: 256 000 logits at k = 64 are 63 workgroups and one
// launch.  Above k = 256 a bitonic sort in LDS (topk_sort_kernel).
#include <type_traits>

#include "device_utils.h"

namespace tlhip {
namespace {

constexpr float kTopkNegInf = -3.4028234e38f;  // the reference's filler for missing entries

__device__ __forceinline__ uint64_t topk_key(float v, uint32_t index) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  uint32_t k = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  if (v != v) k = 0u;  // NaN: below everything
  return ((uint64_t)k << 32) | (uint64_t)(0xffffffffu - index);
}

__device__ __forceinline__ float topk_value(uint64_t key) {
  const uint32_t k = (uint32_t)(key >> 32);
  const uint32_t b = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __builtin_bit_cast(float, b);
}

constexpr int kTopkChunk = 4096;        // keys a workgroup reduces
constexpr int kSelectThreads = 512;
constexpr int kSelectMaxK = 256;
constexpr int kSelectFused = 8192;      // keys the last workgroup reduces in the same launch

__device__ __forceinline__ uint64_t max_key(uint64_t a, uint64_t b) { return a > b ? a : b; }

// A bound that at least `k` of the wave's 64 * R values reach: the first one tried that no more
// than k + slack reach (`enough`), else the largest.  One bit per step, a chain of 60 clocks.
template <int R>
__device__ __forceinline__ uint32_t bound_of(const uint32_t (&v)[R], const bool (&in)[R], int k, int slack, bool* enough) {
  uint32_t bound = 0;
  *enough = false;
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t trial = bound | (1u << bit);
    int count = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) count += __popcll(__ballot(in[r] && v[r] >= trial));
    if (count >= k) bound = trial;
    if ((uint32_t)(count - k) <= (uint32_t)slack) {
      *enough = true;
      break;
    }
  }
  return bound;
}

// The k largest of the keys the workgroup's threads hold (E each; 0 = none), in order, to
// emit(rank, key); ranks without a key get 0.  Returns with every thread past its LDS reads.
//   1. the maximum of every group of 4 threads (G = 128) or thread (G = 512);
//   2. a bound that k of the G maxima reach, hence at least k keys: for k = 64 of 4096
//      random keys about 100 do, at worst the whole contents of the groups that reach it (4096);
//   3. the keys from the bound on, collected in LDS (a wave counts its own by ballots and takes
//      its places with one atomic: an atomic a key was a chain of E round trips to LDS); the rank
//      of each is the number of larger ones, counted by as many threads as there are for a key.
// The slack of the bound: a quarter of k saves about eight of twenty steps, but the more of the G
// maxima pass the more keys each of them brings, and a rank's time grows with the keys.  Of 512, up
// to 224 (k = 256, us: no slack / a sixteenth / a quarter 10.6 / 10.2 / 11.0 of 4096 logits, 32.6 /
// 30.6 / 31.8 of 256 000; k = 160 7.8 / 7.3 / 7.0 and 21.8 / 20.9 / 20.0).
template <int G, int E, typename Emit>
__device__ __forceinline__ void select_keys(const uint64_t (&key)[E], int k, uint64_t* maxima, uint64_t* found, int* n_found, Emit emit) {
  constexpr int R = G / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  uint64_t best = key[0];
#pragma unroll
  for (int e = 1; e < E; ++e) best = max_key(best, key[e]);
  if (G == kSelectThreads / 4) {
    best = max_key(best, __shfl_xor(best, 1));
    best = max_key(best, __shfl_xor(best, 2));
    if ((tid & 3) == 0) maxima[tid >> 2] = best;
  } else {
    maxima[tid] = best;
  }
  if (tid == 0) *n_found = 0;
  __syncthreads();
  uint32_t hi[R], lo[R];
  bool in[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint64_t m = maxima[r * 64 + lane];
    hi[r] = (uint32_t)(m >> 32);
    lo[r] = (uint32_t)m;
    in[r] = true;
  }
  constexpr int kMostGroups = kTopkChunk / (E * kSelectThreads / G);  // whose whole contents `found` holds
  const int slack = max(0, min(max(min(k / 4, 224 - k), k / 16), kMostGroups - k));
  bool enough;
  const uint32_t bound_hi = bound_of<R>(hi, in, k, slack, &enough);
  uint32_t bound_lo = 0;
  if (!enough) {  // equal values around the bound: the index decides
    int larger = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      larger += __popcll(__ballot(hi[r] > bound_hi));
      in[r] = hi[r] == bound_hi;
    }
    bound_lo = bound_of<R>(lo, in, k - larger, slack, &enough);
  }
  const uint64_t bound = ((uint64_t)bound_hi << 32) | bound_lo;
  uint64_t hits[E];  // of the wave
  int mine = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    hits[e] = __ballot(key[e] != 0 && key[e] >= bound);
    mine += __popcll(hits[e]);
  }
  if (mine) {
    int at = 0;
    if (lane == 0) at = atomicAdd(n_found, mine);
    at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (hits[e]) {
        if (key[e] != 0 && key[e] >= bound)
          found[at + __builtin_amdgcn_mbcnt_hi((uint32_t)(hits[e] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hits[e], 0u))] = key[e];
        at += __popcll(hits[e]);
      }
  }
  __syncthreads();
  const int c = *n_found;
  auto rank_keys = [&](auto threads) {
    constexpr int T = decltype(threads)::value;  // of a key, neighbours in a wave
    for (int i0 = 0; i0 < c; i0 += kSelectThreads / T) {
      const int i = i0 + tid / T;
      const uint64_t own = found[min(i, c - 1)];
      int rank = 0;
#pragma unroll 8
      for (int j = tid % T; j < c; j += T) rank += found[j] > own ? 1 : 0;
      if (T > 1) rank += __builtin_amdgcn_update_dpp(0, rank, 0xB1, 0xf, 0xf, true);  // quad_perm [1,0,3,2]
      if (T > 2) rank += __builtin_amdgcn_update_dpp(0, rank, 0x4E, 0xf, 0xf, true);  // quad_perm [2,3,0,1]
      if (tid % T == 0 && i < c && rank < k) emit(rank, own);
    }
  };
  if (c <= kSelectThreads / 4) rank_keys(std::integral_constant<int, 4>());
  else if (c <= kSelectThreads / 2) rank_keys(std::integral_constant<int, 2>());
  else rank_keys(std::integral_constant<int, 1>());
  for (int i = c + tid; i < k; i += kSelectThreads) emit(i, (uint64_t)0);
  __syncthreads();
}

__device__ __forceinline__ void write_result(int i, uint64_t key, float* out_values, void* out_indices, int index_dtype) {
  const bool real = key != 0;
  out_values[i] = real ? topk_value(key) : kTopkNegInf;
  const int32_t idx = real ? (int32_t)(0xffffffffu - (uint32_t)key) : -1;
  if (index_dtype == TLHIP_F32) ((float*)out_indices)[i] = (float)idx;  // token ids as f32 (deviceTopK)
  else ((int32_t*)out_indices)[i] = idx;
}

// FROM_FLOAT: keys are made from `logits[offset + i]` with index i; else read from `keys_in`.
// The chunk's k keys go to keys_out[rank * gridDim.x + block].  With `counter` the workgroup that arrives
// last reduces all of them to the result (gridDim.x * k <= kSelectFused); a launch of one
// workgroup writes the result at once.
// 256 000 logits, k = 64, 8 rows behind each other: 35 us a row with three launches of sorted
// chunks of 1024 at first, 14 us with this launch, 9.6 us since a bound may let a few more keys pass,
// a wave takes its places with one atomic and up to four threads count a rank (k = 256: 33.6 -> 30.2):
// what is left is the launch, two loads of keys, the stores and the counter, each a round trip to
// memory behind the other.
template <bool FROM_FLOAT, int G>
__global__ __launch_bounds__(kSelectThreads) void topk_select_kernel(const float* __restrict__ logits, int64_t offset,
                                                                     const uint64_t* __restrict__ keys_in, int64_t count, int k,
                                                                     uint64_t* keys_out, int* counter,
                                                                     float* __restrict__ out_values,
                                                                     void* __restrict__ out_indices, int index_dtype) {
  __shared__ uint64_t maxima[G];
  __shared__ uint64_t found[kTopkChunk];
  __shared__ int n_found, arrived;
  constexpr int E = kTopkChunk / kSelectThreads;
  const int64_t base = (int64_t)blockIdx.x * kTopkChunk + threadIdx.x;
  uint64_t key[E];
#pragma unroll
  for (int e = 0; e < E; ++e) key[e] = 0;  // padding is below every key: the index part of a real key is at least 1
  if (count > 0) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int64_t at = base + e * kSelectThreads, clamped = at < count ? at : count - 1;
      const uint64_t v = FROM_FLOAT ? topk_key(logits[offset + clamped], (uint32_t)at) : keys_in[clamped];
      key[e] = at < count ? v : 0;
    }
  }
  if (gridDim.x == 1) {
    select_keys<G, E>(key, k, maxima, found, &n_found, [&](int i, uint64_t v) { write_result(i, v, out_values, out_indices, index_dtype); });
    return;
  }
  // Device-scope accesses only, as for the K slices of the matrix-core GEMV: coherent between
  // the L2 caches by themselves, without a fence that writes back and invalidates them.
  // Largest first over all chunks: the next selection's groups of neighbours then hold keys of
  // one rank.  (Chunk after chunk a few groups held every chunk's largest, so that its bound
  // let thousands of keys pass: 68 us a row.)
  uint64_t* mine = keys_out + blockIdx.x;
  select_keys<G, E>(key, k, maxima, found, &n_found,
                    [&](int i, uint64_t v) { __hip_atomic_store(mine + (size_t)i * gridDim.x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); });
  if (!counter) return;
  // select_keys ends with a barrier, but a wave's stores are complete only once they are acknowledged
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
  if (threadIdx.x == 0) arrived = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (arrived != (int)gridDim.x - 1) return;
  if (threadIdx.x == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
  const int total = (int)gridDim.x * k;
  auto last = [&](auto per_thread) {
    constexpr int E2 = decltype(per_thread)::value;
    uint64_t all[E2];
#pragma unroll
    for (int e = 0; e < E2; ++e) {
      const int at = e * kSelectThreads + (int)threadIdx.x;
      const uint64_t v = __hip_atomic_load(keys_out + (at < total ? at : total - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      all[e] = at < total ? v : 0;
    }
    select_keys<G, E2>(all, k, maxima, found, &n_found, [&](int i, uint64_t v) { write_result(i, v, out_values, out_indices, index_dtype); });
  };
  // as few keys a thread as hold them all
  if (total <= 2 * kSelectThreads) last(std::integral_constant<int, 2>());
  else if (total <= 8 * kSelectThreads) last(std::integral_constant<int, 8>());
  else last(std::integral_constant<int, kSelectFused / kSelectThreads>());
}

// k above kSelectMaxK: the chunk sorted in LDS, its first k keys to keys_out[block * k ..] or,
// with `final`, decoded to the result.
template <bool FROM_FLOAT>
__global__ __launch_bounds__(kTopkChunk / 4) void topk_sort_kernel(const float* __restrict__ logits, int64_t offset,
                                                        const uint64_t* __restrict__ keys_in, int64_t count, int k,
                                                        uint64_t* __restrict__ keys_out, int final,
                                                        float* __restrict__ out_values,
                                                        void* __restrict__ out_indices, int index_dtype) {
  __shared__ uint64_t keys[kTopkChunk];
  const int64_t base = (int64_t)blockIdx.x * kTopkChunk;
  constexpr int THREADS = kTopkChunk / 4;
#pragma unroll
  for (int i = threadIdx.x; i < kTopkChunk; i += THREADS) {
    const int64_t e = base + i;
    uint64_t key = 0;  // padding sorts last: the index part of a real key is at least 1
    if (e < count) key = FROM_FLOAT ? topk_key(logits[offset + e], (uint32_t)e) : keys_in[e];
    keys[i] = key;
  }
  __syncthreads();
  // bitonic sort, descending
  for (int size = 2; size <= kTopkChunk; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      // two compare-exchanges per thread, both pairs read before either is written
      const int t0 = threadIdx.x, t1 = threadIdx.x + THREADS;
      const int lo0 = 2 * t0 - (t0 & (stride - 1)), lo1 = 2 * t1 - (t1 & (stride - 1));
      const uint64_t a0 = keys[lo0], b0 = keys[lo0 + stride], a1 = keys[lo1], b1 = keys[lo1 + stride];
      const bool swap0 = (a0 < b0) == ((lo0 & size) == 0), swap1 = (a1 < b1) == ((lo1 & size) == 0);
      keys[lo0] = swap0 ? b0 : a0;
      keys[lo0 + stride] = swap0 ? a0 : b0;
      keys[lo1] = swap1 ? b1 : a1;
      keys[lo1 + stride] = swap1 ? a1 : b1;
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < k; i += THREADS) {
    const uint64_t key = keys[i];
    if (final) {
      write_result(i, key, out_values, out_indices, index_dtype);
    } else {
      keys_out[(int64_t)blockIdx.x * k + i] = key;
    }
  }
}

}  // namespace
}  // namespace tlhip

using namespace tlhip;

extern "C" int tlhip_topk(const float* logits, int64_t offset, int64_t length, int k, float* out_values,
                          void* out_indices, int index_dtype, tlhip_stream_t stream) {
  TLHIP_REQUIRE_INIT();
  if (k < 1 || k > 1024) return set_error(TLHIP_ERR_INVALID, "topk: k=%d must be 1..1024", k);
  if (index_dtype != TLHIP_F32 && index_dtype != TLHIP_I32)
    return set_error(TLHIP_ERR_INVALID, "topk: indices are TLHIP_I32 or TLHIP_F32");
  if (offset < 0 || length < 0) return set_error(TLHIP_ERR_INVALID, "topk: negative offset or length");
  if (length > (int64_t)0xfffffffe) return set_error(TLHIP_ERR_INVALID, "topk: length above 2^32-2");
  if (!out_values || !out_indices || (length > 0 && !logits)) return set_error(TLHIP_ERR_INVALID, "topk: null pointer");
  hipStream_t s = resolve_stream(stream);
  // level 0 reads the floats; later levels read the keys the level before wrote
  // into the stream's workspace, alternating between its two halves
  const bool select = k <= kSelectMaxK;
  float* ws = nullptr;
  int* counters = nullptr;
  const size_t half = kSplitWorkspaceFloats / 4;  // uint64 keys per half
  // the lengths a call takes, and from which it works through the workspace: one row of k
  // keys per 1024 logits (k <= 256; the levels below need a quarter of it) or per 4096
  const int64_t limit_chunk = select ? 1024 : kTopkChunk;
  const int64_t limit_blocks = (length + limit_chunk - 1) / limit_chunk;
  if (limit_blocks > 1) {
    if ((size_t)limit_blocks * k > half)
      return set_error(TLHIP_ERR_INVALID, "topk: length %lld with k=%d needs more workspace than the library holds",
                       (long long)length, k);
    const int rc = split_workspace(s, &ws, &counters);
    if (rc) return rc;
  }
  uint64_t* bufs[2] = {(uint64_t*)ws, (uint64_t*)ws + half};
  int64_t count = length;
  const uint64_t* keys_in = nullptr;
  for (int level = 0;; ++level) {
    int64_t blocks = (count + kTopkChunk - 1) / kTopkChunk;
    if (blocks < 1) blocks = 1;
    const int64_t survivors = blocks * k;
    uint64_t* keys_out = blocks == 1 ? nullptr : bufs[level & 1];
    const dim3 grid((unsigned)blocks);
    bool final = blocks == 1;
    if (select) {
      int* counter = !final && survivors <= kSelectFused ? counters : nullptr;
      final = final || counter;
      // groups of 4 threads are enough maxima up to k = 64
      auto kernel = level == 0 ? (k <= 64 ? topk_select_kernel<true, 128> : topk_select_kernel<true, 512>)
                               : (k <= 64 ? topk_select_kernel<false, 128> : topk_select_kernel<false, 512>);
      hipLaunchKernelGGL(kernel, grid, dim3(kSelectThreads), 0, s, logits, offset, keys_in, count, k, keys_out, counter,
                         out_values, out_indices, index_dtype);
    } else {
      auto kernel = level == 0 ? topk_sort_kernel<true> : topk_sort_kernel<false>;
      hipLaunchKernelGGL(kernel, grid, dim3(kTopkChunk / 4), 0, s, logits, offset, keys_in, count, k, keys_out, (int)final,
                         out_values, out_indices, index_dtype);
    }
    TLHIP_CHECK_HIP(hipGetLastError());
    if (final) break;
    keys_in = keys_out;
    count = survivors;
  }
  return TLHIP_OK;
}
