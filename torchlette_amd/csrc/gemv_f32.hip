// Decode GEMV / skinny GEMM on f32 activations, 2 to 16 rows, on the matrix cores without
// giving up their 24 bits.  Same contract and reference route as gemv.hip
// (src/backend/webgpu/matmul/gemv.ts:365-466).
//
// An f32 value is the sum of three bf16 values (its significand in three pieces of eight bits,
// cut and not rounded: no bit is lost above 2^-133), an int4 or int8 weight is a bf16 value, and
// the product of the two is exact in f32.  So row m becomes three rows of a bf16 product and its
// sum the sum of theirs: the arithmetic of the VALU kernel with the sums in another order.
// One launch, us, VALU kernel -> here, 5 rows: int8-64 2304 x 9216 33.6 -> 19.1, 9216 x 2304 34.4 ->
// 15.7, 1024 x 768 8.6 -> 7.3; int4-32 12288 x 4096 81.5 -> 28.7; 16 rows of int8-64 12288 x 4096
// 98.9 -> 38.6.
//
// What bounds it: the weights' bytes, and behind them the trip of the activations into LDS.
// The VALU kernel streams the weights once per four rows, or per two where four rows of f32 do
// not fit its LDS (K = 9216), and multiplies every weight by every row on the VALU.  Here a
// weight is read and converted once (1.5 VALU instructions for an int8) whatever M is.
//   * A workgroup of eight waves owns 128 columns of Y and a slice of K: 16 columns a wave.
//   * It cuts its slice of X into pieces in LDS, row 3 m + p holding piece p of row m: five
//     rows of X are one 16-row MFMA operand, ten are two, sixteen are three.
//   * A lane loads 16 bytes of its weight row at a time, the first loads ahead of the pieces.
//     int8: 64 k are two v_mfma_f32_16x16x32_bf16 and one group scale; int4: the words of four
//     lanes are exchanged so that one instruction multiplies 32 k of one group.
//   * K slices meet through device-scope accesses; the last workgroup adds them in order.
#include <algorithm>
#include <cstring>

#include "gemv_mfma_common.h"

namespace tlhip {
namespace {

constexpr int kCols = 128;       // columns of Y per workgroup
constexpr int kThreads = 512;
constexpr int kPatch = kCols + 4;
constexpr int kMaxSlices = 64;
constexpr size_t kLdsPerWorkgroup = 78 * 1024;  // two workgroups share a CU

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct F32Args {
  const u32x4* packed;
  const void* scales;
  const float* x;
  void* y;
  int m, n, k;
  int row_chunks;       // 16-byte chunks of a weight row
  int group_shift;      // log2(group size / 64) for int8, / 32 for int4
  int groups_per_row;
  int blocks;           // K in blocks of one 16-byte chunk on each of four lanes, rounded up
  int slices;
  int cols, block_cols;  // all of K in a workgroup: its columns, and those of a block
  float* workspace;     // slices > 1: [tile][slice][M][128]
  int* counters;        // one per tile, zero between launches
  float alpha, scale_mul;
  int y_dtype;
  DevEpilogue epi;
};

// x in three pieces, each in the upper half of a word
__device__ __forceinline__ void pieces_of(uint32_t b, uint32_t (&piece)[3]) {
  const uint32_t h1 = b & 0xffff0000u;
  const float r1 = as_float(b) - as_float(h1);
  const uint32_t h2 = __builtin_bit_cast(uint32_t, r1) & 0xffff0000u;
  const float r2 = r1 - as_float(h2);
  const bool finite = (b & 0x7f800000u) != 0x7f800000u;  // else inf - inf, and a NaN's payload may be cut to none
  piece[0] = finite ? h1 : ((b & 0x007fffffu) ? (b | 0x00400000u) : b);
  piece[1] = finite ? h2 : 0u;
  piece[2] = finite ? __builtin_bit_cast(uint32_t, r2) : 0u;
}

__device__ __forceinline__ uint32_t upper_halves(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }

template <int FMT>
__device__ __forceinline__ void weight_bf16(uint32_t w, uint32_t* out) {  // 4 (int8) or 8 (int4) weights
  constexpr int COUNT = FMT == TLHIP_FMT_INT4_GROUPED ? 8 : 4;
  uint32_t f[COUNT];
#pragma unroll
  for (int j = 0; j < COUNT; ++j) {
    const int q = FMT == TLHIP_FMT_INT4_GROUPED ? (int)(w << (28 - 4 * j)) >> 28 : (int)(int8_t)(w >> (8 * j));
    f[j] = __builtin_bit_cast(uint32_t, (float)q);
  }
#pragma unroll
  for (int j = 0; j < COUNT / 2; ++j) out[j] = upper_halves(f[2 * j], f[2 * j + 1]);
}

// T: tiles of 16 piece rows (3 M <= 16 T)
template <int FMT, int T>
__global__ __launch_bounds__(kThreads, 4) void gemv_f32_kernel(const F32Args a) {
  constexpr bool INT4 = FMT == TLHIP_FMT_INT4_GROUPED, ROW = FMT == TLHIP_FMT_INT8_ROW;
  constexpr int BK = INT4 ? 128 : 64;      // k of a block
  constexpr int STEPS = BK / 32;           // MFMAs of a block and tile
  constexpr int SCALES = ROW ? 0 : (INT4 ? 4 : 1);
  constexpr int U = 4;                     // blocks in flight ahead
  extern __shared__ u32x4 lds[];
  __shared__ int arrived;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, lg = lane >> 4;
  const int slice = (int)blockIdx.x % a.slices, tile = (int)blockIdx.x / a.slices;
  const int b0 = (int)((int64_t)a.blocks * slice / a.slices), b1 = (int)((int64_t)a.blocks * (slice + 1) / a.slices);
  const int nb = b1 - b0, k0 = b0 * BK, ks = nb * BK;
  const int stride = ks * 2 + 16;          // bytes of a piece row: 16 more, so that rows start in other banks
  const int n0 = tile * kCols;

  // ---- weights ----------------------------------------------------------------------------
  const int64_t wrow = min(n0 + wave * 16 + l16, a.n - 1);  // columns past N compute the last one, not stored
  const u32x4* const wp = a.packed + wrow * a.row_chunks;
  const uint16_t* const sp = (const uint16_t*)a.scales + wrow * a.groups_per_row;
  struct Batch {
    u32x4 w[U];
    uint16_t s[U][SCALES ? SCALES : 1];
  };
  auto load = [&](Batch& t, int b) {  // blocks b .. b + U - 1 of the slice; past its end the last one again
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int bb = b0 + min(b + u, nb - 1);
      // past K (a last block that is not whole) the last chunk again: the pieces there are 0
      t.w[u] = __builtin_nontemporal_load(wp + min(bb * 4 + lg, a.row_chunks - 1));
#pragma unroll
      for (int i = 0; i < SCALES; ++i) t.s[u][i] = sp[min((bb * (INT4 ? 4 : 1) + i) >> a.group_shift, a.groups_per_row - 1)];
    }
  };

  // ---- X: the first units requested, then the first weights, then cut into pieces -----------
  const int upr = ks / 4;  // units of 4 floats in a row
  const int units = a.m * upr;
  constexpr int XS = 4;
  u32x4 xr[XS];
  auto request = [&](int base) {
#pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int idx = min(base + tid + i * kThreads, units - 1), row = idx / upr, at = k0 + (idx - row * upr) * 4;
      xr[i] = *(const u32x4*)(a.x + (int64_t)row * a.k + min(at, a.k - 4));
    }
  };
  auto cut = [&](int base) {
#pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int idx = base + tid + i * kThreads;
      if (idx < units) {
        const int row = idx / upr, u = idx - row * upr;
        const bool in = k0 + u * 4 < a.k;  // K is a multiple of 4: a unit is whole or past the end
        uint32_t p[4][3];
        pieces_of(in ? xr[i].x : 0u, p[0]);
        pieces_of(in ? xr[i].y : 0u, p[1]);
        pieces_of(in ? xr[i].z : 0u, p[2]);
        pieces_of(in ? xr[i].w : 0u, p[3]);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const uint64_t v = (uint64_t)upper_halves(p[0][q], p[1][q]) | ((uint64_t)upper_halves(p[2][q], p[3][q]) << 32);
          *(uint64_t*)((char*)lds + (row * 3 + q) * stride + u * 8) = v;
        }
      }
    }
  };
  Batch cur, next;
  request(0);
  load(cur, 0);
  cut(0);
  for (int base = XS * kThreads; base < units; base += XS * kThreads) {
    request(base);
    cut(base);
  }
  lds_barrier();

  // ---- products ---------------------------------------------------------------------------
  float4_t acc[T], acc2[T];  // batches in turn: chains half as long, and so their rounding error smaller
  const char* arow[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    acc[t] = acc2[t] = (float4_t){0.f, 0.f, 0.f, 0.f};
    arow[t] = (const char*)lds + min(t * 16 + l16, a.m * 3 - 1) * stride + lg * (INT4 ? 16 : 32);
  }
  auto multiply = [&](const Batch& v, int b, float4_t (&acc)[T]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (b + u >= nb) break;
      uint32_t words[4] = {v.w[u].x, v.w[u].y, v.w[u].z, v.w[u].w};
      // int4: a lane holds a whole group of its row; afterwards word i is its eighth of group i
      if constexpr (INT4) transpose4(words[0], words[1], words[2], words[3]);
      float4_t chain[T];
#pragma unroll
      for (int t = 0; t < T; ++t) chain[t] = ROW ? acc[t] : (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < STEPS; ++i) {
        u32x4 wv;
        uint32_t wb[4];
        if constexpr (INT4) {
          weight_bf16<FMT>(words[i], wb);
        } else {
          weight_bf16<FMT>(words[2 * i], wb);
          weight_bf16<FMT>(words[2 * i + 1], wb + 2);
        }
        wv = (u32x4){wb[0], wb[1], wb[2], wb[3]};
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const u32x4 xv = *(const u32x4*)(arow[t] + (b + u) * (BK * 2) + i * (INT4 ? 64 : 16));
          chain[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xv), __builtin_bit_cast(bf16x8, wv), chain[t], 0, 0, 0);
        }
        if constexpr (INT4) {
          const float s = half_bits_to_float(v.s[u][i]);
#pragma unroll
          for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[t][e] = fmaf(s, chain[t][e], acc[t][e]);
            chain[t] = (float4_t){0.f, 0.f, 0.f, 0.f};
          }
        }
      }
      if constexpr (ROW) {
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t] = chain[t];
      } else if constexpr (!INT4) {
        const float s = half_bits_to_float(v.s[u][0]);
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][e] = fmaf(s, chain[t][e], acc[t][e]);
      }
    }
  };
  for (int b = 0; b < nb; b += 2 * U) {
    load(next, b + U);
    multiply(cur, b, acc);
    if (b + U >= nb) break;
    load(cur, b + 2 * U);
    multiply(next, b + U, acc2);
  }

  // ---- the pieces' sums together, slices, epilogue -------------------------------------------
  float* const patch = (float*)lds;
  lds_barrier();  // the pieces are read
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) patch[(t * 16 + lg * 4 + e) * kPatch + wave * 16 + l16] = acc[t][e] + acc2[t][e];
  lds_barrier();
  constexpr int MR = (16 * T / 3 + 3) / 4;  // rows of Y a thread finishes: four rows of 128 columns at a time
  const int c = tid & (kCols - 1), m_first = tid / kCols;
  float v[MR];
#pragma unroll
  for (int i = 0; i < MR; ++i) {
    const float* p = patch + min(m_first + 4 * i, a.m - 1) * 3 * kPatch + c;
    v[i] = p[0] + (p[kPatch] + p[2 * kPatch]);
  }
  if (a.slices > 1) {
    // Device-scope accesses only: coherent between the L2 caches by themselves, without a
    // fence that writes back and invalidates them.
    const int plane = a.m * kCols;
    float* const planes = a.workspace + (int64_t)tile * a.slices * plane;
#pragma unroll
    for (int i = 0; i < MR; ++i)
      if (m_first + 4 * i < a.m)
        __hip_atomic_store(planes + slice * plane + (m_first + 4 * i) * kCols + c, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the stores are acknowledged
    __syncthreads();
    if (tid == 0) arrived = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (arrived != a.slices - 1) return;
    if (tid == 0) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
#pragma unroll
    for (int i = 0; i < MR; ++i) {
      if (m_first + 4 * i >= a.m) break;
      const float* p = planes + (m_first + 4 * i) * kCols + c;
      float sum = 0.f;
      for (int s = 0; s < a.slices; s += 8) {
        float part[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) part[j] = __hip_atomic_load(p + min(s + j, a.slices - 1) * plane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int j = 0; j < 8; ++j) sum += s + j < a.slices ? part[j] : 0.f;
      }
      v[i] = sum;
    }
  }
  const int col = n0 + c;
  if (col >= a.n) return;
  const float factor = ROW ? ((const float*)a.scales)[col] * a.scale_mul : a.scale_mul;
#pragma unroll
  for (int i = 0; i < MR; ++i) v[i] = v[i] * factor * a.alpha;
  apply_epilogue_all<MR>(a.epi, v, col, [&](int i) { return m_first + 4 * i < a.m ? (int64_t)(m_first + 4 * i) * a.n + col : (int64_t)-1; });
#pragma unroll
  for (int i = 0; i < MR; ++i)
    if (m_first + 4 * i < a.m) store_out(a.y, a.y_dtype, (int64_t)(m_first + 4 * i) * a.n + col, v[i]);
}

// ---- all of K in one workgroup ------------------------------------------------------------------
// The same products where K slices across workgroups cost more than they give (the pieces of a
// slice behind a barrier, then planes of partial sums through memory and a counter: 4-5 us of 9-17):
// a workgroup owns up to 16 NB columns, an even share of them, and all of K.  Each of its eight waves has
// a range of K: it reads the range's group scales once, cuts its rows of X into pieces in a patch of LDS
// that belongs to it, 128 of K at a time, and meets the others once.  No workspace.  What bounds it: the
// VALU, in cutting X in every workgroup (more columns share it) and in converting the weights.  Values
// that are not finite are cut apart only where a wave finds one.
constexpr int kWhole = 8;                     // waves; the config's p0, with p1 blocks of 16 columns
constexpr int kWholeStep = 128;
constexpr int kWholeRow = kWholeStep * 2 + 16;  // bytes of a piece row in LDS
constexpr int kWholeMaxCols = 4;
constexpr int kWholeMaxSteps = 16;              // of a wave
constexpr int kWholeScaleRow = kWholeMaxSteps * 8 + 16;  // bytes of a column's scales in LDS

typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t buffer_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ u32x4 load16(rsrc_t r, uint32_t at, uint32_t step_at) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, (int)step_at, 0));
}

// x in three pieces, x finite (pieces_of without its selects): each in the upper half of a word
__device__ __forceinline__ void finite_pieces_of(uint32_t b, uint32_t (&piece)[3]) {
  const float r1 = as_float(b) - as_float(b & 0xffff0000u);
  const uint32_t r1b = __builtin_bit_cast(uint32_t, r1);
  piece[0] = b;
  piece[1] = r1b;
  piece[2] = __builtin_bit_cast(uint32_t, r1 - as_float(r1b & 0xffff0000u));
}

// T: tiles of 16 piece rows; XV: loads of X, two rows each.  WIDE: a group's scales are whole words (int4,
// int8 in groups of 64)
template <int FMT, int T, int XV, int NB, bool WIDE>
__global__ __launch_bounds__(kWhole * 64) void gemv_f32_whole_kernel(const F32Args a) {
  constexpr bool INT4 = FMT == TLHIP_FMT_INT4_GROUPED, ROW = FMT == TLHIP_FMT_INT8_ROW;
  constexpr int WV = INT4 ? 1 : 2;         // 16-byte loads of a step, lane and column block
  constexpr int SB = INT4 ? 8 : 4;         // bytes of a step and column in the patch of scales
  extern __shared__ u32x4 lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4, m = a.m;
  const int n0 = (int)blockIdx.x * a.cols, have = min(a.cols, a.n - n0), block_cols = a.block_cols;
  const int steps = a.k / kWholeStep;
  const uint32_t row_bytes = (uint32_t)a.row_chunks * 16u, scale_row_bytes = ROW ? 4u : (uint32_t)a.groups_per_row * 2u;

  // A lane's place in a step is fixed, the step is a scalar offset.
  const rsrc_t wb = buffer_of((const uint8_t*)a.packed + (int64_t)n0 * row_bytes, (uint32_t)have * row_bytes);
  const rsrc_t sb = buffer_of((const uint8_t*)a.scales + (int64_t)n0 * scale_row_bytes, (uint32_t)have * scale_row_bytes);
  const rsrc_t xb = buffer_of(a.x, (uint32_t)m * (uint32_t)a.k * 4u);
  uint32_t w_at[NB], s_at[NB], x_at[XV];
#pragma unroll
  for (int b = 0; b < NB; ++b) {  // columns past the block's or the matrix's: the last one again, not stored
    const uint32_t col = (uint32_t)min(b * block_cols + min(l16, block_cols - 1), have - 1);
    w_at[b] = col * row_bytes + (uint32_t)lg * 16u;
    s_at[b] = col * scale_row_bytes;
  }
  const int half = lane >> 5, unit = lane & 31;
#pragma unroll
  for (int i = 0; i < XV; ++i) x_at[i] = (uint32_t)min(2 * i + half, m - 1) * (uint32_t)a.k * 4u + (uint32_t)unit * 16u;
  struct Step {
    u32x4 x[XV];
    u32x4 w[NB][WV];
  };
  auto load_x = [&](Step& v, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XV; ++i) v.x[i] = load16(xb, x_at[i], (uint32_t)st * (kWholeStep * 4u));
  };
  auto load_w = [&](Step& v, int b, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WV; ++i) v.w[b][i] = load16(wb, w_at[b] + (uint32_t)i * 64u, (uint32_t)st * (WV * 64u));
  };
  auto load = [&](Step& v, int st) __attribute__((always_inline)) {
    load_x(v, st);
#pragma unroll
    for (int b = 0; b < NB; ++b) load_w(v, b, st);
  };

  // ---- the wave's range of steps and its scales (workgroups of an XCD start at different ranges: all on
  // the same lines of X at a time is 10-15 % slower)
  const int range = (wave + ((int)blockIdx.x >> 3)) & (kWhole - 1);
  // (the first ranges are the longer ones: waves four apart share a SIMD, two long ones there are a step more)
  const int each = steps / kWhole, more = steps % kWhole;
  const int st0 = range * each + min(range, more), left = each + (range < more ? 1 : 0);
  constexpr int PER = WIDE ? 64 / SB : 4;  // steps of a load: a quarter of them on each of a column's four lanes
  constexpr int SL = kWholeMaxSteps / PER;
  char* const patch = (char*)lds + wave * (16 * T * kWholeRow);
  char* const scale_patch = (char*)lds + kWhole * (16 * T * kWholeRow) + wave * (NB * 16 * kWholeScaleRow);
  struct Scales {
    u32x4 v[NB];
  };
  auto load_scales = [&](Scales& v, int from) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if constexpr (WIDE) v.v[b] = load16(sb, s_at[b] + (uint32_t)lg * 16u, (uint32_t)(st0 + from) * SB);
      else v.v[b].x = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sb, (int)(s_at[b] + ((uint32_t)(2 * (st0 + from + lg)) >> a.group_shift) * 2u), 0, 0);
    }
  };
  auto lay_scales = [&](const Scales& v, int from) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      char* const to = scale_patch + (b * 16 + l16) * kWholeScaleRow;
      if constexpr (WIDE) *(u32x4*)(to + from * SB + lg * 16) = v.v[b];
      else *(uint32_t*)(to + (from + lg) * 4) = v.v[b].x | v.v[b].x << 16;
    }
  };

  auto cut = [&](const Step& v) __attribute__((always_inline)) {
    bool odd = false;  // anything not finite
#pragma unroll
    for (int i = 0; i < XV; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) odd = odd | __builtin_amdgcn_classf(as_float(v.x[i][e]), 0x207);
    const bool any = __builtin_amdgcn_ballot_w64(odd) != 0;
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int row = 2 * i + half;
      uint32_t p[4][3];
#pragma unroll
      for (int e = 0; e < 4; ++e) finite_pieces_of(v.x[i][e], p[e]);
      if (any)
#pragma unroll
        for (int e = 0; e < 4; ++e) pieces_of(v.x[i][e], p[e]);
      if (row < m) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const uint64_t w = (uint64_t)upper_halves(p[0][q], p[1][q]) | ((uint64_t)upper_halves(p[2][q], p[3][q]) << 32);
          *(uint64_t*)(patch + (row * 3 + q) * kWholeRow + unit * 8) = w;
        }
      }
    }
  };
  float4_t acc[NB][T];
  const char* arow[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    arow[t] = patch + min(t * 16 + l16, m * 3 - 1) * kWholeRow + lg * (INT4 ? 16 : 32);
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
  }
  // `next`: the step whose loads take the registers as they become free, or -1
  auto consume = [&](Step& v, int i_step, int next) __attribute__((always_inline)) {
    cut(v);
    if (next >= 0) load_x(v, next);
    bf16x8 xa[4][T];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < T; ++t) xa[i][t] = __builtin_bit_cast(bf16x8, *(const u32x4*)(arow[t] + (INT4 ? 64 * i : 128 * (i >> 1) + 16 * (i & 1))));
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      uint32_t words[4 * WV];
#pragma unroll
      for (int i = 0; i < WV; ++i) {
        words[4 * i + 0] = v.w[b][i].x;
        words[4 * i + 1] = v.w[b][i].y;
        words[4 * i + 2] = v.w[b][i].z;
        words[4 * i + 3] = v.w[b][i].w;
      }
      if (next >= 0) load_w(v, b, next);
      if constexpr (INT4) transpose4(words[0], words[1], words[2], words[3]);
      uint32_t sc2[2] = {0u, 0u};  // int4: four group scales; int8: one per half step
      if constexpr (!ROW) {
        const char* const from = scale_patch + (b * 16 + l16) * kWholeScaleRow + i_step * SB;
        sc2[0] = *(const uint32_t*)from;
        if constexpr (INT4) sc2[1] = *(const uint32_t*)(from + 4);
      }
      float4_t chain[T], sum[T];  // a step's own sum first: the long one takes a step at a time
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t wq[4];
        if constexpr (INT4) {
          weight_bf16<FMT>(words[i], wq);
        } else {
          weight_bf16<FMT>(words[2 * i], wq);
          weight_bf16<FMT>(words[2 * i + 1], wq + 2);
        }
        const bf16x8 wv = __builtin_bit_cast(bf16x8, (u32x4){wq[0], wq[1], wq[2], wq[3]});
        constexpr int GROUP = INT4 ? 1 : (ROW ? 4 : 2);  // products of one scale
        const bool first = i % GROUP == 0, last = i % GROUP == GROUP - 1;
#pragma unroll
        for (int t = 0; t < T; ++t)
          chain[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][t], wv, first ? (float4_t){0.f, 0.f, 0.f, 0.f} : chain[t], 0, 0, 0);
        if (last) {
          const float s = ROW ? 1.f : half_bits_to_float(INT4 ? ((i & 1) ? sc2[i >> 1] >> 16 : sc2[i >> 1] & 0xffffu) : (i >> 1 ? sc2[0] >> 16 : sc2[0] & 0xffffu));
#pragma unroll
          for (int t = 0; t < T; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[t][e] = ROW ? chain[t][e] : (i < GROUP ? s * chain[t][e] : fmaf(s, chain[t][e], sum[t][e]));
        }
      }
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b][t][e] += sum[t][e];
    }
  };

  // ---- one step in flight, or two where a step is short; none past the end, every load unconditional (a
  // wait at a join would count it as not issued), the scales ahead of them
  if (left > 0) {
    Scales sv[SL];
    if constexpr (!ROW) {
#pragma unroll
      for (int q = 0; q < SL; ++q)
        if (q == 0 || q * PER < left) load_scales(sv[q], q * PER);
    }
    auto lay_all = [&]() __attribute__((always_inline)) {
      if constexpr (!ROW) {
#pragma unroll
        for (int q = 0; q < SL; ++q)
          if (q == 0 || q * PER < left) lay_scales(sv[q], q * PER);
      }
    };
    Step v0;
    load(v0, st0);
    int i = 0;
    if constexpr (NB * T > 2) {
      lay_all();
      for (; i + 1 < left; ++i) consume(v0, i, st0 + i + 1);
      consume(v0, i, -1);
    } else if (left == 1) {
      lay_all();
      consume(v0, 0, -1);
    } else {
      Step v1;
      load(v1, st0 + 1);
      lay_all();
      for (; i + 3 < left; i += 2) {
        consume(v0, i, -1);
        load(v0, st0 + i + 2);
        consume(v1, i + 1, -1);
        load(v1, st0 + i + 3);
      }
      if (left & 1) {
        consume(v0, i, -1);
        load(v0, st0 + i + 2);
        consume(v1, i + 1, -1);
        consume(v0, i + 2, -1);
      } else {
        consume(v0, i, -1);
        consume(v1, i + 1, -1);
      }
    }
  }

  lds_barrier();  // every wave has read its patch
  float* const sums = (float*)lds;  // [range][tile][block][16 x 16]
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) sums[((range * T + t) * NB + b) * 256 + (4 * lg + e) * 16 + l16] = acc[b][t][e];
  lds_barrier();
  for (int e = tid; e < m * have; e += kWhole * 64) {
    const int row = e / have, oc = e - row * have, col = n0 + oc, ob = oc / block_cols, c = oc - ob * block_cols;
    float part[kWhole];
#pragma unroll
    for (int w = 0; w < kWhole; ++w) {
      float p[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int r = row * 3 + q;
        p[q] = sums[((w * T + (r >> 4)) * NB + ob) * 256 + (r & 15) * 16 + c];
      }
      part[w] = p[0] + (p[1] + p[2]);
    }
    const float v = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    const float factor = ROW ? ((const float*)a.scales)[col] * a.scale_mul : a.scale_mul;
    const int64_t at = (int64_t)row * a.n + col;
    store_out(a.y, a.y_dtype, at, apply_epilogue(a.epi, v * factor * a.alpha, col, at));
  }
}

template <int FMT, int T, int XV, bool WIDE>
const void* whole_fn_nb(int nb) {
  if (nb == 1) return (const void*)gemv_f32_whole_kernel<FMT, T, XV, 1, WIDE>;
  if (nb == 2) return (const void*)gemv_f32_whole_kernel<FMT, T, XV, 2, WIDE>;
  if (nb == 3) return (const void*)gemv_f32_whole_kernel<FMT, T, XV, 3, WIDE>;
  if constexpr (T < 3)  // three tiles of pieces and four blocks: more registers than a lane has
    if (nb == 4) return (const void*)gemv_f32_whole_kernel<FMT, T, XV, 4, WIDE>;
  return nullptr;
}
template <int FMT, bool WIDE>
const void* whole_fn_rows(int64_t m, int nb) {
  if (m <= 4) return whole_fn_nb<FMT, 1, 2, WIDE>(nb);
  if (m == 5) return whole_fn_nb<FMT, 1, 3, WIDE>(nb);
  if (m <= 8) return whole_fn_nb<FMT, 2, 4, WIDE>(nb);
  if (m <= 10) return whole_fn_nb<FMT, 2, 5, WIDE>(nb);
  if (m <= 12) return whole_fn_nb<FMT, 3, 6, WIDE>(nb);
  return whole_fn_nb<FMT, 3, 8, WIDE>(nb);
}
const void* whole_fn(const Problem& p, int nb) {
  if (p.format == TLHIP_FMT_INT4_GROUPED) return whole_fn_rows<TLHIP_FMT_INT4_GROUPED, true>(p.m, nb);
  if (p.format == TLHIP_FMT_INT8_ROW) return whole_fn_rows<TLHIP_FMT_INT8_ROW, false>(p.m, nb);
  return p.group_size == 64 ? whole_fn_rows<TLHIP_FMT_INT8_GROUPED, true>(p.m, nb) : whole_fn_rows<TLHIP_FMT_INT8_GROUPED, false>(p.m, nb);
}
size_t whole_lds(const Problem& p, int nb) {
  const size_t tiles = (size_t)((3 * p.m + 15) / 16), scales = p.format == TLHIP_FMT_INT8_ROW ? 0 : (size_t)nb * 16 * kWholeScaleRow;
  return std::max(kWhole * (16 * tiles * kWholeRow + scales), (size_t)kWhole * tiles * nb * 1024);
}
// Columns of a workgroup (p2; 0: 16 p1), its blocks, and the columns of a block.
int whole_cols(const tlhip_kernel_config_t& c) { return c.p2 ? c.p2 : 16 * c.p1; }
int whole_blocks(const tlhip_kernel_config_t& c) { return (whole_cols(c) + 15) / 16; }
int whole_block_cols(const tlhip_kernel_config_t& c) { return (whole_cols(c) + whole_blocks(c) - 1) / whole_blocks(c); }

template <int FMT>
const void* fn_of(int tiles) {
  return tiles == 1 ? (const void*)gemv_f32_kernel<FMT, 1> : (tiles == 2 ? (const void*)gemv_f32_kernel<FMT, 2> : (const void*)gemv_f32_kernel<FMT, 3>);
}
const void* fn_of(int format, int tiles) {
  return format == TLHIP_FMT_INT4_GROUPED ? fn_of<TLHIP_FMT_INT4_GROUPED>(tiles)
         : format == TLHIP_FMT_INT8_ROW   ? fn_of<TLHIP_FMT_INT8_ROW>(tiles)
                                          : fn_of<TLHIP_FMT_INT8_GROUPED>(tiles);
}
int tiles_of(int64_t m) { return (int)((3 * m + 15) / 16); }

int block_k(const Problem& p) { return p.format == TLHIP_FMT_INT4_GROUPED ? 128 : 64; }
int64_t blocks_of(const Problem& p) { return (p.k + block_k(p) - 1) / block_k(p); }
int64_t column_tiles(const Problem& p) { return (p.n + kCols - 1) / kCols; }
size_t lds_of(const Problem& p, int slices) {
  const size_t ks = (size_t)((blocks_of(p) + slices - 1) / slices) * block_k(p);
  return std::max((size_t)p.m * 3 * (ks * 2 + 16), (size_t)tiles_of(p.m) * 16 * kPatch * sizeof(float));
}

}  // namespace

bool gemv_f32_config_applicable(const Problem& p, const tlhip_kernel_config_t& c, const char** why) {
  static const char* reasons[] = {
      "not the gemv_f32 variant",
      "built for f32 activations, 1..16 rows, without a prologue",
      "K must be a multiple of 32 (int4) or 16 (int8), groups at least 32 (int4) or 64 (int8)",
      "K slices (p0) must be 1..64 and no more than K holds blocks of 128 (int4) or 64 (int8), p1..p6 0; or p0 8 and p1 (blocks of 16 columns) 1, 2 or 4, or p2 (columns) up to 64: K a multiple of 128 up to 16384, int4 in groups of 32; 4 blocks up to 10 rows",
      "the pieces of a K slice do not fit LDS: more slices",
      "the slices' partial sums do not fit the library's workspace",
  };
  auto fail = [&](int i) {
    if (why) *why = reasons[i];
    return false;
  };
  if (c.variant != VARIANT_GEMV_F32) return fail(0);
  if (p.x_dtype != TLHIP_F32 || p.m < 1 || p.m > 16 || p.pro.kind != TLHIP_PRO_NONE) return fail(1);
  const bool int4 = p.format == TLHIP_FMT_INT4_GROUPED;
  if (p.k <= 0 || p.k % (int4 ? 32 : 16) != 0 || (p.format != TLHIP_FMT_INT8_ROW && p.group_size < (int4 ? 32 : 64))) return fail(2);
  if (c.p1 != 0) {  // chains of at most 2048 in a wave: see gemv_f32_default
    return c.p0 == kWhole && (c.p1 == 1 || c.p1 == 2 || c.p1 == 4) && p.k % kWholeStep == 0 && p.k <= kWholeStep * kWholeMaxSteps * kWhole &&
                   (!int4 || p.group_size == 32) && c.p2 >= 0 && c.p2 <= 16 * kWholeMaxCols && whole_fn(p, whole_blocks(c)) &&
                   whole_block_cols(c) * (whole_blocks(c) - 1) < whole_cols(c) && !c.p3 && !c.p4 && !c.p5 && !c.p6
               ? true
               : fail(3);
  }
  if (c.p0 < 1 || c.p0 > kMaxSlices || c.p0 > blocks_of(p) || c.p1 || c.p2 || c.p3 || c.p4 || c.p5 || c.p6) return fail(3);
  if (lds_of(p, c.p0) > kLdsPerWorkgroup) return fail(4);
  const ScratchNeed need = gemv_f32_scratch(p, c);
  if (need.counters > scratch_counters(p) || need.floats > scratch_tile_floats(p)) return fail(5);
  return true;
}

ScratchNeed gemv_f32_scratch(const Problem& p, const tlhip_kernel_config_t& c) {
  if (c.p0 <= 1 || c.p1) return ScratchNeed{0, 0};
  return ScratchNeed{(size_t)column_tiles(p) * (size_t)c.p0 * (size_t)p.m * kCols, column_tiles(p)};
}

// What orders the widths of all of K in one workgroup, `cols` columns of nb blocks: per round of workgroups the
// sums and the barriers, and per 1000 of K the cutting of X, the weights and the products.  Fitted at 2600
// launches (34 matrices of 1024..15340 x 1024..12288, 2..16 rows, four formats, warm): 7 % off (rms); the width it picks
// is 0.5 % behind the best one in the mean, 5 % at worst.  On cold weights it is 5-11 % too low: what the launch takes
// beside K slices is whole_beside_us.
static double packed_mb(const Problem& p) { return (double)p.n * (double)p.k * (p.format == TLHIP_FMT_INT4_GROUPED ? 0.5 : 1.0) / 1e6; }
static int format_index(const Problem& p) { return p.format == TLHIP_FMT_INT4_GROUPED ? 0 : (p.format == TLHIP_FMT_INT8_ROW ? 2 : 1); }
static double whole_us(const Problem& p, int cols) {
  static const double weights[3][3][4] = {  // tiles of pieces, format, blocks
      {{0.404, 0.728, 1.090, 1.388}, {0.314, 0.662, 1.083, 1.376}, {0.162, 0.548, 0.951, 1.217}},
      {{0.463, 0.842, 1.146, 1.671}, {0.406, 0.922, 1.044, 1.419}, {0.240, 0.550, 0.843, 1.159}},
      {{0.519, 0.863, 1.315, 0.0}, {0.471, 0.816, 1.163, 0.0}, {0.362, 0.660, 0.915, 0.0}}};
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256, tiles = tiles_of(p.m), nb = (cols + 15) / 16;
  const int64_t wgs = (p.n + cols - 1) / cols, rounds = (wgs + cus - 1) / cus, steps = p.k / kWholeStep;
  const double k = (double)((steps + kWhole - 1) / kWhole * kWhole * kWholeStep) / 1000.0;
  return 2.02 + (double)rounds * (0.88 + 0.186 * tiles * nb + k * (0.09 * (double)p.m + 0.116 * cols / 16.0 + weights[tiles - 1][format_index(p)][nb - 1]));
}
// Behind each other and on cold weights, the picked width and K slices across workgroups: the weights' way from memory,
// per round the sums and, per 1000 of K, the cutting of X and the blocks' products; of slices the longest one's pieces
// and weights and, for every row of every slice, what the last arrival adds.  Fitted at 2287 launches of either (106
// matrices of 768..16384 x 1024..16384, 3..16 rows, three formats): 2-7 % and 4-9 % rms; the cheaper one is 0.05-0.3 % behind the faster
// in the mean and more than 3 % at 1-4 % of the problems (2-7 % by warm prices: five rows of int8 per row at
// 5120 x 12288 21.4 us in slices, 30.1 so).  Most of those K are multiples of 1024, whose rows crowd onto a part of the memory's channels:
// at others slices of int4 take 0.86 of it for an odd number of steps (16 rows at 1712 x 8064 16.9 us, 20.9 so), and up to
// eight rows of int8 per row in one workgroup 0.83-0.93 (five at 4384 x 7424 15.0 us in slices, 12.3 so).
static double whole_beside_us(const Problem& p, int cols) {
  struct Cost {
    double launch, mb, round, sums, k, k_rows, k_blocks;
  };
  static const Cost costs[3][3] = {  // format, tiles of pieces
      {{0.0, 0.073, 2.511, 0.415, 0.0, 0.080, 0.446}, {2.925, 0.084, 0.0, 0.343, 0.084, 0.057, 0.617}, {1.159, 0.091, 0.883, 0.985, 0.335, 0.079, 0.458}},
      {{0.0, 0.063, 2.817, 0.348, 0.0, 0.071, 0.374}, {3.447, 0.079, 0.0, 0.043, 0.0, 0.045, 0.644}, {1.246, 0.068, 1.205, 0.701, 0.587, 0.070, 0.392}},
      {{2.604, 0.059, 0.0, 0.348, 0.0, 0.063, 0.407}, {3.179, 0.081, 0.0, 0.080, 0.0, 0.045, 0.587}, {1.157, 0.080, 0.861, 0.687, 0.672, 0.068, 0.293}}};
  const Cost& t = costs[format_index(p)][tiles_of(p.m) - 1];
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256, nb = (cols + 15) / 16;
  const int64_t wgs = (p.n + cols - 1) / cols, steps = p.k / kWholeStep;
  const double rounds = (double)((wgs + cus - 1) / cus), k = (double)((steps + kWhole - 1) / kWhole * kWhole * kWholeStep) / 1000.0;
  const double spread = p.format == TLHIP_FMT_INT8_ROW && p.m <= 8 && p.k % 1024 ? 0.93 : 1.0;
  return spread * (t.launch + t.mb * packed_mb(p) + rounds * (t.round + t.sums * nb + k * (t.k + t.k_rows * (double)p.m + t.k_blocks * nb)));
}
static double slices_us(const Problem& p, int slices) {
  struct Cost {
    double launch, mb, weights, cut, slice, sum, out;
  };
  static const Cost costs[3] = {{10.40, 0.103, 6.152, 0.256, 0.022, 0.010, 0.064}, {5.73, 0.096, 6.809, 0.113, 0.097, 0.012, 0.057}, {5.06, 0.091, 3.680, 0.113, 0.093, 0.010, 0.065}};
  const Cost& t = costs[format_index(p)];
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const int64_t wgs = column_tiles(p) * slices, rounds = (wgs + cus - 1) / cus, slice = (blocks_of(p) + slices - 1) / slices * block_k(p);
  const double rows = (double)(slices * p.m);
  const double spread = p.format == TLHIP_FMT_INT4_GROUPED && p.k % 256 ? 0.87 : 1.0;
  return spread * (t.launch + t.mb * packed_mb(p) + (double)(rounds * slice) / 1000.0 * (t.weights + t.cut * (double)p.m) + t.slice * slices + t.sum * rows +
                   t.out * (double)column_tiles(p) * rows / 100.0);
}

// All of K in one workgroup, at the cheapest number of columns (whole blocks, or an even share that
// leaves no round half empty: 9216 columns in 256 workgroups of 36, not 576 of 16), or false where K slices stay.
// Us, slices / here, cold weights: ten rows of int8-64 at 3072 x 8192 19.9 / 16.3; 16 rows of int4 at 12288 x 4096 45 / 20.
// Three exceptions, where the routes of longer standing are kept though this form has caught up with them:
// more than 16384 columns; fewer than 1024 of a K beyond 8192 of int8 (5 rows at 512 x 16384 17.3 / 15.3; of int4 at 768 x 9728
// 18.9 / 12.7, which goes by the price); and int4 with more than ten rows, 8192 columns and K an odd number of steps (10208 x
// 3712, 16 rows 27 / 18; 12748 x 4224, 14 rows 26.5 / 30).
static bool whole_default(const Problem& p, tlhip_kernel_config_t* out, double* us) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  if (p.n > 16384 || (p.n < 1024 && p.k > 8192 && p.format != TLHIP_FMT_INT4_GROUPED)) return false;
  if (p.format == TLHIP_FMT_INT4_GROUPED && p.m > 10 && p.n > 8192 && p.k / kWholeStep % 2) return false;
  memset(out, 0, sizeof *out);
  out->variant = VARIANT_GEMV_F32;
  out->p0 = kWhole;
  bool found = false;
  for (int nb = 1; nb <= kWholeMaxCols; ++nb) {
    const int64_t rounds = (p.n + (int64_t)cus * 16 * nb - 1) / ((int64_t)cus * 16 * nb);
    const int even = (int)((p.n + rounds * cus - 1) / (rounds * cus)), cols = even > 16 * (nb - 1) && nb > 1 ? even : 16 * nb;
    tlhip_kernel_config_t c = *out;
    c.p2 = cols == 16 * nb && nb != 3 ? 0 : cols;
    c.p1 = c.p2 ? (cols < 48 ? 1 : 2) : nb;  // beside p2 only the mark of the form
    if (!gemv_f32_config_applicable(p, c, nullptr) || (found && whole_us(p, cols) >= *us)) continue;
    *out = c;
    *us = whole_us(p, cols);
    found = true;
  }
  return found;
}

static bool slices_default(const Problem& p, tlhip_kernel_config_t* out) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  memset(out, 0, sizeof *out);
  out->variant = VARIANT_GEMV_F32;
  const int64_t tiles = std::max<int64_t>(1, column_tiles(p));
  // a workgroup to a CU (2304 x 9216, int8-64, 5 rows: 27.6 / 19.1 / 24.3 us in 4 / 8 / 16
  // slices of 18 tiles; 9216 x 2304: 21.0 / 15.7 / 18.0 us in 1 / 2 / 4 of 72), each slice at
  // least two blocks, and none longer than 2048: there the sums' rounding error (rel-L2
  // 1.0-1.2e-7) would pass the VALU kernel's (1.0-1.4e-7; 2.0e-7 at one chain of 4096)
  int64_t s = std::max<int64_t>(std::min<int64_t>({cus / tiles, blocks_of(p) / 2, 16}), (p.k + 2047) / 2048);
  for (s = std::max<int64_t>(s, 1); s <= kMaxSlices; ++s) {
    out->p0 = (int)s;
    if (gemv_f32_config_applicable(p, *out, nullptr)) return true;
  }
  return false;
}

bool gemv_f32_whole_default(const Problem& p, tlhip_kernel_config_t* out) {
  double us = 0.0;
  return whole_default(p, out, &us);
}

bool gemv_f32_default(const Problem& p, tlhip_kernel_config_t* out) {
  tlhip_kernel_config_t whole;
  double us = 0.0;
  const bool found = slices_default(p, out);
  if (!whole_default(p, &whole, &us) || (found && whole_beside_us(p, whole_cols(whole)) >= slices_us(p, out->p0))) return found;
  *out = whole;
  return true;
}

int launch_gemv_f32(const Problem& p, const tlhip_kernel_config_t& c, hipStream_t stream) {
  const char* why = nullptr;
  if (!gemv_f32_config_applicable(p, c, &why))
    return set_error(TLHIP_ERR_INVALID, "gemv_f32: config not applicable: %s", why ? why : "?");
  if (p.n == 0 || p.m == 0) return TLHIP_OK;
  const bool int4 = p.format == TLHIP_FMT_INT4_GROUPED, row = p.format == TLHIP_FMT_INT8_ROW;
  F32Args a;
  memset(&a, 0, sizeof a);
  a.packed = (const u32x4*)p.packed;
  a.scales = p.scales;
  a.x = (const float*)p.x;
  a.y = p.y;
  a.m = (int)p.m;
  a.n = (int)p.n;
  a.k = (int)p.k;
  a.row_chunks = (int)(int4 ? p.k / 32 : p.k / 16);
  a.group_shift = row ? 0 : __builtin_ctz((unsigned)(p.group_size / (int4 ? 32 : 64)));
  a.groups_per_row = row ? 0 : (int)(p.k / p.group_size);
  a.blocks = (int)blocks_of(p);
  a.slices = c.p1 ? 1 : c.p0;
  if (a.slices > 1) {
    const int rc = problem_scratch(p, stream, &a.workspace, &a.counters);
    if (rc) return rc;
  }
  a.alpha = p.alpha;
  a.scale_mul = p.format == TLHIP_FMT_INT8_GROUPED ? 1.0f / 127.0f : 1.0f;
  a.y_dtype = p.y_dtype;
  a.epi = p.epi;
  void* args[] = {(void*)&a};
  const int tiles = tiles_of(p.m);
  if (c.p1) {
    a.cols = whole_cols(c);
    a.block_cols = whole_block_cols(c);
  }
  const int rc = c.p1 ? launch_kernel(whole_fn(p, whole_blocks(c)), dim3((unsigned)((p.n + a.cols - 1) / a.cols)), dim3(kWhole * 64), args, whole_lds(p, whole_blocks(c)), stream)
                      : launch_kernel(fn_of(p.format, tiles), dim3((unsigned)(column_tiles(p) * a.slices)), dim3(kThreads), args,
                                      lds_of(p, a.slices), stream);
  if (rc) return rc;
  count_gemv_dispatch();
  return TLHIP_OK;
}

// Every instance launch_gemv_f32 can reach, in prepare mode (see launch_kernel).
int prepare_gemv_f32_kernels() {
  for (int format : {TLHIP_FMT_INT4_GROUPED, TLHIP_FMT_INT8_GROUPED, TLHIP_FMT_INT8_ROW})
    for (int tiles = 1; tiles <= 3; ++tiles) {
      int rc = launch_kernel(fn_of(format, tiles), dim3(1), dim3(64), nullptr, 0, nullptr);
      if (rc) return rc;
    }
  Problem p;
  memset(&p, 0, sizeof p);
  for (p.format = 0; p.format < 3; ++p.format)
    for (p.group_size = 64; p.group_size <= 128; p.group_size *= 2)
      for (p.m = 1; p.m <= 16; ++p.m)
        for (int nb = 1; nb <= kWholeMaxCols; ++nb)
          if (const void* fn = whole_fn(p, nb)) {
            const int rc = launch_kernel(fn, dim3(1), dim3(64), nullptr, 0, nullptr);
            if (rc) return rc;
          }
  return TLHIP_OK;
}

}  // namespace tlhip
