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
// a workgroup owns 16 NB columns and all of K, which its eight waves take in turn, 128 at a time,
// each cutting its own rows of X into pieces in a patch of LDS that belongs to it; they meet once.
// No workspace.  What bounds it: the VALU, in cutting X (45 instructions for 4 values of a row, in
// every workgroup: more columns share them) and in converting the weights.
// One launch, us, K slices -> here: 5 rows of int8-64 at 9216 x 2304 13.0 -> 11.2, at 2304 x 9216 16.8 ->
// 15.3, at 2048 x 2304 10.8 -> 5.8; 10 rows of int4 at 4096 x 4096 16.3 -> 11.3 (0.8 TB/s of weights).
constexpr int kWhole = 8;                     // waves; the config's p0, with p1 blocks of 16 columns
constexpr int kWholeStep = 128;
constexpr int kWholeRow = kWholeStep * 2 + 16;  // bytes of a piece row in LDS
constexpr int kWholeMaxCols = 4;

typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t buffer_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ u32x4 load16(rsrc_t r, uint32_t at, uint32_t step_at) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, (int)step_at, 0));
}

template <int FMT, int T, int NB>
__global__ __launch_bounds__(kWhole * 64) void gemv_f32_whole_kernel(const F32Args a) {
  constexpr bool INT4 = FMT == TLHIP_FMT_INT4_GROUPED, ROW = FMT == TLHIP_FMT_INT8_ROW;
  constexpr int WV = INT4 ? 1 : 2;         // 16-byte loads of a step, lane and column block
  constexpr int XV = (16 * T / 3 + 1) / 2; // loads of X: two rows each
  extern __shared__ u32x4 lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int n0 = (int)blockIdx.x * (16 * NB);
  const int cols = min(16 * NB, a.n - n0);
  const int steps = a.k / kWholeStep;
  const uint32_t row_bytes = (uint32_t)a.row_chunks * 16u, scale_row_bytes = ROW ? 4u : (uint32_t)a.groups_per_row * 2u;
  const uint8_t* const packed = (const uint8_t*)a.packed + (int64_t)n0 * row_bytes;
  const uint8_t* const scales = (const uint8_t*)a.scales + (int64_t)n0 * scale_row_bytes;

  // Buffer loads: rows past M, columns past N and steps past K read zero and cost no traffic, so
  // that no load stands under a branch.  A lane's place in a step is fixed, the step is a scalar
  // offset (opaque, or the compiler keeps it in a vector register and loops over the lanes); past
  // the last step a buffer of no bytes at offset 0.
  struct Weights {
    u32x4 w[NB][WV];
    uint32_t s[NB][2];
  };
  auto scalar_step = [&](int st) {
    st = st < steps ? st : -1;
    asm("" : "+s"(st));
    return st;
  };
  auto load_w = [&](Weights& v, int step) {
    const int st = scalar_step(step);
    const uint32_t in = ~(uint32_t)(st >> 31), at = (uint32_t)st & in;
    const rsrc_t wb = buffer_of(packed, (uint32_t)cols * row_bytes & in), sb = buffer_of(scales, (uint32_t)cols * scale_row_bytes & in);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t row = (uint32_t)(16 * b + l16);
#pragma unroll
      for (int i = 0; i < WV; ++i) v.w[b][i] = load16(wb, row * row_bytes + (uint32_t)lg * 16u + (uint32_t)i * 64u, at * (WV * 64u));
      if constexpr (INT4) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 s = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(sb, (int)(row * scale_row_bytes), (int)(at * 8u), 0));
        v.s[b][0] = s.x;
        v.s[b][1] = s.y;
      } else if constexpr (!ROW) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v.s[b][h] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sb, (int)(row * scale_row_bytes), (int)(((2u * at + (uint32_t)h) >> a.group_shift) * 2u), 0);
      }
    }
  };
  struct Rows {
    u32x4 v[XV];
  };
  const int half = lane >> 5, unit = lane & 31;
  auto load_x = [&](Rows& r, int step) {
    const int st = scalar_step(step);
    const uint32_t in = ~(uint32_t)(st >> 31), at = (uint32_t)st * (kWholeStep * 4u) & in;
#pragma unroll
    for (int i = 0; i < XV; ++i)
      r.v[i] = load16(buffer_of(a.x + (int64_t)(2 * i) * a.k, (uint32_t)max(a.m - 2 * i, 0) * (uint32_t)a.k * 4u & in),
                      (uint32_t)half * (uint32_t)a.k * 4u + (uint32_t)unit * 16u, at);
  };
  char* const patch = (char*)lds + wave * (16 * T * kWholeRow);
  auto cut = [&](const Rows& r) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int row = 2 * i + half;
      uint32_t p[4][3];
      pieces_of(r.v[i].x, p[0]);
      pieces_of(r.v[i].y, p[1]);
      pieces_of(r.v[i].z, p[2]);
      pieces_of(r.v[i].w, p[3]);
      if (row < a.m) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const uint64_t v = (uint64_t)upper_halves(p[0][q], p[1][q]) | ((uint64_t)upper_halves(p[2][q], p[3][q]) << 32);
          *(uint64_t*)(patch + (row * 3 + q) * kWholeRow + unit * 8) = v;
        }
      }
    }
  };
  float4_t acc[NB][T];
  const char* arow[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    arow[t] = patch + min(t * 16 + l16, a.m * 3 - 1) * kWholeRow + lg * (INT4 ? 16 : 32);
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
  }
  auto multiply = [&](const Weights& v) __attribute__((always_inline)) {
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
      if constexpr (INT4) transpose4(words[0], words[1], words[2], words[3]);
      float4_t chain[T], sum[T];  // a step's own sum first: the long one takes a step at a time
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t wb[4];
        if constexpr (INT4) {
          weight_bf16<FMT>(words[i], wb);
        } else {
          weight_bf16<FMT>(words[2 * i], wb);
          weight_bf16<FMT>(words[2 * i + 1], wb + 2);
        }
        const bf16x8 wv = __builtin_bit_cast(bf16x8, (u32x4){wb[0], wb[1], wb[2], wb[3]});
        constexpr int GROUP = INT4 ? 1 : (ROW ? 4 : 2);  // products of one scale
        const bool first = i % GROUP == 0, last = i % GROUP == GROUP - 1;
#pragma unroll
        for (int t = 0; t < T; ++t)
          chain[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][t], wv, first ? (float4_t){0.f, 0.f, 0.f, 0.f} : chain[t], 0, 0, 0);
        if (last) {
          const float s = ROW ? 1.f : half_bits_to_float(INT4 ? ((i & 1) ? v.s[b][i >> 1] >> 16 : v.s[b][i >> 1] & 0xffffu) : v.s[b][i >> 1]);
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

  Weights w0, w1;
  Rows x0, x1;
  load_x(x0, wave);
  load_w(w0, wave);
  load_x(x1, wave + kWhole);
  load_w(w1, wave + kWhole);
  for (int st = wave; st < steps; st += 2 * kWhole) {
    cut(x0);
    load_x(x0, st + 2 * kWhole);
    multiply(w0);
    if (st + kWhole >= steps) break;
    load_w(w0, st + 2 * kWhole);
    cut(x1);
    load_x(x1, st + 3 * kWhole);
    multiply(w1);
    load_w(w1, st + 3 * kWhole);
  }

  lds_barrier();  // every wave has read its patch
  float* const sums = (float*)lds;  // [wave][tile][block][16 x 16]
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) sums[((wave * T + t) * NB + b) * 256 + (4 * lg + e) * 16 + l16] = acc[b][t][e];
  lds_barrier();
  for (int e = tid; e < a.m * (16 * NB); e += kWhole * 64) {
    const int row = e / (16 * NB), c = e % (16 * NB), col = n0 + c;
    if (col >= a.n) continue;
    float part[kWhole];
#pragma unroll
    for (int w = 0; w < kWhole; ++w) {
      float p[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int r = row * 3 + q;
        p[q] = sums[((w * T + (r >> 4)) * NB + (c >> 4)) * 256 + (r & 15) * 16 + (c & 15)];
      }
      part[w] = p[0] + (p[1] + p[2]);
    }
    const float v = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    const float factor = ROW ? ((const float*)a.scales)[col] * a.scale_mul : a.scale_mul;
    const int64_t at = (int64_t)row * a.n + col;
    store_out(a.y, a.y_dtype, at, apply_epilogue(a.epi, v * factor * a.alpha, col, at));
  }
}

template <int FMT, int T>
const void* whole_fn(int nb) {
  return nb == 1   ? (const void*)gemv_f32_whole_kernel<FMT, T, 1>
         : nb == 2 ? (const void*)gemv_f32_whole_kernel<FMT, T, 2>
                   : (const void*)gemv_f32_whole_kernel<FMT, T, (T < 3 ? 4 : 2)>;  // three tiles of pieces and four blocks: more registers than a lane has
}
template <int FMT>
const void* whole_fn(int tiles, int nb) {
  return tiles == 1 ? whole_fn<FMT, 1>(nb) : (tiles == 2 ? whole_fn<FMT, 2>(nb) : whole_fn<FMT, 3>(nb));
}
const void* whole_fn(int format, int tiles, int nb) {
  return format == TLHIP_FMT_INT4_GROUPED ? whole_fn<TLHIP_FMT_INT4_GROUPED>(tiles, nb)
         : format == TLHIP_FMT_INT8_ROW   ? whole_fn<TLHIP_FMT_INT8_ROW>(tiles, nb)
                                          : whole_fn<TLHIP_FMT_INT8_GROUPED>(tiles, nb);
}
size_t whole_lds(int tiles, int nb) { return std::max((size_t)kWhole * 16 * tiles * kWholeRow, (size_t)kWhole * tiles * nb * 1024); }

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
      "K slices (p0) must be 1..64 and no more than K holds blocks of 128 (int4) or 64 (int8), p1..p6 0; or p0 8 and p1 (blocks of 16 columns) 1, 2 or 4: K a multiple of 128 up to 16384, int4 in groups of 32; 4 blocks up to 10 rows",
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
    return c.p0 == kWhole && (c.p1 == 1 || c.p1 == 2 || c.p1 == 4) && p.k % kWholeStep == 0 && p.k <= 2048 * kWhole &&
                   (!int4 || p.group_size == 32) && (c.p1 < 4 || p.m <= 10) && !c.p2 && !c.p3 && !c.p4 && !c.p5 && !c.p6
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

// All of K in one workgroup at nb blocks of 16 columns: rounds of workgroups, as the VALU feels them.
// A second workgroup to a CU costs as much as the first (the VALU is what they share), three tiles of
// pieces fill its LDS alone.
static double whole_rounds(const Problem& p, int nb) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const double x = (double)((p.n + 16 * nb - 1) / (16 * nb)) / cus;
  return x <= 1.0 ? 1.0 : (p.m > 10 ? 1.15 * (double)(int64_t)(x + 0.999) : (x <= 2.0 ? 2.0 : 0.4 + 0.95 * x));
}
// ... what orders the widths of a problem, whatever its format: fitted at 1024..13838 x 768..12288, 3..16
// rows; the width it picks is 0.4 % behind the best one in the mean (992 problems).
static double width_us(const Problem& p, int nb) {
  const double m = (double)p.m, c = nb == 1 ? 0.75 + 0.125 * m : (nb == 2 ? 1.35 + 0.135 * m : 2.7 + 0.16 * m);
  return 2.9 + (double)p.k / 1000.0 * c * whole_rounds(p, nb);
}
// ... and the price of the launch beside that of K slices, in microseconds: fitted at 3182 launches of
// the one and 1716 of the other (200 matrices of 400..24576 x 512..12288, 3..16 rows, four formats).
// Per round the sums, 0.27 for every tile of pieces and block, and per 1000 of K the cutting of X and
// the weights of a block: 96 % of the launches take 0.82-1.13 times that.  K slices: the longest one's
// pieces and weights, and 0.010-0.017 for every row of every slice that the last arrival adds:
// 0.85-1.17 times that, int4 (8 % above its fit: its short slices scatter) 0.72-1.2.
static int format_index(const Problem& p) { return p.format == TLHIP_FMT_INT4_GROUPED ? 0 : (p.format == TLHIP_FMT_INT8_ROW ? 2 : 1); }
static double whole_us(const Problem& p, int nb) {
  static const double weights[3][3][3] = {  // tiles of pieces, format, 1 / 2 / 4 blocks
      {{0.61, 1.08, 2.05}, {0.70, 1.24, 2.55}, {0.54, 0.87, 1.84}},
      {{0.70, 1.25, 2.19}, {0.72, 1.37, 2.49}, {0.50, 0.98, 1.74}},
      {{0.92, 1.30, 0.0}, {0.91, 1.31, 0.0}, {0.76, 0.90, 0.0}}};
  const int tiles = tiles_of(p.m);
  const double m = (double)p.m;
  return 2.77 + whole_rounds(p, nb) * (0.29 + 0.27 * tiles * nb + (double)p.k / 1000.0 * (0.074 * m + 0.012 * m * nb + weights[tiles - 1][format_index(p)][nb / 2]));
}
static double slices_us(const Problem& p, int slices) {
  static const double base[3] = {10.7, 6.2, 6.5}, weights[3] = {5.22, 7.86, 4.98}, cut[3] = {0.471, 0.297, 0.324}, sum[3] = {0.010, 0.017, 0.014};
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256, f = format_index(p);
  const int64_t wgs = column_tiles(p) * slices, rounds = (wgs + cus - 1) / cus, slice = (blocks_of(p) + slices - 1) / slices * block_k(p);
  return base[f] + (double)(rounds * slice) / 1000.0 * (weights[f] + cut[f] * (double)p.m) + sum[f] * (double)(slices * p.m);
}

// All of K in one workgroup, at the cheapest number of columns, or false where K slices are ahead.
// Us, slices against here, over 24 matrices of 512..16246 x 768..12288 at 3..16 rows:
//   up to five rows at nearly every one (int8-64 9216 x 2304: 13.0 -> 11.2, 2304 x 9216: 16.8 -> 15.3;
//   int4 at 4096 x 4096 15.4 -> 8.6, at 12288 x 4096 28.8 -> 17.2);
//   more rows of int4 with K up to 4096 or enough columns for every CU (16 rows at 12288 x 4096 50.8 ->
//   33.8, at 4096 x 12288 39.7 -> 36.0; but 12 rows at 789 x 9984: 17.9 against 24.0);
//   more rows of int8 with K up to 4096 where one round of double blocks holds the columns (10 rows
//   at 2048 x 2304: 12.7 -> 7.1, at 7869 x 768 9.7 -> 6.1; but 16 rows at 9216 x 2304: 16.0 against 21.9).
// Within these, where the price says so too: of 1174 problems that both forms were timed at nine are
// more than 3 % behind the slices, by 10 % at most (16 rows of int8-128 at 4114 x 2816: 13.9 against
// 12.7); without it 5 rows of int8 at 512 x 16384 took 23.2 against 17.1, 16 rows of int4 at 10208 x
// 3712 32.4 against 26.8.
static bool whole_default(const Problem& p, tlhip_kernel_config_t* out) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  if (p.n > 16384) return false;
  if (p.m > 5) {
    if (p.format == TLHIP_FMT_INT4_GROUPED ? p.k > 4096 && p.n < (int64_t)cus * 16 : p.k > 4096 || p.n > (int64_t)cus * 32) return false;
  }
  bool found = false;
  double best = 0.0;
  for (int nb = 1; nb <= kWholeMaxCols; nb *= 2) {
    tlhip_kernel_config_t c;
    memset(&c, 0, sizeof c);
    c.variant = VARIANT_GEMV_F32;
    c.p0 = kWhole;
    c.p1 = nb;
    if (!gemv_f32_config_applicable(p, c, nullptr) || (found && width_us(p, nb) >= best)) continue;
    *out = c;
    best = width_us(p, nb);
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

bool gemv_f32_default(const Problem& p, tlhip_kernel_config_t* out) {
  tlhip_kernel_config_t whole;
  const bool found = slices_default(p, out);
  if (!whole_default(p, &whole) || (found && whole_us(p, whole.p1) >= slices_us(p, out->p0))) return found;
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
  const int rc = c.p1 ? launch_kernel(whole_fn(p.format, tiles, c.p1), dim3((unsigned)((p.n + 16 * c.p1 - 1) / (16 * c.p1))), dim3(kWhole * 64), args,
                                      whole_lds(tiles, c.p1), stream)
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
      for (int nb = 1; nb <= kWholeMaxCols && !rc; nb *= 2)
        if (nb < 4 || tiles < 3) rc = launch_kernel(whole_fn(format, tiles, nb), dim3(1), dim3(64), nullptr, 0, nullptr);
      if (rc) return rc;
    }
  return TLHIP_OK;
}

}  // namespace tlhip
