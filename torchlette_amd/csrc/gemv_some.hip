// 2 to 5 f32 activation rows over packed weights on the VALU, every row in one launch.  Same contract and
// reference route as gemv.hip (src/backend/webgpu/matmul/gemv.ts:365-466).
//
// What bounds it: its own instructions, a conversion a weight and a product a row.  Hence:
//   * A lane keeps eight k of every row in registers, for all columns of its workgroup: nothing is cut into
//     pieces, and LDS carries neither activations nor operands.
//   * A workgroup owns an even share of the columns and all of K, each of its eight waves a range of K: no
//     workspace.  The lanes of a wave (16, 32 or 64) cover the range, so that a short K leaves none idle: the
//     others work on the next columns.
//   * The group scales of the columns come once, into LDS, beside the first weights.
//   * The lanes' sums of eight columns are folded by swaps of half and quarter waves, which leave two values of
//     each pair in one register, and the rest through LDS, where a lane adds up an output.
// Us, launches of four, two and one row on the kernel in gemv_kernel.h -> here: 5 rows of int8-64 at 2304 x 2048 10.6 ->
// 5.4, at 1024 x 4096 10.5 -> 5.0; 3 rows of int4 at 4096 x 4096 14.3 -> 6.8, 4 rows at 12288 x 4096 21.0 -> 15.1;
// 2 rows of int8-64 at 4096 x 4096 7.0 -> 6.0 (2.8 TB/s of weights).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "device_utils.h"
#include "gemv_some.h"

namespace tlhip {
namespace {

constexpr int kSomeWaves = 8;
constexpr int kSomeCols = 8;        // columns of a lane between two folds
constexpr int kSomeParts = 4 * kSomeWaves;           // sums of an output that LDS holds
constexpr int kSomePartsRow = kSomeParts + 4;        // ... in other banks than its neighbour's
constexpr int kSomeMaxK = 8192, kSomeMaxCols = 64;

struct SomeArgs {
  const uint8_t* packed;
  const uint8_t* scales;
  const float* x;
  void* y;
  int n, k, cols;
  int row_bytes;     // packed bytes of a weight row
  int groups;        // per row
  int group_shift;   // log2(group size)
  float factor;      // alpha, times what the integers were multiplied by
  int y_dtype;
  DevEpilogue epi;
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ rsrc_t buffer_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ float signed_byte(uint32_t w, int i) { return (float)(int)(int8_t)(w >> (8 * i)); }
// Eight weights in k order; int4: sixteen times each (the nibble on top of its byte).
template <bool INT4>
__device__ __forceinline__ void weights_of(const uint32_t (&w)[2], float (&q)[8]) {
  if constexpr (INT4) {
    const uint32_t even = (w[0] << 4) & 0xf0f0f0f0u, odd = w[0] & 0xf0f0f0f0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      q[2 * i] = signed_byte(even, i);
      q[2 * i + 1] = signed_byte(odd, i);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = signed_byte(w[i >> 2], i & 3);
  }
}
// The sum of two halves (quarters) of a wave: a's in the lower (even) ones, b's in the others.
__device__ __forceinline__ float fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
// M rows; LPC lanes of a column; CH pieces of 8 LPC of K in a wave's range.
template <int FMT, int M, int LPC, int CH>
__global__ __launch_bounds__(kSomeWaves * 64) void gemv_some_kernel(const SomeArgs a) {
  constexpr bool INT4 = FMT == TLHIP_FMT_INT4_GROUPED, ROW = FMT == TLHIP_FMT_INT8_ROW;
  constexpr int LG = 64 / LPC, NV = kSomeCols * M;  // columns side by side; sums of a lane
  extern __shared__ u32x4 lds[];
  uint16_t* const scales = (uint16_t*)lds;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = lane % LPC, sub = lane / LPC;
  const int n0 = (int)blockIdx.x * a.cols, have = min(a.cols, a.n - n0), k = a.k, groups = a.groups, shift = a.group_shift;
  const rsrc_t wb = buffer_of(a.packed + (int64_t)n0 * a.row_bytes, (uint32_t)have * (uint32_t)a.row_bytes);
  const rsrc_t xb = buffer_of(a.x, (uint32_t)(M * k) * 4u);

  // ---- the lane's part of K, its activations (none past K), the first weights
  float x[CH][M][8];
  uint32_t w_at[CH];
  int group[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int k0 = (wave * CH + c) * (8 * LPC) + l * 8, in = min(k0, k - 8);
    w_at[c] = (uint32_t)in >> (INT4 ? 1 : 0);
    group[c] = ROW ? 0 : in >> shift;
#pragma unroll
    for (int r = 0; r < M; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, (r * k + in + 4 * h) * 4, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[c][r][4 * h + e] = k0 < k ? as_float(v[e]) : 0.f;
      }
  }
  struct Weights {
    uint32_t w[kSomeCols][CH][2];
  };
  auto load = [&](Weights& v, int g) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kSomeCols; ++j) {
      const uint32_t col = (uint32_t)min((g * kSomeCols + j) * LG + sub, have - 1) * (uint32_t)a.row_bytes;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        if constexpr (INT4) {
          v.w[j][c][0] = __builtin_amdgcn_raw_buffer_load_b32(wb, (int)(col + w_at[c]), 0, 0);
          v.w[j][c][1] = 0;
        } else {
          const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(wb, (int)(col + w_at[c]), 0, 0));
          v.w[j][c][0] = t.x;
          v.w[j][c][1] = t.y;
        }
      }
    }
  };
  // ---- the columns' scales: adjacent in memory
  if constexpr (!ROW) {
    const rsrc_t sb = buffer_of(a.scales + (int64_t)n0 * groups * 2, (uint32_t)(have * groups) * 2u);
    for (int i = tid; i * 2 < have * groups; i += kSomeWaves * 64)
      ((uint32_t*)lds)[i] = __builtin_amdgcn_raw_buffer_load_b32(sb, i * 4, 0, 0);
  }
  const int parts_at = ROW ? 0 : (a.cols * groups * 2 + 15) / 16 * 16;
  float* const parts = (float*)((char*)lds + parts_at);

  const int count = (have + kSomeCols * LG - 1) / (kSomeCols * LG);
  auto consume = [&](const Weights& v, int g, auto narrow) __attribute__((always_inline)) {
    constexpr bool NARROW = decltype(narrow)::value;
    float acc[NV];
#pragma unroll
    for (int j = 0; j < kSomeCols; ++j) {
      const int col = min((g * kSomeCols + j) * LG + sub, have - 1);
      if constexpr (NARROW) {
#pragma unroll
        for (int r = 0; r < M; ++r) acc[j * M + r] = 0.f;
        if (j > 0 && j * LG >= have) continue;
      }
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        float q[8];
        weights_of<INT4>(v.w[j][c], q);
        const float s = ROW ? 1.f : half_bits_to_float(scales[col * groups + group[c]]);
#pragma unroll
        for (int r = 0; r < M; ++r) {
          float part = q[0] * x[c][r][0];
#pragma unroll
          for (int e = 1; e < 8; ++e) part = fmaf(q[e], x[c][r][e], part);
          float& to = acc[j * M + r];
          if constexpr (ROW) to = c == 0 ? part : to + part;
          else to = c == 0 ? s * part : fmaf(s, part, to);
        }
      }
    }
    // value i of acc: after each fold two of them share a register, by a bit of the lane
    constexpr int N1 = LPC == 64 ? NV / 2 : NV, N2 = LPC >= 32 ? N1 / 2 : N1;
    float* const to = parts + (size_t)(g * LG + sub) * NV * kSomePartsRow + wave * 4 + (lane & 3);
    if constexpr (LPC == 64)
#pragma unroll
      for (int i = 0; i < N1; ++i) acc[i] = fold32(acc[2 * i], acc[2 * i + 1]);
    if constexpr (LPC >= 32)
#pragma unroll
      for (int i = 0; i < N2; ++i) acc[i] = fold16(acc[2 * i], acc[2 * i + 1]);
    const int quarter = LPC >= 32 ? (lane >> 4) & 1 : 0, half = LPC == 64 ? lane >> 5 : 0;
#pragma unroll
    for (int i = 0; i < N2; ++i) {
      const float v = dpp_add<0x124>(dpp_add<0x128>(acc[i]));  // row_ror 8, row_ror 4: lanes four apart
      const int at = LPC == 64 ? 2 * (2 * i + quarter) + half : (LPC == 32 ? 2 * i + quarter : i);
      if ((lane & 15) < 4) to[at * kSomePartsRow] = v;
    }
  };
  Weights v;
  load(v, 0);
  if constexpr (!ROW) lds_barrier();
  // Up to six of the eight columns of a lane: a branch for each (1024 columns of K = 1024, 5 rows: 5.9 -> 4.6 us);
  // more: none, which keeps the columns' chains side by side (4096 x 4096, 3 rows: 6.5 us, 9.5 with branches).
  if (have <= 6 * LG) {
    consume(v, 0, std::true_type());
  } else {
    for (int g = 0; g + 1 < count; ++g) {
      Weights next;
      load(next, g + 1);
      consume(v, g, std::false_type());
      v = next;
    }
    consume(v, count - 1, std::false_type());
  }
  lds_barrier();

  for (int o = tid; o < count * LG * NV; o += kSomeWaves * 64) {
    const int i = o % NV, gs = o / NV, row = i % M, c = (gs / LG * kSomeCols + i / M) * LG + gs % LG;
    if (c >= have) continue;
    const float4_t* p = (const float4_t*)(parts + (size_t)o * kSomePartsRow);
    float part[kSomeWaves];
#pragma unroll
    for (int w = 0; w < kSomeWaves; ++w) part[w] = (p[w][0] + p[w][1]) + (p[w][2] + p[w][3]);
    const float sum = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    const int col = n0 + c;
    const float factor = ROW ? ((const float*)a.scales)[col] * a.factor : a.factor;
    const int64_t at = (int64_t)row * a.n + col;
    store_out(a.y, a.y_dtype, at, apply_epilogue(a.epi, sum * factor, col, at));
  }
}

template <int FMT, int M>
const void* some_fn(int lanes, int pieces) {
  if (pieces == 2) return lanes == 64 ? (const void*)gemv_some_kernel<FMT, M, 64, 2> : nullptr;
  return lanes == 16 ? (const void*)gemv_some_kernel<FMT, M, 16, 1> : (lanes == 32 ? (const void*)gemv_some_kernel<FMT, M, 32, 1> : (const void*)gemv_some_kernel<FMT, M, 64, 1>);
}
template <int FMT>
const void* some_fn(int64_t m, int lanes, int pieces) {
  return m == 2 ? some_fn<FMT, 2>(lanes, pieces) : (m == 3 ? some_fn<FMT, 3>(lanes, pieces) : (m == 4 ? some_fn<FMT, 4>(lanes, pieces) : some_fn<FMT, 5>(lanes, pieces)));
}
const void* instance(int format, int64_t m, int lanes, int pieces) {
  return format == TLHIP_FMT_INT4_GROUPED ? some_fn<TLHIP_FMT_INT4_GROUPED>(m, lanes, pieces)
         : format == TLHIP_FMT_INT8_ROW   ? some_fn<TLHIP_FMT_INT8_ROW>(m, lanes, pieces)
                                          : some_fn<TLHIP_FMT_INT8_GROUPED>(m, lanes, pieces);
}
int pieces_of(const Problem& p, int lanes) { return (int)((p.k + kSomeWaves * 8 * lanes - 1) / (kSomeWaves * 8 * lanes)); }
int groups_of(const Problem& p) { return p.format == TLHIP_FMT_INT8_ROW ? 0 : (int)(p.k / p.group_size); }
size_t lds_of(const Problem& p, const tlhip_kernel_config_t& c) {
  const int lg = 64 / c.p0, count = (c.p4 + kSomeCols * lg - 1) / (kSomeCols * lg);
  return (size_t)((c.p4 * groups_of(p) * 2 + 15) / 16 * 16) + (size_t)count * lg * kSomeCols * (size_t)p.m * kSomePartsRow * 4;
}

}  // namespace

bool is_some_config(const tlhip_kernel_config_t& c) { return c.variant == VARIANT_GEMV && c.p5 == 4; }

bool gemv_some_config_applicable(const Problem& p, const tlhip_kernel_config_t& c, const char** why) {
  auto fail = [&](const char* text) {
    if (why) *why = text;
    return false;
  };
  if (!is_some_config(c) || p.x_dtype != TLHIP_F32 || p.m < 2 || p.m > 5 || p.pro.kind != TLHIP_PRO_NONE)
    return fail("the form for f32 rows (p5 = 4) is built for 2..5 of them and no prologue");
  if (p.k <= 0 || p.k > kSomeMaxK || p.k % 32 != 0) return fail("K must be a multiple of 32 up to 8192");
  if (p.format != TLHIP_FMT_INT8_ROW && (p.group_size < 32 || groups_of(p) % 2 != 0)) return fail("groups must be of 32 or more, an even number of them to a row");
  if (c.p1 != 1 || c.p2 != kSomeWaves || c.p3 != 1 || c.p6 || (c.p0 != 16 && c.p0 != 32 && c.p0 != 64) || c.p4 < 1 || c.p4 > kSomeMaxCols)
    return fail("lanes of a column (p0) 16, 32 or 64; p1 1, p2 8, p3 1; columns (p4) 1..64");
  if (pieces_of(p, c.p0) > (c.p0 == 64 ? 2 : 1)) return fail("more of K than the lanes of eight waves hold");
  if (lds_of(p, c) > (size_t)160 * 1024) return fail("the sums of a workgroup do not fit LDS");
  return true;
}

bool gemv_some_default(const Problem& p, tlhip_kernel_config_t* out) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  memset(out, 0, sizeof *out);
  out->variant = VARIANT_GEMV;
  out->p0 = p.k <= kSomeWaves * 8 * 16 ? 16 : (p.k <= kSomeWaves * 8 * 32 ? 32 : 64);
  out->p1 = 1;
  out->p2 = kSomeWaves;
  out->p3 = 1;
  out->p5 = 4;
  // An even share of the columns, at most what a lane's registers hold between two folds: eight columns for
  // each group of lanes (two workgroups a CU hide more than a second turn: 2 rows of int8-64 at 4096 x 4096 6.0 us
  // with 8 columns, 6.6 with 16), twice that where two pieces of K leave room for one workgroup.
  const int64_t most = (int64_t)kSomeCols * (64 / out->p0) * std::min(pieces_of(p, out->p0), 2);
  const int64_t rounds = std::max<int64_t>(1, (p.n + cus * most - 1) / (cus * most));
  out->p4 = (int)std::max<int64_t>(1, (p.n + cus * rounds - 1) / (cus * rounds));
  return gemv_some_config_applicable(p, *out, nullptr);
}

int launch_gemv_some(const Problem& p, const tlhip_kernel_config_t& c, hipStream_t stream) {
  const char* why = nullptr;
  if (!gemv_some_config_applicable(p, c, &why)) return set_error(TLHIP_ERR_INVALID, "gemv_some: config not applicable: %s", why ? why : "?");
  if (p.n == 0) return TLHIP_OK;
  SomeArgs a;
  memset(&a, 0, sizeof a);
  a.packed = (const uint8_t*)p.packed;
  a.scales = (const uint8_t*)p.scales;
  a.x = (const float*)p.x;
  a.y = p.y;
  a.n = (int)p.n;
  a.k = (int)p.k;
  a.cols = c.p4;
  a.row_bytes = (int)(p.format == TLHIP_FMT_INT4_GROUPED ? p.k / 2 : p.k);
  a.groups = groups_of(p);
  a.group_shift = p.format == TLHIP_FMT_INT8_ROW ? 0 : __builtin_ctz((unsigned)p.group_size);
  a.factor = p.alpha * (p.format == TLHIP_FMT_INT8_GROUPED ? 1.0f / 127.0f : (p.format == TLHIP_FMT_INT4_GROUPED ? 0.0625f : 1.0f));
  a.y_dtype = p.y_dtype;
  a.epi = p.epi;
  void* args[] = {(void*)&a};
  const int rc = launch_kernel(instance(p.format, p.m, c.p0, pieces_of(p, c.p0)), dim3((unsigned)((p.n + c.p4 - 1) / c.p4)), dim3(kSomeWaves * 64), args,
                               lds_of(p, c), stream);
  if (rc) return rc;
  count_gemv_dispatch();
  return TLHIP_OK;
}

// Every instance launch_gemv_some can reach, in prepare mode (see launch_kernel).
int prepare_gemv_some_kernels() {
  for (int format = 0; format < 3; ++format)
    for (int m = 2; m <= 5; ++m)
      for (int lanes : {16, 32, 64})
        for (int pieces = 1; pieces <= (lanes == 64 ? 2 : 1); ++pieces) {
          const int rc = launch_kernel(instance(format, m, lanes, pieces), dim3(1), dim3(64), nullptr, 0, nullptr);
          if (rc) return rc;
        }
  return TLHIP_OK;
}

}  // namespace tlhip
