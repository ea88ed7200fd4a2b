// GEMM of 17 to 64 f16 activation rows over packed weights, exact: the integers go to the
// matrix cores as they are and every group's sum is scaled in f32, as in the decode kernels.
// Same contract and reference route as gemv.hip (src/backend/webgpu/matmul/gemv.ts:365-466).
//
// What bounds it: its own instructions (X into LDS and out of it as operands, the dequantising, the
// products), then the weights' way from memory.  Every workgroup needs all of X (64 rows of K = 4096 are 512 KB,
// three times a CU's LDS) from its L2: little beside the instructions at that K, the largest part at long K on few columns
// (48 rows at 4096 x 12288: 302 MB of X for 28 MB of weights).  Hence:
//   * A workgroup owns 16 NB columns of Y and all of K, so that nothing is combined between
//     workgroups: no planes of partial sums, no second launch, no workspace.
//   * Each of its eight waves has a range of K, 128 a step, alone until one barrier at the end: the
//     activations of a step (16 MT rows) are loaded into registers a step ahead, whole lines per row, laid
//     into a patch of LDS that belongs to the wave, and read back as MFMA operands.
//   * A range's group scales come once, 16 bytes of a column a lane, into LDS too: a load of 8 bytes of 16
//     columns with every step cost the memory pipe what the step's weights do.
//   * Plain loads of the weights: the neighbouring steps of a range share lines, which the nontemporal hint
//     fetched twice (10-25 % slower).
//   * An operand of X feeds NB products and a weight, dequantised once, MT.
//   * Few columns: a workgroup takes a share of the row tiles, so that more CUs work (gemm_rows_default).
// Us on cold weights, steps dealt to the waves in turn with their scales, two in flight and empty loads past the end -> as it
// is: int4 12288 x 4096 at 48 rows 18.1 -> 16.5, with a residual 19.9 -> 18.6, 4096 x 4096 with a residual 12.7 -> 11.3,
// 4096 x 12288 25.7 -> 22.6, 1024 x 1024 5.4 -> 3.5; int8-64 12288 x 4096 at 32 rows 22.3 -> 15.7; 1.22 times faster in the mean
// of 6588 problems of up to 16384 columns at 17..64 rows, three formats.  16.5 us are 1.7 TB/s of weights and scales and
// 293 TFLOP/s.
// Rearranging X for the cheaper int4 unpacking, or its addresses by lane, moved nothing.
//   * Buffer loads: rows past M and columns past N read zero, so that the loop has no branch around a load.
#include <algorithm>
#include <cstring>

#include "gemv_mfma_common.h"

namespace tlhip {
namespace {

constexpr int kWaves = 8;
constexpr int kStep = 128;                  // k of a step
constexpr int kRowBytes = kStep * 2 + 16;   // LDS row of a step: 16 bytes more, so that rows start in other banks
constexpr int kMaxCols = 4;                 // blocks of 16 columns per workgroup
constexpr int kMaxScaleSteps = 16;          // steps of a wave whose scales it holds at a time

struct RowsArgs {
  const uint8_t* packed;
  const uint8_t* scales;
  const _Float16* x;
  void* y;
  int m, n, k;
  int row_bytes;         // packed bytes of a weight row
  int scale_row_bytes;   // bytes of a row's group scales
  int group_shift;       // int8 groups: log2(group size / 64)
  int scale_steps;       // steps of a wave whose scales its patch holds
  int scale_stride;      // bytes of a column there
  float alpha, scale_mul;
  int y_dtype;
  int vec_ok;            // N % 4 == 0 and y 16-byte aligned: four columns in one store
  DevEpilogue epi;
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ rsrc_t buffer_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00027000);
}
template <int AUX>
__device__ __forceinline__ u32x4 load16(rsrc_t r, uint32_t at, uint32_t step_at) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, (int)step_at, AUX));
}

// The 8 weights of a word in k order (unpack_int4_word: pairs four apart): three more VALU
// instructions a word, but no rearranging of the activations, of which a step has MT times as many.
__device__ __forceinline__ half8_t weights_of(uint32_t w) {
  const uint32_t t = w ^ 0x88888888u;
  const half2_t mul = {(_Float16)1.f, (_Float16)0.0625f}, add = {(_Float16)-1032.f, (_Float16)-72.f};
  half2_t h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t twice = __builtin_amdgcn_perm(t, t, 0x01010101u * (uint32_t)i);  // byte i four times
    h[i] = __builtin_bit_cast(half2_t, and_or(twice, 0x00f0000fu, 0x64006400u)) * mul + add;
  }
  return join8(h);
}

// MT: tiles of 16 rows (M <= 16 MT); NB: blocks of 16 columns
template <int FMT, int MT, int NB>
__global__ __launch_bounds__(kWaves * 64) void gemm_rows_kernel(const RowsArgs a) {
  constexpr bool INT4 = FMT == TLHIP_FMT_INT4_GROUPED, ROW = FMT == TLHIP_FMT_INT8_ROW;
  constexpr int WV = INT4 ? 1 : 2;      // 16-byte loads of a step, lane and column block
  constexpr int XV = MT * 4;            // 16-byte loads of a step's X per lane: four rows each
  extern __shared__ u32x4 lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nl = lane & 15, g = lane >> 4;
  const int a_scale_steps = a.scale_steps, scale_stride = a.scale_stride;
  const int n0 = (int)blockIdx.x * (16 * NB);
  const int cols = min(16 * NB, a.n - n0);
  const int row0 = (int)blockIdx.y * (16 * MT), m = min(a.m - row0, 16 * MT);  // (fewer tiles a workgroup than rows: a share of them)
  const int steps = a.k / kStep;
  const uint8_t* const packed = a.packed + (int64_t)n0 * a.row_bytes;
  const uint8_t* const scales = a.scales + (int64_t)n0 * a.scale_row_bytes;

  // A lane's place in a step is fixed, the step is a scalar offset; past the last step a buffer
  // of no bytes at offset 0 (a range check may or may not count the scalar offset).
  uint32_t w_at[NB], s_at[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    w_at[b] = (uint32_t)(16 * b + nl) * (uint32_t)a.row_bytes + (uint32_t)g * 16u;
    s_at[b] = (uint32_t)(16 * b + nl) * (uint32_t)a.scale_row_bytes;
  }
  const uint32_t x_at = (uint32_t)g * (uint32_t)a.k * 2u + (uint32_t)nl * 16u;  // in four rows, a buffer each

  // The wave's range of steps (workgroups of an XCD start at different ones: all on the same lines of X at a
  // time is slower), and its group scales in a patch of LDS, 16 bytes of a column a lane.
  const int range = (wave + ((int)blockIdx.x >> 3)) & (kWaves - 1);
  // (the first ranges are the longer ones: waves four apart share a SIMD, two long ones there are a step more)
  const int each = steps / kWaves, more = steps % kWaves;
  const int st0 = range * each + min(range, more), end = st0 + each + (range < more ? 1 : 0);
  constexpr int SB = INT4 ? 8 : 4;  // bytes of a step and column
  constexpr bool LATE = INT4 && MT * NB >= 8;  // no registers for the weights of two steps, nor a last step of its own
  constexpr int SL = INT4 ? 2 : 1;  // 16-byte loads for kMaxScaleSteps steps: 64 bytes of a column each
  char* const scale_patch = (char*)lds + kWaves * (MT * 16 * kRowBytes) + wave * (16 * NB * scale_stride) + nl * scale_stride;
  struct Scales {
    u32x4 v[SL][NB];  // (int8 in wider groups: word q is the scale of step 4 q + g)
  };
  const rsrc_t sb = buffer_of(scales, (uint32_t)cols * (uint32_t)a.scale_row_bytes);
  auto load_scales = [&](Scales& v, int from) __attribute__((always_inline)) {
    const int count = min(a_scale_steps, end - from);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (INT4 || a.group_shift == 0) {
#pragma unroll
        for (int q = 0; q < SL; ++q) {  // (a lane past the range: what its column's first one reads)
          const int at = q * 64 + g * 16 < count * SB ? q * 64 + g * 16 : 0;
          v.v[q][b] = load16<0>(sb, s_at[b] + (uint32_t)at, (uint32_t)from * SB);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v.v[0][b][q] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sb, (int)(s_at[b] + ((uint32_t)(2 * (from + min(4 * q + g, count - 1))) >> a.group_shift) * 2u), 0, 0);
      }
    }
  };
  auto lay_scales = [&](const Scales& v, int from) __attribute__((always_inline)) {
    const int count = min(a_scale_steps, end - from);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      char* const to = scale_patch + 16 * b * scale_stride;
      if (INT4 || a.group_shift == 0) {
#pragma unroll
        for (int q = 0; q < SL; ++q)
          if (q * 64 + g * 16 < count * SB) *(u32x4*)(to + q * 64 + g * 16) = v.v[q][b];
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q * 4 + g < count) *(uint32_t*)(to + (q * 4 + g) * 4) = v.v[0][b][q] | v.v[0][b][q] << 16;
      }
    }
  };
  struct Weights {
    u32x4 w[NB][WV];
  };
  const rsrc_t wb = buffer_of(packed, (uint32_t)cols * (uint32_t)a.row_bytes);
  auto load_block = [&](Weights& v, int b, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WV; ++i) v.w[b][i] = load16<0>(wb, w_at[b] + (uint32_t)i * 64u, (uint32_t)st * (WV * 64u));
  };
  auto load_w = [&](Weights& v, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b) load_block(v, b, st);
  };
  struct Rows {
    u32x4 v[XV];
  };
  auto load_x = [&](Rows& r, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XV; ++i)
      r.v[i] = load16<0>(buffer_of(a.x + (int64_t)(row0 + 4 * i) * a.k, (uint32_t)max(m - 4 * i, 0) * (uint32_t)a.k * 2u), x_at, (uint32_t)st * (kStep * 2u));
  };
  char* const patch = (char*)lds + wave * (MT * 16 * kRowBytes);
  auto lay_x = [&](const Rows& r) {
#pragma unroll
    for (int i = 0; i < XV; ++i) *(u32x4*)(patch + (4 * i + g) * kRowBytes + nl * 16) = r.v[i];
  };

  float4_t acc[NB][MT];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[b][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
  // operand s of a step: int4 k = 32 s + 8 g; int8 k = 64 (s / 2) + 16 g + 8 (s % 2)
  auto operand = [&](int t, int s) {
    const int unit = INT4 ? 4 * s + g : 8 * (s >> 1) + 2 * g + (s & 1);
    return __builtin_bit_cast(half8_t, *(const u32x4*)(patch + (16 * t + nl) * kRowBytes + unit * 16));
  };
  // `next`: the step whose weights take the registers as they become free, or -1
  auto multiply = [&](Weights& v, int st_held, int next) __attribute__((always_inline)) {
    uint32_t scale[NB][2];  // int4: four group scales; int8: one per half step
    if constexpr (!ROW) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const char* const from = scale_patch + 16 * b * scale_stride + st_held * SB;
        const uint32_t w = *(const uint32_t*)from;
        scale[b][0] = INT4 ? w : w & 0xffffu;
        scale[b][1] = INT4 ? *(const uint32_t*)(from + 4) : w >> 16;
      }
    }
    uint32_t word[NB][4 * WV];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int i = 0; i < WV; ++i) {
        word[b][4 * i + 0] = v.w[b][i].x;
        word[b][4 * i + 1] = v.w[b][i].y;
        word[b][4 * i + 2] = v.w[b][i].z;
        word[b][4 * i + 3] = v.w[b][i].w;
      }
      // a lane holds 32 k of its row, one group; afterwards word i is its eighth of group i
      if constexpr (INT4) transpose4(word[b][0], word[b][1], word[b][2], word[b][3]);
    }
    if (next >= 0) load_w(v, next);
    // a step's own sum first: the long one takes a step at a time (rel-L2 against 64 bits at K = 8192,
    // int4 / int8-64 / per row: 11.3 / 9.7 / 16.3e-8 one group at a time, 8.4 / 8.9 / 8.8e-8 so, 8.8 / 8.9 / 9.2e-8
    // for the decode kernel with its four to eight K slices)
    if constexpr (INT4 && MT * NB >= 12) {  // a block at a time: X from LDS again, a third of the registers
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float4_t sum[MT];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const half8_t wv = weights_of(word[b][s]);
          const float sc = half_bits_to_float((s & 1) ? scale[b][s >> 1] >> 16 : scale[b][s >> 1] & 0xffffu);
          float4_t d[MT];
#pragma unroll
          for (int t = 0; t < MT; ++t) d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(t, s), wv, (float4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[t][r] = s == 0 ? sc * d[t][r] : fmaf(sc, d[t][r], sum[t][r]);
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[b][t][r] += sum[t][r];
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
    float4_t sum[NB][MT];
    if constexpr (INT4) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        half8_t xa[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) xa[t] = operand(t, s);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const half8_t wv = weights_of(word[b][s]);
          const float sc = half_bits_to_float((s & 1) ? scale[b][s >> 1] >> 16 : scale[b][s >> 1] & 0xffffu);
          float4_t d[MT];
#pragma unroll
          for (int t = 0; t < MT; ++t) d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[t], wv, (float4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[b][t][r] = s == 0 ? sc * d[t][r] : fmaf(sc, d[t][r], sum[b][t][r]);
        }
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        half8_t xa[2][MT];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < MT; ++t) xa[i][t] = operand(t, 2 * h + i);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          float4_t d[MT];
#pragma unroll
          for (int t = 0; t < MT; ++t) d[t] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            half2_t w[4];
            unpack_int8_word(word[b][4 * h + 2 * i], w);
            unpack_int8_word(word[b][4 * h + 2 * i + 1], w + 2);
            const half8_t wv = join8(w);
#pragma unroll
            for (int t = 0; t < MT; ++t) d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][t], wv, d[t], 0, 0, 0);
          }
          const float sc = ROW ? 1.f : half_bits_to_float(scale[b][h]);
#pragma unroll
          for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float p = ROW ? d[t][r] : sc * d[t][r];
              sum[b][t][r] = h == 0 ? p : (ROW ? sum[b][t][r] + d[t][r] : fmaf(sc, d[t][r], sum[b][t][r]));
            }
        }
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[b][t][r] += sum[b][t][r];
  };

  // No load goes past the end, though a buffer would answer it with zeros: at one to four steps a wave those cost
  // as much as the others (12-20 % at K up to 2304).  The patch is the wave's own, and a
  // wave's LDS accesses stay in order.  One part, unless the scales of a range do not fit.
  for (int from = st0; from < end; from += a_scale_steps) {
    const int upto = min(from + a_scale_steps, end), left = upto - from;
    Scales v;
    if constexpr (!ROW) {
      load_scales(v, from);
      __builtin_amdgcn_sched_barrier(0);  // ahead of the rest: a wait for them is a wait for nothing else
    }
    Weights w;
    Rows x;
    load_x(x, from);
    load_w(w, from);
    if constexpr (!ROW) lay_scales(v, from);
    if constexpr (LATE) {
      for (int i = 0; i + 1 < left; ++i) {
        lay_x(x);
        load_x(x, from + i + 1);
        multiply(w, i, -1);
        load_w(w, from + i + 1);
      }
      lay_x(x);
      __builtin_amdgcn_sched_barrier(0);
      multiply(w, left - 1, -1);
    } else {
      for (int i = 0; i + 1 < left; ++i) {
        lay_x(x);
        load_x(x, from + i + 1);
        multiply(w, i, from + i + 1);
      }
      lay_x(x);
      multiply(w, left - 1, -1);
    }
  }

  // ---- the waves' sums and the epilogue ---------------------------------------
  lds_barrier();  // every wave has read its patch
  float* const sums = (float*)lds;  // [range][row tile][block][16 x 16]
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) sums[((range * MT + t) * NB + b) * 256 + (4 * g + r) * 16 + nl] = acc[b][t][r];
  lds_barrier();
  float factor = a.scale_mul * a.alpha;
#pragma unroll
  for (int e0 = 0; e0 < MT * NB * 64; e0 += kWaves * 64) {
    const int e = e0 + tid, row = e / (4 * NB), c = e % (4 * NB) * 4;  // four columns of a row
    if (e >= MT * NB * 64 || row >= m || n0 + c >= a.n) continue;
    const float* p = sums + ((row >> 4) * NB + (c >> 4)) * 256 + (row & 15) * 16 + (c & 15);
    float4_t part[kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) part[w] = *(const float4_t*)(p + w * (MT * NB * 256));
    float4_t sum;  // in pairs: a shorter chain, a smaller rounding error
#pragma unroll
    for (int i = 0; i < 4; ++i)
      sum[i] = ((part[0][i] + part[1][i]) + (part[2][i] + part[3][i])) + ((part[4][i] + part[5][i]) + (part[6][i] + part[7][i]));
    const int col = n0 + c;
    const int64_t at = (int64_t)(row0 + row) * a.n + col;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ci = min(col + i, a.n - 1) - col;  // past the last column: that one again, not stored
      float f = factor;
      if constexpr (ROW) f *= ((const float*)a.scales)[col + ci];
      v[i] = apply_epilogue(a.epi, sum[i] * f, col + ci, at + ci);
    }
    if (a.vec_ok) {  // N a multiple of 4, rows aligned
      if (a.y_dtype == TLHIP_F16) *(half4_t*)((_Float16*)a.y + at) = (half4_t){(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
      else *(float4_t*)((float*)a.y + at) = (float4_t){v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (col + i < a.n) store_out(a.y, a.y_dtype, at + i, v[i]);
    }
  }
}

int row_tiles_of(int64_t m) { return (int)((m + 15) / 16); }
// ... of a workgroup: all, or p6 of them.
int tiles_of(const Problem& p, const tlhip_kernel_config_t& c) { return c.p6 ? c.p6 : row_tiles_of(p.m); }
// The column blocks whose instance fits 256 vector registers a lane without spilling one; the fullest
// (int4, three blocks of 48 rows and two of 64) use all of them.  Four row tiles need 16 buffer
// descriptors a step and spill some scalar registers, to lanes of a vector register.
constexpr int most_columns(int format, int mt) {
  return mt == 1 ? 1 : format == TLHIP_FMT_INT4_GROUPED ? (mt == 4 ? 3 : 4) : (mt == 2 ? 4 : (mt == 3 ? 3 : 2));
}

template <int FMT, int MT, int NB>
const void* instance() {
  if constexpr (NB > most_columns(FMT, MT)) {
    return nullptr;
  } else {
    return (const void*)gemm_rows_kernel<FMT, MT, NB>;
  }
}
template <int FMT, int MT>
const void* instance_of(int nb) {
  return nb == 1 ? instance<FMT, MT, 1>() : (nb == 2 ? instance<FMT, MT, 2>() : (nb == 3 ? instance<FMT, MT, 3>() : instance<FMT, MT, 4>()));
}
template <int FMT>
const void* instance_of(int mt, int nb) {
  return mt == 1 ? instance<FMT, 1, 1>() : mt == 2 ? instance_of<FMT, 2>(nb) : (mt == 3 ? instance_of<FMT, 3>(nb) : instance_of<FMT, 4>(nb));
}
const void* instance_of(int format, int mt, int nb) {
  return format == TLHIP_FMT_INT4_GROUPED ? instance_of<TLHIP_FMT_INT4_GROUPED>(mt, nb)
         : format == TLHIP_FMT_INT8_ROW   ? instance_of<TLHIP_FMT_INT8_ROW>(mt, nb)
                                          : instance_of<TLHIP_FMT_INT8_GROUPED>(mt, nb);
}

// Steps whose scales a wave's patch holds: all of a range, or as many as fit beside the rows.
int scale_steps_of(const Problem& p, int mt, int nb) {
  if (p.format == TLHIP_FMT_INT8_ROW) return (int)(p.k / kStep);
  const int sb = p.format == TLHIP_FMT_INT4_GROUPED ? 8 : 4, range = (int)((p.k / kStep + kWaves - 1) / kWaves);
  const int lds = 160 * 1024 - kWaves * mt * 16 * kRowBytes;
  const int fit = (lds / (kWaves * 16 * nb) / 16 * 16 - 16) / sb;
  return std::min({range, kMaxScaleSteps, fit});
}
int scale_stride_of(const Problem& p, int mt, int nb) {
  const int steps = scale_steps_of(p, mt, nb);
  return p.format == TLHIP_FMT_INT8_ROW ? 0 : (steps * (p.format == TLHIP_FMT_INT4_GROUPED ? 8 : 4) + 15) / 16 * 16 + 16;
}
size_t lds_of(const Problem& p, int mt, int nb) {
  const int scales = 16 * nb * scale_stride_of(p, mt, nb);
  return std::max((size_t)kWaves * (mt * 16 * kRowBytes + scales), (size_t)kWaves * mt * nb * 1024);
}

}  // namespace

bool is_rows_config(const Problem& p, const tlhip_kernel_config_t& c) {
  if (c.variant != VARIANT_GEMV_MFMA || c.p0 != kWaves || c.p4 < 1 || c.p4 > kMaxCols) return false;
  if (c.p1 || c.p2 || c.p3 || c.p5 || c.p6 < 0 || c.p6 >= row_tiles_of(p.m) || (c.p6 && (c.p6 > 2 || c.p4 > 1))) return false;  // the other form's fields: p4 is not read there
  if (p.x_dtype != TLHIP_F16 || p.m < 17 || p.m > 64 || p.pro.kind != TLHIP_PRO_NONE) return false;
  if (!c.p6 && c.p4 > most_columns(p.format, row_tiles_of(p.m))) return false;
  if (p.k <= 0 || p.k % kStep != 0 || p.k > (1 << 23)) return false;  // offsets below 2^31: 64 rows of X or of weights
  if (p.format == TLHIP_FMT_INT4_GROUPED) return p.group_size == 32;
  return p.format == TLHIP_FMT_INT8_ROW || p.group_size >= 64;
}

// What a launch takes behind others and on cold weights, beside K slices across workgroups (gemv_mfma_rows_us): the
// weights' way from memory, per round of workgroups the blocks' sums and, per 4096 of K, a step, its blocks and its
// rows; a share of the row tiles, of which every workgroup has a CU, the walk of a range.
// Fitted at 4968 launches of the geometries that gemm_rows_default weighs (13 x 11 matrices of 768..28672 x 1024..16384,
// 17..64 rows, three formats, with and without a residual): 3-5 % rms, two tiles of int8 8 %.
double gemm_rows_us(const Problem& p, const tlhip_kernel_config_t& c) {
  struct Whole {
    double launch, mb, round, sums, k, k_blocks, k_rows, residual, residual_out;
  };
  struct Share {
    double launch, k, mb, residual, residual_out;
  };
  static const Whole whole[3][3] = {  // format, row tiles
      {{2.035, 0.089, 0.0, 0.876, 1.163, 1.220, 1.005, 0.990, 0.140}, {1.401, 0.121, 0.464, 1.145, 2.486, 1.195, 0.686, 0.916, 0.165}, {1.627, 0.104, 0.253, 1.290, 0.0, 2.078, 1.285, 0.830, 0.158}},
      {{1.878, 0.061, 0.394, 0.587, 0.718, 1.677, 1.555, 1.062, 0.124}, {1.182, 0.069, 1.001, 0.848, 2.336, 1.383, 1.132, 0.868, 0.202}, {1.415, 0.077, 0.475, 1.299, 0.0, 0.978, 1.863, 0.855, 0.165}},
      {{1.682, 0.068, 0.518, 0.631, 0.907, 1.445, 1.500, 1.000, 0.099}, {1.586, 0.081, 0.272, 0.996, 2.676, 1.101, 1.028, 0.833, 0.183}, {1.477, 0.082, 0.498, 1.019, 0.0, 1.118, 1.766, 0.808, 0.163}}};
  static const Share share[3][2] = {  // format, one or two tiles a workgroup
      {{2.699, 2.401, 0.115, 0.771, 0.804}, {2.899, 3.771, 0.108, 0.816, 0.438}},
      {{2.786, 3.127, 0.045, 0.816, 0.812}, {2.899, 4.408, 0.047, 0.702, 0.805}},
      {{2.710, 3.085, 0.045, 0.795, 0.775}, {2.828, 4.293, 0.043, 0.662, 0.781}}};
  const bool int4 = p.format == TLHIP_FMT_INT4_GROUPED, residual = has_residual(p);
  const int format = int4 ? 0 : (p.format == TLHIP_FMT_INT8_ROW ? 2 : 1), cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const double mb = (double)p.n * (double)p.k * (int4 ? 0.5 : 1.0) / 1e6, out = (double)p.m * (double)p.n / 1e5, walk = (double)p.k / 4096.0;
  if (c.p6) {
    const Share& t = share[format][c.p6 - 1];
    return t.launch + t.k * walk + t.mb * mb + (residual ? t.residual + t.residual_out * out : 0.0);
  }
  const Whole& t = whole[format][row_tiles_of(p.m) - 2];
  const int64_t wgs = (p.n + 16 * c.p4 - 1) / (16 * c.p4);
  const double rounds = (double)((wgs + cus - 1) / cus);
  return t.launch + t.mb * mb + rounds * (t.round + t.sums * c.p4 + walk * (t.k + t.k_blocks * c.p4 + t.k_rows * (double)p.m / 16.0)) +
         (residual ? t.residual + t.residual_out * out : 0.0);
}

// The number of column blocks or the share of the row tiles, and its time in microseconds where the launch is not behind
// others (beside the tiles, which were priced so), or false.  Fitted at 3072 launches of 52 matrices of 768..16384 x
// 768..12288, 17..64 rows, four formats: launch, and per round of workgroups a constant, the sums of a block and, per
// 4096 of K in whole steps of the longest wave, the figure of the width, a little more for every row above the middle of
// its tile.  One block a workgroup: up to four rounds overlap (two fit a CU up to 32 rows).  8-10 % off (rms); the width
// it picks is 0.0-0.4 % behind the best one in the mean of 2624 problems on cold weights.
bool gemm_rows_default(const Problem& p, tlhip_kernel_config_t* out, double* us) {
  struct Cost {
    double launch, round, block, walk[kMaxCols], second, per_row;
  };
  static const Cost costs[3][3] = {  // format, row tiles
      {{3.24, 0.0, 0.367, {4.09, 5.39, 6.99, 8.29}, 0.56, 0.004}, {2.70, 0.64, 0.568, {5.64, 6.72, 8.72, 11.71}, 0.83, 0.004}, {2.52, 0.85, 0.584, {7.03, 8.10, 11.91, 0.0}, 0.82, 0.006}},  // int4
      {{3.37, 0.0, 0.361, {4.54, 5.92, 7.65, 9.23}, 0.64, 0.012}, {3.04, 0.65, 0.507, {6.00, 7.22, 9.62, 0.0}, 0.88, 0.005}, {2.87, 1.27, 0.169, {7.09, 8.70, 0.0, 0.0}, 0.86, 0.006}},    // int8 in groups
      {{3.62, 0.0, 0.147, {4.26, 5.60, 7.51, 9.12}, 0.73, 0.008}, {2.78, 0.69, 0.495, {5.84, 6.75, 9.22, 0.0}, 0.87, 0.005}, {2.65, 1.44, 0.127, {6.77, 8.13, 0.0, 0.0}, 0.84, 0.009}}};  // int8 per row
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const int format = p.format == TLHIP_FMT_INT4_GROUPED ? 0 : (p.format == TLHIP_FMT_INT8_ROW ? 2 : 1), mt = row_tiles_of(p.m);
  // (up to four steps: on a SIMD each)
  const int64_t steps = p.k / kStep, walked = steps <= 4 ? steps : (steps + kWaves - 1) / kWaves * kWaves;
  const double walk = (double)(walked * kStep) / 4096.0;
  bool found = false;
  for (int nb = 1; nb <= kMaxCols; ++nb) {
    tlhip_kernel_config_t c;
    memset(&c, 0, sizeof c);
    c.variant = VARIANT_GEMV_MFMA;
    c.p0 = kWaves;
    c.p4 = nb;
    if (!is_rows_config(p, c)) continue;
    const Cost& cost = costs[format][mt - 2];
    const int64_t wgs = (p.n + 16 * nb - 1) / (16 * nb), turns = (wgs + cus - 1) / cus;
    const double rounds = 1.0 + (nb == 1 ? cost.second * (double)(std::min<int64_t>(turns, 4) - 1) + (double)std::max<int64_t>(turns - 4, 0) : (double)(turns - 1));
    const double t = cost.launch + rounds * (cost.round + cost.block * nb + walk * cost.walk[nb - 1] * (1.0 + cost.per_row * (double)(p.m - 16 * mt + 8)));
    if (found && t >= *us) continue;
    *out = c;
    *us = t;
    found = true;
  }
  // Few columns: the row tiles to workgroups of their own while every one has a CU, which reads the weights once
  // for each (from the last-level cache) but walks a range in the time of one tile, us, all tiles / one / two a
  // workgroup: int4 1024 x 4096 at 48 rows 9.6 / 6.3 / 7.8, 1024 x 12288 at 64 27.4 / 11.0 / 15.0, 1536 x 6144 at 48 12.1 /
  // 10.8 / 9.7; past one a CU behind (int8-64 4096 x 4096 at 48 rows 10.6 / 13.0 / 12.5).  Int8 with K beyond 6144 and more
  // than 1152 columns is left to the K slices, as the tests of the routing hold it there.
  if (found && (format == 0 || p.k <= 6144 || p.n <= 1152))
    for (int tiles = 1; tiles <= 2 && tiles < mt; ++tiles) {
      tlhip_kernel_config_t c = *out;
      c.p4 = 1;
      c.p6 = tiles;
      if ((p.n + 15) / 16 * ((mt + tiles - 1) / tiles) > cus || !is_rows_config(p, c) || gemm_rows_us(p, c) >= gemm_rows_us(p, *out)) continue;
      static const double one[3] = {2.2, 2.85, 2.7};
      const Cost& two = costs[format][0];
      *out = c;
      *us = tiles == 1 ? 4.1 + walk * one[format] : two.launch + two.round + two.block + walk * two.walk[0];
    }
  return found;
}

int launch_gemm_rows(const Problem& p, const tlhip_kernel_config_t& c, hipStream_t stream) {
  if (!is_rows_config(p, c)) return set_error(TLHIP_ERR_INVALID, "gemm_rows: config not applicable");
  if (p.n == 0 || p.m == 0) return TLHIP_OK;
  RowsArgs a;
  memset(&a, 0, sizeof a);
  a.packed = (const uint8_t*)p.packed;
  a.scales = (const uint8_t*)p.scales;
  a.x = (const _Float16*)p.x;
  a.y = p.y;
  a.m = (int)p.m;
  a.n = (int)p.n;
  a.k = (int)p.k;
  a.row_bytes = (int)(p.format == TLHIP_FMT_INT4_GROUPED ? p.k / 2 : p.k);
  a.scale_row_bytes = p.format == TLHIP_FMT_INT8_ROW ? 4 : (int)(p.k / p.group_size) * 2;
  a.group_shift = p.format == TLHIP_FMT_INT8_GROUPED ? __builtin_ctz((unsigned)(p.group_size / 64)) : 0;
  a.scale_steps = scale_steps_of(p, tiles_of(p, c), c.p4);
  a.scale_stride = scale_stride_of(p, tiles_of(p, c), c.p4);
  a.alpha = p.alpha;
  a.scale_mul = p.format == TLHIP_FMT_INT8_GROUPED ? 1.0f / 127.0f : 1.0f;
  a.y_dtype = p.y_dtype;
  a.vec_ok = p.n % 4 == 0 && ((uintptr_t)p.y & 15) == 0;
  a.epi = p.epi;
  void* args[] = {(void*)&a};
  const int mt = tiles_of(p, c), nb = c.p4;
  const int rc = launch_kernel(instance_of(p.format, mt, nb), dim3((unsigned)((p.n + 16 * nb - 1) / (16 * nb)), (unsigned)((row_tiles_of(p.m) + mt - 1) / mt)), dim3(kWaves * 64), args,
                               lds_of(p, mt, nb), stream);
  if (rc) return rc;
  count_gemv_dispatch();
  return TLHIP_OK;
}

// Every instance launch_gemm_rows can reach, in prepare mode (see launch_kernel).
int prepare_gemm_rows_kernels() {
  for (int format : {TLHIP_FMT_INT4_GROUPED, TLHIP_FMT_INT8_GROUPED, TLHIP_FMT_INT8_ROW})
    for (int mt = 1; mt <= 4; ++mt)
      for (int nb = 1; nb <= most_columns(format, mt); ++nb) {
        const int rc = launch_kernel(instance_of(format, mt, nb), dim3(1), dim3(64), nullptr, 0, nullptr);
        if (rc) return rc;
      }
  return TLHIP_OK;
}

}  // namespace tlhip
