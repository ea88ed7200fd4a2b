// 2 to 16 f16 activation rows over packed weights, all of K in one workgroup, exact: the integers go to
// the matrix cores as they are and every group's sum is scaled in f32.  Same contract and reference
// route as gemv.hip (src/backend/webgpu/matmul/gemv.ts:365-466).
//
// What bounds it: the weights' way from memory where a workgroup has many columns, else the chain of
// one step after the other in a wave.  Hence:
//   * A workgroup owns up to 16 NB columns and all of K: no slices to combine between workgroups, no
//     workspace.  Its waves take K in turn, 128 at a time, each alone until one barrier at the end, so
//     that nothing waits for the slowest wave's activations.
//   * The columns are dealt evenly over the chip, in blocks of at most 16: a block with fewer loads
//     fewer (its other lanes load a neighbour's), where a last block of a few columns would be a round.
//   * A wave's part of K is one range.  Its group scales come once, 16 bytes of a column a lane, into a
//     patch of LDS: a load of 8 bytes of 16 columns per step costs the memory pipe what the step's weights
//     do (gate and up of 12288 x 4096 at 16 rows 21.6 us with, 16.4 without them).
//   * A step's activations go through a patch of the wave's own as well; two steps are in flight, and no
//     load goes past the end.
//   * Plain loads: the nontemporal hint cost 0.5-4 us a launch, as neighbouring steps share lines.
//   * A pair's gate and up are blocks of one workgroup, which writes their product.
#pragma once
#include "gemv_few_args.h"
#include "gemv_mfma_common.h"

namespace tlhip {
namespace {

typedef __amdgpu_buffer_rsrc_t few_rsrc_t;
__device__ __forceinline__ few_rsrc_t few_buffer(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ u32x4 few_load16(few_rsrc_t r, uint32_t at, uint32_t step_at) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, (int)step_at, 0));
}

// Scalars that are to be in registers from here on: arguments read where they are first used are a
// trip to memory each, one behind the other.
template <typename T>
__device__ __forceinline__ void few_in_register(T v) {
  asm volatile("" ::"s"(v));
}
template <typename... Ts>
__device__ __forceinline__ void few_in_registers(const Ts&... v) {
  (few_in_register(v), ...);
}

// XV: 16-byte loads of a step's activations per lane, four rows each (M <= 4 XV).  NB: blocks of columns
// (a pair: of both projections).  WIDE: a group's scales are whole words (int4, int8 in groups of 64).
template <int FMT, int XV, int NB, int KIND, bool WIDE>
__global__ __launch_bounds__(kFewWaves * 64) void gemv_few_kernel(const FewArgs<KIND> a) {
  constexpr bool INT4 = FMT == TLHIP_FMT_INT4_GROUPED, ROW = FMT == TLHIP_FMT_INT8_ROW;
  constexpr bool GROUP = KIND == FEW_GROUP, PAIR = KIND == FEW_PAIR;
  constexpr int NP = FewArgs<KIND>::NP, NA = PAIR ? 2 : 1, BP = NB / NA;  // blocks of a projection
  constexpr int WV = INT4 ? 1 : 2;  // 16-byte loads of a step, lane and block
  constexpr int SB = INT4 ? 8 : 4;  // bytes of a step and column in the patch of scales
  extern __shared__ u32x4 lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nl = lane & 15, g = lane >> 4, wg = (int)blockIdx.x;
  const int m = a.m, k = a.k, steps = a.steps, cols = a.cols, block_cols = a.block_cols, y_dtype = a.y_dtype, vec = a.vec;
  const uint32_t row_bytes = a.row_bytes, scale_row_bytes = a.scale_row_bytes;
  const int group_shift = a.group_shift;
  const float factor = a.factor;
  const _Float16* const xp = a.x;

  // ---- this workgroup's problem, selected between scalars
  int first = 0, n = a.n[0], pre_kind = a.pre_kind[0], pre_row = a.pre_row[0], n_ops = a.n_ops[0], pi = 0;
  const uint8_t *packed[NA] = {a.packed[0]}, *scales[NA] = {a.scales[0]};
  const void* pre = a.pre[0];
  void* y = a.y[0];
  if constexpr (GROUP) {
#pragma unroll
    for (int j = 0; j < NP; ++j)
      few_in_registers(a.first[j], a.n[j], a.pre_kind[j], a.pre_row[j], a.n_ops[j], a.packed[j], a.scales[j], a.pre[j], a.y[j]);
    few_in_registers(a.count);
  }
  if constexpr (PAIR) {
    packed[1] = a.packed[1];
    scales[1] = a.scales[1];
    few_in_registers(packed[1], scales[1], a.unary);
  }
  few_in_registers(m, k, steps, cols, block_cols, y_dtype, vec, row_bytes, scale_row_bytes, group_shift, factor, xp, n, pre_kind,
                   pre_row, n_ops, packed[0], scales[0], pre, y);
  if constexpr (GROUP) {
#pragma unroll
    for (int j = 1; j < NP; ++j) {
      const bool here = j < a.count && wg >= a.first[j];
      first = here ? a.first[j] : first;
      n = here ? a.n[j] : n;
      pre_kind = here ? a.pre_kind[j] : pre_kind;
      pre_row = here ? a.pre_row[j] : pre_row;
      n_ops = here ? a.n_ops[j] : n_ops;
      packed[0] = here ? a.packed[j] : packed[0];
      scales[0] = here ? a.scales[j] : scales[0];
      pre = here ? a.pre[j] : pre;
      y = here ? a.y[j] : y;
      pi = here ? j : pi;
    }
  }
  const int n0 = (wg - first) * cols, have = min(cols, n - n0);

  // ---- loads.  A lane's place in a step is fixed, the step is a scalar offset.
  uint32_t w_at[BP], s_at[BP];
#pragma unroll
  for (int b = 0; b < BP; ++b) {  // columns past the block's or the matrix's: the last one again, not stored
    const uint32_t col = (uint32_t)min(b * block_cols + min(nl, block_cols - 1), have - 1);
    w_at[b] = col * row_bytes + (uint32_t)g * 16u;
    s_at[b] = col * scale_row_bytes;
  }
  few_rsrc_t wb[NA], sb[NA];
#pragma unroll
  for (int p = 0; p < NA; ++p) {
    wb[p] = few_buffer(packed[p] + (int64_t)n0 * row_bytes, (uint32_t)have * row_bytes);
    sb[p] = few_buffer(scales[p] + (int64_t)n0 * scale_row_bytes, (uint32_t)have * scale_row_bytes);
  }
  uint32_t x_at[XV];
#pragma unroll
  for (int i = 0; i < XV; ++i) x_at[i] = (uint32_t)min(4 * i + g, m - 1) * (uint32_t)k * 2u + (uint32_t)nl * 16u;
  const few_rsrc_t xb = few_buffer(xp, (uint32_t)m * (uint32_t)k * 2u);
  struct Step {
    u32x4 x[XV];
    u32x4 w[NB][WV];
  };
  auto load_x = [&](Step& v, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XV; ++i) v.x[i] = few_load16(xb, x_at[i], (uint32_t)st * (kFewStep * 2u));
  };
  auto load_w = [&](Step& v, int b, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WV; ++i) v.w[b][i] = few_load16(wb[b / BP], w_at[b % BP] + (uint32_t)i * 64u, (uint32_t)st * (WV * 64u));
  };
  auto load = [&](Step& v, int st) __attribute__((always_inline)) {
    load_x(v, st);
#pragma unroll
    for (int b = 0; b < NB; ++b) load_w(v, b, st);
  };

  // ---- the wave's range of steps and its scales
  // (workgroups of an XCD start at different ranges: all on the same lines at a time is 10-15 % slower)
  const int range = (wave + (wg >> 3)) & (kFewWaves - 1);
  // (the first ranges are the longer ones: waves four apart share a SIMD, two long ones there are a step more)
  const int each = steps / kFewWaves, more = steps % kFewWaves;
  const int st0 = range * each + min(range, more), left = each + (range < more ? 1 : 0);
  constexpr int PER = WIDE ? 64 / SB : 4;        // steps of a load: a quarter of them on each of a column's four lanes
  constexpr int SL = WIDE ? kFewMaxSteps / PER : kFewMaxSteps / 4;
  char* const scale_patch = (char*)lds + kFewWaves * (4 * XV * kFewRowBytes) + wave * (NB * 16 * kFewScaleRow);
  struct Scales {
    u32x4 v[NB];
  };
  auto load_scales = [&](Scales& v, int from) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if constexpr (WIDE) {
        v.v[b] = few_load16(sb[b / BP], s_at[b % BP] + (uint32_t)g * 16u, (uint32_t)(st0 + from) * SB);
      } else {
        const uint32_t at = (uint32_t)(2 * (st0 + from + g)) >> group_shift;
        v.v[b].x = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sb[b / BP], (int)(s_at[b % BP] + at * 2u), 0, 0);
      }
    }
  };
  auto lay_scales = [&](const Scales& v, int from) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      char* const to = scale_patch + (b * 16 + nl) * kFewScaleRow;
      if constexpr (WIDE) *(u32x4*)(to + from * SB + g * 16) = v.v[b];
      else *(uint32_t*)(to + (from + g) * 4) = v.v[b].x | v.v[b].x << 16;
    }
  };

  // ---- what this thread stores in the end: four columns of a row.  Its first epilogue input.
  const int quads = (cols + 3) >> 2;
  const int orow = tid / quads, oc = (tid - orow * quads) * 4;
  const bool stores = orow < m && oc < have;
  const int64_t oat = (int64_t)orow * n + n0 + oc;
  float4_t prev = {0.f, 0.f, 0.f, 0.f};
  if constexpr (!PAIR) {
    if (pre_kind != FEW_PRE_NONE && stores) {
      const int64_t at = (int64_t)orow * pre_row + n0 + oc;
      if (vec && pre_kind == FEW_PRE_F16) {
        const half4_t h = *(const half4_t*)((const _Float16*)pre + at);
        prev = (float4_t){(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
      } else if (vec) {
        prev = *(const float4_t*)((const float*)pre + at);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int64_t e = at + min(i, have - 1 - oc);
          prev[i] = pre_kind == FEW_PRE_F16 ? (float)((const _Float16*)pre)[e] : ((const float*)pre)[e];
        }
      }
    }
  }

  char* const patch = (char*)lds + wave * (4 * XV * kFewRowBytes);
  float4_t acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = (float4_t){0.f, 0.f, 0.f, 0.f};
  // `next`: the step whose loads take the registers as they become free, or -1
  auto consume = [&](Step& v, int i_step, int next) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XV; ++i) *(u32x4*)(patch + (4 * i + g) * kFewRowBytes + nl * 16) = INT4 ? permute_x_for_int4(v.x[i]) : v.x[i];
    if (next >= 0) load_x(v, next);
    half8_t xa[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {  // int4 k = 32 s + 8 g; int8 k = 64 (s / 2) + 16 g + 8 (s % 2)
      const int unit = INT4 ? 4 * s + g : 8 * (s >> 1) + 2 * g + (s & 1);
      xa[s] = __builtin_bit_cast(half8_t, *(const u32x4*)(patch + (XV == 4 ? nl : nl & (4 * XV - 1)) * kFewRowBytes + unit * 16));
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      uint32_t word[4 * WV];
#pragma unroll
      for (int i = 0; i < WV; ++i) {
        word[4 * i + 0] = v.w[b][i].x;
        word[4 * i + 1] = v.w[b][i].y;
        word[4 * i + 2] = v.w[b][i].z;
        word[4 * i + 3] = v.w[b][i].w;
      }
      if (next >= 0) load_w(v, b, next);
      // a lane holds 32 k of its row, one group; afterwards word i is its eighth of group i
      if constexpr (INT4) transpose4(word[0], word[1], word[2], word[3]);
      uint32_t sc2[2] = {0u, 0u};  // int4: four group scales; int8: one per half step
      if constexpr (!ROW) {
        const char* const from = scale_patch + (b * 16 + nl) * kFewScaleRow + i_step * SB;
        sc2[0] = *(const uint32_t*)from;
        if constexpr (INT4) sc2[1] = *(const uint32_t*)(from + 4);
      }
      float4_t sum;  // a step's own sum first: the long one takes a step at a time
      if constexpr (INT4) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          half2_t h[4];
          unpack_int4_word(word[s], h);
          const float sc = half_bits_to_float((s & 1) ? sc2[s >> 1] >> 16 : sc2[s >> 1] & 0xffffu);
          const float4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[s], join8(h), (float4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) sum[r] = s == 0 ? sc * d[r] : fmaf(sc, d[r], sum[r]);
        }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            half2_t w[4];
            unpack_int8_word(word[4 * h + 2 * i], w);
            unpack_int8_word(word[4 * h + 2 * i + 1], w + 2);
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[2 * h + i], join8(w), d, 0, 0, 0);
          }
          const float sc = ROW ? 1.f : half_bits_to_float(h ? sc2[0] >> 16 : sc2[0] & 0xffffu);
#pragma unroll
          for (int r = 0; r < 4; ++r) sum[r] = h == 0 ? (ROW ? d[r] : sc * d[r]) : (ROW ? sum[r] + d[r] : fmaf(sc, d[r], sum[r]));
        }
      }
      acc[b] += sum;
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
    if constexpr (NB > 1) {
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

  // ---- the waves' sums and the epilogue
  lds_barrier();  // every wave has read its patch
  float* const sums = (float*)lds;  // [range][block][16 x 16]
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) sums[(range * NB + b) * 256 + (4 * g + r) * 16 + nl] = acc[b][r];
  lds_barrier();
  if (!stores) return;
  float4_t v[NA];
#pragma unroll
  for (int p = 0; p < NA; ++p) {
    // the columns of a quad lie in one block: block_cols is a multiple of four
    const int ob = oc / block_cols, c = oc - ob * block_cols;
    const float* from = sums + (p * BP + ob) * 256 + orow * 16 + c;
    float4_t s[kFewWaves];  // in pairs: a shorter chain, a smaller rounding error
#pragma unroll
    for (int w = 0; w < kFewWaves; ++w) s[w] = *(const float4_t*)(from + w * (NB * 256));
    v[p] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float f = factor;
      if constexpr (ROW) f *= ((const float*)scales[p])[n0 + min(oc + i, have - 1)];
      v[p][i] *= f;
    }
  }
  if constexpr (PAIR) {  // both rounded to f16, as the projections on their own would be
    half4_t h;
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = (_Float16)(apply_unary(a.unary, (float)(_Float16)v[0][i]) * (float)(_Float16)v[1][i]);
    if (vec) {
      *(half4_t*)((_Float16*)y + oat) = h;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (oc + i < have) ((_Float16*)y)[oat + i] = h[i];
    }
  } else {
    if (n_ops < 0) {
      v[0] += prev;
    } else if (n_ops > 0) {
      const DevEpilogue& ep = a.epi[pi];
      const int at = a.pre_at[pi];
      for (int s = 0; s < n_ops; ++s) {
        if (pre_kind != FEW_PRE_NONE && s == at) {
          const int op = ep.kind[s] == TLHIP_EPI_BIAS ? (int)TLHIP_BINARY_ADD : ep.unary[s];
          v[0] = op == TLHIP_BINARY_ADD ? v[0] + prev : (op == TLHIP_BINARY_SUB ? v[0] - prev : v[0] * prev);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int e = min(i, have - 1 - oc);
            v[0][i] = apply_epilogue_step(ep.kind[s], ep.unary[s], ep.input[s], ep.input_dtype[s], v[0][i], n0 + oc + e, oat + e);
          }
        }
      }
    }
    if (vec) {
      if (y_dtype == TLHIP_F16) *(half4_t*)((_Float16*)y + oat) = (half4_t){(_Float16)v[0][0], (_Float16)v[0][1], (_Float16)v[0][2], (_Float16)v[0][3]};
      else *(float4_t*)((float*)y + oat) = v[0];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (oc + i < have) store_out(y, y_dtype, oat + i, v[0][i]);
    }
  }
}

template <int FMT, bool WIDE, int XV, int KIND>
const void* few_instance_nb(int nb) {
  if constexpr (KIND != FEW_PAIR) {
    if (nb == 1) return (const void*)gemv_few_kernel<FMT, XV, 1, KIND, WIDE>;
    if (nb == 3) return (const void*)gemv_few_kernel<FMT, XV, 3, KIND, WIDE>;
  }
  if (nb == 2) return (const void*)gemv_few_kernel<FMT, XV, 2, KIND, WIDE>;
  if (nb == 4) return (const void*)gemv_few_kernel<FMT, XV, 4, KIND, WIDE>;
  if (nb == 6) return (const void*)gemv_few_kernel<FMT, XV, 6, KIND, WIDE>;
  return nullptr;
}
template <int FMT, bool WIDE, int XV>
const void* few_instance_kind(int nb, int kind) {
  return kind == FEW_SINGLE ? few_instance_nb<FMT, WIDE, XV, FEW_SINGLE>(nb)
         : kind == FEW_GROUP ? few_instance_nb<FMT, WIDE, XV, FEW_GROUP>(nb) : few_instance_nb<FMT, WIDE, XV, FEW_PAIR>(nb);
}
template <int FMT, bool WIDE>
const void* few_instance(int xv, int nb, int kind) {
  return xv == 1 ? few_instance_kind<FMT, WIDE, 1>(nb, kind) : (xv == 2 ? few_instance_kind<FMT, WIDE, 2>(nb, kind) : few_instance_kind<FMT, WIDE, 4>(nb, kind));
}

}  // namespace
}  // namespace tlhip
