// Decode GEMV of ONE activation row over packed weights with fused dequant.  Same contract and
// reference route as gemv.hip (src/backend/webgpu/matmul/gemv.ts:365-466).
//
// What bounds it: a launch of 1-3 MB is a chain of dependent steps (arguments, activations,
// barrier, weights, sums, store), each some hundred cycles, and a wave on its own issues a dependent
// VALU instruction every 8 cycles: instructions in the chain cost as much as memory does.  Hence:
//   * A lane keeps ITS chunks of the activations in registers (P chunks of 16 packed bytes, for
//     every row it works on) and all the weights of a row are one batch of loads, issued before the
//     activations are staged: no second trip to memory behind the barrier.
//   * The first epilogue input comes with the weights instead of behind the sum.
//   * A group's problem is selected between scalars, not read through an index.
//   * Sums over 32 and 64 lanes use the VALU's lane swaps instead of LDS.
// Everything else is as in gemv_kernel.h: exact integers in f16 (f32 activations: in f32), f32
// sums, the group's scale on a chunk's sum, activations (or what a prologue makes of them) staged
// once per workgroup, `kw` waves sharing a long row through LDS.
#pragma once
#include "device_utils.h"
#include "gemv_one_args.h"

namespace tlhip {
namespace {

// Sum over groups of 1 << shift consecutive lanes (16, 32 or 64), in every lane of the group.
__device__ __forceinline__ float lanes_sum(float v, int shift) {
  v = dpp_add<0xB1>(v);
  v = dpp_add<0x4E>(v);
  v = dpp_add<0x141>(v);
  v = dpp_add<0x140>(v);
  if (shift >= 5) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    v = as_float(r[0]) + as_float(r[1]);
  }
  if (shift >= 6) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    v = as_float(r[0]) + as_float(r[1]);
  }
  return v;
}

// The op's branch outside the loop over the values.
template <int N>
__device__ __forceinline__ void unary_all(int op, float (&v)[N]) {
  if (op == TLHIP_UNARY_SILU) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = apply_unary(TLHIP_UNARY_SILU, v[e]);
  } else if (op == TLHIP_UNARY_GELU_TANH) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = apply_unary(TLHIP_UNARY_GELU_TANH, v[e]);
  } else {
    for (int e = 0; e < N; ++e) v[e] = apply_unary(op, v[e]);
  }
}

// Sum of products of one 16-byte chunk with its activations, two chains.
template <int FMT, typename XT>
struct OneDot {
  static constexpr bool INT4 = FMT == TLHIP_FMT_INT4_GROUPED, F16 = sizeof(XT) == 2;
  static constexpr int NQ = (INT4 ? 32 : 16) * (int)sizeof(XT) / 16;  // 16-byte units of activations per chunk
  static __device__ __forceinline__ float of(const u32x4& w, const u32x4 (&x)[NQ]) {
    const uint32_t word[4] = {w.x, w.y, w.z, w.w};
    float d0 = 0.f, d1 = 0.f;
    if constexpr (F16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (INT4) {
          half2_t h[4];
          unpack_int4_word(word[i], h);
          d0 = __builtin_amdgcn_fdot2(h[0], as_half2(x[i].x), d0, false);
          d1 = __builtin_amdgcn_fdot2(h[1], as_half2(x[i].y), d1, false);
          d0 = __builtin_amdgcn_fdot2(h[2], as_half2(x[i].z), d0, false);
          d1 = __builtin_amdgcn_fdot2(h[3], as_half2(x[i].w), d1, false);
        } else {
          half2_t h[2];
          unpack_int8_word(word[i], h);
          const u32x4 xv = x[i / 2];
          d0 = __builtin_amdgcn_fdot2(h[0], as_half2((i & 1) ? xv.z : xv.x), d0, false);
          d1 = __builtin_amdgcn_fdot2(h[1], as_half2((i & 1) ? xv.w : xv.y), d1, false);
        }
      }
    } else {
      auto four = [&](float a, float b, float c, float d, const u32x4& xv) {
        d0 = fmaf(a, as_float(xv.x), d0);
        d1 = fmaf(b, as_float(xv.y), d1);
        d0 = fmaf(c, as_float(xv.z), d0);
        d1 = fmaf(d, as_float(xv.w), d1);
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (INT4) {
          float f[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) f[j] = (float)(((int)(word[i] << (28 - 4 * j))) >> 28);
          four(f[0], f[1], f[2], f[3], x[2 * i]);
          four(f[4], f[5], f[6], f[7], x[2 * i + 1]);
        } else {
          four((float)(int8_t)(word[i] & 0xffu), (float)(int8_t)((word[i] >> 8) & 0xffu), (float)(int8_t)((word[i] >> 16) & 0xffu),
               (float)(int8_t)(word[i] >> 24), x[i]);
        }
      }
    }
    return d0 + d1;
  }
};

// Scalars that are to be in registers from here on: arguments read where they are first used are a
// trip to memory each, one behind the other.
template <typename T>
__device__ __forceinline__ void in_register(T v) {
  asm volatile("" ::"s"(v));
}
template <typename... Ts>
__device__ __forceinline__ void in_registers(const Ts&... v) {
  (in_register(v), ...);
}

// P: chunks of a row per lane.  XS: 16-byte units of activations a thread stages at a time, one or two
// where those are all.  PRO: the prologue (f16 activations only).  KIND: see OneArgs.
template <int FMT, typename XT, int P, int XS, int PRO, int KIND>
__global__ __launch_bounds__(512) void gemv_one_kernel(const OneArgs<KIND> a) {
  using Dot = OneDot<FMT, XT>;
  constexpr int NQ = Dot::NQ, NP = OneArgs<KIND>::NP;
  constexpr bool GROUPED = FMT != TLHIP_FMT_INT8_ROW, PAIR = KIND == ONE_PAIR, GROUP = KIND == ONE_GROUP;
  constexpr bool PERMUTE = FMT == TLHIP_FMT_INT4_GROUPED && sizeof(XT) == 2;
  constexpr bool ALL = XS < 4;  // one round stages everything
  constexpr int NA = PAIR ? 2 : 1;
  extern __shared__ u32x4 lds[];
  __shared__ float4_t red[2];  // a sum of squares per wave

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T = a.threads, nchunks = a.nchunks, lpr_shift = a.lpr_shift, kw_shift = a.kw_shift, cpg_shift = a.cpg_shift;
  const int groups_per_row = a.groups_per_row, rows_per_wg = a.rows_per_wg, y_dtype = a.y_dtype, wg = (int)blockIdx.x;
  const float factor = a.factor;
  const void *xp = a.x, *const operand = a.operand;

  // ---- this workgroup's problem, selected between scalars
  int first = 0, last = a.first[GROUP ? 1 : NP], rounds = a.rounds[0], longer = a.longer[0], n = a.n[0], pre_kind = a.pre_kind[0];
  int n_ops = a.n_ops[0], pi = 0;
  const u32x4* packed[NA] = {a.packed[0]};
  const void* scales[NA] = {a.scales[0]};
  const void* pre = a.pre[0];
  void* y = a.y[0];
  if constexpr (GROUP) {
#pragma unroll
    for (int j = 0; j < NP; ++j)
      in_registers(a.first[j + 1], a.rounds[j], a.longer[j], a.n[j], a.pre_kind[j], a.n_ops[j], a.packed[j], a.scales[j], a.pre[j], a.y[j]);
    in_registers(a.own_x, a.count);
  }
  if constexpr (PAIR) {
    packed[1] = a.packed[1];
    scales[1] = a.scales[1];
    in_registers(packed[1], scales[1], a.unary);
  }
  in_registers(T, nchunks, lpr_shift, kw_shift, cpg_shift, groups_per_row, rows_per_wg, y_dtype, factor, xp, operand, first, last, rounds,
               longer, n, pre_kind, n_ops, packed[0], scales[0], pre, y);
  if constexpr (PRO == TLHIP_PRO_RMSNORM) in_registers(a.k, a.eps);
  if constexpr (PRO == TLHIP_PRO_GATED_MUL) in_registers(a.unary);
  if constexpr (GROUP) {
    if (a.own_x)
#pragma unroll
      for (int j = 1; j < NP; ++j)
        if (j < a.count && wg >= a.first[j]) xp = a.xs[j];
  }

  // ---- the first activation loads: units of 16 bytes, one a thread and round, the last one again past
  // the end (every load in front of the weights is unconditional, so that the waits count them exactly)
  const int units = nchunks * NQ;
  const u32x4* const xg = (const u32x4*)xp;
  u32x4 xr[XS], ur[XS], nw[XS][2];
  auto issue_x = [&](int base) {
#pragma unroll
    for (int i = 0; i < XS; ++i) {
      const uint32_t u = (uint32_t)min(base + i * T + tid, units - 1);
      xr[i] = xg[u];
      if constexpr (PRO == TLHIP_PRO_GATED_MUL) ur[i] = ((const u32x4*)operand)[u];
      if constexpr (PRO == TLHIP_PRO_RMSNORM) {
        nw[i][0] = ((const u32x4*)operand)[2 * u];
        nw[i][1] = ((const u32x4*)operand)[2 * u + 1];
      }
    }
  };
  issue_x(0);

  if constexpr (GROUP) {
#pragma unroll
    for (int j = 1; j < NP; ++j) {
      const bool here = j < a.count && wg >= a.first[j];
      first = here ? a.first[j] : first;
      last = here ? a.first[j + 1] : last;
      rounds = here ? a.rounds[j] : rounds;
      longer = here ? a.longer[j] : longer;
      n = here ? a.n[j] : n;
      pre_kind = here ? a.pre_kind[j] : pre_kind;
      n_ops = here ? a.n_ops[j] : n_ops;
      packed[0] = here ? a.packed[j] : packed[0];
      scales[0] = here ? a.scales[j] : scales[0];
      pre = here ? a.pre[j] : pre;
      y = here ? a.y[j] : y;
      pi = here ? j : pi;
    }
  }
  const int bid = wg - first, nblk = last - first;

  // ---- a row's weights: P chunks a lane
  const int lpr = 1 << lpr_shift, kw = 1 << kw_shift;
  const int sub = lane >> lpr_shift, lj = lane & (lpr - 1);
  const int kwi = wave & (kw - 1);
  const int row_in_wg = (wave >> kw_shift) * (64 >> lpr_shift) + sub;
  int cc[P], xc[P];
  bool in[P];
#pragma unroll
  for (int j = 0; j < P; ++j) {  // past the row's end: its last chunk again, times activations of zero (and a scale of zero)
    const int c = (kwi * P + j) * lpr + lj;
    in[j] = c < nchunks;
    cc[j] = min(c, nchunks - 1);
    xc[j] = min(c, nchunks);
  }
  struct Batch {
    u32x4 w[NA][P];
    uint16_t s[NA][P];
    float rs[NA];
    uint32_t pre;
  };
  auto load_batch = [&](Batch& b, int rb) {
    const int row = min(rb * rows_per_wg + row_in_wg, n - 1);  // rows past the end: the last again, not stored
    if constexpr (!PAIR) {
      if (pre_kind == ONE_PRE_F16) b.pre = ((const uint16_t*)pre)[row];
      else if (pre_kind == ONE_PRE_F32) b.pre = ((const uint32_t*)pre)[row];
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
#pragma unroll
      for (int j = 0; j < P; ++j) {
        b.w[i][j] = __builtin_nontemporal_load(packed[i] + (int64_t)row * nchunks + cc[j]);
        if constexpr (GROUPED) b.s[i][j] = ((const uint16_t*)scales[i])[(int64_t)row * groups_per_row + (cc[j] >> cpg_shift)];
      }
      if constexpr (!GROUPED) b.rs[i] = ((const float*)scales[i])[row];
    }
  };
  int rb = bid;
  Batch cur, other;
  load_batch(cur, rb);

  // ---- staging: unit q of chunk c at q * stride + c, so that lanes on consecutive chunks read
  // consecutive units (a thread's neighbours write to other banks).  A thread past the last unit writes it
  // again, the same value.  Behind the last chunk one of zeros for the lanes past the row's end: a scale of zero alone
  // leaves NaN where the last chunk's sum is infinite, and a select behind every sum is up to 10 % of a launch.
  const uint32_t stride = (uint32_t)nchunks + 1;
  if (tid < NQ) lds[tid * stride + (uint32_t)nchunks] = (u32x4){0u, 0u, 0u, 0u};
  auto place = [&](int u) {
    const uint32_t c = (uint32_t)u / NQ, q = (uint32_t)u % NQ;
    return lds + q * stride + c;
  };
  if constexpr (PRO == TLHIP_PRO_RMSNORM) {
    float ss = 0.f;
    auto squares = [&](int base) {
#pragma unroll
      for (int i = 0; i < XS; ++i) {
        float f[8];
        unit_to_floats<_Float16>(xr[i], f);
        float s0 = f[0] * f[0], s1 = f[1] * f[1];
#pragma unroll
        for (int e = 2; e < 8; e += 2) {
          s0 = fmaf(f[e], f[e], s0);
          s1 = fmaf(f[e + 1], f[e + 1], s1);
        }
        ss += base + i * T + tid < units ? s0 + s1 : 0.f;
      }
    };
    squares(0);
    if constexpr (!ALL)
      for (int base = XS * T; base < units; base += XS * T) {
        issue_x(base);
        squares(base);
      }
    ss = lanes_sum(ss, 6);
    if (lane == 0) ((float*)red)[wave] = ss;
    lds_barrier();
    const float4_t r0 = red[0];
    float t = (r0[0] + r0[1]) + (r0[2] + r0[3]);  // four or eight waves
    if (T > 256) {
      const float4_t r1 = red[1];
      t += (r1[0] + r1[1]) + (r1[2] + r1[3]);
    }
    const float inv = 1.f / sqrtf(t / (float)a.k + a.eps);
    auto norm = [&](int base) {
#pragma unroll
      for (int i = 0; i < XS; ++i) {
        float f[8];
        unit_to_floats<_Float16>(xr[i], f);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f[4 * h + 0] = (f[4 * h + 0] * inv) * as_float(nw[i][h].x);
          f[4 * h + 1] = (f[4 * h + 1] * inv) * as_float(nw[i][h].y);
          f[4 * h + 2] = (f[4 * h + 2] * inv) * as_float(nw[i][h].z);
          f[4 * h + 3] = (f[4 * h + 3] * inv) * as_float(nw[i][h].w);
        }
        u32x4 v = floats_to_unit<_Float16>(f);
        if constexpr (PERMUTE) v = permute_x_for_int4(v);
        *place(min(base + i * T + tid, units - 1)) = v;
      }
    };
    if (ALL || units <= XS * T) {
      norm(0);  // still in registers
    } else {
      for (int base = 0; base < units; base += XS * T) {
        issue_x(base);
        norm(base);
      }
    }
  } else {
    auto stage = [&](int base) {
#pragma unroll
      for (int i = 0; i < XS; ++i) {
        u32x4 v = xr[i];
        if constexpr (PRO == TLHIP_PRO_GATED_MUL) {
          float g[8], up[8];
          unit_to_floats<_Float16>(v, g);
          unit_to_floats<_Float16>(ur[i], up);
          unary_all(a.unary, g);
#pragma unroll
          for (int e = 0; e < 8; ++e) g[e] *= up[e];
          v = floats_to_unit<_Float16>(g);
        }
        if constexpr (PERMUTE) v = permute_x_for_int4(v);
        *place(min(base + i * T + tid, units - 1)) = v;
      }
    };
    stage(0);
    if constexpr (!ALL)
      for (int base = XS * T; base < units; base += XS * T) {
        issue_x(base);
        stage(base);
      }
  }
  lds_barrier();
  u32x4 x[P][NQ];
#pragma unroll
  for (int j = 0; j < P; ++j)
#pragma unroll
    for (int q = 0; q < NQ; ++q) x[j][q] = lds[q * stride + (uint32_t)xc[j]];
  float* const partial = (float*)(lds + stride * NQ);  // [kw][row][NA]

  auto consume = [&](const Batch& b, int rb) {
    float acc[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      acc[i] = 0.f;
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const float d = Dot::of(b.w[i][j], x[j]);
        if constexpr (GROUPED) acc[i] = fmaf(in[j] ? half_bits_to_float(b.s[i][j]) : 0.f, d, acc[i]);
        else acc[i] += d;
        if constexpr (sizeof(XT) == 4) __builtin_amdgcn_sched_barrier(0);  // one chunk's 32 floats at a time
      }
      acc[i] = lanes_sum(acc[i], lpr_shift);
    }
    if (kw > 1) {
      lds_barrier();
      if (lj == 0)
#pragma unroll
        for (int i = 0; i < NA; ++i) partial[(kwi * rows_per_wg + row_in_wg) * NA + i] = acc[i];
      lds_barrier();
      if (kwi == 0 && lj == 0)
        for (int w = 1; w < kw; ++w)
#pragma unroll
          for (int i = 0; i < NA; ++i) acc[i] += partial[(w * rows_per_wg + row_in_wg) * NA + i];
    }
    const int row = rb * rows_per_wg + row_in_wg;
    if (kwi != 0 || lj != 0 || row >= n) return;
    float v[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) v[i] = acc[i] * (GROUPED ? factor : b.rs[i] * factor);
    if constexpr (PAIR) {  // both rounded to f16, as the projections on their own would be
      const float g = apply_unary(a.unary, (float)(_Float16)v[0]);
      ((_Float16*)y)[row] = (_Float16)(g * (float)(_Float16)v[1]);
    } else {
      if (n_ops > 0) {
        const DevEpilogue& ep = a.epi[pi];
        const int at = a.pre_at[pi];
        const float o = pre_kind == ONE_PRE_F32 ? as_float(b.pre) : half_bits_to_float(b.pre);
        for (int i = 0; i < n_ops; ++i) {
          if (pre_kind != ONE_PRE_NONE && i == at) {
            const int op = ep.kind[i] == TLHIP_EPI_BIAS ? (int)TLHIP_BINARY_ADD : ep.unary[i];
            v[0] = op == TLHIP_BINARY_ADD ? v[0] + o : (op == TLHIP_BINARY_SUB ? v[0] - o : v[0] * o);
          } else {
            v[0] = apply_epilogue_step(ep.kind[i], ep.unary[i], ep.input[i], ep.input_dtype[i], v[0], row, row);
          }
        }
      } else if (n_ops < 0) {  // a bias or a residual, and nothing else
        v[0] += pre_kind == ONE_PRE_F32 ? as_float(b.pre) : half_bits_to_float(b.pre);
      }
      store_out(y, y_dtype, row, v[0]);
    }
  };

  // Rows of this workgroup, `nblk` row blocks apart; the next batch is loaded before the current one
  // is consumed, and every load in the loop is unconditional.
  int left = rounds + (bid < longer ? 1 : 0);
  while (left >= 3) {
    load_batch(other, rb + nblk);
    consume(cur, rb);
    rb += nblk;
    load_batch(cur, rb + nblk);
    consume(other, rb);
    rb += nblk;
    left -= 2;
  }
  if (left == 2) {
    load_batch(other, rb + nblk);
    consume(cur, rb);
    consume(other, rb + nblk);
  } else if (left == 1) {
    consume(cur, rb);
  }
}

template <int FMT, typename XT, int XS, int PRO, int KIND>
const void* one_instance_p(int p) {
  // at most 96 registers of activations
  constexpr int NQ = OneDot<FMT, XT>::NQ;
  if (p == 1) return (const void*)gemv_one_kernel<FMT, XT, 1, XS, PRO, KIND>;
  if (p == 2) return (const void*)gemv_one_kernel<FMT, XT, 2, XS, PRO, KIND>;
  if (p == 3) return (const void*)gemv_one_kernel<FMT, XT, 3, XS, PRO, KIND>;
  if constexpr (NQ <= 4) {
    if (p == 4) return (const void*)gemv_one_kernel<FMT, XT, 4, XS, PRO, KIND>;
    if constexpr (KIND != ONE_PAIR) {  // (two weights' batches as well: spills)
      if (p == 5) return (const void*)gemv_one_kernel<FMT, XT, 5, XS, PRO, KIND>;
      if (p == 6) return (const void*)gemv_one_kernel<FMT, XT, 6, XS, PRO, KIND>;
    }
  }
  return nullptr;
}

template <int FMT, typename XT, int PRO, int KIND>
const void* one_instance_x(int p, int units) {
  return units == 1 ? one_instance_p<FMT, XT, 1, PRO, KIND>(p) : (units == 2 ? one_instance_p<FMT, XT, 2, PRO, KIND>(p) : one_instance_p<FMT, XT, 4, PRO, KIND>(p));
}

template <int FMT>
const void* one_instance(int x_dtype, int p, int units, int prologue, int kind) {
  if (x_dtype == TLHIP_F32)
    return prologue == TLHIP_PRO_NONE && kind == ONE_SINGLE ? one_instance_x<FMT, float, TLHIP_PRO_NONE, ONE_SINGLE>(p, units) : nullptr;
  if (kind == ONE_PAIR) return prologue == TLHIP_PRO_NONE ? one_instance_x<FMT, _Float16, TLHIP_PRO_NONE, ONE_PAIR>(p, units) : nullptr;
  if (kind == ONE_SINGLE) {
    if (prologue == TLHIP_PRO_RMSNORM) return one_instance_x<FMT, _Float16, TLHIP_PRO_RMSNORM, ONE_SINGLE>(p, units);
    if (prologue == TLHIP_PRO_GATED_MUL) return one_instance_x<FMT, _Float16, TLHIP_PRO_GATED_MUL, ONE_SINGLE>(p, units);
    return one_instance_x<FMT, _Float16, TLHIP_PRO_NONE, ONE_SINGLE>(p, units);
  }
  if (prologue == TLHIP_PRO_RMSNORM) return one_instance_x<FMT, _Float16, TLHIP_PRO_RMSNORM, ONE_GROUP>(p, units);
  if (prologue == TLHIP_PRO_GATED_MUL) return one_instance_p<FMT, _Float16, 4, TLHIP_PRO_GATED_MUL, ONE_GROUP>(p);
  return one_instance_x<FMT, _Float16, TLHIP_PRO_NONE, ONE_GROUP>(p, units);
}

}  // namespace
}  // namespace tlhip
