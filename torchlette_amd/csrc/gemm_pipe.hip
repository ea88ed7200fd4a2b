// Prefill GEMM over packed weights, third form: Y[M,N] = epilogue(alpha * X[M,K] * W[N,K]^T)
// for launches that fill the chip with tiles.  Same contract and reference route as
// gemm_prefill.hip (src/backend/webgpu/ops/matmul-ops.ts:163-181;
// src/schedule/matmul-skeleton.ts:738-966).
//
// What bounds it: the matrix cores and, next to them, LDS.  Per step of 64 k a workgroup of
// eight waves
//   * brings its X tile into LDS without registers (global_load_lds_dwordx4, two steps
//     ahead, three buffers; the XOR swizzle of the 16-byte units is applied by which unit a
//     lane fetches, so a row of a wave's request is still one whole 128-byte line);
//   * dequantises its W tile ONCE (the form in gemm_direct.hip does it in every wave that
//     needs the column: twice to eight times per workgroup) from registers loaded two steps
//     ahead into f16 LDS tiles, two buffers, one rounding of q * scale as there;
//   * multiplies with v_mfma_f32_16x16x32_f16 (2.44 PFLOP/s in a pure-MFMA loop on data,
//     where 32x32x16 holds 2.2: the chip clocks down less).
// The two waves of a SIMD belong to different halves of the workgroup, which run one phase
// apart ("ping-pong"): while one wave issues the MFMAs of 32 k from registers, the other
// reads its next operands from LDS, dequantises and issues loads; every phase ends with a
// workgroup barrier, so the matrix pipe of a SIMD always has one wave's whole block of
// MFMAs queued and neither wave waits for LDS inside it.
#include <cstring>
#include <type_traits>
#include <utility>

#include "gemm_common.h"

namespace tlhip {
namespace {

constexpr int PK = 64;     // k per step
constexpr int UPR = 8;     // 16-byte units of an LDS row (64 f16)
enum { PIPE_INT4 = 0, PIPE_INT8 = 1, PIPE_INT8_ROW = 2 };

struct PipeArgs {
  const uint8_t* packed;
  const uint16_t* scales;  // f16 bits, groups_per_row per row (not PIPE_INT8_ROW)
  const _Float16* x;
  int m, n, k;
  int w_row_bytes;
  int group_shift;         // log2(group size / 32)
  int groups_per_row;
  int ksteps;              // K / 64
  int ksplit;              // workgroups that share a tile, each walking a slice of the steps (1 = none)
  float* workspace;        // ksplit > 1: the slices' partial sums, [slice][M][N] f32
  TileMap map;
  OutArgs out;
};

// 16 bytes a lane from global memory to LDS at lds_byte + 16 * lane.  Written out because the
// compiler, given the builtin, waits for every such load before any later LDS read.
__device__ __forceinline__ void load_to_lds(uint32_t lds_byte, uint32_t offset, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_byte), "v"(offset), "s"(base) : "memory");
}
// Loads whose wait is counted by hand (wait_loads): the compiler does not know that the
// registers fill later, so a value goes from its load to its wait as one whole operand and
// nothing touches it in between.
__device__ __forceinline__ void load_packed(u32x4& v, uint32_t offset, const void* base) {
  asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(offset), "s"(base));
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void load_packed(u32x2& v, uint32_t offset, const void* base) {
  asm volatile("global_load_dwordx2 %0, %1, %2" : "=v"(v) : "v"(offset), "s"(base));
}
__device__ __forceinline__ void load_scale(uint32_t& v, uint32_t offset, const void* base) {
  asm volatile("global_load_ushort %0, %1, %2" : "=v"(v) : "v"(offset), "s"(base));
}

// One step's share of the packed W tile of a thread: WORDS words of weights and their scale.
template <int WORDS>
struct WRegs {
  typedef std::conditional_t<WORDS == 2, u32x2, u32x4> Vec;
  Vec v[WORDS == 8 ? 2 : 1];
  uint32_t scale;
  __device__ __forceinline__ uint32_t word(int i) const { return v[i >> 2][i & 3]; }
};

// At most N of the wave's global loads are still in flight behind this.
template <int N, int WORDS>
__device__ __forceinline__ void wait_loads(WRegs<WORDS>& r) {
  if constexpr (WORDS == 8) asm volatile("s_waitcnt vmcnt(%c3)" : "+v"(r.v[0]), "+v"(r.v[1]), "+v"(r.scale) : "n"(N));
  else asm volatile("s_waitcnt vmcnt(%c2)" : "+v"(r.v[0]), "+v"(r.scale) : "n"(N));
}

// The ROWS x COLS block of one wave in its LDS patch (rows of COLS + 4 floats) to the output:
// alpha (and the column factors of int8 per row), the chain, the store.  Small loops for every
// block: the same written out per block was 57 000 lines of assembly, and a tile's end waited
// for its own code (a 256 x 256 tile of two steps: 20 us).
// vec_ok (N a multiple of 8, y and every input of the chain 16-byte aligned): eight columns a
// lane, 16-byte pieces.
template <int ROWS, int COLS, bool COLSCALE>
__device__ __forceinline__ void store_block8(const float* patch, int lane, int row0, int col0, const OutArgs& o, float* plane) {
  constexpr int PW = COLS + 4;
  constexpr int LPR = COLS / 8;  // lanes per row
  constexpr int RPP = 64 / LPR;  // rows per pass (48 columns: 10 rows on 60 lanes)
  constexpr int PASSES = (ROWS + RPP - 1) / RPP;
  const int rr0 = lane / LPR, cc = (lane % LPR) * 8;
  const int col = col0 + cc;
  if (rr0 >= RPP || col >= o.n) return;
  const bool bare = plane != nullptr;
  const bool f16 = !bare && o.y_dtype == TLHIP_F16;
  const int n_ops = bare ? 0 : o.epi.n_ops;
  // a leading bias needs no loads in the loop: the lane's columns are the same in every row
  const int first = n_ops > 0 && o.epi.kind[0] == TLHIP_EPI_BIAS ? 1 : 0;
  float scale[8], bias[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    scale[e] = bare ? 1.f : (COLSCALE ? o.alpha * o.col_scale[col + e] : o.alpha);
    bias[e] = !first ? 0.f : (o.epi.input_dtype[0] == TLHIP_F16 ? (float)((const _Float16*)o.epi.input[0])[col + e] : ((const float*)o.epi.input[0])[col + e]);
  }
#pragma unroll 1
  for (int p = 0; p < PASSES; ++p) {
    const int rr = p * RPP + rr0, row = row0 + rr;
    if (rr >= ROWS || row >= o.m) break;
    const float4_t a = *(const float4_t*)(patch + rr * PW + cc), b = *(const float4_t*)(patch + rr * PW + cc + 4);
    float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    const int64_t idx = (int64_t)row * o.n + col;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = v[e] * scale[e] + bias[e];
#pragma unroll
    for (int i = 0; i < TLHIP_MAX_EPILOGUE_OPS; ++i) {
      if (i < first || i >= n_ops) continue;
      const int kind = o.epi.kind[i];
      if (kind == TLHIP_EPI_UNARY) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = apply_unary(o.epi.unary[i], v[e]);
      } else if (kind == TLHIP_EPI_CAST_F16) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (float)(_Float16)v[e];
      } else if (kind != TLHIP_EPI_NONE) {
        const int64_t at = kind == TLHIP_EPI_BIAS ? col : idx;
        float w[8];
        if (o.epi.input_dtype[i] == TLHIP_F16) {
          const half8_t h = *(const half8_t*)((const _Float16*)o.epi.input[i] + at);
#pragma unroll
          for (int e = 0; e < 8; ++e) w[e] = (float)h[e];
        } else {
          const float4_t lo = *(const float4_t*)((const float*)o.epi.input[i] + at), hi = *(const float4_t*)((const float*)o.epi.input[i] + at + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = lo[e], w[4 + e] = hi[e];
        }
        const int op = kind == TLHIP_EPI_BIAS ? (int)TLHIP_BINARY_ADD : o.epi.unary[i];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = op == TLHIP_BINARY_ADD ? v[e] + w[e] : (op == TLHIP_BINARY_SUB ? v[e] - w[e] : v[e] * w[e]);
      }
    }
    if (f16) {
      half8_t h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = (_Float16)v[e];
      __builtin_nontemporal_store(h, (half8_t*)((_Float16*)o.y + idx));
    } else {
      float* dst = (bare ? plane : (float*)o.y) + idx;
      __builtin_nontemporal_store((float4_t){v[0], v[1], v[2], v[3]}, (float4_t*)dst);
      __builtin_nontemporal_store((float4_t){v[4], v[5], v[6], v[7]}, (float4_t*)(dst + 4));
    }
  }
}

// Any N and any alignment: one column a lane, four rows at a time.
template <int ROWS, int COLS, bool COLSCALE>
__device__ __forceinline__ void store_block1(const float* patch, int lane, int row0, int col0, const OutArgs& o, float* plane) {
  constexpr int PW = COLS + 4;
  const bool bare = plane != nullptr;
  const int n_ops = bare ? 0 : o.epi.n_ops;
  const int lrow = COLS <= 32 ? lane / 32 : 0, rpp = COLS <= 32 ? 2 : 1;  // two rows of 32 columns side by side
  const int cc = COLS <= 32 ? lane % 32 : lane, col = col0 + cc;
  if (cc >= COLS || col >= o.n) return;
  const float scale = bare ? 1.f : (COLSCALE ? o.alpha * o.col_scale[col] : o.alpha);
#pragma unroll 1
  for (int r = lrow; r < ROWS && row0 + r < o.m; r += 4 * rpp) {
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int rr = r + q * rpp;  // ROWS is a multiple of 8; rows past M load the last row's inputs and are not stored
      const int64_t idx = (int64_t)min(row0 + rr, o.m - 1) * o.n + col;
      v[q] = patch[rr * PW + cc] * scale;
#pragma unroll
      for (int i = 0; i < TLHIP_MAX_EPILOGUE_OPS; ++i)
        if (i < n_ops) v[q] = apply_epilogue_step(o.epi.kind[i], o.epi.unary[i], o.epi.input[i], o.epi.input_dtype[i], v[q], col, idx);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = row0 + r + q * rpp;
      if (row < o.m) {
        if (bare) plane[(int64_t)row * o.n + col] = v[q];
        else store_out(o.y, o.y_dtype, (int64_t)row * o.n + col, v[q]);
      }
    }
  }
}

// WM x WN waves; BM x BN outputs; a wave owns TM x TN MFMA tiles of 16 x 16.
template <int BM, int BN, int WM, int WN, int F>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_pipe_kernel(const PipeArgs a) {
  static_assert(WM * WN == 8, "eight waves: two per SIMD, one of each half");
  constexpr int THREADS = 512;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  static_assert(TM % 2 == 0 && BM % 64 == 0 && BN % 64 == 0, "whole patches of 32 rows");
  constexpr int NX = BM / 64;              // X loads of a wave per step (1 KB each)
  constexpr int UW = BN > 128 ? 4 : 2;     // units of 8 weights a thread dequantises per step
  constexpr int TPR = UPR / UW;            // threads per weight row
  constexpr bool W_PART = THREADS / TPR != BN;  // more threads than weights: the rest idle
  constexpr int WORDS = F == PIPE_INT4 ? UW : 2 * UW;
  constexpr int UB = WORDS * 4;            // packed bytes of a thread per step
  constexpr int STEP_BYTES = F == PIPE_INT4 ? PK / 2 : PK;
  constexpr int NW = (WORDS + 3) / 4 + (F == PIPE_INT8_ROW ? 0 : 1);  // W loads of a wave per step
  constexpr uint32_t X_BYTES = BM * 128, W_BYTES = BN * 128;
  extern __shared__ u32x4 lds[];  // three X buffers, two W buffers

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int l16 = lane & 15, lg = lane >> 4;

  const int slice = a.ksplit > 1 ? (int)(blockIdx.x % (unsigned)a.ksplit) : 0;
  const int tile_id = a.ksplit > 1 ? (int)(blockIdx.x / (unsigned)a.ksplit) : (int)blockIdx.x;
  const int nsteps = a.ksteps / a.ksplit;
  const int step0 = slice * nsteps;
  int tm_idx, tn_idx;
  if (!tile_of(a.map, tile_id, tm_idx, tn_idx)) return;  // padding of the tile map (whole workgroup)
  const int m0 = tm_idx * BM, n0 = tn_idx * BN;

  // ---- X: global -> LDS ----------------------------------------------------------------
  // load i of a wave: rows 8 * (wave * NX + i) .. + 7, one 128-byte line each; lane l brings
  // unit (l % 8) ^ f(row) of its row to position l % 8, f(row) = (row / 2) % 8
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)(void*)lds;
  uint32_t xoff[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int r = (wave * NX + i) * 8 + (lane >> 3);
    const int rc = min(r, a.m - 1 - m0);
    xoff[i] = (uint32_t)rc * (uint32_t)(a.k * 2) + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
  }
  const char* const x_tile = (const char*)(a.x + (size_t)m0 * a.k) + (size_t)step0 * (PK * 2);
  auto load_x = [&](int step, uint32_t buf, int from, int to) {
    const char* base = x_tile + (size_t)min(step, nsteps - 1) * (PK * 2);  // past the end: a harmless reload
#pragma unroll
    for (int i = from; i < to; ++i) load_to_lds(buf + (uint32_t)(wave * NX + i) * 1024u, xoff[i], base);
  };

  // ---- W: global -> registers -> f16 in LDS ----------------------------------------------
  const int wr = tid / TPR, wp = tid % TPR;
  const int wrc = min(min(wr, BN - 1), a.n - 1 - n0);
  const uint32_t woff = (uint32_t)wrc * (uint32_t)a.w_row_bytes + (uint32_t)(wp * UB);
  const uint32_t soff = (uint32_t)wrc * (uint32_t)(a.groups_per_row * 2);
  const char* const w_tile = (const char*)a.packed + (size_t)n0 * a.w_row_bytes + (size_t)step0 * STEP_BYTES;
  const char* const s_tile = (const char*)a.scales + (size_t)n0 * a.groups_per_row * 2;
  typedef WRegs<WORDS> Regs;
  auto load_w = [&](int step, Regs& r) {
    const int st = min(step, nsteps - 1);
    const char* base = w_tile + (size_t)st * STEP_BYTES;
    load_packed(r.v[0], woff, base);
    if constexpr (WORDS == 8) load_packed(r.v[1], woff + 16u, base);
    if constexpr (F != PIPE_INT8_ROW) {
      const int g = ((step0 + st) * 2 + (wp * UW) / 4) >> a.group_shift;
      load_scale(r.scale, soff + (uint32_t)g * 2u, s_tile);
    } else {
      r.scale = 0;
    }
  };
  // units u0, u0 + 1 of the thread's share, to W buffer `buf` (a u32x4 index into lds)
  const int wf = (wr >> 1) & 7;
  auto dequant = [&](const Regs& r, int buf, int u0, int count) {
    const half2_t s2 = {__builtin_bit_cast(_Float16, (uint16_t)r.scale), __builtin_bit_cast(_Float16, (uint16_t)r.scale)};
#pragma unroll
    for (int u = u0; u < u0 + count; ++u) {
      half2_t h[4];
      u32x4 unit;
      if constexpr (F == PIPE_INT4) {
        unpack_int4_word(r.word(u), h);  // pairs (k0,k4) (k1,k5) (k2,k6) (k3,k7)
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = h[e] * s2;
        const uint32_t p0 = __builtin_bit_cast(uint32_t, h[0]), p1 = __builtin_bit_cast(uint32_t, h[1]);
        const uint32_t p2 = __builtin_bit_cast(uint32_t, h[2]), p3 = __builtin_bit_cast(uint32_t, h[3]);
        unit.x = __builtin_amdgcn_perm(p1, p0, 0x05040100u);  // (k0, k1)
        unit.y = __builtin_amdgcn_perm(p3, p2, 0x05040100u);  // (k2, k3)
        unit.z = __builtin_amdgcn_perm(p1, p0, 0x07060302u);  // (k4, k5)
        unit.w = __builtin_amdgcn_perm(p3, p2, 0x07060302u);  // (k6, k7)
      } else {
        unpack_int8_word(r.word(2 * u), h);
        unpack_int8_word(r.word(2 * u + 1), h + 2);
        if constexpr (F == PIPE_INT8) {
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = h[e] * s2;
        }
        unit.x = __builtin_bit_cast(uint32_t, h[0]);
        unit.y = __builtin_bit_cast(uint32_t, h[1]);
        unit.z = __builtin_bit_cast(uint32_t, h[2]);
        unit.w = __builtin_bit_cast(uint32_t, h[3]);
      }
      if (!W_PART || wr < BN) lds[buf + wr * UPR + ((wp * UW + u) ^ wf)] = unit;
    }
  };

  // ---- operands ---------------------------------------------------------------------------
  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
  half8_t af[TM], bf[TN];
  const int frag = lg ^ ((l16 >> 1) & 7);  // unit of k group lg in a row's swizzled order; kk = 1: the other four
  const int a_row = (wm * TM * 16 + l16) * UPR, b_row = (wn * TN * 16 + l16) * UPR;

  // Buffers by index into lds (16-byte units); X: 0, 1, 2, then W: 0, 1
  constexpr int XU = X_BYTES / 16, WU = W_BYTES / 16;
  constexpr int DEQUANT_OPS = (F == PIPE_INT4 ? 20 : 16) * UW / 2;
  constexpr int VALU_PER_MFMA = (DEQUANT_OPS + TM * TN - 1) / (TM * TN);

  int xb = 0;   // X buffer of the step being multiplied
  int wb = 0;   // W buffer of it
  // One phase of loading: the operands of k half kk of step s.  In the first half the wave also
  // dequantises half of its share of W(s+1) and does not wait for anything (its MFMAs wait for
  // their operands one by one); in the second half it issues the loads of X two steps ahead and
  // of W three steps ahead and leaves only those in flight: X of the next step, W of the one
  // after and its own LDS accesses are done, so that behind the barrier every buffer of the
  // step before may be written.
  auto load_phase = [&](int s, int kk, Regs& next, Regs& later) {
    const u32x4* xs = lds + xb * XU + a_row + (frag ^ (kk * 4));
    const u32x4* ws = lds + 3 * XU + wb * WU + b_row + (frag ^ (kk * 4));
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[j] = __builtin_bit_cast(half8_t, ws[j * 16 * UPR]);
#pragma unroll
    for (int i = 0; i < TM; ++i) af[i] = __builtin_bit_cast(half8_t, xs[i * 16 * UPR]);
    __builtin_amdgcn_sched_barrier(0);
    if (kk == 0) {
      dequant(next, 3 * XU + (wb ^ 1) * WU, 0, UW / 2);
    } else {
      const int xn = xb == 0 ? 2 : xb - 1;  // (xb + 2) % 3
      load_x(s + 2, lds_base + (uint32_t)xn * X_BYTES, 0, NX);
      load_w(s + 3, next);
      wait_loads<NX + NW, WORDS>(later);
      __builtin_amdgcn_s_waitcnt(0xc07f);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
  };
  // The MFMAs of a phase; in the first half of a step the other half of W(s+1) is dequantised
  // in their shadow.  Two VALU instructions per MFMA of the SIMD are free (measured: 16.8 clocks
  // per MFMA with none to two, 21 with three), so a step's dequantisation is spread over two
  // phases of each half of the workgroup.
  auto multiply_phase = [&](int kk, const Regs& next) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    if (kk == 0) dequant(next, 3 * XU + (wb ^ 1) * WU, UW / 2, UW / 2);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
    if (kk == 0) {
#pragma unroll
      for (int u = 0; u < UW / 2; ++u) {
#pragma unroll
        for (int e = 0; e < TM * TN / (UW / 2); ++e) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, VALU_PER_MFMA, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // an LDS write
      }
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
  };
  // `next`: registers of W(s+1), refilled with W(s+3); `later`: those of W(s+2)
  auto step = [&](int s, Regs& next, Regs& later) {
    load_phase(s, 0, next, later);
    multiply_phase(0, next);
    load_phase(s, 1, next, later);
    multiply_phase(1, next);
    xb = xb == 2 ? 0 : xb + 1;
    wb ^= 1;
  };

  // ---- pipeline ---------------------------------------------------------------------------
  Regs w0, w1;
  load_w(0, w0);
  load_x(0, lds_base, 0, NX);
  load_w(1, w1);
  load_x(1, lds_base + X_BYTES, 0, NX);
  wait_loads<2 * NX + NW, WORDS>(w0);
  dequant(w0, 3 * XU, 0, UW);
  load_w(2, w0);
  wait_loads<NX + NW, WORDS>(w1);  // X(0) and W(1)
  lds_barrier();
  if (wave >= 4) __builtin_amdgcn_s_barrier();  // this half runs one phase behind
  for (int s = 0; s < nsteps; s += 2) {
    step(s, w1, w0);
    if (s + 1 < nsteps) step(s + 1, w0, w1);
  }
  if (wave < 4) __builtin_amdgcn_s_barrier();

  // the loads past the end have landed before their buffers become the epilogue's patches
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();

  // ---- epilogue: blocks of ER rows through a private LDS patch ------------------------------
  constexpr int ER = BM == 256 && TM % 4 == 0 ? 64 : 32, EB = TM * 16 / ER, PW = TN * 16 + 4;
  float* const patch = (float*)lds + wave * (ER * PW);
  float* const plane = a.ksplit > 1 ? a.workspace + (size_t)slice * a.m * a.n : nullptr;
  auto fill = [&](auto block) {  // a lane holds row l16, columns 4 lg .. 4 lg + 3 of a tile
#pragma unroll
    for (int i = 0; i < ER / 16; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) *(float4_t*)(patch + (i * 16 + l16) * PW + j * 16 + lg * 4) = acc[block * (ER / 16) + i][j];
  };
#pragma unroll 1
  for (int b = 0; b < EB; ++b) {
    if (b == 0) fill(std::integral_constant<int, 0>{});
    if constexpr (EB > 1) { if (b == 1) fill(std::integral_constant<int, 1>{}); }
    if constexpr (EB > 2) { if (b == 2) fill(std::integral_constant<int, 2>{}); }
    if constexpr (EB > 3) { if (b == 3) fill(std::integral_constant<int, 3>{}); }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // the patch is this wave's alone
    const int row0 = m0 + wm * TM * 16 + b * ER, col0 = n0 + wn * TN * 16;
    if (a.out.vec_ok) store_block8<ER, TN * 16, F == PIPE_INT8_ROW>(patch, lane, row0, col0, a.out, plane);
    else store_block1<ER, TN * 16, F == PIPE_INT8_ROW>(patch, lane, row0, col0, a.out, plane);
    __builtin_amdgcn_s_waitcnt(0xc07f);
  }
}

template <int BM, int BN, int WM, int WN>
int launch_pipe_tile(const PipeArgs& a, int f, hipStream_t stream) {
  const void* fn = f == PIPE_INT4 ? (const void*)gemm_pipe_kernel<BM, BN, WM, WN, PIPE_INT4>
                   : f == PIPE_INT8 ? (const void*)gemm_pipe_kernel<BM, BN, WM, WN, PIPE_INT8>
                                    : (const void*)gemm_pipe_kernel<BM, BN, WM, WN, PIPE_INT8_ROW>;
  size_t lds_bytes = (size_t)(3 * BM + 2 * BN) * 128;
  constexpr size_t patch_bytes = (size_t)8 * (BM == 256 && BM / WM % 64 == 0 ? 64 : 32) * (BN / WN + 4) * sizeof(float);
  if (lds_bytes < patch_bytes) lds_bytes = patch_bytes;
  static_assert(patch_bytes <= 160 * 1024, "the patches fit LDS");
  PipeArgs b = a;
  int grid = 0;
  b.map = make_tile_map((a.m + BM - 1) / BM, (a.n + BN - 1) / BN, TileCost{BM * 2, f == PIPE_INT4 ? BN / 2 : BN}, &grid);
  void* args[] = {(void*)&b};
  return launch_kernel(fn, dim3(grid * (a.ksplit > 1 ? a.ksplit : 1)), dim3(WM * WN * 64), args, lds_bytes, stream);
}

struct PipeTile {
  int bm, bn, wm, wn;
  int (*launch)(const PipeArgs&, int, hipStream_t);
};
// tile M, tile N, waves M, waves N
const PipeTile kPipeTiles[] = {
    {256, 256, 2, 4, launch_pipe_tile<256, 256, 2, 4>},  // wave tile 128 x 64
    {256, 192, 2, 4, launch_pipe_tile<256, 192, 2, 4>},  // 128 x 48
    {256, 128, 4, 2, launch_pipe_tile<256, 128, 4, 2>},  // 64 x 64
    {128, 128, 2, 4, launch_pipe_tile<128, 128, 2, 4>},  // 64 x 32, 80 KB of LDS: two workgroups share a CU
    {64, 128, 2, 4, launch_pipe_tile<64, 128, 2, 4>},    // 32 x 32
};

}  // namespace

bool gemm_pipe_config_applicable(const Problem& p, const tlhip_kernel_config_t& c, const char** why) {
  static const char* reasons[] = {
      "not a tile K 64 configuration of the tiled_direct variant",
      "activations must be f16",
      "K must be a multiple of 64",
      "the group size must be 32 x a power of two for int4-grouped, 64 x a power of two for int8-grouped",
      "K split across workgroups (p5) must be 0, 1 or a power of two up to 16 that divides K / 64, with the slices' "
      "partial sums (p5 x M x N, f32) inside the library's workspace",
      "tile (M, N, waves M, waves N) must be one of 256x256 2x4, 256x192 2x4, 256x128 4x2, 128x128 2x4, 64x128 2x4 with tile K 64",
  };
  auto fail = [&](int i) {
    if (why) *why = reasons[i];
    return false;
  };
  if (!is_pipe_config(c)) return fail(0);
  if (p.x_dtype != TLHIP_F16) return fail(1);
  if (p.k % PK != 0 || p.k == 0) return fail(2);
  if (p.format != TLHIP_FMT_INT8_ROW) {
    const int unit = p.format == TLHIP_FMT_INT4_GROUPED ? 32 : 64;
    const int groups = p.group_size / unit;
    if (p.group_size % unit != 0 || groups == 0 || (groups & (groups - 1)) != 0) return fail(3);
  }
  for (const auto& t : kPipeTiles)
    if (t.bm == c.p0 && t.bn == c.p1 && t.wm == c.p3 && t.wn == c.p4) {
      const int ks = c.p5 < 1 ? 1 : c.p5;
      if (ks > 1) {
        if (ks > 16 || (ks & (ks - 1)) != 0 || (p.k / PK) % ks != 0) return fail(4);
        if ((size_t)p.m * (size_t)p.n * ks > scratch_tile_floats(p)) return fail(4);
      }
      return true;
    }
  return fail(5);
}

int launch_gemm_pipe(const Problem& p, const tlhip_kernel_config_t& c, hipStream_t stream) {
  const char* why = nullptr;
  if (!gemm_pipe_config_applicable(p, c, &why))
    return set_error(TLHIP_ERR_INVALID, "gemm_pipe: config not applicable: %s", why ? why : "?");
  if (p.m == 0 || p.n == 0) return TLHIP_OK;
  PipeArgs a;
  const bool row = p.format == TLHIP_FMT_INT8_ROW, int4 = p.format == TLHIP_FMT_INT4_GROUPED;
  a.packed = (const uint8_t*)p.packed;
  a.scales = (const uint16_t*)p.scales;
  a.x = (const _Float16*)p.x;
  a.m = (int)p.m;
  a.n = (int)p.n;
  a.k = (int)p.k;
  a.w_row_bytes = (int)(int4 ? p.k / 2 : p.k);
  a.group_shift = row ? 0 : __builtin_ctz((unsigned)(p.group_size / 32));
  a.groups_per_row = row ? 0 : (int)(p.k / p.group_size);
  a.ksteps = (int)(p.k / PK);
  a.ksplit = c.p5 < 1 ? 1 : c.p5;
  a.workspace = nullptr;
  if (a.ksplit > 1) {
    int* counters = nullptr;
    const int rc = problem_scratch(p, stream, &a.workspace, &counters);
    if (rc) return rc;
  }
  a.out.y = p.y;
  a.out.y_dtype = p.y_dtype;
  a.out.vec_ok = (p.n % 8 == 0) && ((uintptr_t)p.y % 16 == 0);
  for (int i = 0; i < p.epi.n_ops; ++i)
    if (p.epi.kind[i] == TLHIP_EPI_BIAS || p.epi.kind[i] == TLHIP_EPI_BINARY) a.out.vec_ok = a.out.vec_ok && (uintptr_t)p.epi.input[i] % 16 == 0;
  a.out.m = (int)p.m;
  a.out.n = (int)p.n;
  a.out.alpha = p.format == TLHIP_FMT_INT8_GROUPED ? p.alpha * (1.0f / 127.0f) : p.alpha;
  a.out.epi = p.epi;
  a.out.col_scale = row ? (const float*)p.scales : nullptr;
  const int f = int4 ? PIPE_INT4 : (row ? PIPE_INT8_ROW : PIPE_INT8);
  int rc = TLHIP_ERR_INVALID;
  for (const auto& t : kPipeTiles)
    if (t.bm == c.p0 && t.bn == c.p1 && t.wm == c.p3 && t.wn == c.p4) rc = t.launch(a, f, stream);
  if (rc) return rc;
  if (a.ksplit > 1) {
    const int rr = launch_k_slice_reduce(a.ksplit, a.workspace, a.out, stream);
    if (rr) return rr;
  }
  count_gemm_dispatch();
  return TLHIP_OK;
}

// Every instance launch_gemm_pipe can reach, in prepare mode (see launch_kernel).
int prepare_gemm_pipe_kernels() {
  PipeArgs a;
  memset(&a, 0, sizeof a);
  a.m = a.n = 1;
  a.ksplit = 1;
  for (const auto& t : kPipeTiles)
    for (int f : {PIPE_INT4, PIPE_INT8, PIPE_INT8_ROW}) {
      const int rc = t.launch(a, f, nullptr);
      if (rc) return rc;
    }
  return TLHIP_OK;
}

}  // namespace tlhip
