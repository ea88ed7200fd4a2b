// Kernel arguments of the decode GEMV of one activation row, shared by the kernels
// (gemv_one_kernel.h) and the host side (gemv_one.hip).
#pragma once
#include "device_utils.h"
#include "gemv_one.h"

namespace tlhip {

constexpr int kOneProblems[] = {1, 4, 2};  // of a launch, by ONE_*

// The input of the first epilogue step that has one, loaded with the weights.
enum { ONE_PRE_NONE = 0, ONE_PRE_F16 = 1, ONE_PRE_F32 = 2 };

template <int KIND>
struct OneArgs {
  static constexpr int NP = kOneProblems[KIND];
  const void* x;        // of every problem, or with own_x of the first
  const void* operand;  // the prologue's
  int threads;
  int nchunks;          // 16-byte chunks per weight row
  int lpr_shift;        // log2(lanes per row)
  int kw_shift;         // log2(waves that share a row's K)
  int cpg_shift;        // grouped formats: log2(chunks sharing one scale)
  int groups_per_row;
  int rows_per_wg;
  int y_dtype;
  float factor;         // alpha, times 1/127 for INT8_GROUPED
  int count;
  int own_x;
  int k;
  int unary;            // of the gated prologue, or of the pair's gate
  float eps;
  // workgroups [first[i], first[i + 1]) work on problem i (a pair's all on both): each of them on
  // `rounds` blocks of rows, the first `longer` on one more
  int first[NP + 1];
  int rounds[NP];
  int longer[NP];
  int n[NP];
  int pre_kind[NP];
  int n_ops[NP];
  const u32x4* packed[NP];
  const void* scales[NP];
  void* y[NP];
  const void* pre[NP];
  const void* xs[NP];
  int pre_at[NP];       // the step whose input `pre` is
  DevEpilogue epi[NP];
};

// Defined once per weight format (gemv_one_int4.hip, ...); a null pointer where an
// instance is not built.
const void* gemv_one_instance_int4(int x_dtype, int positions, int units, int prologue, int kind);
const void* gemv_one_instance_int8_grouped(int x_dtype, int positions, int units, int prologue, int kind);
const void* gemv_one_instance_int8_row(int x_dtype, int positions, int units, int prologue, int kind);

}  // namespace tlhip
