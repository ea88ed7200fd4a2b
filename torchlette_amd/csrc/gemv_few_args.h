// Kernel arguments of the decode kernel for 2 to 16 f16 rows that keeps all of K in a workgroup, shared
// by the kernels (gemv_few_kernel.h) and the host side (gemv_few.hip).
#pragma once
#include "device_utils.h"
#include "gemv_few.h"

namespace tlhip {

constexpr int kFewStep = 128;                     // k of a step
constexpr int kFewRowBytes = kFewStep * 2 + 16;   // LDS row of a step: 16 bytes more, so that rows start in other banks
constexpr int kFewWaves = 8;
constexpr int kFewMaxSteps = 16;                  // steps of a wave: its scales are in LDS
constexpr int kFewScaleRow = kFewMaxSteps * 8 + 16;  // LDS row of a column's scales
constexpr int kFewMaxBlocks = 6;                  // blocks of columns per workgroup
constexpr int kFewProblems[] = {1, 4, 2};         // of a launch, by FEW_*

// The input of the first epilogue step that has one, loaded ahead of the sums.
enum { FEW_PRE_NONE = 0, FEW_PRE_F16 = 1, FEW_PRE_F32 = 2 };

template <int KIND>
struct FewArgs {
  static constexpr int NP = kFewProblems[KIND];
  const _Float16* x;
  int m, k;
  int steps;             // K / 128
  int cols;              // columns of a workgroup (of either projection of a pair)
  int block_cols;        // ... of a block: at most 16
  uint32_t row_bytes;        // packed bytes of a weight row
  uint32_t scale_row_bytes;  // bytes of a row's group scales
  int group_shift;       // int8 groups: log2(group size / 64)
  float factor;          // alpha, times 1/127 for INT8_GROUPED
  int y_dtype;
  int vec;               // N % 4 == 0 and outputs and inputs aligned for four columns at a time
  int unary;             // of a pair's gate
  int count;
  int first[NP + 1];     // workgroups [first[i], first[i + 1]) work on problem i (a pair's all on both)
  int n[NP];
  int pre_kind[NP];
  int pre_row[NP];       // elements of a row of that input: N, or 0 for a bias
  int n_ops[NP];         // -1: that input is added, and nothing else
  const uint8_t* packed[NP];
  const uint8_t* scales[NP];
  void* y[NP];
  const void* pre[NP];
  int pre_at[NP];
  DevEpilogue epi[NP];
};

// Defined once per weight format (gemv_few_int4.hip, ...): `xv` loads of four rows each, `nb` blocks of columns
// (a pair: of both projections); a null pointer where an instance is not built.
const void* gemv_few_instance_int4(int xv, int nb, int kind);
const void* gemv_few_instance_int8_64(int xv, int nb, int kind);
const void* gemv_few_instance_int8_grouped(int xv, int nb, int kind);
const void* gemv_few_instance_int8_row(int xv, int nb, int kind);

}  // namespace tlhip
