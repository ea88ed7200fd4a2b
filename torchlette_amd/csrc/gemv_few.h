// The decode kernel for 2 to 16 f16 rows with all of K in a workgroup (gemv_few.hip), as the callers that
// choose its launches see it: a form of the gemv_mfma variant with p0 = 8, p1 = 0, p2 columns and p4 blocks of
// columns per workgroup.
#pragma once
#include "common.h"

namespace tlhip {

// What a launch works on: one problem, up to four on the same activations, or a gate and an up
// projection whose product it writes.
enum { FEW_SINGLE = 0, FEW_GROUP = 1, FEW_PAIR = 2 };

bool is_few_config(const Problem& p, const tlhip_kernel_config_t& c, int kind);
// The cheapest geometry for a launch of `count` problems (a pair: its gate's) and its time in microseconds, or false.
bool gemv_few_default(const Problem* ps, int count, int kind, tlhip_kernel_config_t* out, double* us);
// What the launch c of one problem takes beside other kernels, in microseconds (see gemv_mfma_us).
double gemv_few_us(const Problem& p, const tlhip_kernel_config_t& c);
int launch_gemv_few(const Problem* ps, int count, int kind, int unary, const tlhip_kernel_config_t& c, hipStream_t stream);
int prepare_gemv_few_kernels();  // gemv_few.hip (+ the per-format units)

}  // namespace tlhip
