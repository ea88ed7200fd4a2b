// The VALU kernel for 2 to 5 f32 rows in one launch (gemv_some.hip), as its callers see it: a form of the gemv
// variant with p5 = 4, p0 lanes of a column and p4 columns of a workgroup.
#pragma once
#include "common.h"

namespace tlhip {

bool is_some_config(const tlhip_kernel_config_t& c);
bool gemv_some_config_applicable(const Problem& p, const tlhip_kernel_config_t& c, const char** why);
// The geometry for p's rows, sizes and format, or false.
bool gemv_some_default(const Problem& p, tlhip_kernel_config_t* out);
int launch_gemv_some(const Problem& p, const tlhip_kernel_config_t& c, hipStream_t stream);
int prepare_gemv_some_kernels();

}  // namespace tlhip
