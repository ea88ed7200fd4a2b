// The one-row decode GEMV (gemv_one.hip) as the callers that choose its launches see it.
#pragma once
#include "common.h"

namespace tlhip {

// What a launch works on: one problem, up to four of one K, or a gate and an
// up projection whose product it writes.
enum { ONE_SINGLE = 0, ONE_GROUP = 1, ONE_PAIR = 2 };

// The geometry for p's K, format and types with `rows` rows of weights in all, or false.
bool gemv_one_default(const Problem& p, int64_t rows, int kind, tlhip_kernel_config_t* out);
// The launch of a group whose longest problem runs as `alone` on its own, or false.
bool gemv_one_group_config(const Problem* ps, int count, const tlhip_kernel_config_t& alone, tlhip_kernel_config_t* out);
// gate.y (f16) = unary(gate) * up, both rounded to f16 first; no epilogue, no prologue.
bool gemv_pair_applicable(const Problem& gate, const Problem& up, const tlhip_kernel_config_t& c);
int launch_gemv_pair(const Problem& gate, const Problem& up, int unary, const tlhip_kernel_config_t& c, hipStream_t stream);

}  // namespace tlhip
