// The one-row decode GEMV for one weight format (a unit of its own, so that the formats compile in parallel).
#include "gemv_one_kernel.h"

namespace tlhip {
const void* gemv_one_instance_int8_row(int x_dtype, int positions, int units, int prologue, int kind) {
  return one_instance<TLHIP_FMT_INT8_ROW>(x_dtype, positions, units, prologue, kind);
}
}  // namespace tlhip
