// gemv_few for one weight format (a unit of its own, so that the formats compile in parallel).
#include "gemv_few_kernel.h"

namespace tlhip {
const void* gemv_few_instance_int4(int xv, int nb, int kind) { return few_instance<TLHIP_FMT_INT4_GROUPED, true>(xv, nb, kind); }
}  // namespace tlhip
