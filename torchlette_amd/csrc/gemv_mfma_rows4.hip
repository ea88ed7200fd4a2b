// The instances of the skinny matrix-core GEMV for 33..64 activation rows: four tiles of 16
// rows per weight row block (gemv_mfma_kernel.h).  Apart from gemv_mfma_rows.hip, so that the
// two, the longest to compile, are compiled side by side.
#include "gemv_mfma_kernel.h"

namespace tlhip {

int launch_mfma_rows4(int format, int group_size, int64_t k, int unroll, int line, const MfmaArgs& a, int grid, int threads,
                      size_t lds_bytes, hipStream_t stream) {
  return launch_mfma_instance<false, 4>(format, group_size, k, unroll, line, a, grid, threads, lds_bytes, stream);
}

int prepare_mfma_rows4() { return prepare_mfma_instances<false, 4>(); }

}  // namespace tlhip
