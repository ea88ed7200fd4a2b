// Host side of the decode kernel for 2 to 16 f16 rows (stands in for dispatchQuantizedGemvNT,
// src/backend/webgpu/matmul/dispatch.ts:875-931): configuration checks, the default geometry and the
// launches.  The kernel is in gemv_few_kernel.h.
#include <algorithm>
#include <cstring>

#include "gemv_few_args.h"

namespace tlhip {
namespace {

constexpr int kLds = 160 * 1024;
int x_loads(const Problem& p) { return p.m <= 4 ? 1 : (p.m <= 8 ? 2 : 4); }
const void* instance(const Problem& p, int xv, int nb, int kind) {
  if (p.format == TLHIP_FMT_INT4_GROUPED) return gemv_few_instance_int4(xv, nb, kind);
  if (p.format == TLHIP_FMT_INT8_ROW) return gemv_few_instance_int8_row(xv, nb, kind);
  return p.group_size == 64 ? gemv_few_instance_int8_64(xv, nb, kind) : gemv_few_instance_int8_grouped(xv, nb, kind);
}
size_t lds_of(const Problem& p, int nb) {
  const size_t scales = p.format == TLHIP_FMT_INT8_ROW ? 0 : (size_t)nb * 16 * kFewScaleRow;
  return std::max(kFewWaves * ((size_t)4 * x_loads(p) * kFewRowBytes + scales), (size_t)kFewWaves * nb * 1024);
}
// Columns of a block: a quarter of four at least, all blocks alike.
int block_cols(int cols, int blocks) { return ((cols + blocks - 1) / blocks + 3) / 4 * 4; }

template <int KIND>
int launch(const Problem* ps, int count, int unary, const tlhip_kernel_config_t& c, hipStream_t stream) {
  constexpr bool pair = KIND == FEW_PAIR;
  const Problem& p = ps[0];
  FewArgs<KIND> a;
  memset(&a, 0, sizeof a);
  a.x = (const _Float16*)p.x;
  a.m = (int)p.m;
  a.k = (int)p.k;
  a.steps = (int)(p.k / kFewStep);
  a.cols = c.p2;
  a.block_cols = block_cols(c.p2, pair ? c.p4 / 2 : c.p4);
  a.row_bytes = (uint32_t)(p.format == TLHIP_FMT_INT4_GROUPED ? p.k / 2 : p.k);
  a.scale_row_bytes = p.format == TLHIP_FMT_INT8_ROW ? 4 : (uint32_t)(p.k / p.group_size) * 2;
  a.group_shift = p.format == TLHIP_FMT_INT8_GROUPED ? __builtin_ctz((unsigned)(p.group_size / 64)) : 0;
  a.factor = p.alpha * (p.format == TLHIP_FMT_INT8_GROUPED ? 1.0f / 127.0f : 1.0f);
  a.y_dtype = p.y_dtype;
  a.unary = unary;
  a.vec = 1;
  for (int i = 0; i < count; ++i) {
    if (ps[i].n == 0) continue;
    const int at = a.count++;
    a.packed[at] = (const uint8_t*)ps[i].packed;
    a.scales[at] = (const uint8_t*)ps[i].scales;
    a.y[at] = ps[i].y;
    a.n[at] = (int)ps[i].n;
    a.first[at + 1] = a.first[at] + (pair && at ? 0 : (int)((ps[i].n + c.p2 - 1) / c.p2));
    if (ps[i].n % 4 != 0 || ((uintptr_t)ps[i].y & (p.y_dtype == TLHIP_F16 ? 7 : 15)) != 0) a.vec = 0;
    if (pair) continue;
    a.epi[at] = ps[i].epi;
    a.n_ops[at] = ps[i].epi.n_ops;
    // the first step with an input, which comes ahead of the sums; n_ops -1: it is added and the only step
    for (int s = 0; s < ps[i].epi.n_ops; ++s) {
      const int kind = ps[i].epi.kind[s];
      if (kind != TLHIP_EPI_BIAS && kind != TLHIP_EPI_BINARY) continue;
      const bool f16 = ps[i].epi.input_dtype[s] == TLHIP_F16;
      a.pre[at] = ps[i].epi.input[s];
      a.pre_kind[at] = f16 ? FEW_PRE_F16 : FEW_PRE_F32;
      a.pre_row[at] = kind == TLHIP_EPI_BIAS ? 0 : (int)ps[i].n;
      a.pre_at[at] = s;
      if (((uintptr_t)a.pre[at] & (f16 ? 7 : 15)) != 0) a.vec = 0;
      if (ps[i].epi.n_ops == 1 && (kind == TLHIP_EPI_BIAS || ps[i].epi.unary[s] == TLHIP_BINARY_ADD)) a.n_ops[at] = -1;
      break;
    }
  }
  if (a.count == 0 || p.m == 0) return TLHIP_OK;
  void* args[] = {(void*)&a};
  const int rc = launch_kernel(instance(p, x_loads(p), c.p4, KIND), dim3((unsigned)a.first[a.count]), dim3(kFewWaves * 64), args,
                               lds_of(p, c.p4), stream);
  if (rc) return rc;
  for (int i = 0; i < a.count; ++i) count_gemv_dispatch();
  return TLHIP_OK;
}

}  // namespace

bool is_few_config(const Problem& p, const tlhip_kernel_config_t& c, int kind) {
  if (c.variant != VARIANT_GEMV_MFMA || c.p0 != kFewWaves || c.p4 < 1 || c.p4 > kFewMaxBlocks) return false;
  if (c.p1 || c.p3 || c.p5 || c.p6) return false;  // the other form's fields
  if (p.x_dtype != TLHIP_F16 || p.m < 2 || p.m > 16 || p.pro.kind != TLHIP_PRO_NONE) return false;
  if (p.k <= 0 || p.k % kFewStep != 0 || p.k > kFewStep * kFewWaves * kFewMaxSteps) return false;
  if (p.format == TLHIP_FMT_INT4_GROUPED ? p.group_size != 32 : (p.format != TLHIP_FMT_INT8_ROW && p.group_size < 64)) return false;
  const int blocks = kind == FEW_PAIR ? c.p4 / 2 : c.p4;
  if (blocks < 1 || c.p2 < 4 || c.p2 % 4 != 0) return false;
  const int each = block_cols(c.p2, blocks);
  if (each > 16 || each * (blocks - 1) >= c.p2) return false;  // no empty block
  return instance(p, x_loads(p), c.p4, kind) && lds_of(p, c.p4) <= kLds;
}

// What orders the geometries of a problem: per round of workgroups a constant, a little more for more rows, and
// per 1000 of K the step, the rows and the width of the blocks.  Fitted at 27 matrices of 1024..18432 x
// 1024..12288, 2..16 rows, four formats (3600 launches, 3.6-7.1 % rms each, warm); the geometry it picks is 0.6-1.2 %
// behind the best one in the mean of 1700 problems (18084 launches on cold weights, where it is 15 % too low: what a
// launch takes beside another kernel's is gemv_few_us).
static double few_us(const Problem* ps, int count, int kind, const tlhip_kernel_config_t& c) {
  const Problem& p = ps[0];
  struct Cost {
    double launch, round, rows, k, k_rows, k_width;
  };
  static const Cost costs[3][5] = {  // format, 1 / 2 / 3 / 4 / 6 blocks
      {{2.36, 0.30, 0.47, 0.224, 0.280, 0.115}, {2.73, 0.20, 0.11, 0.655, 0.195, 0.129}, {2.33, 0.78, 0.58, 1.103, 0.194, 0.0}, {0.50, 3.05, 0.16, 1.418, 0.255, 0.0}, {2.64, 1.47, 0.30, 1.240, 0.229, 0.880}},   // int4
      {{2.16, 0.48, 0.53, 0.154, 0.276, 0.334}, {2.42, 0.37, 0.49, 0.488, 0.240, 0.483}, {1.27, 2.12, 0.0, 1.102, 0.348, 0.233}, {0.50, 3.10, 0.05, 1.825, 0.359, 0.0}, {2.61, 1.40, 0.23, 1.529, 0.355, 1.204}},   // int8 in groups
      {{2.29, 0.39, 0.33, 0.125, 0.302, 0.346}, {2.34, 0.39, 0.40, 0.460, 0.258, 0.479}, {1.30, 2.00, 0.0, 1.252, 0.344, 0.019}, {0.50, 2.95, 0.16, 1.693, 0.393, 0.0}, {2.47, 1.22, 0.47, 1.486, 0.287, 1.124}}};  // int8 per row
  const Cost& t = costs[p.format == TLHIP_FMT_INT4_GROUPED ? 0 : (p.format == TLHIP_FMT_INT8_ROW ? 2 : 1)][c.p4 == 6 ? 4 : c.p4 - 1];
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  int64_t wgs = 0;
  for (int i = 0; i < count; ++i) wgs += (ps[i].n + c.p2 - 1) / c.p2;
  const double rows = 0.25 * x_loads(p), width = (double)c.p2 * (kind == FEW_PAIR ? 2 : 1) / (16.0 * c.p4);
  return t.launch + (double)((wgs + cus - 1) / cus) * (t.round + t.rows * rows + (double)p.k / 1000.0 * (t.k + t.k_rows * rows + t.k_width * width));
}

// Beside other kernels, behind each other and on cold weights: the weights' way from memory, the activations' into every
// workgroup (16 rows of K = 12288 are 100 MB at 256 workgroups, four times the int4 weights of 4096 columns), and per
// round the blocks' sums and, per 1000 of K, the blocks, the rows and the columns.
// A residual costs next to nothing: it is loaded ahead of the sums.  Fitted at 7919 launches of the geometries it
// is asked for (17 x 13 matrices of 768..28672 x 1024..14336, 2..16 rows, with and without a residual): 4.3-4.6 % rms.
double gemv_few_us(const Problem& p, const tlhip_kernel_config_t& c) {
  struct Cost {
    double launch, mb, x, sums, sums_rows, k_blocks, k_rows, k_both, k_cols, residual, residual_out;
  };
  static const Cost costs[3] = {{2.583, 0.0801, 0.0382, 0.226, 0.104, 0.273, 0.106, 0.030, 0.049, 0.067, 0.034},   // int4
                                {2.602, 0.0564, 0.0592, 0.224, 0.071, 0.126, 0.173, 0.0, 0.306, 0.118, 0.001},    // int8 in groups
                                {2.628, 0.0633, 0.0526, 0.232, 0.065, 0.125, 0.187, 0.0, 0.261, 0.045, 0.015}};   // int8 per row
  const bool int4 = p.format == TLHIP_FMT_INT4_GROUPED;
  const Cost& t = costs[int4 ? 0 : (p.format == TLHIP_FMT_INT8_ROW ? 2 : 1)];
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const int64_t wgs = (p.n + c.p2 - 1) / c.p2;
  const double rounds = (double)((wgs + cus - 1) / cus), rows = 0.25 * x_loads(p), nb = c.p4, k = (double)p.k / 1000.0;
  const double mb = (double)p.n * (double)p.k * (int4 ? 0.5 : 1.0) / 1e6;
  return t.launch + t.mb * mb + t.x * (double)(wgs * p.m) * (double)p.k / 1e6 +
         rounds * (nb * (t.sums + t.sums_rows * rows) + k * (t.k_blocks * nb + t.k_rows * rows + t.k_both * rows * nb + t.k_cols * c.p2 / 16.0)) +
         (has_residual(p) ? t.residual + t.residual_out * (double)p.m * (double)p.n / 1e5 : 0.0);
}

// Full blocks, or the columns dealt evenly over one to six rounds of workgroups (several problems: the
// next wider shares too, as each ends with a workgroup of its own).
bool gemv_few_default(const Problem* ps, int count, int kind, tlhip_kernel_config_t* out, double* us) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  int64_t n = 0;
  for (int i = 0; i < count; ++i) n += ps[i].n;
  bool found = false;
  auto weigh = [&](int64_t cols, int nb) {
    tlhip_kernel_config_t c;
    memset(&c, 0, sizeof c);
    c.variant = VARIANT_GEMV_MFMA;
    c.p0 = kFewWaves;
    c.p2 = (int)cols;
    c.p4 = nb;
    if (!is_few_config(ps[0], c, kind)) return;
    const double t = few_us(ps, count, kind, c);
    if (found && t >= *us) return;
    *out = c;
    *us = t;
    found = true;
  };
  for (int nb : {1, 2, 3, 4, 6}) {
    const int64_t most = 16 * (kind == FEW_PAIR ? nb / 2 : nb);
    weigh(most, nb);
    for (int rounds = 1; rounds <= 6; ++rounds) {
      const int64_t even = ((n + (int64_t)cus * rounds - 1) / ((int64_t)cus * rounds) + 3) / 4 * 4;
      for (int64_t cols = even; cols < most && cols <= even + (count > 1 ? 8 : 0); cols += 4) weigh(cols, nb);
    }
  }
  return found;
}

int launch_gemv_few(const Problem* ps, int count, int kind, int unary, const tlhip_kernel_config_t& c, hipStream_t stream) {
  if (!is_few_config(ps[0], c, kind)) return set_error(TLHIP_ERR_INVALID, "gemv_few: config not applicable");
  return kind == FEW_SINGLE  ? launch<FEW_SINGLE>(ps, count, unary, c, stream)
         : kind == FEW_GROUP ? launch<FEW_GROUP>(ps, count, unary, c, stream)
                             : launch<FEW_PAIR>(ps, count, unary, c, stream);
}

// Every instance launch_gemv_few can reach, in prepare mode (see launch_kernel).
int prepare_gemv_few_kernels() {
  Problem p;
  memset(&p, 0, sizeof p);
  for (p.format = 0; p.format < 3; ++p.format)
    for (p.group_size = 64; p.group_size <= 128; p.group_size *= 2)
      for (int xv : {1, 2, 4})
        for (int nb = 1; nb <= kFewMaxBlocks; ++nb)
          for (int kind : {FEW_SINGLE, FEW_GROUP, FEW_PAIR})
            if (const void* fn = instance(p, xv, nb, kind)) {
              const int rc = launch_kernel(fn, dim3(1), dim3(64), nullptr, 0, nullptr);
              if (rc) return rc;
            }
  return TLHIP_OK;
}

}  // namespace tlhip
