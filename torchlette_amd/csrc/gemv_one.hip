// Host side of the one-row decode GEMV (stands in for dispatchQuantizedGemvNT at M = 1,
// src/backend/webgpu/matmul/dispatch.ts:875-931): configuration checks, the default geometry and
// the launches.  The kernel is in gemv_one_kernel.h.
#include <algorithm>
#include <cstring>

#include "gemv_one.h"
#include "gemv_one_args.h"

namespace tlhip {
namespace {

constexpr size_t kLdsBudget = 128 * 1024;
int chunk_weights(int format) { return format == TLHIP_FMT_INT4_GROUPED ? 32 : 16; }
int x_units(const Problem& p) { return chunk_weights(p.format) * (p.x_dtype == TLHIP_F16 ? 2 : 4) / 16; }  // of a chunk
int64_t chunks_of(const Problem& p) { return p.k / chunk_weights(p.format); }

// Chunks a lane holds (seven: more than any instance is built for).
int positions(const Problem& p, const tlhip_kernel_config_t& c) {
  const int64_t lanes = (int64_t)c.p0 * c.p3, n = (chunks_of(p) + lanes - 1) / lanes;
  return (int)std::min<int64_t>(n, 7);
}
// Units of activations a thread stages: one, two, or four at a time.
int units(const Problem& p, const tlhip_kernel_config_t& c) {
  const int64_t all = chunks_of(p) * x_units(p), threads = (int64_t)c.p2 * 64;
  return all <= threads ? 1 : (all <= 2 * threads ? 2 : 4);
}
const void* instance(const Problem& p, int pos, int units, int prologue, int kind) {
  if (p.format == TLHIP_FMT_INT4_GROUPED) return gemv_one_instance_int4(p.x_dtype, pos, units, prologue, kind);
  if (p.format == TLHIP_FMT_INT8_GROUPED) return gemv_one_instance_int8_grouped(p.x_dtype, pos, units, prologue, kind);
  return gemv_one_instance_int8_row(p.x_dtype, pos, units, prologue, kind);
}
int rows_per_wg(const tlhip_kernel_config_t& c) { return c.p2 / c.p3 * (64 / c.p0); }
size_t lds_bytes(const Problem& p, const tlhip_kernel_config_t& c, int kind) {
  return (size_t)(chunks_of(p) + 1) * x_units(p) * 16 + (size_t)c.p3 * rows_per_wg(c) * (kind == ONE_PAIR ? 8 : 4);
}

const char* refusal(const Problem& p, const tlhip_kernel_config_t& c, int kind) {
  if (p.m != 1) return "the one-row form (p5 = 3) takes M = 1";
  if (c.p0 != 16 && c.p0 != 32 && c.p0 != 64) return "lanes per row must be 16, 32 or 64";
  if (c.p1 != 1) return "the one-row form has one row per lane group";
  if (c.p2 != 4 && c.p2 != 8) return "the one-row form has four or eight waves per workgroup";
  if (c.p3 < 1 || (c.p3 & (c.p3 - 1)) != 0 || c.p3 > c.p2) return "K-split waves must be 1, 2, 4 or 8 and divide waves per workgroup";
  if (c.p4 < 1 || c.p4 > 8 || c.p4 * c.p2 > 32) return "the one-row form has 1..8 workgroups, at most 32 waves, per CU";
  const int cw = chunk_weights(p.format);
  if (p.k <= 0 || p.k % cw != 0) return "K must be a whole number of 16-byte chunks (K % 32 for int4, K % 16 for int8)";
  if (p.format != TLHIP_FMT_INT8_ROW && p.group_size % cw != 0) return "group size must be a multiple of the chunk (32 for int4, 16 for int8)";
  if (!instance(p, positions(p, c), units(p, c), p.pro.kind, kind)) return "more chunks per lane than the one-row form is built for";
  if (lds_bytes(p, c, kind) > kLdsBudget) return "the activation row does not fit LDS";
  return nullptr;
}

// The first step with an input, which the kernel loads with the weights; n_ops is -1 where it adds
// that input and is the only step.
template <int KIND>
void fill_epilogue(const Problem& p, int i, OneArgs<KIND>& a) {
  a.epi[i] = p.epi;
  a.n_ops[i] = p.epi.n_ops;
  for (int s = 0; s < p.epi.n_ops; ++s) {
    if (p.epi.kind[s] != TLHIP_EPI_BIAS && p.epi.kind[s] != TLHIP_EPI_BINARY) continue;
    a.pre[i] = p.epi.input[s];
    a.pre_kind[i] = p.epi.input_dtype[s] == TLHIP_F16 ? ONE_PRE_F16 : ONE_PRE_F32;
    a.pre_at[i] = s;
    if (p.epi.n_ops == 1 && (p.epi.kind[s] == TLHIP_EPI_BIAS || p.epi.unary[s] == TLHIP_BINARY_ADD)) a.n_ops[i] = -1;
    return;
  }
}

template <int KIND>
int launch(const Problem* ps, int count, int unary, const tlhip_kernel_config_t& c, hipStream_t stream) {
  constexpr bool pair = KIND == ONE_PAIR;
  OneArgs<KIND> a;
  memset(&a, 0, sizeof a);
  const Problem& p = ps[0];
  const int cw = chunk_weights(p.format), cus = device_cu_count() > 0 ? device_cu_count() : 256;
  a.operand = p.pro.operand;
  a.threads = c.p2 * 64;
  a.k = (int)p.k;
  a.nchunks = (int)chunks_of(p);
  a.lpr_shift = __builtin_ctz((unsigned)c.p0);
  a.kw_shift = __builtin_ctz((unsigned)c.p3);
  a.cpg_shift = p.format == TLHIP_FMT_INT8_ROW ? 0 : __builtin_ctz((unsigned)(p.group_size / cw));
  a.groups_per_row = p.format == TLHIP_FMT_INT8_ROW ? 0 : (int)(p.k / p.group_size);
  a.rows_per_wg = rows_per_wg(c);
  a.unary = pair ? unary : p.pro.unary;
  a.eps = p.pro.eps;
  a.factor = p.alpha * (p.format == TLHIP_FMT_INT8_GROUPED ? 1.0f / 127.0f : 1.0f);
  a.y_dtype = p.y_dtype;
  // a workgroup for every block of rows, or as many as are resident, in proportion
  int64_t total = 0, blocks[4] = {0, 0, 0, 0};
  for (int i = 0; i < (pair ? 1 : count); ++i) total += blocks[i] = (ps[i].n + a.rows_per_wg - 1) / a.rows_per_wg;
  const int64_t resident = (int64_t)cus * c.p4;
  for (int i = 0; i < count; ++i) {
    if (ps[i].n == 0) continue;
    const int at = a.count++;
    a.xs[at] = ps[i].x;
    if (at == 0) a.x = ps[i].x;
    if (ps[i].x != a.x) a.own_x = 1;
    a.packed[at] = (const u32x4*)ps[i].packed;
    a.scales[at] = ps[i].scales;
    a.y[at] = ps[i].y;
    a.n[at] = (int)ps[i].n;
    if (!pair) fill_epilogue(ps[i], at, a);
    if (pair && at == 1) {  // the first's workgroups, no more
      a.first[at + 1] = a.first[at];
      continue;
    }
    const int64_t wgs = total > resident ? std::max<int64_t>(1, blocks[i] * resident / total) : blocks[i];
    a.first[at + 1] = a.first[at] + (int)wgs;
    a.rounds[at] = (int)(blocks[i] / wgs);
    a.longer[at] = (int)(blocks[i] % wgs);
  }
  if (a.count == 0) return TLHIP_OK;
  const int grid = a.first[a.count];
  void* args[] = {(void*)&a};
  const int rc = launch_kernel(instance(p, positions(p, c), units(p, c), p.pro.kind, KIND), dim3((unsigned)grid), dim3((unsigned)c.p2 * 64),
                               args, lds_bytes(p, c, KIND), stream);
  if (rc) return rc;
  for (int i = 0; i < a.count; ++i) count_gemv_dispatch();
  return TLHIP_OK;
}

}  // namespace

bool is_one_config(const tlhip_kernel_config_t& c) { return c.variant == VARIANT_GEMV && c.p5 == 3; }

bool gemv_one_config_applicable(const Problem& p, const tlhip_kernel_config_t& c, const char** why) {
  const char* r = refusal(p, c, ONE_SINGLE);
  if (why && r) *why = r;
  return !r;
}

int launch_gemv_one(const Problem& p, const tlhip_kernel_config_t& c, hipStream_t stream) {
  if (const char* r = refusal(p, c, ONE_SINGLE)) return set_error(TLHIP_ERR_INVALID, "gemv: config not applicable: %s", r);
  return launch<ONE_SINGLE>(&p, 1, 0, c, stream);
}

// Grouped launch: problems of one K, format, types and prologue; rows, pointers and epilogues are each one's own.
bool gemv_group_compatible(const Problem* ps, int count, const tlhip_kernel_config_t& c, const char** why) {
  const char* r = nullptr;
  if (count < 1 || count > 4) r = "a group holds 1..4 problems";
  for (int i = 0; !r && i < count; ++i) {
    if (ps[i].x_dtype != TLHIP_F16) r = "grouped launches are built for M = 1 and f16 activations";
    else if (ps[i].format != ps[0].format || ps[i].group_size != ps[0].group_size || ps[i].k != ps[0].k ||
             ps[i].y_dtype != ps[0].y_dtype)
      r = "all problems of a group must share format, group size, K and output type";
    else if (!is_one_config(c)) r = "grouped launches are built for the one-row form";
    else r = refusal(ps[i], c, ONE_GROUP);
  }
  if (why && r) *why = r;
  return !r;
}

int launch_gemv_grouped(const Problem* ps, int count, const tlhip_kernel_config_t& c, hipStream_t stream) {
  const char* why = nullptr;
  if (!gemv_group_compatible(ps, count, c, &why)) return set_error(TLHIP_ERR_INVALID, "gemv_grouped: %s", why);
  return launch<ONE_GROUP>(ps, count, 0, c, stream);
}

bool gemv_pair_applicable(const Problem& gate, const Problem& up, const tlhip_kernel_config_t& c) {
  return is_one_config(c) && gate.x_dtype == TLHIP_F16 && gate.pro.kind == TLHIP_PRO_NONE && gate.x == up.x && gate.n == up.n &&
         gate.k == up.k && gate.format == up.format && gate.group_size == up.group_size && !refusal(gate, c, ONE_PAIR);
}

int launch_gemv_pair(const Problem& gate, const Problem& up, int unary, const tlhip_kernel_config_t& c, hipStream_t stream) {
  if (!gemv_pair_applicable(gate, up, c)) return set_error(TLHIP_ERR_INVALID, "gemv_pair: config not applicable");
  const Problem ps[2] = {gate, up};
  return launch<ONE_PAIR>(ps, 2, unary, c, stream);
}

// Waves of a workgroup and workgroups of a CU for c's lanes.
static void set_waves(const Problem& p, int kind, tlhip_kernel_config_t* c) {
  const bool alone = kind == ONE_SINGLE && p.pro.kind == TLHIP_PRO_NONE;
  c->p2 = c->p3 > 1 || p.k >= (alone ? 4096 : 8192) ? 8 : 4;
  // activations in registers decide how many waves fit; a gated prologue of a long row costs every workgroup much
  const bool few = positions(p, *c) * x_units(p) > (kind == ONE_PAIR ? 8 : (alone ? 16 : 12)) ||
                   (p.pro.kind == TLHIP_PRO_GATED_MUL && p.k > 4096);
  c->p4 = (few ? 8 : 16) / c->p2;
}

// A group's: the lanes of its longest problem on its own, so that its results are those of separate launches.
bool gemv_one_group_config(const Problem* ps, int count, const tlhip_kernel_config_t& alone, tlhip_kernel_config_t* out) {
  *out = alone;
  if (!is_one_config(alone)) return false;
  set_waves(ps[0], ONE_GROUP, out);
  return gemv_group_compatible(ps, count, *out, nullptr);
}

// Lanes and waves for `rows` rows of K in all: the fewest lanes that keep a row's chunks in registers
// (three chunks of f16 rows each, two of f32 ones, before more lanes are better), that waste few of
// them past the row's end and give the chip 1024 waves, but not many more; a wave less in the row
// where a workgroup pays for a prologue, or the lanes can be few because a group has many rows.
// Against the best of 60 geometries at 19 matrices of 1024..151936 x 1024..12288, five pairs of format
// and type: 1.8 % behind it in the mean.  What it does not take, and long rows of many (one_row_config in dispatch.cpp), are
// left to gemv_kernel.h; us, that kernel -> here, cold weights, one f16 row of int4 1024 x 1024 2.8 -> 2.3, 12288 x 4096 7.8 -> 7.2,
// 65536 x 2048 22.0 -> 16.3; int8-64 1024 x 3072 3.7 -> 2.9, 12288 x 4096 11.2 -> 10.7, level at 4096 x 12288 (10.8-11.0); per
// row 2048 x 5120 4.9 -> 3.9; one f32 row of int8-64 1024 x 9728 7.4 -> 5.1.  Five chunks have an instance of their own: run
// as six they took 8 % more at 5120 and 9728 of int8 (2048 x 5120 4.4 us).  The rows of a long matrix (an LM head) go to
// fewer lanes: 256000 x 2304 per row 95 us on 64 lanes, 88 on 32.
bool gemv_one_default(const Problem& p, int64_t rows, int kind, tlhip_kernel_config_t* out) {
  if (p.m != 1) return false;
  const bool f16 = p.x_dtype == TLHIP_F16;
  const bool alone = kind == ONE_SINGLE && p.pro.kind == TLHIP_PRO_NONE;
  if (!f16 && p.k > 10240) return false;
  const int64_t chunks = chunks_of(p);
  const bool longer = rows >= 32768;
  double best = 0.0;
  bool found = false;
  for (int lanes = 16; lanes <= 512; lanes *= 2) {
    tlhip_kernel_config_t c;
    memset(&c, 0, sizeof c);
    c.variant = VARIANT_GEMV;
    c.p0 = std::min(lanes, 64);
    c.p1 = 1;
    c.p3 = lanes / c.p0;
    c.p5 = 3;
    set_waves(p, kind, &c);
    const int pos = positions(p, c);
    if (refusal(p, c, kind)) continue;
    double cost = 0.3 * ((double)(lanes * pos) / (double)chunks - 1.0) + (longer ? 0.01 : (alone ? 0.05 : 0.02)) * std::max(0, pos - (f16 ? 3 : 2));
    double waves = (double)rows * lanes / 64.0;
    for (; waves < 1024.0; waves *= 2.0) cost += 0.1 * std::min(1.0, 1024.0 / waves - 1.0);
    for (; waves > 1024.0; waves *= 0.5) cost += (alone && !longer ? 0.03 : 0.05) * std::min(1.0, waves / 1024.0 - 1.0);
    for (int l = lanes; l > 64; l /= 2) cost += 0.06;
    if (found && cost >= best) continue;
    best = cost;
    *out = c;
    found = true;
  }
  return found;
}

// Every instance the launches above can reach, in prepare mode (see launch_kernel).
int prepare_gemv_one_kernels() {
  Problem p;
  memset(&p, 0, sizeof p);
  for (p.format = 0; p.format < 3; ++p.format)
    for (p.x_dtype = 0; p.x_dtype < 2; ++p.x_dtype)
      for (int kind : {ONE_SINGLE, ONE_GROUP, ONE_PAIR})
        for (int pro : {TLHIP_PRO_NONE, TLHIP_PRO_RMSNORM, TLHIP_PRO_GATED_MUL})
          for (int pos = 1; pos <= 6; ++pos)
            for (int units : {1, 2, 4})
              if (const void* fn = instance(p, pos, units, pro, kind)) {
                const int rc = launch_kernel(fn, dim3(1), dim3(64), nullptr, 0, nullptr);
                if (rc) return rc;
              }
  return TLHIP_OK;
}

}  // namespace tlhip
