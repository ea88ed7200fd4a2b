// quantizeLinearWeight (src/backend/quantize.ts:77-131) on the device, for
// quantize-at-load of weights that are already resident: same bits as the host
// routine for every input (f64 arithmetic for the scale reciprocal and the
// product, Math.round ties toward +infinity, the reference's f16 encoder with
// its round-half-up subnormals).
//
// HBM-bound: 4 bytes read and 1 + 2/G written per weight, if the f64 arithmetic keeps up.
// quantize_int8_groups_kernel (groups of 16..256, a power of two): a lane holds 4 weights of a
// group in registers, the lanes of a group find its maximum by exchanges, and one lane of four
// divides for each of the wave's four pieces in flight: one read, no LDS, no barrier, a quarter of
// a division per 4 weights.  quantize_int8_grouped_kernel (any other group size): one workgroup
// per weight row at a time, the group's maximum in LDS by an unsigned atomic max on the float bits
// (non-negative floats order like their bit patterns; NaN is skipped, as `a > max` is false for
// NaN in the reference), the weights read twice, a division per 4 weights.  12288 x 4096 in groups
// of 64: 81.8 us with the latter, 45.7 us (5.5 TB/s) with the former.
#include <type_traits>

#include "device_utils.h"

namespace tlhip {
namespace {

// quantize.ts:22-47
__device__ __forceinline__ uint32_t encode_f16_ref(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const uint32_t sign = (u >> 16) & 0x8000u;
  const int e16 = int((u >> 23) & 0xffu) - 112;
  const uint32_t frac = u & 0x007fffffu;
  if (e16 >= 31) return sign | 0x7c00u;
  if (e16 >= 1) {
    uint32_t h = sign | (uint32_t(e16) << 10) | (frac >> 13);
    const uint32_t rem = frac & 0x1fffu;
    if (rem > 0x1000u || (rem == 0x1000u && (h & 1u))) h += 1;
    return h;
  }
  if (e16 < -10) return sign;
  const uint32_t shifted = (frac | 0x00800000u) >> uint32_t(1 - e16);
  return sign | ((shifted >> 13) + ((shifted >> 12) & 1u));
}

// quantize.ts:50-60 for a non-negative pattern; exact in double
__device__ __forceinline__ double decode_f16_ref(uint32_t h) {
  const int e = (h >> 10) & 0x1f;
  const int f = h & 0x3ff;
  if (e == 0) return ldexp((double)f, -24);
  if (e == 31) return f ? __builtin_nan("") : __builtin_inf();
  return ldexp((double)(1024 + f), e - 25);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}

__device__ __forceinline__ uint32_t quantize_one(float w, double inv) {
#pragma clang fp contract(off)  // t is the rounded product, in t - f as well
  const double t = (double)w * inv;
  // Math.round: up from a half on.  f beyond the integers saturates, t - f of an infinity is NaN;
  // the clamp before the step keeps it from overflowing.
  const double f = floor(t);
  int q = t == t ? (int)fmin(fmax(f, -128.0), 127.0) : 0;  // NaN -> 0 (NaN & 0xff in JavaScript)
  q += t - f >= 0.5 ? 1 : 0;
  q = q > 127 ? 127 : (q < -127 ? -127 : q);
  return (uint32_t)q & 0xffu;
}

// LANES: lanes of a group (4 weights each)
template <int LANES>
__global__ __launch_bounds__(256) void quantize_int8_groups_kernel(const float4_t* __restrict__ w, int64_t n_words,
                                                                  uint32_t* __restrict__ packed, uint16_t* __restrict__ scales) {
  constexpr int U = 4;
  const int64_t stride = (int64_t)gridDim.x * (256 * U);
  const int quad = threadIdx.x & 3;
  for (int64_t first = (int64_t)blockIdx.x * (256 * U); first < n_words; first += stride) {
    const int64_t base = first + threadIdx.x;
    float4_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(w + (base + u * 256 < n_words ? base + u * 256 : n_words - 1));
    uint32_t top = 0;  // of the piece this lane divides for
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float m = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = fabsf(v[u][e]);
        if (a > m) m = a;  // false for NaN
      }
      uint32_t t = __builtin_bit_cast(uint32_t, m);  // non-negative floats order like their bits
      t = max(t, dpp<0xB1>(t));   // quad_perm [1,0,3,2]
      t = max(t, dpp<0x4E>(t));   // quad_perm [2,3,0,1]
      if (LANES >= 8) t = max(t, dpp<0x141>(t));   // row_half_mirror
      if (LANES >= 16) t = max(t, dpp<0x140>(t));  // row_mirror
      if (LANES >= 32) t = max(t, (uint32_t)__shfl_xor((int)t, 16));
      if (LANES >= 64) t = max(t, (uint32_t)__shfl_xor((int)t, 32));
      top = u == quad ? t : top;
    }
    const uint32_t sbits = encode_f16_ref(__builtin_bit_cast(float, top));
    const double s = (double)half_bits_to_float(sbits);  // exact, never NaN
    const uint64_t inv_bits = __builtin_bit_cast(uint64_t, s > 0 ? 127.0 / s : 0.0);
    const uint32_t lo = (uint32_t)inv_bits, hi = (uint32_t)(inv_bits >> 32);
    auto piece = [&](auto which) {
      constexpr int P = decltype(which)::value, FROM = P * 0x55;  // quad_perm [P,P,P,P]
      const double inv = __builtin_bit_cast(double, ((uint64_t)dpp<FROM>(hi) << 32) | dpp<FROM>(lo));
      const uint32_t scale = dpp<FROM>(sbits);
      const int64_t i = base + P * 256;
      if (i < n_words) {
        packed[i] = quantize_one(v[P][0], inv) | (quantize_one(v[P][1], inv) << 8) | (quantize_one(v[P][2], inv) << 16) |
                    (quantize_one(v[P][3], inv) << 24);
        if ((threadIdx.x & (LANES - 1)) == 0) scales[i / LANES] = (uint16_t)scale;
      }
    };
    piece(std::integral_constant<int, 0>());
    piece(std::integral_constant<int, 1>());
    piece(std::integral_constant<int, 2>());
    piece(std::integral_constant<int, 3>());
  }
}

__global__ __launch_bounds__(256) void quantize_int8_grouped_kernel(const float* __restrict__ w, int64_t n, int k,
                                                                   int g, uint32_t* __restrict__ packed,
                                                                   uint16_t* __restrict__ scales) {
  extern __shared__ uint32_t amax_bits[];  // one per group of the row
  const int groups = k / g, words = k / 4;
  for (int64_t row = blockIdx.x; row < n; row += gridDim.x) {
    const float4_t* wr = (const float4_t*)(w + row * k);
    for (int i = threadIdx.x; i < groups; i += blockDim.x) amax_bits[i] = 0u;
    __syncthreads();
    for (int i = threadIdx.x; i < words; i += blockDim.x) {
      const float4_t v = wr[i];
      float m = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = fabsf(v[e]);
        if (a > m) m = a;  // false for NaN
      }
      // a word never straddles two groups: g is a multiple of 4
      atomicMax(&amax_bits[(i * 4) / g], __builtin_bit_cast(uint32_t, m));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < groups; i += blockDim.x)
      scales[row * groups + i] = (uint16_t)encode_f16_ref(__builtin_bit_cast(float, amax_bits[i]));
    for (int i = threadIdx.x; i < words; i += blockDim.x) {
      const uint32_t sbits = encode_f16_ref(__builtin_bit_cast(float, amax_bits[(i * 4) / g]));
      const double s = decode_f16_ref(sbits);
      const double inv = s > 0 ? 127.0 / s : 0.0;
      const float4_t v = wr[i];
      packed[row * words + i] = quantize_one(v[0], inv) | (quantize_one(v[1], inv) << 8) |
                                (quantize_one(v[2], inv) << 16) | (quantize_one(v[3], inv) << 24);
    }
    __syncthreads();  // amax_bits is reused by the next row
  }
}

}  // namespace
}  // namespace tlhip

using namespace tlhip;

extern "C" int tlhip_quantize_int8_grouped_device(const float* weight, int64_t n, int64_t k, int64_t group_size,
                                                  uint32_t* packed, uint16_t* scales, tlhip_stream_t stream) {
  TLHIP_REQUIRE_INIT();
  if (n < 0 || k < 0) return set_error(TLHIP_ERR_INVALID, "quantize: negative shape");
  if (k % 4 != 0) return set_error(TLHIP_ERR_INVALID, "quantize: K=%lld must be divisible by 4", (long long)k);
  if (group_size <= 0 || k % group_size != 0)
    return set_error(TLHIP_ERR_INVALID, "quantize: K=%lld must be divisible by groupSize=%lld", (long long)k,
                     (long long)group_size);
  if (group_size % 4 != 0)
    return set_error(TLHIP_ERR_INVALID, "quantize (device): groupSize=%lld must be a multiple of 4",
                     (long long)group_size);
  if (n == 0 || k == 0) return TLHIP_OK;
  if (!weight || !packed || !scales) return set_error(TLHIP_ERR_INVALID, "quantize: null pointer");
  if (((uintptr_t)weight & 15) != 0) return set_error(TLHIP_ERR_INVALID, "quantize: weight must be 16-byte aligned");
  if (k > (1 << 22)) return set_error(TLHIP_ERR_INVALID, "quantize (device): K=%lld above 4194304", (long long)k);
  const size_t lds = (size_t)(k / group_size) * sizeof(uint32_t);
  if (lds > 64 * 1024)
    return set_error(TLHIP_ERR_INVALID, "quantize (device): %lld groups per row do not fit LDS",
                     (long long)(k / group_size));
  const int lanes = (int)group_size / 4;
  if (group_size >= 16 && group_size <= 256 && (group_size & (group_size - 1)) == 0) {
    const int64_t words = n * (k / 4), blocks = (words + 1023) / 1024;
    auto kernel = lanes == 4    ? quantize_int8_groups_kernel<4>
                  : lanes == 8  ? quantize_int8_groups_kernel<8>
                  : lanes == 16 ? quantize_int8_groups_kernel<16>
                  : lanes == 32 ? quantize_int8_groups_kernel<32>
                                : quantize_int8_groups_kernel<64>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(blocks < (1 << 20) ? blocks : (1 << 20))), dim3(256), 0, resolve_stream(stream),
                       (const float4_t*)weight, words, packed, scales);
    TLHIP_CHECK_HIP(hipGetLastError());
    return TLHIP_OK;
  }
  const int64_t cap = (int64_t)device_cu_count() * 8;
  const int grid = (int)(n < cap ? n : cap);
  hipLaunchKernelGGL(quantize_int8_grouped_kernel, dim3(grid), dim3(256), lds, resolve_stream(stream), weight, n,
                     (int)k, (int)group_size, packed, scales);
  TLHIP_CHECK_HIP(hipGetLastError());
  return TLHIP_OK;
}
