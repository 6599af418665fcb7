// Three-way bf16 split of fp32 values, shared by the fp32 kernels on the bf16 matrix cores.
#pragma once

#include "qconv_device.h"

namespace miq {
namespace {

typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef __bf16 v2b __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int kSplitLds = 160 * 1024;           // bytes per CU
constexpr unsigned kSmall2 = (17u << 24) - 1u;  // 2 * bits(2^-110) - 1
constexpr unsigned kNone = 0x80000000u;         // a buffer offset that reads zero

struct Split8 {
  v4u p[3];
};

// Eight fp32 values as three bf16 each; `mn` collects the smallest 2 * bits - 1 (zero wraps to the
// largest unsigned value).
__device__ __forceinline__ Split8 split8(const v4f& lo, const v4f& hi, unsigned& mn) {
  Split8 out;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const v2f v = j < 2 ? v2f{lo[2 * j], lo[2 * j + 1]} : v2f{hi[2 * j - 4], hi[2 * j - 3]};
    const unsigned u0 = (__builtin_bit_cast(unsigned, static_cast<float>(v[0])) << 1) - 1u;
    const unsigned u1 = (__builtin_bit_cast(unsigned, static_cast<float>(v[1])) << 1) - 1u;
    mn = min(mn, min(u0, u1));
    const v2b h = __builtin_convertvector(v, v2b);
    const v2f r1 = v2f{v[0] - static_cast<float>(h[0]), v[1] - static_cast<float>(h[1])};
    const v2b m = __builtin_convertvector(r1, v2b);
    const v2f r2 = v2f{r1[0] - static_cast<float>(m[0]), r1[1] - static_cast<float>(m[1])};
    const v2b l = __builtin_convertvector(r2, v2b);
    out.p[0][j] = __builtin_bit_cast(unsigned, h);
    out.p[1][j] = __builtin_bit_cast(unsigned, m);
    out.p[2][j] = __builtin_bit_cast(unsigned, l);
  }
  return out;
}

// 16 and 4 bytes at byte offset voff + soff of a buffer; zero where voff is past its 2^31 - 1 bytes
__device__ __forceinline__ v4f buffer_load16(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
  return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ float buffer_load4(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

}  // namespace
}  // namespace miq
