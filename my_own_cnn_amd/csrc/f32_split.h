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
constexpr float kSplitScale = 8388608.0f;       // 2^23: the scale of staged values
constexpr float kSplitUnscale = 0x1p-46f;       // of a product's two
constexpr float kFltMax = 3.4028234663852886e38f;
constexpr unsigned kNone = 0x80000000u;         // a buffer offset that reads zero

struct Split8 {
  v4u p[3];
};

// Eight fp32 values times `scale` as three bf16 each.  With a scale of 2^23 every fp32 value below
// 2^104 is carried exactly, subnormals among them: a residual of the scaled value is a multiple of
// 2^-126, so each piece is zero or a normal bf16, and the corrections of a product that fp32 holds
// stay above the subnormal range.  From about 2^105 a value becomes infinite, and whatever it reaches infinite
// or NaN.
__device__ __forceinline__ Split8 split8(const v4f& lo, const v4f& hi, float scale) {
  Split8 out;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const v2f v = j < 2 ? v2f{lo[2 * j] * scale, lo[2 * j + 1] * scale} : v2f{hi[2 * j - 4] * scale, hi[2 * j - 3] * scale};
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
