// fp32 operands as three bfloat16 parts for v_mfma_f32_32x32x16_bf16 (conv_split.hip has the reasons)
#ifndef SINGA_AMD_CSRC_SPLIT_PARTS_H_
#define SINGA_AMD_CSRC_SPLIT_PARTS_H_

// Operands are multiplied by this before they are split, results by the square of its inverse: three bfloat16 values hold 24 bits
// of a number from 2^-110 on, and with this all bits of every fp32 number down to the smallest subnormal one.  What comes out
// beyond 2^96 is formed again anyway.
constexpr float kSplitScale = 65536.f, kSplitUnscale = 1.f / kSplitScale / kSplitScale;

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ v16f mfma(v4u a, v4u b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ unsigned pack2(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{a, b}, bf16x2));
}
__device__ __forceinline__ float lo_f(unsigned p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float hi_f(unsigned p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// The parts of two fp32 values, packed
struct Parts {
  unsigned p[3];
};
__device__ __forceinline__ Parts split2(float a, float b) {
  a *= kSplitScale, b *= kSplitScale;
  const unsigned p0 = pack2(a, b);
  const float ra = a - lo_f(p0), rb = b - hi_f(p0);
  const unsigned p1 = pack2(ra, rb);
  return {{p0, p1, pack2(ra - lo_f(p1), rb - hi_f(p1))}};
}

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) < __builtin_inff(); }

}  // namespace

#endif  // SINGA_AMD_CSRC_SPLIT_PARTS_H_
