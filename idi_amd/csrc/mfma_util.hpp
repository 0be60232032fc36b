// FP16 operand fragments of the matrix instructions and the split of FP32 phasors into them, shared
// by the separable forward (separable.hip) and adjoint (adjoint_sep.hip).
#pragma once
#include "device_util.hpp"

namespace idisim {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

union Frag {
    half8_t v;
    half2_t p[4];
};

template <int T>
struct SepTraits;
template <>
struct SepTraits<32> {
    using acc_t = float16_t;
    static constexpr int kStep = 8, kRegs = 16;
    static __device__ __forceinline__ void mma(const Frag& a, const Frag& b, acc_t& c)
    {
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, b.v, c, 0, 0, 0);
    }
    // row of accumulator register i in lane group g = lane / 32
    static __device__ __forceinline__ int row(int i, int g) { return 8 * (i >> 2) + 4 * g + (i & 3); }
};
template <>
struct SepTraits<16> {
    using acc_t = float4_t;
    static constexpr int kStep = 16, kRegs = 4;
    static __device__ __forceinline__ void mma(const Frag& a, const Frag& b, acc_t& c)
    {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v, b.v, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int i, int g) { return 4 * g + i; }
};

// (c, s) as FP16 pairs: h rounded to nearest, l the remainder rounded to nearest.
__device__ __forceinline__ void split_half(float c, float s, half2_t& h, half2_t& l)
{
    h = __builtin_convertvector((float2_t{c, s}), half2_t);
    asm("v_fma_mixlo_f16 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %0, -%1, 1.0, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=&v"(l)
        : "v"(h), "v"(c), "v"(s));
}

// (x, y) -> (-y, x)
__device__ __forceinline__ half2_t rot90(half2_t v)
{
    half2_t r;
    asm("v_pk_mul_f16 %0, %1, 1.0 op_sel:[1,0] op_sel_hi:[0,0] neg_lo:[1,0]" : "=v"(r) : "v"(v));
    return r;
}

}  // namespace idisim
