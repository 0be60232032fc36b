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

// Amplitudes and weights are scaled by the power of two that brings the largest of a range to
// [2^(kHalfTop - 1), 2^kHalfTop) before they are split.  FP16's smallest step is 2^-24 whatever the value, so
// what the two parts leave of a value is 2^-23 of itself down to 2^-16 of the largest, and 2^-39 of the
// largest below.  Scaled to [1/2, 1) it was 2^-25 of the largest: 1.5e-6 to 2.1e-6 of the field of 100000 emitters
// of 1 beside one of 1000, and 6e-7 to 1e-6 of the gradients with one bright pixel a square, where FP32
// phasors and weights leave 3.6e-7.
constexpr int kHalfTop = 14;

// (c, s) as FP16 pairs: h rounded to nearest, l the remainder (exact in FP32) rounded to nearest.
// No instruction that writes an operand stands in an asm (the empty ones write none): the compiler keeps
// the wait states in front of a matrix instruction only for writers that it sees.  `one`, hidden from it,
// keeps a remainder one instruction (v_fma_mix_f32 reads h as it is).  MIX: v_fma_mixlo/hi_f16 round it as
// well; otherwise both are packed by one conversion, as each write of half a register costs its reader a
// wait.  100000 emitters on 512 x 512: 1.068 ms with MIX, 1.042 without; with amplitudes, where the
// products fill the waits, 78.4 ms without and 77.4 with it (two shots of 1e6 on 1024 x 1024).
template <bool MIX = false>
__device__ __forceinline__ void split_half(float c, float s, half2_t& h, half2_t& l)
{
    h = __builtin_convertvector((float2_t{c, s}), half2_t);
    float one = 1.f;
    asm("" : "+s"(one));
    float lc = __builtin_fmaf(-(float)h.x, one, c), ls = __builtin_fmaf(-(float)h.y, one, s);
    if (!MIX) asm("" : "+v"(lc), "+v"(ls));
    l = __builtin_convertvector((float2_t{lc, ls}), half2_t);
    asm("" : "+v"(l));  // rot90 turns the pair, and does not form it anew in the other order
}

// (x, y) -> (-y, x): one v_pk_mul_f16 that reads v turned (the factors are hidden as above, or the turn
// would become an instruction of its own)
__device__ __forceinline__ half2_t rot90(half2_t v)
{
    unsigned sign = 0x3c00bc00u;  // (-1, 1)
    asm("" : "+s"(sign));
    return half2_t{v.y, v.x} * __builtin_bit_cast(half2_t, sign);
}

}  // namespace idisim
