// ifa_dequant_q4.h -- the dequantised halves of eight 4-bit codes, value = half(q * scale + base) rounded ONCE.  A byte 0..15 read as
// an FP8 E4M3 number is b * 2^-9 exactly (codes 0..7 are its subnormals m * 2^-9, codes 8..15 the first binade (8 + m) * 2^-9: one
// linear ramp), so v_cvt_scalef32_pk_f16_fp8 with the scale 2^9 turns two codes into two exact halves, and v_pk_fma_f16 forms two
// values: 11 VALU instructions per 8 weights in the MO layout's order, 15 in the tiled order.  The fp32 form before (two codes per
// conversion to float, eight v_fma_f32, four conversions to half: 19) took 78 cycles a word on a SIMD, this one 46
// (Llama-2-7B: nine queries 2.80 -> 2.65 ms, a prompt of 37 tokens 3.53 -> 3.43, of 512 10.34 -> 10.04; the same outputs).
// The reference's dequantisation kernels round twice (the fp32 sum, then the half): the sum is exact in fp32 -- and the halves the
// same -- unless scale and base are more than 2^9 apart; there the single rounding is the nearer one.
#pragma once
#include <stdint.h>
#include <hip/hip_runtime.h>

namespace ifa {

typedef _Float16 q4_h2 __attribute__((ext_vector_type(2)));

// a block's (base, scale) word: base in the low half, scale in the high half
__device__ __forceinline__ q4_h2 q4_base2(uint32_t w) { const q4_h2 h = __builtin_bit_cast(q4_h2, w); return __builtin_shufflevector(h, h, 0, 0); }
__device__ __forceinline__ q4_h2 q4_scale2(uint32_t w) { const q4_h2 h = __builtin_bit_cast(q4_h2, w); return __builtin_shufflevector(h, h, 1, 1); }

// values of the codes in bytes 0, 1 (HI = false) or 2, 3 of a word of bytes 0..15
template <bool HI>
__device__ __forceinline__ q4_h2 q4_value2(uint32_t bytes, q4_h2 scale2, q4_h2 base2)
{
    return __builtin_elementwise_fma(__builtin_bit_cast(q4_h2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)bytes, 512.0f, HI)), scale2, base2);
}

// MO layout (ifa_gemm_rows_mfma.h): byte b of the word holds element b (low nibble) and element 4 + b (high nibble)
// w[i] = (element 2i, element 2i + 1)
__device__ __forceinline__ void q4x8_dequant_mo(uint32_t cw, q4_h2 scale2, q4_h2 base2, q4_h2 (&w)[4])
{
    const uint32_t lo = cw & 0x0F0F0F0Fu, hi = (cw >> 4) & 0x0F0F0F0Fu;
    w[0] = q4_value2<false>(lo, scale2, base2); w[1] = q4_value2<true>(lo, scale2, base2);
    w[2] = q4_value2<false>(hi, scale2, base2); w[3] = q4_value2<true>(hi, scale2, base2);
}

// tiled and reference layouts: byte b of the word holds element 2b (low nibble) and 2b + 1 (high nibble)
__device__ __forceinline__ void q4x8_dequant(uint32_t cw, q4_h2 scale2, q4_h2 base2, q4_h2 (&w)[4])
{
    q4_h2 v[4];
    q4x8_dequant_mo(cw, scale2, base2, v);                       // elements (0, 2), (4, 6), (1, 3), (5, 7)
    w[0] = __builtin_shufflevector(v[0], v[2], 0, 2); w[1] = __builtin_shufflevector(v[0], v[2], 1, 3);
    w[2] = __builtin_shufflevector(v[1], v[3], 0, 2); w[3] = __builtin_shufflevector(v[1], v[3], 1, 3);
}

// eight codes from the tiled order to the MO order
__device__ __forceinline__ uint32_t q4_word_to_mo(uint32_t cw)
{
    uint32_t o = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) o |= ((cw >> (4 * e)) & 0xFu) << (e < 4 ? 8 * e : 8 * (e - 4) + 4);
    return o;
}

} // namespace ifa
