// sx8_gemm_ops.h -- what the prefill GEMM kernels share: the weight sources, and the decode of
// a sub-block's levels into fp16 MFMA operands.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sx8_device.h"

namespace sx8 {

// Weight sources: the v4.4 layout (hdr + levels) or the kb-major split arrays.
struct WeightSrc {
    const uint8_t* hdr;
    const uint8_t* levels;
    const uint16_t* dmin;
    const uint16_t* dmax;
    const uint8_t* config;
    const uint8_t* coeff;
    const uint8_t* hi;
    const uint8_t* lo;
};

}  // namespace sx8

// c as an exact fp16 pair (c, c)
__device__ __forceinline__ uint32_t sx8_coeff_pair_f16(int c) {
    const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)(float)c);
    return h | (h << 16);
}

// The 6-bit levels of a sub-block's 8 weights, two per word: weight i in the low half of lv[i],
// weight i + 4 in the high half (i < 4).  H: its hi-nibble word; P, sel: its two lo-quad bytes
// are the low half of P (sel = kQuadLo) or the high half (kQuadHi).  The halves are read as
// fp16 bit patterns by sx8_dec_weights: a level is then the subnormal lv 2^-24, exact, so no
// integer conversion is needed (12 instructions; byte-wise unpacking and eight conversions to
// float took 21).
constexpr uint32_t kQuadLo = 0x0C010C00u, kQuadHi = 0x0C030C02u;
__device__ __forceinline__ void sx8_dec_levels(uint32_t H, uint32_t P, uint32_t sel, uint32_t (&lv)[4]) {
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
    const us2 q = __builtin_bit_cast(us2, __builtin_amdgcn_perm(0u, P, sel));    // P0, P1 as halves
    const us2 s6 = {6, 6}, s4 = {4, 4}, s2 = {2, 2};
    // bits 2 .. 5 of each half from the nibble word, the rest from the quad word: one v_bfi_b32
    // (the compiler makes two instructions of the masks it can narrow)
    auto merge = [](uint32_t nib, uint32_t qua) {
        uint32_t r;
        asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "s"(0x003C003Cu), "v"(nib), "v"(qua));
        return r;
    };
    lv[0] = merge(H << 2, __builtin_bit_cast(uint32_t, (us2)(q >> s6)));
    lv[1] = merge(H >> 2, __builtin_bit_cast(uint32_t, (us2)(q >> s4)));
    lv[2] = merge(H >> 6, __builtin_bit_cast(uint32_t, (us2)(q >> s2)));
    lv[3] = merge(H >> 10, __builtin_bit_cast(uint32_t, q) & 0x00030003u);
}

// Step of a sub-block as sx8_dec_weights takes it: 2^24 step, undoing the levels' scale (both
// factors exact, so step lv is the same product).
constexpr int kStepExp = 24;
constexpr float kStepFloor = 1e-10f * 16777216.0f;

// The sub-block's weights rlo + step lv, each multiply-add rounded once to fp16, in order.
typedef uint32_t sx8_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ sx8_u32x4 sx8_dec_weights(const uint32_t (&lv)[4], float rlo, float step24) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const sx8_half2 a = __builtin_bit_cast(sx8_half2, lv[2 * (i & 1)]);
        const sx8_half2 b = __builtin_bit_cast(sx8_half2, lv[2 * (i & 1) + 1]);
        const float we = __builtin_fmaf(step24, (float)(i < 2 ? a.x : a.y), rlo);
        const float wo = __builtin_fmaf(step24, (float)(i < 2 ? b.x : b.y), rlo);
        const sx8_half2 v = {(_Float16)we, (_Float16)wo};
        w[i] = __builtin_bit_cast(uint32_t, v);
    }
    return sx8_u32x4{w[0], w[1], w[2], w[3]};
}
