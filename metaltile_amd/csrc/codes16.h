// Sixteen packed codes of any width as operands of the 16x16x32 matrix instruction.
#pragma once
#include "mfma16.h"

namespace mtq {

// What the conversion adds to every code: the power of two in whose mantissa (10 bits in f16, 7 in bf16) a code that stands AT bits up is the
// code itself. The f32 sums carry the offset, so it is to be small, and AT large. LEAST: the one that leaves no more room than the
// code needs, and 8-bit codes with the offset taken out again by a packed subtraction; else the largest that leaves one of the shifts below
// free, as AT = 0 does. Error of the sums of a row of 1024 f16 4-bit codes, of a result of 2.9, with 1024, 64 and 16: 1.0e-4, 6.4e-6 and 2.2e-6;
// 2.0e-6 in the kernels whose calls LEAST is for. It costs a shift in eight or an addition to each pair (67882 x 2304, 4 bits, norm included, 22.3 ->
// 23.0 us; 14336 x 1664, 8 bits, 9.3 -> 9.8).
template <int DT, int BITS, bool LEAST> struct QcCodes {
    static_assert(!LEAST || DT == DT_F16, "bf16: 128 and less in every kernel");
    static constexpr int ROOM = (DT == DT_F16 ? 10 : 7) - BITS;
    static constexpr int AT = DT == DT_F16 ? (BITS == 4 && !LEAST ? 4 : ROOM) : BITS == 2 ? 4 : BITS == 3 ? 3 : BITS == 5 ? 1 : 0;
    static constexpr bool TAKEN_OUT = BITS == 8 && (LEAST || DT == DT_BF16);
    static constexpr int LOG2 = (DT == DT_F16 ? 10 : 7) - (TAKEN_OUT ? 0 : AT);
    static constexpr float MAGIC = TAKEN_OUT ? 0.0f : (float)(1 << LOG2);
    static constexpr uint32_t KOR = (DT == DT_F16 ? (uint32_t)(15 + LOG2) << 10 : (uint32_t)(127 + LOG2) << 7) * 0x10001u;   // twice, in the element type
};

// 16 consecutive codes (2 * BITS bytes) -> two MFMA operands of MAGIC + code, as pairs (i, i + 8): the eight codes between
// them are whole bytes at every width, so that one byte permute puts a 16-bit window of the one half of the codes
// into the lower half of a dword and the same window of the other half into the upper one. kor: QcCodes::KOR, opaque.
template <int DT, int BITS, bool LEAST> __device__ __forceinline__ void qc_convert(const uint32_t* d, uint32_t kor, kr_u32x4 (&o)[2]) {
    using C = QcCodes<DT, BITS, LEAST>;
    constexpr int AT = C::AT;
    constexpr uint32_t m = ((1u << BITS) - 1u) * 0x10001u << AT;
    // (a shift to the left carries less than AT bits of the lower half into the upper one: the mask takes them away)
    auto put = [&](int i, uint32_t window, int shift) { o[i / 4][i % 4] = ((shift >= AT ? window >> (shift - AT) : window << (AT - shift)) & m) | kor; };
    if constexpr (BITS == 2) {
#pragma unroll
        for (int i = 0; i < 8; i++) put(i, d[0], 2 * i);
    } else if constexpr (BITS == 3) {
        const uint32_t a = __builtin_amdgcn_perm(d[1], d[0], 0x04030100u), b = __builtin_amdgcn_perm(d[1], d[0], 0x05040201u);
#pragma unroll
        for (int i = 0; i < 5; i++) put(i, a, 3 * i);
#pragma unroll
        for (int i = 5; i < 8; i++) put(i, b, 3 * i - 8);
    } else if constexpr (BITS == 4) {
        const uint32_t a = __builtin_amdgcn_perm(d[1], d[0], 0x05040100u), b = __builtin_amdgcn_perm(d[1], d[0], 0x07060302u);
#pragma unroll
        for (int i = 0; i < 4; i++) put(i, a, 4 * i);
#pragma unroll
        for (int i = 0; i < 4; i++) put(i + 4, b, 4 * i);
    } else if constexpr (BITS == 5) {
        const uint32_t h = __builtin_amdgcn_alignbyte(d[2], d[1], 1), t = __builtin_amdgcn_alignbyte(d[1], d[0], 3);   // bytes 5..8, 3..6
        const uint32_t w0 = __builtin_amdgcn_perm(h, d[0], 0x05040100u), w1 = __builtin_amdgcn_perm(h, d[0], 0x06050201u);
        const uint32_t w2 = __builtin_amdgcn_perm(h, d[0], 0x07060302u), w3 = __builtin_amdgcn_perm(d[2], t, 0x05040100u);
        put(0, w0, 0); put(1, w0, 5); put(2, w0, 10); put(3, w1, 7); put(4, w2, 4); put(5, w3, 1); put(6, w3, 6); put(7, w3, 11);
    } else if constexpr (BITS == 6) {
        const uint32_t h = __builtin_amdgcn_alignbyte(d[2], d[1], 2), t = __builtin_amdgcn_alignbyte(d[1], d[0], 3);   // bytes 6..9, 3..6
        const uint32_t w0 = __builtin_amdgcn_perm(h, d[0], 0x05040100u), w1 = __builtin_amdgcn_perm(h, d[0], 0x06050201u);
        const uint32_t w2 = __builtin_amdgcn_perm(d[2], t, 0x06050100u), w3 = __builtin_amdgcn_perm(d[2], d[1], 0x07060100u);
        put(0, w0, 0); put(1, w0, 6); put(2, w1, 4); put(3, w1, 10); put(4, w2, 0); put(5, w2, 6); put(6, w3, 4); put(7, w3, 10);
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t lo = d[i / 4], hi = d[2 + i / 4];
            if constexpr (DT == DT_F16) {
                typedef _Float16 half2 __attribute__((ext_vector_type(2)));
                const uint32_t v = __builtin_amdgcn_perm(hi, lo, 0x0C040C00u + 0x00010001u * (uint32_t)(i % 4));
                o[i / 4][i % 4] = C::TAKEN_OUT ? __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2, v | kor) - (half2)(_Float16)1024.0f) : (v << AT) | kor;
            } else {   // integers up to 255 are exact in bf16: the upper halves of their f32 forms
                const uint32_t f0 = __float_as_uint((float)((lo >> (8 * (i % 4))) & 0xFFu)), f1 = __float_as_uint((float)((hi >> (8 * (i % 4))) & 0xFFu));
                o[i / 4][i % 4] = __builtin_amdgcn_perm(f1, f0, 0x07060302u);
            }
        }
    }
}

// A lane's 16 codes out of LDS: 2 * BITS bytes at `at` (4-byte aligned but for odd quarters of 3- and 5-bit codes, which
// start 2 bytes behind it).
template <int BITS> __device__ __forceinline__ void qc_read(const unsigned char* at, uint32_t odd, uint32_t (&d)[4]) {
    if constexpr (BITS == 8) {
        const kr_u32x4 v = *(const kr_u32x4*)at;
        d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
    } else if constexpr (BITS == 4) {
        const kr_u32x2 v = *(const kr_u32x2*)at;
        d[0] = v.x; d[1] = v.y;
    } else {
        constexpr int n = BITS == 2 ? 1 : BITS == 3 ? 2 : 3;
#pragma unroll
        for (int i = 0; i < n; i++) d[i] = ((const uint32_t*)at)[i];
        if constexpr (BITS == 3) {
            d[0] = __builtin_amdgcn_alignbyte(d[1], d[0], odd);
            d[1] = __builtin_amdgcn_alignbyte(0u, d[1], odd);
        }
        if constexpr (BITS == 5) {
            d[0] = __builtin_amdgcn_alignbyte(d[1], d[0], odd);
            d[1] = __builtin_amdgcn_alignbyte(d[2], d[1], odd);
            d[2] = __builtin_amdgcn_alignbyte(0u, d[2], odd);
        }
    }
}

}  // namespace mtq
