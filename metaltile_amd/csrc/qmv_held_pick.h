// The instances of the GEMV with its activations in LDS, a translation unit per element type and kind of group.
#pragma once
#include "qmv_held_impl.h"

namespace mtq {

struct HeldInstance {
    const void* fn;
    uint32_t (*lds)(uint32_t K, uint32_t rpl, uint32_t waves);
};

// rows: 1, or more (up to 16); least: the smallest offset of the codes (f16, 4 bits plain or RMS-normalised, 8 bits plain, one row)
template <int DT, int BITS, bool G32> static HeldInstance held_instance(int mode, uint32_t rows, bool least) {
    HeldInstance k{nullptr, [](uint32_t K, uint32_t rpl, uint32_t waves) { return QhLds<BITS, G32>::bytes(K, rpl, waves); }};
    constexpr bool L1 = DT == DT_F16 && (BITS == 4 || BITS == 8), LN = DT == DT_F16 && BITS == 4;
    if (mode == HELD_NORM) k.fn = least ? (const void*)qmv_held_kernel<DT, BITS, G32, 2, HELD_NORM, LN> : (const void*)qmv_held_kernel<DT, BITS, G32, 2, HELD_NORM, false>;
    else if (mode == HELD_PLAIN) k.fn = rows == 1 ? (const void*)qmv_held_kernel<DT, BITS, G32, 1, HELD_PLAIN, L1> : (const void*)qmv_held_kernel<DT, BITS, G32, 4, HELD_PLAIN, false>;
    else if constexpr (BITS == 4) k.fn = (const void*)qmv_held_kernel<DT, BITS, G32, 2, HELD_GATED, false>;
    return k;
}
template <int DT, bool G32> static HeldInstance held_pick_bits(int bits, int mode, uint32_t rows, bool least) {
    switch (bits) {
        case 2: return held_instance<DT, 2, G32>(mode, rows, least);
        case 3: return held_instance<DT, 3, G32>(mode, rows, least);
        case 4: return held_instance<DT, 4, G32>(mode, rows, least);
        case 5: return held_instance<DT, 5, G32>(mode, rows, least);
        case 6: return held_instance<DT, 6, G32>(mode, rows, least);
        default: return held_instance<DT, 8, G32>(mode, rows, least);
    }
}

}  // namespace mtq
