// The instances of the GEMV with its activations in LDS, a translation unit per element type and kind of group.
#pragma once
#include "qmv_held_impl.h"

namespace mtq {

struct HeldInstance {
    const void* fn;
    uint32_t (*lds)(uint32_t K, uint32_t rpl, uint32_t waves);
};

// rows: 1, or more (up to 16)
template <int DT, int BITS, bool G32> static HeldInstance held_instance(int mode, uint32_t rows) {
    HeldInstance k{nullptr, [](uint32_t K, uint32_t rpl, uint32_t waves) { return QhLds<BITS, G32>::bytes(K, rpl, waves); }};
    if (mode == HELD_NORM) k.fn = (const void*)qmv_held_kernel<DT, BITS, G32, 2, HELD_NORM>;
    else if (mode == HELD_PLAIN) k.fn = rows == 1 ? (const void*)qmv_held_kernel<DT, BITS, G32, 1, HELD_PLAIN> : (const void*)qmv_held_kernel<DT, BITS, G32, 4, HELD_PLAIN>;
    else if constexpr (BITS == 4) k.fn = (const void*)qmv_held_kernel<DT, BITS, G32, 2, HELD_GATED>;
    return k;
}
template <int DT, bool G32> static HeldInstance held_pick_bits(int bits, int mode, uint32_t rows) {
    switch (bits) {
        case 2: return held_instance<DT, 2, G32>(mode, rows);
        case 3: return held_instance<DT, 3, G32>(mode, rows);
        case 4: return held_instance<DT, 4, G32>(mode, rows);
        case 5: return held_instance<DT, 5, G32>(mode, rows);
        case 6: return held_instance<DT, 6, G32>(mode, rows);
        default: return held_instance<DT, 8, G32>(mode, rows);
    }
}

}  // namespace mtq
