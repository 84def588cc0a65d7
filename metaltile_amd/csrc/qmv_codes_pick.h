// The instances of the matrix-core GEMV on codes, a translation unit per element type and kind of group.
#pragma once
#include "qmv_codes_impl.h"

namespace mtq {

struct CodesInstance {
    const void* fn;
    uint32_t stage;   // steps of activations between barriers, at most
    uint32_t (*lds)(uint32_t kw, uint32_t stage, uint32_t waves);
};

template <int DT, int BITS, bool G32, int MT> static CodesInstance codes_instance() {
    return {(const void*)qmv_codes_kernel<DT, BITS, G32, MT>, QcShape<MT>::STAGE, [](uint32_t kw, uint32_t stage, uint32_t waves) { return QcLds<BITS, G32, MT>::bytes(kw, stage, waves); }};
}
template <int DT, bool G32, int MT> static CodesInstance codes_pick_bits(int bits) {
    switch (bits) {
        case 2: return codes_instance<DT, 2, G32, MT>();
        case 3: return codes_instance<DT, 3, G32, MT>();
        case 4: return codes_instance<DT, 4, G32, MT>();
        case 5: return codes_instance<DT, 5, G32, MT>();
        case 6: return codes_instance<DT, 6, G32, MT>();
        default: return codes_instance<DT, 8, G32, MT>();
    }
}
template <int DT, bool G32> static CodesInstance codes_pick(int bits, uint32_t mt) {
    return mt == 1 ? codes_pick_bits<DT, G32, 1>(bits) : mt == 2 ? codes_pick_bits<DT, G32, 2>(bits) : codes_pick_bits<DT, G32, 3>(bits);
}

}  // namespace mtq
