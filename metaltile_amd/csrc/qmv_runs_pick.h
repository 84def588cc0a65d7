// The instances of the K-run matrix-core GEMV for one element type.
#pragma once
#include "qmv_runs_impl.h"

namespace mtq {

// Blocks in flight: as many as the registers of a wave hold beside the activations. Eight waves to a block where sixteen do
// not hold four steps each (8192 x 8192, 16 rows 18.4 us, eight waves 15.7), and on short rows, where they have one step each.
template <int DT, int BITS, int G> static const void* runs_pick_steps(bool sliced, uint32_t xs) {
    if constexpr (BITS == 4) {
        if (sliced) return (const void*)qmv_slices_kernel<DT, 4, G, 5, G == 32 ? 2 : 3>;
        return xs <= 1 ? (const void*)qmv_runs_kernel<8, DT, 4, G, 1, 3> : xs == 2 ? (const void*)qmv_runs_kernel<16, DT, 4, G, 2, 2> :
               xs == 3 ? (const void*)qmv_runs_kernel<16, DT, 4, G, 3, 1> : (const void*)qmv_runs_kernel<8, DT, 4, G, 4, 1>;
    } else {
        if (sliced) return (const void*)qmv_slices_kernel<DT, 8, G, 10, 1>;
        return xs <= 2 ? (const void*)qmv_runs_kernel<16, DT, 8, G, 2, 2> : xs <= 4 ? (const void*)qmv_runs_kernel<16, DT, 8, G, 4, 1> : (const void*)qmv_runs_kernel<16, DT, 8, G, 5, 1>;
    }
}
template <int DT> static const void* runs_pick_type(int bits, uint32_t G, bool sliced, uint32_t xs) {
    if (bits == 4) return G == 32 ? runs_pick_steps<DT, 4, 32>(sliced, xs) : G == 64 ? runs_pick_steps<DT, 4, 64>(sliced, xs) : runs_pick_steps<DT, 4, 128>(sliced, xs);
    return G == 32 ? runs_pick_steps<DT, 8, 32>(sliced, xs) : G == 64 ? runs_pick_steps<DT, 8, 64>(sliced, xs) : runs_pick_steps<DT, 8, 128>(sliced, xs);
}

}  // namespace mtq
