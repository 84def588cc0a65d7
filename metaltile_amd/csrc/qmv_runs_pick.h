// The instances of the K-run matrix-core GEMV for one element type.
#pragma once
#include "qmv_runs_impl.h"

namespace mtq {

// Blocks in flight: as many as the registers of a wave hold beside the activations. Eight waves to a block where sixteen do
// not hold four steps each (8192 x 8192, 16 rows 18.4 us, eight waves 15.7), and on short rows, where they have one step each (8 bits, 5
// rows: 16384 x 512 9.1 us, eight waves 6.6; 4096 x 1024 6.0, 4.6). few: up to 8 activation rows.
template <bool PAIRED, int DT, int BITS, int G> static RunsInstance runs_pick_steps(bool sliced, uint32_t xs, bool few) {
    if constexpr (BITS == 4) {
        if (sliced) return {(const void*)qmv_slices_kernel<PAIRED, DT, 4, G, 5, G == 32 ? 2 : 3>, 512};
        if (xs <= 1) return {(const void*)qmv_runs_kernel<PAIRED, false, 8, DT, 4, G, 1, 3>, 512};
        if (xs == 2) return {few ? (const void*)qmv_runs_kernel<PAIRED, false, 16, DT, 4, G, 2, 2> : (const void*)qmv_runs_kernel<PAIRED, true, 16, DT, 4, G, 2, 2>, 1024};
        if (xs == 3) return {(const void*)qmv_runs_kernel<PAIRED, true, 16, DT, 4, G, 3, 1>, 1024};
        return {(const void*)qmv_runs_kernel<PAIRED, true, 8, DT, 4, G, 4, 1>, 512};
    } else {
        if (sliced) return {(const void*)qmv_slices_kernel<PAIRED, DT, 8, G, 10, 1>, 512};
        if (xs <= 1) return {(const void*)qmv_runs_kernel<PAIRED, false, 8, DT, 8, G, 1, 3>, 512};
        if (xs == 2) return {(const void*)qmv_runs_kernel<PAIRED, false, 16, DT, 8, G, 2, 2>, 1024};
        return {xs <= 4 ? (const void*)qmv_runs_kernel<PAIRED, true, 16, DT, 8, G, 4, 1> : (const void*)qmv_runs_kernel<PAIRED, true, 16, DT, 8, G, 5, 1>, 1024};
    }
}
// paired: rows are whole numbers of 128 bytes (of 8-bit codes every row is)
template <bool PAIRED, int DT> static RunsInstance runs_pick_type(int bits, uint32_t G, bool sliced, uint32_t xs, bool few) {
    if constexpr (PAIRED)
        if (bits == 8) return G == 32 ? runs_pick_steps<true, DT, 8, 32>(sliced, xs, few) : G == 64 ? runs_pick_steps<true, DT, 8, 64>(sliced, xs, few) : runs_pick_steps<true, DT, 8, 128>(sliced, xs, few);
    return G == 32 ? runs_pick_steps<PAIRED, DT, 4, 32>(sliced, xs, few) : G == 64 ? runs_pick_steps<PAIRED, DT, 4, 64>(sliced, xs, few) : runs_pick_steps<PAIRED, DT, 4, 128>(sliced, xs, few);
}
template <int DT> static RunsInstance runs_pick_type(bool paired, int bits, uint32_t G, bool sliced, uint32_t xs, bool few) {
    return paired ? runs_pick_type<true, DT>(bits, G, sliced, xs, few) : runs_pick_type<false, DT>(bits, G, sliced, xs, few);
}

}  // namespace mtq
