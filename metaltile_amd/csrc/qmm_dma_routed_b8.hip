// Expert-routed rows on row tiles of up to 160 rows, 8-bit codes (qmm_dma_impl.h): replaces, with many rows per expert, the
// same reference kernels as the 64-row tiles (crates/metaltile-std/src/ffai/moe.rs:2256). A translation unit of its own so that
// it compiles beside the others.
#include "qmm_dma_impl.h"

namespace mtq {

template <int BITS> static const void* routed_t(int dtype, bool windowed) {
    if (dtype == DT_BF16) return windowed ? (const void*)tall::qmm_dma_kernel<DT_BF16, 2, 2, 8, 2, true, false, true, BITS> : (const void*)tall::qmm_dma_kernel<DT_BF16, 2, 2, 8, 2, true, false, false, BITS>;
    if (dtype == DT_F16) return windowed ? (const void*)tall::qmm_dma_kernel<DT_F16, 2, 2, 8, 2, true, false, true, BITS> : (const void*)tall::qmm_dma_kernel<DT_F16, 2, 2, 8, 2, true, false, false, BITS>;
    return nullptr;
}

const void* qmm_dma_routed_pick_b8(int dtype, bool windowed) { return routed_t<8>(dtype, windowed); }

}  // namespace mtq
