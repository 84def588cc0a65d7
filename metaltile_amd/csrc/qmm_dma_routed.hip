// Expert-routed rows on row tiles of up to 160 rows, 4-bit codes (qmm_dma_impl.h): replaces, with many rows per expert, the
// same reference kernels as the 64-row tiles (crates/metaltile-std/src/ffai/moe.rs:2256). A translation unit of its own so that
// it compiles beside the others.
#include "qmm_dma_impl.h"

namespace mtq {

size_t qmm_dma_routed_lds_bytes(uint32_t gpr, bool windowed) {
    const size_t sb = windowed ? 32768 : (size_t)2 * 128 * (((gpr + 3) & ~3u) + 2) * 2;
    return (size_t)3 * QD_ROUTED_ROWS * 2 * 128 + sb;   // (the epilogue's 120 KB fit the ring of three)
}

const void* qmm_dma_routed_pick_b8(int dtype, bool windowed);
const void* qmm_dma_routed_pick(int bits, int dtype, bool windowed) {
    if (bits == 8) return qmm_dma_routed_pick_b8(dtype, windowed);
    return qmm_dma_routed_instance<4>(dtype, windowed);
}

}  // namespace mtq
