// Expert-routed rows on row tiles of up to 160 rows, 8-bit codes (qmm_dma_impl.h): replaces, with many rows per expert, the
// same reference kernels as the 64-row tiles (crates/metaltile-std/src/ffai/moe.rs:2256). A translation unit of its own so that
// it compiles beside the others.
#include "qmm_dma_impl.h"

namespace mtq {

const void* qmm_dma_routed_pick_b8(int dtype, bool windowed) { return qmm_dma_routed_instance<8>(dtype, windowed); }

}  // namespace mtq
