#include "qmv_held_pick.h"

namespace mtq {

HeldInstance qmv_held_pick_bf16(int bits, int mode, uint32_t rows) { return held_pick_bits<DT_BF16, false>(bits, mode, rows); }

}  // namespace mtq
