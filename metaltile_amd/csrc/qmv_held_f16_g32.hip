#include "qmv_held_pick.h"

namespace mtq {

HeldInstance qmv_held_pick_f16_g32(int bits, int mode, uint32_t rows) { return held_pick_bits<DT_F16, true>(bits, mode, rows); }

}  // namespace mtq
