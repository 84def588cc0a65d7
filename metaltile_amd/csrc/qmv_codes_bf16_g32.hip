#include "qmv_codes_pick.h"

namespace mtq {

CodesInstance qmv_codes_pick_bf16_g32(int bits, uint32_t mt) { return codes_pick<DT_BF16, true>(bits, mt); }

}  // namespace mtq
