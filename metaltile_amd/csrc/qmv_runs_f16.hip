// The K-run matrix-core GEMV, f16 instances.
#include "qmv_runs_pick.h"

namespace mtq {

RunsInstance qmv_runs_pick_f16(bool paired, int bits, uint32_t G, bool sliced, uint32_t xs, bool few) { return runs_pick_type<DT_F16>(paired, bits, G, sliced, xs, few); }

}  // namespace mtq
