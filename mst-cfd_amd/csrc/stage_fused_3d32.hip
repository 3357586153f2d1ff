// Fused strategy, 3D, the mixed form.
#include "stage_fused.hpp"

namespace mstk {
template int run_fused_t<3, float>(mst_ctx *, int, int, int, const Stage &, int);
}
