// Fused strategy, 2D, FP64.
#include "stage_fused.hpp"

namespace mstk {
template int run_fused_t<2, double>(mst_ctx *, int, int, int, const Stage &, int);
}
