// Host-only build of the plan's graph check (no device code, no GPU), with a mistake that can be planted in
// the tile-column op list: every lu reads the list's last tile.
#define tile_order_ops tile_order_ops_made
#include "../../sparse-operator-graph-lu_amd/csrc/device/tile_order.h"
#undef tile_order_ops

static int plant = 0;

namespace sogl_dev {
inline bool tile_order_ops(const sogl_factor_desc* d, const int32_t* in_bi, const int32_t* in_bj, TileOrderOps& out) {
    if (!tile_order_ops_made(d, in_bi, in_bj, out)) return false;
    if (plant)
        for (sogl_op& o : out.ops)
            if (o.op == SOGL_OP_LU || o.op == SOGL_OP_LLT) o.src = out.ops.back().result;
    return true;
}
void noalloc_scratch_init(int) {}
}  // namespace sogl_dev

#include "../../sparse-operator-graph-lu_amd/csrc/device/factor.hip"
#include "no_device.h"

extern "C" {
int check_planted(const sogl_plan* plan, int32_t precision, int p) {
    plant = p;
    return sogl_graph_check_plan(plan, precision, nullptr);
}
}
