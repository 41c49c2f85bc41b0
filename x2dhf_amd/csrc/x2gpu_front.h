// Ordered SOR sweeps as moving fronts (x2gpu_front.hip).
#pragma once
#include "x2gpu_internal.h"

namespace x2g {

// One problem's ordered SOR sweeps; `work` is padded (row stride nni + 8) and
// relaxed in place.
struct FrontItem {
    x2g_grid *g;
    double *work;
    const double *lhs, *rhs;
    double omega;
    int bkind, isym, method, ordering;
};
// Whether (method, ordering) on a grid of nni x nmu runs as fronts.
bool front_fits(const x2g_ctx *ctx, int nni, int nmu, int method, int ordering);
// Reserve the workspace of launch_fronts.
int front_reserve(x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps);
// nsweeps sweeps of every item (each must fit, and the workspace be reserved).
int launch_fronts(x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps);
int front_lds_attr(x2g_ctx *ctx);

}  // namespace x2g
