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
// Whether (method, ordering) on a grid of nni x nmu can run as fronts.
bool front_fits(const x2g_ctx *ctx, int nni, int nmu, int method, int ordering);
// Whether nsweeps sweeps of the items (each fits) are faster as fronts than on
// the level tables.
bool front_pays(const x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps);
// Bytes that one problem's fronts add to the workspace at most, however many
// sweeps (0: does not run as fronts).
size_t front_workspace_bytes(int nni, int nmu, int method, int ordering);
// Reserve the workspace of launch_fronts.
int front_reserve(x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps);
// Launches of nsweeps sweeps of every item (each must fit, and the workspace
// be reserved), their descriptors staged.
struct FrontDesc;
struct FrontPlan {
    const FrontDesc *descs = nullptr;
    int n = 0, nsweeps = 0, threads = 0, most = 0;   // most: elements of the longest array by level
    size_t lds = 0;
    double bytes = 0;          // algorithmic, of a launch: the arrays once, however many sweeps
};
int plan_fronts(x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps, FrontPlan &plan);
// The sweeps.  Stages nothing, so it can run any number of times in a call.
int launch_fronts(x2g_ctx *ctx, const FrontPlan &plan);
int front_lds_attr(x2g_ctx *ctx);

}  // namespace x2g
