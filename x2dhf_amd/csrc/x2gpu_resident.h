// Col-wise FP64 MCSOR of small grids, resident in LDS (x2gpu_resident.hip).
#pragma once
#include "x2gpu_internal.h"

namespace x2g {

struct ResidentDesc {
    double *work;              // padded, row stride nni + 8; relaxed in place
    const double *lr;          // (omega/lhs, rhs) pairs in the colour order of k_pack
    const double *bmu, *dnu;
    double c[16], ex[5], omega1;
    int nni, nmu, even, per;   // per: threads of a row
};
// Whether a grid fits one compute unit.
bool resident_fits(const x2g_ctx *ctx, int nni, int nmu);
// Everything of a problem but its arrays.
ResidentDesc resident_desc(const x2g_grid *g, int bkind, int isym, double omega);
// A launch of all problems (each must fit), its descriptors staged.
struct ResidentPlan {
    const ResidentDesc *descs = nullptr;
    int n = 0, groups = 1, threads = 64;
    size_t lds = 0;
    double bytes = 0;          // algorithmic: the grids and pairs once, however many sweeps
};
int plan_resident(x2g_ctx *ctx, std::vector<ResidentDesc> &v, ResidentPlan &plan);
// nsweeps sweeps of every problem.  Stages nothing, so it can run any number
// of times in a call.
int launch_resident(x2g_ctx *ctx, const ResidentPlan &plan, int nsweeps);
int resident_lds_attr(x2g_ctx *ctx);

}  // namespace x2g
