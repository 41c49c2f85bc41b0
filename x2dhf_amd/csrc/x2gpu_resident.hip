// Col-wise FP64 MCSOR of small grids, resident in LDS.
//
// k_sweep streams a strip of rows through its five passes and recomputes 16
// rows on each side: on a small grid a sweep is those 36 or more serial steps
// whatever the chip could hold (31 microseconds at 91 x 121, with its
// launch).  Here one workgroup keeps the whole grid in LDS and runs all
// sweeps of a call: a colour pass is one phase over the grid, every thread
// relaxing one point in each of its groups of five along nu, then a barrier.
// A thread's groups lie in one row, so its row weights stay in registers; the
// (omega/lhs, rhs) pairs of a pass are loaded during the pass before.
//
// 10 sweeps of one 91 x 121 function through x2g_mcsor: 313 -> 112 microseconds,
// 106 of them the kernel: 50 passes and 20 boundary phases, bound by the LDS
// reads (17 values of each of 2070 points a pass; waves wait for LDS in three
// quarters of the cycles that an instruction waits) and the arithmetic of one
// compute unit.  Four groups a thread spill 14 registers.
//
// The point and the boundary values are k_sweep's own, rounding for rounding,
// so a problem's result does not depend on which of the two a batch's sizes
// choose.  (Both end at 336 columns: one wider FP64 grid sends the whole batch
// to k_strip or k_phase, which round differently.)
#include "x2gpu_resident.h"
#include <algorithm>

namespace x2g {

constexpr int kResidentThreads = 1024;
constexpr int kMaxGroups = 4;   // groups of a thread (more do not fit its registers)

typedef double res_d2 __attribute__((ext_vector_type(2)));
typedef const res_d2 __attribute__((address_space(1))) *gd2ptr;

__host__ __device__ inline int res_groups(int nni) { return (nni - 2 + 4) / 5; }

// Threads of a row with `G` groups each.
static int res_per(int nni, int G) { return (res_groups(nni) + G - 1) / G; }

// LDS: rows mu = -2 .. nmu of columns nu = -2 .. nni + 3, then d(nu).
static size_t res_lds(int nni, int nmu)
{
    return ((size_t)(nni + 6) * (nmu + 3) + nni) * sizeof(double);
}

template <int G>
__global__ void __launch_bounds__(kResidentThreads) k_resident(const ResidentDesc *__restrict__ rd, int nsweeps)
{
    extern __shared__ double lds[];
    const ResidentDesc &d = rd[blockIdx.x];
    const int nni = d.nni, nmu = d.nmu, S = nni + 6, M = res_groups(nni), s1 = nni + 8, per = d.per;
    double *const f = lds;                                  // (mu + 2) * S + nu + 2
    double *const dnu = lds + (size_t)S * (nmu + 3);        // at nu - 1
    const int tid = threadIdx.x, nth = blockDim.x;
    const gdptr_w work = gmem_w(d.work);
    for (int e = tid; e < S * (nmu + 3); e += nth) {
        const int r = e / S;
        f[e] = work[(r + 1) * s1 + (e - r * S) + 1];
    }
    for (int e = tid; e < nni; e += nth) dnu[e] = d.dnu[e];

    // this thread's row (past the grid: none) and its groups t, t + per, ...
    const int row = tid / per, t0 = tid - row * per;
    const bool on = row < nmu - 5;
    const int mu = 2 + (on ? row : 0);
    const int cA = (nni - 2) % 5 == 0 ? 4 : (nni - 2) % 5;
    const double b = d.bmu[mu - 1];
    double am[4], ap[4];   // rows mu -+ 4 .. 1
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        am[k] = mcsor_row_weight(b, d.c[k], d.c[4 + k]);
        ap[k] = mcsor_row_weight(-b, d.c[k], d.c[4 + k]);
    }
    const double om1 = d.omega1;
    int col[G], left[G];      // LDS place of a group's first point; points from there to nu = nni - 1
    unsigned at[G];           // its pair of pass 0
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int t = min(t0 + g * per, M - 1);
        col[g] = (mu + 2) * S + 4 + 5 * t;
        left[g] = on && t0 + g * per < M ? nni - 2 - 5 * t : 0;
        at[g] = (unsigned)((mu - 2) * 5 * M + t);
    }
    const gd2ptr lr = (gd2ptr)(unsigned long long)d.lr;
    res_d2 pr[G];
#pragma unroll
    for (int g = 0; g < G; ++g) pr[g] = lr[at[g]];
    int j = (5 * cA - cA * ((mu - 2) % 5) % 5) % 5;   // place in its group of the point of the pass
    __syncthreads();
    for (int sw = 0; sw < nsweeps; ++sw) {
        for (int p = 0; p < 5; ++p) {
            res_d2 pn[G];
            const int np = p == 4 ? 0 : p + 1;
#pragma unroll
            for (int g = 0; g < G; ++g) pn[g] = lr[at[g] + (unsigned)(np * M)];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                if (j < left[g]) {
                    double *const q = f + col[g] + j;
                    const int nu = col[g] + j - (mu + 2) * S - 2;
                    double x[17];
#pragma unroll
                    for (int k = 0; k < 9; ++k) x[k] = q[k - 4];
#pragma unroll
                    for (int k = 1; k <= 4; ++k) {
                        x[8 + k] = q[-k * S];
                        x[12 + k] = q[k * S];
                    }
                    q[0] = mcsor_point(x, am, ap, d.c + 8, d.c + 12, dnu[nu - 1], pr[g].x, pr[g].y, om1);
                }
            }
#pragma unroll
            for (int g = 0; g < G; ++g) pr[g] = pn[g];
            j = j == 4 ? 0 : j + 1;
            __syncthreads();
        }
        // mu = 1, then nu = 1 and nu = nni (sormcsor.F90:333-383)
        for (int e = tid; e < nni - 2; e += nth) {
            double *const q = f + 3 * S + 4 + e;
            const double v = mcsor_edge_mu(d.ex, q[S], q[2 * S], q[3 * S], q[4 * S], q[5 * S]);
            q[0] = d.even ? v : 0.0;
        }
        __syncthreads();
        for (int e = tid; e < 2 * (nmu - 4); e += nth) {
            const int r = e >> 1, to = e & 1 ? -1 : 1;
            double *const q = f + (r + 3) * S + (e & 1 ? nni + 2 : 3);
            const double v = mcsor_edge_nu(d.ex, q[to], q[2 * to], q[3 * to], q[4 * to], q[5 * to]);
            q[0] = d.even ? v : 0.0;
        }
        __syncthreads();
    }
    // mu = 1 .. nmu - 4, nu = 1 .. nni
    for (int e = tid; e < nni * (nmu - 4); e += nth) {
        const int r = e / nni, k = e - r * nni;
        work[(r + 4) * s1 + k + 4] = f[(r + 3) * S + k + 3];
    }
}

static int res_pick(int nni, int nmu)
{
    for (int G = 1; G <= kMaxGroups; ++G)
        if ((nmu - 5) * res_per(nni, G) <= kResidentThreads) return G;
    return 0;
}

bool resident_fits(const x2g_ctx *ctx, int nni, int nmu)
{
    return res_lds(nni, nmu) <= ctx->max_lds && res_pick(nni, nmu) > 0;
}

ResidentDesc resident_desc(const x2g_grid *g, int bkind, int isym, double omega)
{
    ResidentDesc d{};
    d.bmu = bkind == 0 ? g->bmu_orb : g->bmu_pot;
    d.dnu = g->dnu;
    for (int i = 0; i < 16; ++i) d.c[i] = g->coef[i];
    for (int i = 0; i < 5; ++i) d.ex[i] = g->coef[16 + i];
    d.omega1 = 1.0 - omega;
    d.nni = g->nni;
    d.nmu = g->nmu;
    d.even = isym == 1;
    return d;
}

int resident_lds_attr(x2g_ctx *ctx)
{
    const void *ks[] = {(const void *)k_resident<1>, (const void *)k_resident<2>, (const void *)k_resident<3>,
                        (const void *)k_resident<4>};
    for (const void *k : ks)
        X2G_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ctx->max_lds));
    return X2G_OK;
}

int plan_resident(x2g_ctx *ctx, std::vector<ResidentDesc> &v, ResidentPlan &plan)
{
    plan = ResidentPlan{};
    if (v.empty()) return X2G_OK;
    for (auto &d : v) plan.groups = std::max(plan.groups, res_pick(d.nni, d.nmu));
    for (auto &d : v) {
        d.per = res_per(d.nni, plan.groups);
        plan.threads = std::max(plan.threads, ((d.nmu - 5) * d.per + 63) & ~63);
        plan.lds = std::max(plan.lds, res_lds(d.nni, d.nmu));
        plan.bytes += 32.0 * (double)(d.nni - 2) * (double)(d.nmu - 5);
    }
    plan.n = (int)v.size();
    return stage_n(ctx, v.data(), v.size(), &plan.descs);
}

int launch_resident(x2g_ctx *ctx, const ResidentPlan &plan, int nsweeps)
{
    if (plan.n == 0 || nsweeps <= 0) return X2G_OK;
    int rc = stage_flush(ctx);
    if (rc) return rc;
    hipEvent_t ea, eb;
    if ((rc = stats_begin(ctx, &ea, &eb))) return rc;
    const dim3 wgs((unsigned)plan.n), th((unsigned)plan.threads);
    const ResidentDesc *dd = plan.descs;
    switch (plan.groups) {
    case 1: X2G_LAUNCH(ctx, k_resident<1>, wgs, th, plan.lds, dd, nsweeps); break;
    case 2: X2G_LAUNCH(ctx, k_resident<2>, wgs, th, plan.lds, dd, nsweeps); break;
    case 3: X2G_LAUNCH(ctx, k_resident<3>, wgs, th, plan.lds, dd, nsweeps); break;
    default: X2G_LAUNCH(ctx, k_resident<4>, wgs, th, plan.lds, dd, nsweeps); break;
    }
    ++ctx->counts[X2G_COUNT_RESIDENT];
    X2G_HIP(hipGetLastError());
    return stats_end(ctx, ea, eb, plan.bytes, 0, X2G_COUNT_RESIDENT, 1);
}

}  // namespace x2g
