// The chained MCSOR sweep in FP32 (correction sweeps).
#include "x2gpu_chain.h"

namespace x2g {

// A workgroup runs its segments side by side, each as a chain of `sweeps`
// sweeps (one wave per sweep and tile).  first: the chain's first sweep
// takes its input's boundary values as they are.
__global__ void __launch_bounds__(64 * kChainWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_chain_f32(const ChainPack *__restrict__ packs, const ChainSeg *__restrict__ segs,
            const ChainWg *__restrict__ wgs, int sweeps, int first)
{
    __shared__ ChainLds lds;
    const ChainWg wg = wgs[blockIdx.x];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // waves by stage, segment and tile
    const int row = wg.wt * wg.nseg, k = wave / row;
    const int sub = (wave - k * row) / wg.wt;
    if (k >= sweeps) {
        for (int i = 0; i < wg.nstep + kChainU; ++i) chain_barrier();
        return;
    }
    const ChainSeg sg = segs[wg.seg0 + sub];
    ChainRole ro;
    ro.wave = wave;
    ro.tile = wave % wg.wt;
    ro.next = row;
    ro.ntile = wg.wt;
    ro.delay = k * kChainLag;
    ro.extrap = !(first && k == 0);
    const auto &pk = ((const ChainPack __attribute__((address_space(4))) *)(unsigned long long)
                          packs)[__builtin_amdgcn_readfirstlane(sg.pack)];
    // stage k relaxes the rows that the later stages' cones reach
    const int a = __builtin_amdgcn_readfirstlane(sg.a), b = __builtin_amdgcn_readfirstlane(sg.b);
    const int lo0 = a - 16 - 20 * (sweeps - 1 - k), hi0 = b + 16 + 20 * (sweeps - 1 - k);
    const int s00 = chain_s00(a - 16 - 20 * (sweeps - 1));
    const bool fst = k == 0, lst = k == sweeps - 1;
#define X2G_STAGE(R)                                                                                                \
    if (fst && lst) chain_stage<R, true, true>(pk, ro, lo0, hi0, a, b, s00, wg.nstep, lds);            \
    else if (fst) chain_stage<R, true, false>(pk, ro, lo0, hi0, a, b, s00, wg.nstep, lds);             \
    else if (lst) chain_stage<R, false, true>(pk, ro, lo0, hi0, a, b, s00, wg.nstep, lds);             \
    else chain_stage<R, false, false>(pk, ro, lo0, hi0, a, b, s00, wg.nstep, lds)
    switch ((pk.nni - 2) % 5) {
    case 0: X2G_STAGE(0); break;
    case 1: X2G_STAGE(1); break;
    case 2: X2G_STAGE(2); break;
    case 3: X2G_STAGE(3); break;
    default: X2G_STAGE(4); break;
    }
#undef X2G_STAGE
}

int chain_kernel(x2g_ctx *ctx, const ChainPack *packs, const ChainSeg *segs, const ChainWg *wgs, int nwg,
                 int sweeps, int first)
{
    X2G_LAUNCH(ctx, k_chain_f32, dim3(nwg), dim3(64 * kChainWaves), 0, packs, segs, wgs, sweeps, first);
    ++ctx->counts[X2G_COUNT_CHAIN];
    X2G_HIP(hipGetLastError());
    return X2G_OK;
}

}  // namespace x2g
