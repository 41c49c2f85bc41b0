// Chained MCSOR sweeps in FP32: several sweeps of a batch per launch.
//
// One launch per sweep reads u and the (omega/lhs, rhs) pairs and writes u
// each time: 16 bytes per point and sweep, which bound it on large batches
// (312 microseconds for 352 grids of 331 x 601).  Here a wave relaxes one
// sweep of a tile, a lane holding a group of five consecutive nu points, and
// streams the rows through registers: in step s it reads row s + 4 and runs
// colour pass i on row s - 4 i (one point per lane and pass), so a row
// is read once for the five passes, and the colours are known at compile time
// in a loop of ten steps.  Its finished rows go through LDS to the wave of the
// next sweep, so a workgroup of eight waves runs (tiles of a row) x (sweeps)
// of a segment of rows, and only the first sweep reads u and only the last
// writes it.  Neighbours in nu are the next lanes' (DPP shifts in the
// multiply-adds), or come from the next tile's wave through LDS; weights of
// rows are scalar.  Segments recompute 16 + 20 (sweeps - 1) rows at each end;
// grids with the same b(mu) lie side by side in a row, so tiles are full.
//
// A point's operations and their order are k_sweep's, so a result does not
// depend on which of the two a batch's size chooses.
//
// Bound by the length of a step, 168 VALU instructions per wave with two waves
// on a SIMD and a barrier at its end, and where all CUs stream by memory as
// well: pairs of sweeps over 352 grids of 331 x 601 are 390 steps in 389
// microseconds that move 2.0 GB (5.2 TB/s), 1.8 times the arrays' size, as
// every sweep of a launch reads the pairs and the segments' ends are read
// twice.  Per sweep that is 195 microseconds, 315 with one launch per sweep;
// 104 grids of 169 x 241 .. 505 x 901 take 110 and took 127.
//
// The 256 registers of a wave do not hold all: 14 are spilled, and their
// scratch traffic counts with the loads that a first stage waits for.
#pragma once
#include "x2gpu_internal.h"
#include <type_traits>
#include <utility>

namespace x2g {

constexpr int kChainWaves = 8;        // of a workgroup: two per SIMD
constexpr int kTileLanes = 62;        // lanes of a wave that hold groups of their own
constexpr int kChainMinNu = 17;       // narrowest grid: three groups of five per row

// One pack of problems on one grid (same b(mu)): consecutive problems lie
// a fixed stride apart in the work buffers.
struct ChainPack {
    const float *src;        // padded input rows, src_row elements apart (row mu at (mu+3)*src_row); null: zero
    float *dst;              // padded output rows, dst_row elements apart
    const float *lr;         const float *rowc;       // 8 weights per row mu, at rowc + 8*mu
    const double *dnu;
    double c1[4], c2[4]; // d/dnu and d2/dnu2 weights at distance 4, 3, 2, 1
    double ex[5];        // boundary extrapolation weights
    unsigned lr_stride;  // elements between consecutive problems' pairs
    int src_row, dst_row;
    int nni, nmu, nprob;
    int even;            // bit q: problem q is even
    int full_out;        // dst gets halos and fixed rows too (a later chain reads it)
    float om1[8];            // 1 - omega of each problem
};

// One segment: rows [a, b) of a pack.
struct ChainSeg {
    int pack, a, b;
};
// A workgroup: nseg segments of packs that take wt tiles of a row each, run
// side by side for nstep steps.
struct ChainWg {
    int seg0, nseg, wt, nstep;
};

// Launch one chain kernel of `sweeps` sweeps.
int chain_kernel(x2g_ctx *ctx, const ChainPack *packs, const ChainSeg *segs, const ChainWg *wgs, int nwg,
                 int sweeps, int first);

// One relaxation problem of a chained batch.  The problems of a grid and
// b(mu) follow each other in the list, and their (omega/lhs, rhs) pairs lie
// one stride apart; `A`, `B` and `in` (null: a zero input) are areas of
// (nmu + 8) rows of chain_row(nni) elements which also follow each other: a
// pack of problems shares those of its members.
struct ChainProblem {
    x2g_grid *g;
    int bkind, isym;
    double omega;
    const float *lr, *in;
    float *A, *B;
};
// Groups of five of a row, with the halo group at each end, and the elements
// of a row of `groups` groups (ChainRow's planes over all of them, in whole
// 16-byte chunks).
__host__ __device__ inline int chain_groups(int nni) { return (nni - 2 + 4) / 5 + 2; }
__host__ __device__ inline int chain_row(int groups) { return (5 * groups + 3) & ~3; }
// Element of value j of group g in such a row.
__host__ __device__ inline int chain_elem(int groups, int g, int j)
{
    return j < 4 ? 4 * g + j : 4 * groups + g;
}
// Where a planned batch leaves a problem: the value nu of row mu is value
// (nu + 3) % 5 of group first + (nu + 3) / 5 in row mu + 3 of `e`.
struct ChainOut {
    const float *e;
    int groups, first;
};
// Whether the batch (pointers not needed yet) can go through chains and is
// expected to run faster that way than with one launch per sweep.
struct ChainCut {
    int sweeps, steps;   // sweeps per launch, steps of a workgroup
};
bool chain_pays(x2g_ctx *ctx, const std::vector<ChainProblem> &probs, int nsweeps, ChainCut &cut);

// A planned batch: its chunks of sweeps (one launch each).
struct ChainPlan {
    struct Chunk {
        int sweeps, nwg;
        const ChainPack *packs;
        const ChainSeg *segs;
        const ChainWg *wgs;
    };
    std::vector<Chunk> chunks;
    std::vector<ChainOut> out;   // by problem
    double bytes = 0;          // algorithmic bytes of all launches
};
// Plan nsweeps sweeps of the problems and stage the launch descriptors.
int chain_plan(x2g_ctx *ctx, const std::vector<ChainProblem> &probs, int nsweeps, const ChainCut &cut,
               ChainPlan &plan);
int chain_run(x2g_ctx *ctx, const ChainPlan &plan);

// (lane i) <- lane i-1 / i+1 of the wave; 0 beyond its ends.
__device__ __forceinline__ float lane_left(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_right(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x130, 0xf, 0xf, true));
}

// A scalar in registers of its own (loaded with its neighbours it would keep
// their whole register tuple alive).
template <typename V>
__device__ __forceinline__ V own(V x)
{
    asm("" : "+s"(x));
    return x;
}

typedef float chain_f2 __attribute__((ext_vector_type(2)));
typedef float chain_f4 __attribute__((ext_vector_type(4)));
typedef unsigned chain_u4 __attribute__((ext_vector_type(4)));

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

constexpr int kLead = 4;      // steps the input rows of a first stage are loaded ahead
constexpr int kRing = 5;      // its ring of rows (a divisor of kChainU, more than kLead)
constexpr int kRowPadLo = 32; // rows of weights below and above the grid: the steps
constexpr int kRowPadHi = 480;// before and after a segment read them without effect
constexpr int kChainLag = 23; // steps a stage runs behind the stage it reads from
constexpr int kChainU = 10;   // unrolled steps: a multiple of 5 (the colours' period) and 2 (the LDS buffers)
constexpr int cmod(int a, int b) { return ((a % b) + b) % b; }

// lane in mask ? y : x
__device__ __forceinline__ float lane_select(unsigned long long mask, float x, float y)
{
    float r;
    asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "s"(mask));
    return r;
}
// mask if bit BIT of flags is set, else no lane
template <int BIT>
__device__ __forceinline__ unsigned long long mask_if(unsigned flags, unsigned long long mask)
{
    unsigned long long r;
    asm("s_bitcmp1_b32 %1, %3\n\ts_cselect_b64 %0, %2, 0" : "=s"(r) : "s"(flags), "s"(mask), "n"(BIT) : "scc");
    return r;
}

// A row of a tile in LDS or in a chain's global buffers: the groups' first
// four values, then the last value of every group.
struct ChainRow {
    float4 c[64];
    float last[64];
};
__device__ __forceinline__ void row_get(const ChainRow &r, int lane, float (&w)[5])
{
    const float4 a = r.c[lane];
    w[0] = a.x;
    w[1] = a.y;
    w[2] = a.z;
    w[3] = a.w;
    w[4] = r.last[lane];
}
__device__ __forceinline__ void row_put(ChainRow &r, int lane, const float (&w)[5])
{
    r.c[lane] = make_float4(w[0], w[1], w[2], w[3]);
    r.last[lane] = w[4];
}

// The LDS of a workgroup: a first stage's ring of input rows, and by step
// parity a wave's input rows and its passes' new values (read at lanes 1 and
// 62).
struct ChainLds {
    ChainRow ring[kChainWaves][kRing];
    ChainRow fifo[kChainWaves][2];
    float edge[kChainWaves][2][5][64];
};

// Global memory into LDS: a 16-byte chunk / a word per lane, to lds_byte + 16
// (4) * lane.  No register holds it; it counts as a vector memory load.
__device__ __forceinline__ void chunk_to_lds(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff, unsigned lds_byte)
{
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rs),
                 "s"(soff), "s"(lds_byte)
                 : "m0", "memory");
}
__device__ __forceinline__ void word_to_lds(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff, unsigned lds_byte)
{
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds" ::"v"(voff), "s"(rs), "s"(soff),
                 "s"(lds_byte)
                 : "m0", "memory");
}

// A wave's place in its chain.
struct ChainRole {
    int wave, tile, ntile;   // wave of the workgroup, tile of the row
    int next;                // waves from this one to the next stage's of the same tile
    int delay;               // steps it starts behind the chain's first wave
    bool extrap;             // the input rows' boundary values are to be extrapolated
};

constexpr unsigned kChainAll = 0x7fffffffu;   // no bound: in range by construction
__device__ __forceinline__ __amdgpu_buffer_rsrc_t chain_rsrc(const void *p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ chain_f2 chain_load_pair(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff)
{
    return __builtin_bit_cast(chain_f2, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, 0));
}
// A group's five values into a global row, the last one at vlast.
__device__ __forceinline__ void chain_store5(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned vlast, unsigned soff,
                                             const float (&w)[5])
{
    const chain_f4 a = {w[0], w[1], w[2], w[3]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(chain_u4, a), rs, voff, soff, 0);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, w[4]), rs, vlast, soff, 0);
    // A 16-byte store reads its registers late: written by the very next
    // instruction they reach memory changed (seen in lanes 12-15 and 28-31
    // when two waves shared a SIMD).  The compiler guards against it only when
    // the scalar offset is a constant.
    asm volatile("s_nop 1" ::"v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]));
}

__device__ __forceinline__ void chain_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One sweep over rows [lo0, hi0) of a pack, as one stage of a chain whose last stage writes rows [a, b).  FIRST / LAST: the
// stage reads / writes global memory (else its neighbours' LDS): separate
// code, so that the waits for a stage's loads count exactly its own.
template <int REM, bool FIRST, bool LAST>
__device__ __forceinline__ void chain_stage(const ChainPack __attribute__((address_space(4))) &pk,
                                            const ChainRole &ro, const int lo0, const int hi0, const int a,
                                            const int b, const int s00, const int nstep, ChainLds &lds)
{
    constexpr int NP = 5, U = kChainU;
    constexpr int PD = FIRST ? 4 : 3;          // steps the (omega/lhs, rhs) pairs are loaded ahead
    constexpr int CA = REM == 0 ? 4 : REM;
    constexpr int EMIT = 4 * (NP - 1) + 1;     // the row s - EMIT is final in step s
    constexpr int BASE = 4 * NP;               // the window holds rows s - BASE .. s + 5
    constexpr int WN = BASE + 6;
    typedef const float __attribute__((address_space(4))) *cptr;

    const int lane = threadIdx.x & 63;
    const int nni = own(pk.nni), nmu = own(pk.nmu), nprob = pk.nprob;
    const int M = (nni - 2 + 4) / 5, gp = M + 2;
    const int v = kTileLanes * ro.tile + lane;
    const int q = min(v / gp, nprob - 1);
    const int g = min(v - q * gp, M + 1);
    const bool have = v < nprob * gp;
    const bool real = (g >= 1) & (g <= M) & have;
    const int t = max(0, min(g - 1, M - 1));
    const bool even = (pk.even >> q) & 1;
    const float om1 = pk.om1[q];
    // lanes 0 and 63 of a tile hold copies of the neighbouring tiles' edge
    // groups, whose new values are injected a step later
    const bool is_copy = ((lane == 0) & (ro.tile > 0)) | ((lane == 63) & (ro.tile < ro.ntile - 1));
    const bool full_out = pk.full_out != 0;
    const bool store = have & !is_copy & (real | full_out);
    const unsigned long long inj = __ballot(is_copy);
    const unsigned long long gl_on = __ballot(ro.extrap & (g == 0));
    const unsigned long long gr_on = __ballot(ro.extrap & (REM == 0 ? g == M + 1 : (real & (t == M - 1))));
    // lanes that relax the points before / from position REM of their group
    const unsigned long long act_last = __ballot(real & !is_copy);
    const unsigned long long act_full = __ballot(real & !is_copy & (REM == 0 || t < M - 1));

    // d(nu) of the group's points, d/dnu and d2/dnu2 weights at distance 4 .. 1
    float dn[5], cf[8];
#pragma unroll
    for (int j = 0; j < 5; ++j) dn[j] = (float)pk.dnu[min(2 + 5 * t + j, nni - 1) - 1];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        cf[k] = (float)pk.c1[k];
        cf[4 + k] = (float)pk.c2[k];
        asm("" : "+v"(cf[k]), "+v"(cf[4 + k]));   // in vector registers
    }
    const unsigned long long is_even = __ballot(even);
    const float ex0 = (float)pk.ex[0], ex1 = (float)pk.ex[1], ex2 = (float)pk.ex[2], ex3 = (float)pk.ex[3],
                ex4 = (float)pk.ex[4];
    // the five values next to nu = 1 or nu = nni, nearest first
    auto extrap = [&](float v0, float v1, float v2, float v3, float v4) {
        return __builtin_fmaf(
            ex4, v4, __builtin_fmaf(ex3, v3, __builtin_fmaf(ex2, v2, __builtin_fmaf(ex0, v0, ex1 * v1))));
    };

    float win[WN + U][5];   // row s + d in step u of a loop: win[BASE + u + d]
#pragma unroll
    for (int k = 0; k < WN + U; ++k)
#pragma unroll
        for (int j = 0; j < 5; ++j) win[k][j] = 0.0f;

    // Addresses: buffer resources, a scalar offset per row and the lane's byte
    // offset.  A wave issues the same memory operations in every step, so that
    // its waits count exactly: what is not to be read or written is out of
    // its resource's range (a load gives 0, a store is dropped).
    const unsigned lastp = 16 * (unsigned)(gp * nprob);
    const int vg = q * gp + g;   // group of the pack's row
    const unsigned usrc = (unsigned)(16 * vg), lsrc = lastp + (unsigned)(vg * 4);
    const unsigned udst = store ? usrc : 0x80000000u, ldst = store ? lsrc : 0x80000000u;
    const unsigned src_rowb = own((unsigned)(pk.src_row * 4));
    const unsigned dst_rowb = own((unsigned)(pk.dst_row * 4));
    const unsigned lr_rowb = own((unsigned)(10 * M * 4));
    const __amdgpu_buffer_rsrc_t rs_src = chain_rsrc(pk.src, pk.src ? kChainAll : 0u);
    const unsigned long long dst0 = own((unsigned long long)pk.dst);
    // Pairs of pass i in step s: row s - 4i, from a base kRowPadLo rows below
    // row 2 (the B buffer's memory); reads past the last row return 0.
    const __amdgpu_buffer_rsrc_t rs_lr =
        chain_rsrc(reinterpret_cast<const char *>(pk.lr) - (size_t)kRowPadLo * lr_rowb,
                   (unsigned)kRowPadLo * lr_rowb + (unsigned)(((size_t)(nprob - 1) * pk.lr_stride) * 4) +
                       (unsigned)(nmu - 5) * lr_rowb);
    // lane offset of pass i: its row is 4i above the first pass's
    unsigned lro[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i)
        lro[i] = (unsigned)((q * pk.lr_stride + 2 * (i * M + t)) * 4) + 4 * (NP - 1 - i) * lr_rowb;

    ChainRow *const fin = FIRST ? lds.ring[ro.wave] : lds.fifo[ro.wave];
    ChainRow *const fout = lds.fifo[LAST ? ro.wave : ro.wave + ro.next];
    // new values of a tile's edge groups: lane 0 takes the left tile's lane
    // 62, lane 63 the right tile's lane 1
    float(*const eout)[5][64] = lds.edge[ro.wave];
    const float *const ein = is_copy ? (lane == 0 ? &lds.edge[ro.wave - 1][0][0][62] : &lds.edge[ro.wave + 1][0][0][1])
                                 : &lds.edge[ro.wave][0][0][1];

    const int lo = max(2, lo0);
    const unsigned len = (unsigned)(min(nmu - 3, hi0) - lo);
    const int a_out = full_out && a == 2 ? -2 : a;
    const unsigned n_out = (unsigned)((full_out && b == nmu - 3 ? nmu + 1 : b) - a_out);

    int s = s00;
    const int smax = nmu + 12;   // the last step that relaxes anything
    // The first stage's input rows go from global memory to its LDS ring, kLead
    // steps ahead (rows -3 .. nmu exist, others are not used); a zero input
    // is cleared there once.
    const bool fetch = pk.src != nullptr;
    const unsigned ring_byte =
        own((unsigned)(unsigned long long)(__attribute__((address_space(3))) char *)reinterpret_cast<char *>(fin));
    auto fetch_row = [&](int r, int slot) {
        const unsigned row = (unsigned)(max(-3, min(r, nmu)) + 3) * src_rowb;
        const unsigned to = ring_byte + (unsigned)(slot * (int)sizeof(ChainRow));
        chunk_to_lds(rs_src, usrc, row, to);
        word_to_lds(rs_src, lsrc, row, to + 1024u);
    };
    constexpr int kFetch = 2;   // loads per row
    if constexpr (FIRST) {
        if (fetch) {
#pragma unroll
            for (int d = 1; d < kLead; ++d) fetch_row(s00 + 4 + d, (4 + d) % kRing);
        } else {
            const float z[5] = {};
            for (int k = 0; k < kRing; ++k) row_put(fin[k], lane, z);
        }
    }
    // Pairs are loaded PD steps ahead, a pass's next ones as soon as it has
    // used the last.
    unsigned lrs = (unsigned)(s00 - 2 + kRowPadLo - 4 * (NP - 1)) * lr_rowb;
    chain_f2 lr[PD + U][NP];
#pragma unroll
    for (int d = 0; d < PD; ++d) {
#pragma unroll
        for (int i = 0; i < NP; ++i) lr[d][i] = chain_load_pair(rs_lr, lro[i], lrs);
        lrs += lr_rowb;
    }
    // Row weights: a pass's eight are loaded (scalar) during the pass before.
    // The lines come from the scalar cache, which touch_rows fills once per U
    // steps, U steps ahead: a miss inside a step would stall the whole chain.
    cptr rowp = (cptr)own((unsigned long long)(pk.rowc + 8 * (s00 - 4 * (NP - 1))));   // row s - 4 (NP-1)
    float rc[2][8];
    auto load_rows = [&](int off, float(&w)[8]) {
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = rowp[8 * off + k];
    };
    auto touch_rows = [&]() {
        constexpr int per = 2;   // rows per line
        float x[U / per + 1];   // of the rows a loop further on
#pragma unroll
        for (int k = 0; k <= U / per; ++k) x[k] = rowp[8 * (4 * (NP - 1) + U + 1 + k * per)];
#pragma unroll
        for (int k = 0; k <= U / per; ++k) asm volatile("" ::"s"(x[k]));
    };
    load_rows(4 * (NP - 1), rc[0]);
    unsigned inside = 0;   // bit k: row s - k is to be relaxed

    auto step = [&](auto uc) {
        constexpr int u = decltype(uc)::value, cur = u & 1, prev = cur ^ 1, c = BASE + u;   // c: row s
        if constexpr (FIRST) {
            // row s + 5 is in: at least the pairs of kLead - 1 steps and kLead - 2
            // rows were issued after it (spilled registers add to them, which only
            // lengthens the wait: operations complete in order)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NP * (kLead - 1) + kFetch * (kLead - 2)) : "memory");
            row_get(fin[(u + 5) % kRing], lane, win[c + 5]);
            if (fetch) fetch_row(s + 4 + kLead, (u + 4 + kLead) % kRing);
        } else {
            // written a step ago; the lag is odd, so the parity is this step's own
            static_assert(kChainLag % 2 == 1, "parity of the input rows");
            row_get(fin[cur], lane, win[c + 5]);
        }
        {
            if constexpr (u == 0) {
                // the mu = 1 row before the first update of row 2 (s00 = -8 there)
                if (ro.extrap & (s == 2)) {
#pragma unroll
                    for (int j = 0; j < 5; ++j) {
                        float x = 0.0f;
#pragma unroll
                        for (int k = 0; k < 5; ++k) x = __builtin_fmaf((float)pk.ex[k], win[c + k][j], x);
                        win[c - 1][j] = even ? x : 0.0f;
                    }
                }
            }
            // nu = 1 and nu = nni of the next row
            const float(&w)[5] = win[c + 1];
            float xl[5];   // the left lane's values REM .. 4
#pragma unroll
            for (int j = 0; j < 5; ++j) xl[j] = REM > 0 && j >= REM ? lane_left(w[j]) : w[j];
            constexpr int q = REM + 4;   // position of nu = nni - 1, the left lane's included
            const float x1 = lane_right(extrap(w[0], w[1], w[2], w[3], w[4]));
            const float x2 = extrap(xl[q % 5], xl[(q - 1) % 5], xl[(q - 2) % 5], xl[(q - 3) % 5], xl[(q - 4) % 5]);
            const float e1 = lane_select(is_even, 0.0f, x1);
            win[c + 1][4] = lane_select(gl_on, win[c + 1][4], e1);
            const float e2 = lane_select(is_even, 0.0f, REM == 0 ? lane_left(x2) : x2);
            win[c + 1][REM] = lane_select(gr_on, win[c + 1][REM], e2);
        }
        inside = (inside << 1) | ((unsigned)(s - lo) < len ? 1u : 0u);
        float ev[NP];   // neighbours' edge values of the previous step
        static_for<NP>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            constexpr int r0 = c - 4 * i, j = cmod(i - CA * (u + i), 5);
            if constexpr (i == NP - 1) {
#pragma unroll
                for (int k = 0; k < NP; ++k) ev[k] = ein[(prev * 5 + k) * 64];
            }
            constexpr int rb = (NP * u + i) % 2;
            // of the next pass
            load_rows(4 * (NP - 1 - (i + 1) % NP) + (i + 1) / NP, rc[rb ^ 1]);
            const chain_f2 pr = lr[u][i];
            // in k_sweep's order, so that a batch's results do not depend on the
            // kernel its size chooses
            const float f = win[r0][j];
            float acc = rc[rb][0] * win[r0 - 4][j];
            acc = __builtin_fmaf(rc[rb][4], win[r0 + 4][j], acc);
            static_for<3>([&](auto kc) {
                constexpr int k = decltype(kc)::value + 1;
                acc = __builtin_fmaf(rc[rb][k], win[r0 - (4 - k)][j], acc);
                acc = __builtin_fmaf(rc[rb][4 + k], win[r0 + (4 - k)][j], acc);
            });
            // sums and differences of the neighbours at distance 4 - k
            float sum[4], dif[4];
            static_for<4>([&](auto kc) {
                constexpr int k = decltype(kc)::value, d = 4 - k;
                const float wl = win[r0][cmod(j - d, 5)], wr = win[r0][cmod(j + d, 5)];
                const float l = j - d < 0 ? lane_left(wl) : wl, r = j + d > 4 ? lane_right(wr) : wr;
                sum[k] = l + r;
                dif[k] = l - r;
            });
            float t1 = cf[0] * dif[0];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                acc = __builtin_fmaf(cf[4 + k], sum[k], acc);
                if (k) t1 = __builtin_fmaf(cf[k], dif[k], t1);
            }
            acc = __builtin_fmaf(dn[j], t1, acc);
            const float nv = __builtin_fmaf(pr.y - acc, pr.x, om1 * f);
            win[r0][j] = lane_select(mask_if<4 * i>(inside, REM == 0 || j < REM ? act_last : act_full), f, nv);
            lr[u + PD][i] = chain_load_pair(rs_lr, lro[i], lrs);
#pragma unroll
            for (int k = 0; k < 8; ++k) asm volatile("" : "+s"(rc[rb ^ 1][k]));
            __builtin_amdgcn_sched_barrier(0);   // the pass's loads stay in it
        });
        lrs += s + PD < smax ? lr_rowb : 0u;
        rowp = (cptr)own((unsigned long long)(rowp + 8));
        // the edge values take their places (read three steps on at the earliest)
        static_for<NP>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            constexpr int r = c - 1 - 4 * i, j = cmod(i - CA * (u - 1 + i), 5);
            asm("" : "+v"(ev[i]));   // read by every lane, not in a branch
            win[r][j] = lane_select(inj, win[r][j], ev[i]);
        });
        // the finished row
        if constexpr (LAST) {
            const bool on = (unsigned)(s - EMIT - a_out) < n_out;
            chain_store5(chain_rsrc((const void *)dst0, on ? kChainAll : 0u), udst, ldst,
                         on ? (unsigned)(s - EMIT + 3) * dst_rowb : 0u, win[c - EMIT]);
        } else {
            row_put(fout[cur], lane, win[c - EMIT]);
        }
        static_for<NP>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            eout[cur][i][lane] = win[c - 4 * i][cmod(i - CA * (u + i), 5)];
        });
        ++s;
        chain_barrier();
    };

    for (int k = 0; k < ro.delay; ++k) chain_barrier();
    const int send = s00 + nstep - ro.delay;   // whole loops run
    touch_rows();
    while (s < send) {
        touch_rows();
        static_for<U>([&](auto kc) { step(kc); });
        // the window moves on
#pragma unroll
        for (int k = 0; k < WN; ++k)
#pragma unroll
            for (int j = 0; j < 5; ++j) win[k][j] = win[k + U][j];
#pragma unroll
        for (int d = 0; d < PD; ++d)
#pragma unroll
            for (int i = 0; i < NP; ++i) lr[d][i] = lr[d + U][i];
    }
    // every wave of the workgroup meets the barriers of nstep + U steps
    for (; s < send + U; ++s) chain_barrier();
}

// First step (2 modulo 5, so that a step's colours are known) of a stage whose
// first row relaxed is max(2, lo0): the window fills before it.
__host__ __device__ inline int chain_s00(int lo0)
{
    const int lo = lo0 < 2 ? 2 : lo0;
    const int s = lo - 9;          // at most this
    return s - ((s - 2) % 5 + 5) % 5;
}

}  // namespace x2g
