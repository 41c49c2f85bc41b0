// Ordered SOR sweeps as moving fronts.
//
// sor (sormcsor.F90:20-132) relaxes the points one after another.  A point
// only meets points of its own row and column, so where rows and columns are
// each walked straight, reversed, or from a middle one outwards, the order is
// that of a level R(mu) + C(nu): equal levels are independent, and a level
// along a column is one row on.  A thread therefore holds one column of one
// strand of rows (a strand: a run of rows walked one way; two where the rows
// start in the middle) and goes one row on in every step.  Its neighbours
// along mu are its own last and next rows, in registers; those along nu it
// reads from a ring of 16 rows per column in LDS, which holds eight rows
// ahead of its own (not yet relaxed) and eight behind (relaxed).  The arrays
// are laid out by level beforehand (k_front_in) and put back afterwards
// (k_front_out), so that the threads of a step read and write one row.
//
// A workgroup runs one sweep and the next sweep's follows it kReach levels
// behind, on a progress counter.  Workgroups take their sweeps in the order
// in which they start, so one only ever waits for one that has started.
// Values cross between workgroups (and so between the L2s of two XCDs) by
// agent-scope loads and stores; a wave has waited for its stores before the
// barrier after which the counter moves.
//
// The point update keeps the reference's expression and forms no fused
// multiply-add: the result is the sequential one bit for bit.
//
// Bound by the latency of a step, 0.9 (169 x 241) to 1 microsecond (331 x 601:
// 803 microseconds for 10 sweeps, whose waves wait in 63 % of their cycles), and
// by the levels that must pass.  10 sweeps in the middle ordering against
// one workgroup on a level table: 331 x 601 12.6 -> 0.83 ms, three problems
// of 169 x 241 2.65 -> 0.50 ms.  Blocks of 8 steps: 1.19 and 0.62 ms, as the
// next sweep then follows further behind.
#include "x2gpu_front.h"
#include <algorithm>

namespace x2g {

constexpr int kU = 4;            // steps of a block: loads lead by one, the counter moves once
constexpr int kRingRows = 16;    // of a column in LDS
constexpr int kAhead = 8;        // rows of it not yet reached (the largest level difference of two columns that meet is 7)
constexpr int kLevOff = 16;      // levels of a strand's array before its row 0
constexpr int kFirst = -12;      // first step: the rows behind row 0 pass through the window before it
constexpr int kRowGap = 11;      // a row behind row 0 may be written this many levels after its place
constexpr int kReach = 2 * kU + kAhead + kRowGap;   // levels that must be done before a block's loads
constexpr int kFlagGap = 32;     // words between counters
constexpr int kMinFront = 24;    // least nni, nmu
constexpr int kFrontSweeps = 1024;   // sweeps of a launch at most: they bound the counters' memory

enum { kStraight = 0, kReversed = 1, kMirrored = 2 };

struct Strand {
    int mu0, dir, len, lev0;   // rows mu0 + dir * r, r < len; level of row 0 at C = 0
};
struct FrontDesc {
    double *f;                        // padded
    const double *lhs, *rhs, *bmu, *dnu;
    double *fs, *rs, *ls;             // by level: [strand][lev0-relative level + kLevOff][ld]
    unsigned *done;                   // levels done of each sweep, kFlagGap apart
    double c[16], ex[5], omega, omega1;
    Strand st[2];
    int nni, nmu, even, nst, ckind, cmid, cmax, ld, rows, last;   // cmax: largest C; last: step past the last block
};

// Level of column nu.  The outer columns nu = 1, nni are extrapolated from
// the five next to them; the halos go with them.
__host__ __device__ inline int front_col(int kind, int mid, int nni, int nu)
{
    auto in = [&](int n) {
        return kind == kStraight ? n - 2 : kind == kReversed ? nni - 1 - n : n <= mid ? mid - n : n - mid + 3;
    };
    if (nu <= 1) return max(in(2), in(6)) + 1;
    if (nu >= nni) return max(in(nni - 1), in(nni - 5)) + 1;
    return in(nu);
}

// Through global (not flat) operations: a flat one would also be waited for
// with LDS, at every barrier.
typedef unsigned long long __attribute__((address_space(1))) *gu64;
typedef unsigned __attribute__((address_space(1))) *gu32;
static __device__ __forceinline__ double get_agent(const double *p)
{
    return __builtin_bit_cast(double, __hip_atomic_load((gu64)(unsigned long long)p, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT));
}
static __device__ __forceinline__ void put_agent(double *p, double v)
{
    __hip_atomic_store((gu64)(unsigned long long)p, __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
static __device__ __forceinline__ unsigned get_done(const unsigned *p)
{
    return __hip_atomic_load((gu32)(unsigned long long)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
static __device__ __forceinline__ void front_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Arrays by level, and cleared counters.
__global__ void __launch_bounds__(256) k_front_in(const FrontDesc *__restrict__ fd, unsigned *tickets, int nsweeps)
{
    const FrontDesc &d = fd[blockIdx.y];
    const int tid = blockIdx.x * 256 + threadIdx.x, s1 = d.nni + 8;
    if (blockIdx.y == 0 && tid == 0) *tickets = 0u;
    for (int k = tid; k < nsweeps; k += gridDim.x * 256) d.done[(size_t)k * kFlagGap] = 0u;
    const int n = d.nst * d.rows * d.ld;
    for (int e = tid; e < n; e += gridDim.x * 256) {
        const int q = e / d.ld, j = e - q * d.ld, s = q / d.rows, lr = q - s * d.rows - kLevOff;
        const int nu = j - 3;
        const Strand &st = d.st[s];
        const int r = lr - front_col(d.ckind, d.cmid, d.nni, nu), mu = st.mu0 + st.dir * r;
        const bool have = j < s1 && r >= -4 && r < st.len + 4 && mu >= -3 && mu <= d.nmu + 4;
        d.fs[e] = have ? d.f[(size_t)(mu + 3) * s1 + j] : 0.0;
        const bool own = r >= 0 && r < st.len && mu >= 2 && nu >= 2 && nu <= d.nni - 1;
        const size_t ik = own ? (size_t)(mu - 1) * d.nni + nu - 1 : 0;
        d.rs[e] = own ? d.rhs[ik] : 0.0;
        d.ls[e] = own ? d.lhs[ik] : 1.0;
    }
}

// The relaxed rows mu = 1 .. nmu - 4, nu = 1 .. nni back into the padded array.
__global__ void __launch_bounds__(256) k_front_out(const FrontDesc *__restrict__ fd)
{
    const FrontDesc &d = fd[blockIdx.y];
    const int n = (d.nmu - 4) * d.nni;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256) {
        const int q = e / d.nni, mu = q + 1, nu = e - q * d.nni + 1;
        const int c = front_col(d.ckind, d.cmid, d.nni, nu);
        // the strand of the row; row -1 of an ascending one is mu = 1
        const int s = d.nst == 2 && mu > d.st[0].mu0 ? 1 : 0;
        const int r = (mu - d.st[s].mu0) * d.st[s].dir;
        d.f[(size_t)(mu + 3) * (d.nni + 8) + nu + 3] =
            d.fs[((size_t)s * d.rows + r + c + kLevOff) * d.ld + nu + 3];
    }
}

// One sweep of one problem per workgroup.  NT: threads at most.
template <int NT>
__global__ void __launch_bounds__(NT) k_front(const FrontDesc *__restrict__ fd, unsigned *tickets, int nprob)
{
#pragma clang fp contract(off)
    extern __shared__ double lds[];
    __shared__ unsigned mine;
    if (threadIdx.x == 0) mine = atomicAdd(tickets, 1u);
    __syncthreads();
    const int ticket = __builtin_amdgcn_readfirstlane((int)mine);
    const int sweep = ticket / nprob;
    const FrontDesc &d = fd[ticket - sweep * nprob];
    const int nni = d.nni, nmu = d.nmu, ncol = nni + 8;
    const int W = (ncol + 31) & ~31;                 // columns of a ring row: no bank conflicts along the diagonals
    const int per = (ncol + 63) >> 6;                // waves of a strand
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const bool on = wave < per * d.nst;
    const int sn = on ? wave / per : 0;
    const Strand st = d.st[sn];
    // lanes past the halos do the last halo column's work again, unseen
    const int j0 = (wave - sn * per) * 64 + lane;
    const bool lane_on = on && j0 < ncol;
    const unsigned j = lane_on ? j0 : ncol - 1;
    const int nu = (int)j - 3;
    const bool inner = lane_on && nu >= 2 && nu <= nni - 1;
    const bool edge = lane_on && (nu == 1 || nu == nni);
    const bool any_edge = __any(edge);
    const int C = front_col(d.ckind, d.cmid, nni, nu);
    double *const ring = lds + (size_t)sn * kRingRows * W;
    double *const row1 = lds + (size_t)d.nst * kRingRows * W;  // mu = 1, where the rows start there
    // b(mu) of a strand's rows, its sign the strand's way, from level kFirst of
    // the largest C on
    const int tlo = d.cmax + kLevOff, tn = tlo + d.last;
    double *const tabs = row1 + W;
    for (int q = 0; q < d.nst; ++q)
        for (int k = threadIdx.x; k < tn; k += blockDim.x) {
            const int r = k - tlo, mu = d.st[q].mu0 + d.st[q].dir * r;
            const double b = r >= 0 && r < d.st[q].len ? d.bmu[mu - 1] : 0.0;
            tabs[q * tn + k] = d.st[q].dir > 0 ? b : -b;
        }
    const double c0 = d.c[0], c1 = d.c[1], c2 = d.c[2], c3 = d.c[3], c4 = d.c[4], c5 = d.c[5], c6 = d.c[6],
                 c7 = d.c[7], c8 = d.c[8], c9 = d.c[9], c10 = d.c[10], c11 = d.c[11], c12 = d.c[12], c13 = d.c[13],
                 c14 = d.c[14], c15 = d.c[15];
    const double ex0 = d.ex[0], ex1 = d.ex[1], ex2 = d.ex[2], ex3 = d.ex[3], ex4 = d.ex[4];
    const double omega = d.omega, omega1 = d.omega1;
    const double dn = inner ? d.dnu[nu - 1] : 0.0;
    const bool even = d.even != 0;
    const bool up1 = st.dir > 0 && st.mu0 == 2;           // walks up from mu = 2: mu = 1 follows row 4
    const int r_mu1 = st.dir < 0 ? st.len - 1 : -100000;  // walks down to mu = 1
    const bool second = sn == 1;
    const int last = d.last, ld = d.ld;
    const size_t sbase = (size_t)sn * d.rows * ld;
    double *const fsl = d.fs + sbase;                      // + (level + kLevOff) * ld + column
    const double *const rsl = d.rs + sbase, *const lsl = d.ls + sbase;
    const unsigned len_own = inner || edge ? (unsigned)st.len : 0u;   // rows this lane relaxes
    unsigned *const done = d.done + (size_t)sweep * kFlagGap;
    const unsigned *const before = done - kFlagGap;        // of the sweep before
    const int lev0 = st.lev0;
    const double *const tab = tabs + sn * tn + tlo - C;
    // levels of the wave's columns
    int cmin = C, cmax = C;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        cmin = min(cmin, __shfl_xor(cmin, o, 64));
        cmax = max(cmax, __shfl_xor(cmax, o, 64));
    }
    cmin = __builtin_amdgcn_readfirstlane(cmin);
    cmax = __builtin_amdgcn_readfirstlane(cmax);
    const unsigned W8 = (unsigned)W;
    const unsigned nbj = min(max((int)j, 4), ncol - 5);   // halo columns read within the ring, to no effect

    // wait (first thread) until the sweep before has done `need` levels
    int known = sweep == 0 ? last : 0;
    auto wait_for = [&](int need) {
        need = min(need, last);
        if (known >= need) return;
        // let it get ahead by some blocks, so that the next checks pass
        const int want = min(need + 2 * kU, last);
        while ((known = (int)get_done(before)) < want)
            __builtin_amdgcn_s_sleep(1);
    };
    auto meet = [&]() {   // nothing moves across it
        asm volatile("" ::: "memory");
        __syncthreads();
        asm volatile("" ::: "memory");
    };

    if (threadIdx.x == 0) wait_for(kFirst + kReach);
    meet();
    // w[5 + u + k]: row r + k in step u of a block
    double w[kU + kAhead + 5], nf[kU], cr[kU], cl[kU], nr[kU], nl[kU];
#pragma unroll
    for (int k = 0; k < kU + kAhead + 5; ++k) w[k] = 0.0;
#pragma unroll
    for (int k = 0; k < kU; ++k) {
        const int i = kFirst - lev0 + k + kLevOff;
        nf[k] = on ? get_agent(fsl + (size_t)(i + kAhead) * ld + j) : 0.0;
        nr[k] = on ? gmem(rsl + (size_t)i * ld)[j] : 0.0;
        nl[k] = on ? gmem(lsl + (size_t)i * ld)[j] : 1.0;
    }

    for (int l0 = kFirst; l0 < last; l0 += kU) {
#pragma unroll
        for (int k = 0; k < kU; ++k) {
            w[kAhead + 5 + k] = nf[k];
            cr[k] = nr[k];
            cl[k] = nl[k];
        }
        unsigned prog = 0;
        if (threadIdx.x == 0 && sweep > 0)
            prog = get_done(before);
        if (on) {
#pragma unroll
            for (int k = 0; k < kU; ++k) {
                const int i = l0 - lev0 + kU + k + kLevOff;
                nf[k] = get_agent(fsl + (size_t)(i + kAhead) * ld + j);
                nr[k] = gmem(rsl + (size_t)i * ld)[j];
                nl[k] = gmem(lsl + (size_t)i * ld)[j];
            }
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            // (conditions on a whole wave first: they are scalar)
            const int lr = l0 + u - lev0, r = lr - C;
            const int rmin = lr - cmax, rmax = lr - cmin;
            if (on) {
                const unsigned slot = __umul24((unsigned)r & (kRingRows - 1), W8);
                double *const my = ring + slot + j;
                if (rmax >= 0 && rmin < st.len) {
                    double *const wp = w + 5 + u;
                    if (second && rmin <= 0) {
                        // the rows below the first are the other strand's first four
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const double x = lds[k * W + j];
                            if (r == 0) wp[-1 - k] = x;
                        }
                    }
                    const double *const nb = ring + slot + nbj;
                    const double m4 = nb[-4], p4 = nb[4], m3 = nb[-3], p3 = nb[3], m2 = nb[-2], p2 = nb[2],
                                 m1 = nb[-1], p1 = nb[1];
                    const double b = tab[lr];
                    const double ddmi2 = c4 * (wp[-4] + wp[4]) + c5 * (wp[-3] + wp[3]) + c6 * (wp[-2] + wp[2]) +
                                         c7 * (wp[-1] + wp[1]);
                    const double ddmi1 = c0 * (wp[-4] - wp[4]) + c1 * (wp[-3] - wp[3]) + c2 * (wp[-2] - wp[2]) +
                                         c3 * (wp[-1] - wp[1]);
                    const double ddni2 = c12 * (m4 + p4) + c13 * (m3 + p3) + c14 * (m2 + p2) + c15 * (m1 + p1);
                    const double ddni1 = c8 * (m4 - p4) + c9 * (m3 - p3) + c10 * (m2 - p2) + c11 * (m1 - p1);
                    const double cc = ddmi2 + b * ddmi1 + ddni2 + dn * ddni1;
                    double v = omega * (cr[u] - cc) / cl[u] + omega1 * wp[0];
                    double *const row = fsl + (size_t)(lr + kLevOff) * ld;   // the same for all lanes
                    if ((rmin <= r_mu1 && rmax >= r_mu1) || (up1 && rmin <= 5 && rmax >= 5)) {
                        // mu = 1 from the five rows next to it
                        double x = 0.0;
                        if (even && up1)
                            x = ex0 * wp[-5] + ex1 * wp[-4] + ex2 * wp[-3] + ex3 * wp[-2] + ex4 * wp[-1];
                        else if (even)
                            x = ex0 * wp[-1] + ex1 * wp[-2] + ex2 * wp[-3] + ex3 * wp[-4] + ex4 * wp[-5];
                        if (r == r_mu1) v = x;
                        if (inner && up1 && r == 5) {
                            row1[j] = x;
                            put_agent(row - (size_t)6 * ld + j, x);
                        }
                    }
                    if (any_edge) {
                        if (edge) {
                            const int to = nu == 1 ? 1 : -1;
                            v = even ? ex0 * my[to] + ex1 * my[2 * to] + ex2 * my[3 * to] + ex3 * my[4 * to] +
                                           ex4 * my[5 * to]
                                     : 0.0;
                            if (up1 && r == 5) {
                                const double *const o = row1 + j;
                                put_agent(row - (size_t)6 * ld + j,
                                          even ? ex0 * o[to] + ex1 * o[2 * to] + ex2 * o[3 * to] + ex3 * o[4 * to] +
                                                     ex4 * o[5 * to]
                                               : 0.0);
                            }
                        }
                    }
                    if (((unsigned)r < len_own)) {
                        wp[0] = v;
                        *my = v;
                        put_agent(row + j, v);
                    }
                    // the first rows of the second strand lie behind row 0 of the first
                    if (second && rmin < 4) {
                        if ((unsigned)r < min(len_own, 4u))
                            put_agent(d.fs + (size_t)(C - 1 - r + kLevOff) * ld + j, v);
                    }
                }
                if (lane_on) ring[__umul24(((unsigned)r + kAhead) & (kRingRows - 1), W8) + j] = w[5 + u + kAhead];
            }
            if (u == kU - 1) {
                // this wave's stores are at the agent's coherence point
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (threadIdx.x == 0) {
                    known = max(known, (int)prog);
                    wait_for(l0 + kU + kReach);
                }
                meet();
                if (threadIdx.x == 0)
                    __hip_atomic_store((gu32)(unsigned long long)done, (unsigned)max(0, l0 + kU), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            } else {
                front_barrier();
            }
        }
#pragma unroll
        for (int k = 0; k < kAhead + 5; ++k) w[k] = w[k + kU];
    }
}

// Ways of the rows and of the columns; false: others.
static bool front_ways(int method, int ordering, int &rows, int &cols)
{
    switch (ordering) {
    case X2G_ORDER_COLWISE:
    case X2G_ORDER_ROWWISE: rows = cols = kStraight; break;
    case X2G_ORDER_RROWWISE: rows = cols = kReversed; break;
    case X2G_ORDER_MIDDLE:
    case X2G_ORDER_TEST1:
    case X2G_ORDER_TEST3:
    case X2G_ORDER_MIDDLE2: rows = cols = kMirrored; break;
    case X2G_ORDER_TEST2:
    case X2G_ORDER_TEST4: rows = kReversed; cols = kMirrored; break;
    default: return false;
    }
    if (method == X2G_SOR) return true;
    // backward, a middle row is the last one, met from both sides
    if (method != X2G_SOR_BACKWARD || rows == kMirrored || cols == kMirrored) return false;
    rows = rows == kStraight ? kReversed : kStraight;
    cols = cols == kStraight ? kReversed : kStraight;
    return true;
}

static int front_threads(int nni, int nst) { return ((nni + 8 + 63) & ~63) * nst; }
static size_t front_lds(const FrontDesc &d)
{
    const size_t W = (d.nni + 8 + 31) & ~31;
    return ((size_t)d.nst * kRingRows * W + W + (size_t)d.nst * (d.cmax + kLevOff + d.last)) * sizeof(double);
}

// Strands, levels and sizes of a grid in one order.
static FrontDesc front_shape(int nni, int nmu, int method, int ordering)
{
    int rw = kStraight, cw = kStraight;
    front_ways(method, ordering, rw, cw);
    FrontDesc d{};
    d.nni = nni;
    d.nmu = nmu;
    d.ckind = cw;
    d.cmid = (nni + 7) / 2 - 4;
    const int mid = (nmu + 7) / 2 - 4;
    d.nst = rw == kMirrored ? 2 : 1;
    if (rw == kStraight) {
        d.st[0] = {2, 1, nmu - 5, 0};
    } else if (rw == kReversed) {
        d.st[0] = {nmu - 4, -1, nmu - 4, 0};
    } else {
        d.st[0] = {mid, -1, mid, 0};
        d.st[1] = {mid + 1, 1, nmu - 4 - mid, 4};
    }
    // (the outer columns come after those next to them)
    const int cmax = std::max(front_col(cw, d.cmid, nni, 1), front_col(cw, d.cmid, nni, nni));
    int steps = 0;
    for (int s = 0; s < d.nst; ++s) steps = std::max(steps, d.st[s].lev0 + d.st[s].len + cmax);
    steps -= kFirst;
    d.cmax = cmax;
    d.last = kFirst + (steps + kU - 1) / kU * kU;
    d.ld = (nni + 8 + 7) & ~7;
    d.rows = d.last + kU + kAhead + kLevOff;   // the last block's loads end there
    return d;
}

static bool front_fits_lds(size_t max_lds, int nni, int nmu, int method, int ordering)
{
    int rows, cols;
    if (!front_ways(method, ordering, rows, cols)) return false;
    const int nst = rows == kMirrored ? 2 : 1;
    return nni >= kMinFront && nmu >= kMinFront && (long)nmu * nni < (1L << 28) && front_threads(nni, nst) <= 1024 &&
           front_lds(front_shape(nni, nmu, method, ordering)) + 64 <= max_lds;
}

bool front_fits(const x2g_ctx *ctx, int nni, int nmu, int method, int ordering)
{
    return front_fits_lds(ctx->max_lds, nni, nmu, method, ordering);
}

// The level tables hold a small grid's levels in few steps of one workgroup:
// there a further sweep costs them less than it costs fronts, whose next sweep
// follows kReach levels behind.  Microseconds fitted to 440 calls of both, 24 x
// 24 to 91 x 121 points, 1 to 600 problems, 1 to 40 sweeps (fronts / tables):
// one of 24 x 24 49 / 82 with 1 sweep, 303 / 181 with 10, 1122 / 525 with 40;
// of 61 x 91 128 / 259, 392 / 524, 1253 / 1542.  kStepGain is what a front's
// step saves on the first sweep's, kFrontSweep and kFrontMore a further sweep's
// time and what each problem beside it adds, the rest the tables' (by latency
// for few points, by their one workgroup's rate for many).  The choice is the
// faster one in 431 of the calls and at most 5 % off it in all but one.  The
// tables' workgroups fill a CU each, so more problems than CUs take turns on
// them: 600 take fronts 0.27 to 0.98 of the tables' time at every size.
constexpr double kStepGain = 0.7, kFrontSweep = 30.0, kFrontMore = 0.015;
constexpr double kTableSweep = 13.0, kTablePoint = 0.003, kTableRate = 170.0;

bool front_pays(const x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps)
{
    if ((int)items.size() > ctx->num_cu) return true;
    // (one that gains decides: the others run beside it)
    for (auto &it : items) {
        const double points = (double)it.g->nni * it.g->nmu;
        const FrontDesc d = front_shape(it.g->nni, it.g->nmu, it.method, it.ordering);
        const double table = std::max(kTableSweep + kTablePoint * points, points / kTableRate);
        if (kStepGain * (d.last - kFirst) + nsweeps * (table - kFrontSweep - kFrontMore * items.size()) > 0.0)
            return true;
    }
    return false;
}

int front_lds_attr(x2g_ctx *ctx)
{
    const int lds = (int)ctx->max_lds - 64;   // the static part is one word
    X2G_HIP(hipFuncSetAttribute((const void *)k_front<512>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    X2G_HIP(hipFuncSetAttribute((const void *)k_front<768>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    X2G_HIP(hipFuncSetAttribute((const void *)k_front<1024>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    return X2G_OK;
}

static size_t front_array(const FrontDesc &d) { return (size_t)d.nst * d.rows * d.ld; }
static size_t align256(size_t b) { return (b + 255) & ~size_t(255); }
static size_t front_bytes(const FrontDesc &d, int nsweeps)
{
    return align256(3 * front_array(d) * sizeof(double)) +
           align256((size_t)std::min(nsweeps, kFrontSweeps) * kFlagGap * sizeof(unsigned));
}

size_t front_workspace_bytes(int nni, int nmu, int method, int ordering)
{
    if (!front_fits_lds(kMaxLds, nni, nmu, method, ordering)) return 0;
    return 256 + front_bytes(front_shape(nni, nmu, method, ordering), kFrontSweeps);   // 256: the call's tickets
}

int front_reserve(x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps)
{
    size_t off = 256;   // the tickets first
    for (auto &it : items) off += front_bytes(front_shape(it.g->nni, it.g->nmu, it.method, it.ordering), nsweeps);
    // (a capture cannot allocate)
    if (ctx->cap_arena && ctx->ws[4].bytes < off) return X2G_ENOMEM;
    return ws_reserve(ctx, 4, off);
}

int plan_fronts(x2g_ctx *ctx, const std::vector<FrontItem> &items, int nsweeps, FrontPlan &plan)
{
    plan = FrontPlan{};
    if (items.empty() || nsweeps <= 0) return X2G_OK;
    std::vector<FrontDesc> v;
    size_t off = 256;
    char *base = (char *)ctx->ws[4].ptr;
    for (auto &it : items) {
        const x2g_grid *g = it.g;
        FrontDesc d = front_shape(g->nni, g->nmu, it.method, it.ordering);
        d.f = it.work;
        d.lhs = it.lhs;
        d.rhs = it.rhs;
        d.bmu = it.bkind == 0 ? g->bmu_orb : g->bmu_pot;
        d.dnu = g->dnu;
        for (int i = 0; i < 16; ++i) d.c[i] = g->coef[i];
        for (int i = 0; i < 5; ++i) d.ex[i] = g->coef[16 + i];
        d.omega = it.omega;
        d.omega1 = 1.0 - it.omega;
        d.even = it.isym == 1;
        const size_t n = front_array(d);
        d.fs = (double *)(base + off);
        d.rs = d.fs + n;
        d.ls = d.rs + n;
        d.done = (unsigned *)(base + off + align256(3 * n * sizeof(double)));
        off += front_bytes(d, nsweeps);
        plan.threads = std::max(plan.threads, front_threads(d.nni, d.nst));
        plan.lds = std::max(plan.lds, front_lds(d));
        plan.most = std::max(plan.most, (int)n);
        plan.bytes += 32.0 * (double)(d.nni - 2) * (double)(d.nmu - 5);
        v.push_back(d);
    }
    X2G_CHECK(ctx->ws[4].bytes >= off, "plan_fronts: workspace");
    plan.n = (int)v.size();
    plan.nsweeps = nsweeps;
    return stage_n(ctx, v.data(), v.size(), &plan.descs);
}

int launch_fronts(x2g_ctx *ctx, const FrontPlan &plan)
{
    if (plan.n == 0) return X2G_OK;
    int rc = stage_flush(ctx);
    if (rc) return rc;
    hipEvent_t ea, eb;
    if ((rc = stats_begin(ctx, &ea, &eb))) return rc;
    const FrontDesc *dd = plan.descs;
    unsigned *tickets = (unsigned *)ctx->ws[4].ptr;
    const int np = plan.n, nt = plan.threads, bx = std::min((plan.most + 255) / 256, 1024);
    for (int done = 0; done < plan.nsweeps; done += kFrontSweeps) {
        const int ns = std::min(plan.nsweeps - done, kFrontSweeps);
        X2G_LAUNCH(ctx, k_front_in, dim3(bx, np), dim3(256), 0, dd, tickets, ns);
        const dim3 wgs((unsigned)np * (unsigned)ns);
        if (nt <= 512) X2G_LAUNCH(ctx, k_front<512>, wgs, dim3(nt), plan.lds, dd, tickets, np);
        else if (nt <= 768) X2G_LAUNCH(ctx, k_front<768>, wgs, dim3(nt), plan.lds, dd, tickets, np);
        else X2G_LAUNCH(ctx, k_front<1024>, wgs, dim3(nt), plan.lds, dd, tickets, np);
        ++ctx->counts[X2G_COUNT_FRONT];
        X2G_LAUNCH(ctx, k_front_out, dim3(bx, np), dim3(256), 0, dd);
        X2G_HIP(hipGetLastError());
    }
    const int launches = (plan.nsweeps + kFrontSweeps - 1) / kFrontSweeps;
    return stats_end(ctx, ea, eb, plan.bytes * launches, 0, X2G_COUNT_FRONT, launches);
}

}  // namespace x2g
