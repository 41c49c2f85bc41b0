// Planner of the chained MCSOR sweeps (x2gpu_chain.h): packs, row segments,
// workgroups and launches of a batch.
#include "x2gpu_chain.h"
#include <algorithm>
#include <map>
#include <tuple>

namespace x2g {

// Tiles of a row of `groups` groups: the first and the last lane of a tile
// hold its neighbours' groups.
static int tiles_of(int groups) { return std::max(1, (groups - 2 + kTileLanes - 1) / kTileLanes); }

static bool chain_fits(int nni, int nmu)
{
    return nni >= kChainMinNu && nmu >= 61 && nmu <= 65536 && tiles_of(chain_groups(nni)) <= kChainWaves;
}

// Steps of a chain of `sweeps` sweeps over the segment [a, b).
static int chain_steps(int a, int b, int nmu, int sweeps)
{
    const int s00 = chain_s00(a - 16 - 20 * (sweeps - 1));
    const int last = (b == nmu - 3 ? nmu + 1 : b) - 1;   // a last segment also passes the fixed rows on
    return last + 17 - s00 + (sweeps - 1) * kChainLag + 1;
}

// The problems of one grid and b(mu), and how they are cut.
struct ChainClass {
    int first, count;        // problems
    int nni, nmu, maxprob;   // most problems of a pack (32-bit offsets, ChainPack::om1)
    int npack, wt, rows;     // packs, tiles of a pack's row, rows of a segment

    // packs for chains of `sweeps` sweeps: as many problems side by side as
    // the workgroup's waves hold
    bool pack(int sweeps)
    {
        const int gp = chain_groups(nni), np = std::min(maxprob, (kChainWaves / sweeps * kTileLanes + 2) / gp);
        if (np < 1) return false;
        npack = (count + np - 1) / np;
        wt = tiles_of((count + npack - 1) / npack * gp);
        return true;
    }
    int segments() const { return (nmu - 5 + rows - 1) / rows; }
    long workgroups(int sweeps) const
    {
        const int per = kChainWaves / (wt * sweeps);
        return ((long)npack * segments() + per - 1) / per;
    }
    // longest segments of at most `steps` steps (false: none so short)
    bool fit(int sweeps, int steps)
    {
        const int all = nmu - 5;
        rows = all;
        if (chain_steps(2, nmu - 3, nmu, sweeps) <= steps) return true;
        int n = 2;
        for (;; ++n) {
            rows = (all + n - 1) / n;
            const int mid = chain_steps(1000, 1000 + rows, 1 << 20, sweeps) + 4;
            if (mid <= steps) return true;
            if (rows <= 8) return false;
            n = std::max(n, (int)((long)all / std::max(rows - (mid - steps), 1)) - 1);
        }
    }
};

// Microseconds a step and a launch take, and bytes per microsecond: alone on
// the chip, as the share of the traffic that a step does not hide, and of the
// memory.  Fitted to 22 and 352 problems of 331 x 601 and 104 of 169 x 241 ..
// 505 x 901 with 1 .. 4 sweeps per launch and segments of 20 .. 600 rows:
// within 10 % where the workgroups fill the chip once.
constexpr double kStepTime = 0.82, kLaunchTime = 8.0, kShareRate = 12.5e6, kChainRate = 4.2e6;
// Problems alone or few on their grid share no row weights, which then come from
// memory: steps are longer where problems are alone (0.81 .. 0.91), and hide less
// traffic where workgroups hold several segments of such grids (0.83 .. 1.19 a
// step, which the slowest of their waves ends).  Without these two, 120 problems
// of 331 x 601 on grids of their own took 1443 microseconds in chains and 1256
// with one launch per sweep.
//
// With all of it, 473 calls of 3 .. 1000 problems of 61 x 91 .. 505 x 901 (alone
// on their grids up to all on one, alone and mixed, 2 .. 15 sweeps) against one
// launch per sweep: 212 ran as chains, 1.01 to 2.9 times as fast, and none was
// slower.
constexpr double kStepLone = 0.05, kShareRateFew = 6.3e6;
constexpr int kFewProblems = 3;
// The same for one launch per sweep over the whole batch (k_sweep, as tuned):
// 25 microseconds, and 224 points per ns on wide grids, 0.75 nni on narrow
// ones (measured 10 / 45 / 71 / 130 / 168 / 224 / 231 at nni = 19 / 67 / 91 /
// 163 / 217 / 331 / 505).
constexpr double kSweepTime = 25.0, kSweepRate = 224e3, kSweepRateNu = 0.75e3;
// On mixed grids it runs at the stride of the widest, where a row takes what one
// of the widest grid does: 1.19 ns, more beyond 294 columns.
static double sweep_row(int maxnni) { return std::max(1.19e-3, maxnni / (200e3 + 160.0 * maxnni)); }

static std::vector<ChainClass> chain_classes(const std::vector<ChainProblem> &probs)
{
    std::vector<ChainClass> cls;
    for (size_t i = 0; i < probs.size(); ++i) {
        const ChainProblem &p = probs[i];
        if (i == 0 || p.g != probs[i - 1].g || p.bkind != probs[i - 1].bkind) {
            // 32-bit byte offsets over a pack
            const double bytes = 40.0 * sizeof(float) * chain_groups(p.g->nni) * (p.g->nmu + 64);
            cls.push_back({(int)i, 0, p.g->nni, p.g->nmu, (int)std::max(1.0, std::min(8.0, 0x3fffffff / bytes)), 1, 1, 1});
        }
        ++cls.back().count;
    }
    return cls;
}

// Choose the sweeps per launch and the steps of a workgroup: workgroups of
// equal length that fill the chip as few times as it takes, or once more.
// Only cuts of less than `limit` microseconds count, so that a call which is
// better off without chains pays little for the question.  Returns the time
// (limit: no cut).
static double chain_cut(x2g_ctx *ctx, std::vector<ChainClass> &cls, int nsweeps, double limit, ChainCut &cut)
{
    double best = limit;
    for (int sw = 1; sw <= kChainWaves && sw <= nsweeps; ++sw) {
        if (sw > 1 && (nsweeps + sw - 1) / sw == (nsweeps + sw - 2) / (sw - 1)) continue;   // as many launches
        // the shortest segments there are: a whole grid's 56 rows, or one row with its halos
        const int least = std::min(83 + 23 * (sw - 1), 43 + 43 * (sw - 1));
        if ((nsweeps + sw - 1) / sw * (least * kStepTime + kLaunchTime) >= best) continue;
        bool ok = true;
        for (auto &c : cls) ok = ok && c.pack(sw);
        if (!ok) break;
        const int nch = (nsweeps + sw - 1) / sw;
        auto wgs = [&](int st) {
            long n = 0;
            for (auto &c : cls) {
                if (!c.fit(sw, st)) return 1L << 40;
                n += c.workgroups(sw);
            }
            return n;
        };
        int longest = 1;
        for (auto &c : cls) longest = std::max(longest, chain_steps(2, c.nmu - 3, c.nmu, sw));
        const long whole = wgs(longest);
        double lone = 0, packs = 0;   // packs, and those of a problem alone on its grid
        for (auto &c : cls) {
            packs += c.npack;
            lone += c.count == 1;
        }
        const double step = kStepTime + kStepLone * lone / packs;
        const int r0 = (int)((whole + ctx->num_cu - 1) / ctx->num_cu);
        for (int rounds = r0; rounds < r0 + 2; ++rounds) {
            // least steps with workgroups of `rounds` rounds, where that is a better cut
            const double room = (best / nch - kLaunchTime) / (rounds * step);
            int lo = 1, hi = (int)std::min<double>(longest, room);
            if (hi < least || wgs(hi) > (long)rounds * ctx->num_cu) continue;
            while (lo < hi) {
                const int mid = (lo + hi) / 2;
                if (wgs(mid) <= (long)rounds * ctx->num_cu) hi = mid;
                else lo = mid + 1;
            }
            wgs(hi);
            double bytes = 0, share = 0;
            for (auto &c : cls) {
                const double b = (double)c.count * (c.nni - 2) * sizeof(float) *
                                 (4.0 * (c.nmu - 5) + 3.0 * (c.segments() - 1) * (16 + 20 * (sw - 1)));
                const bool several = kChainWaves / (c.wt * sw) > 1;
                bytes += b;
                share += b / (several && c.count <= kFewProblems ? kShareRateFew : kShareRate);
            }
            const double t = std::max(rounds * hi * step + share, bytes / kChainRate);
            if (nch * (t + kLaunchTime) < best) {
                best = nch * (t + kLaunchTime);
                cut = {sw, hi};
            }
        }
    }
    return best;
}

bool chain_pays(x2g_ctx *ctx, const std::vector<ChainProblem> &probs, int nsweeps, ChainCut &cut)
{
    double t = kSweepTime, rows = 0;
    int maxnni = 0;
    for (auto &p : probs) {
        if (!chain_fits(p.g->nni, p.g->nmu)) return false;
        t += (double)(p.g->nni - 2) * (p.g->nmu - 5) / std::min(kSweepRate, kSweepRateNu * p.g->nni);
        rows += p.g->nmu - 5;
        maxnni = std::max(maxnni, p.g->nni);
    }
    t = std::max(t, kSweepTime + rows * sweep_row(maxnni));
    std::vector<ChainClass> cls = chain_classes(probs);
    // (less the estimates' errors)
    const double limit = nsweeps * t / 1.08;
    return chain_cut(ctx, cls, nsweeps, limit, cut) < limit;
}

int chain_plan(x2g_ctx *ctx, const std::vector<ChainProblem> &probs, int nsweeps, const ChainCut &cut, ChainPlan &plan)
{
    plan.chunks.clear();
    std::vector<ChainClass> cls = chain_classes(probs);
    for (auto &c : cls) X2G_CHECK(c.pack(cut.sweeps) && c.fit(cut.sweeps, cut.steps), "chain_plan: cut");
    const int nch = (nsweeps + cut.sweeps - 1) / cut.sweeps;
    // a launch reads u and the pairs and writes u once, however many sweeps it
    // runs; the first takes a zero u without reading it
    plan.bytes = 0;
    for (auto &p : probs)
        plan.bytes += (4.0 * nch - (p.in ? 0.0 : 1.0)) * sizeof(float) * (double)(p.g->nni - 2) * (p.g->nmu - 5);
    plan.out.resize(probs.size());
    int done = 0;
    // Launches of one direction and length have the same descriptors, which are
    // staged once: what a plan stages does not grow with its sweeps.
    std::map<std::tuple<bool, bool, int, int>, ChainPlan::Chunk> staged;
    for (int k = 0; k < nch; ++k) {
        ChainPlan::Chunk ck{};
        ck.sweeps = (nsweeps - done + nch - k - 1) / (nch - k);
        done += ck.sweeps;
        const auto key = std::make_tuple(k == 0, k == nch - 1, k % 2, ck.sweeps);
        if (const auto it = staged.find(key); it != staged.end()) {
            plan.chunks.push_back(it->second);
            continue;
        }
        std::vector<ChainPack> packs;
        std::vector<ChainSeg> segs;
        std::vector<ChainWg> wgs;
        for (auto &c : cls) {
            std::vector<std::pair<int, ChainSeg>> v;   // (steps, segment)
            const int gp = chain_groups(c.nni);
            int i = c.first;
            for (int q = 0; q < c.npack; ++q) {
                const int np = (c.count - (i - c.first) + c.npack - q - 1) / (c.npack - q);
                const ChainProblem *p = &probs[i];
                const x2g_grid *g = p->g;
                ChainPack d{};
                d.src = k == 0 ? p->in : (k % 2) == 1 ? p->A : p->B;
                d.dst = (k % 2) == 0 ? p->A : p->B;
                d.src_row = d.dst_row = chain_row(gp * np);
                d.lr = p->lr;
                d.lr_stride = np > 1 ? (unsigned)(p[1].lr - p->lr) : 0u;
                d.rowc = g->rowc[p->bkind] + 8 * kRowPadLo;
                d.dnu = g->dnu;
                for (int m = 0; m < 4; ++m) {
                    d.c1[m] = g->coef[8 + m];
                    d.c2[m] = g->coef[12 + m];
                }
                for (int m = 0; m < 5; ++m) d.ex[m] = g->coef[16 + m];
                d.nni = g->nni;
                d.nmu = g->nmu;
                d.nprob = np;
                d.full_out = k < nch - 1;
                for (int m = 0; m < np; ++m) {
                    d.even |= (p[m].isym == 1) << m;
                    d.om1[m] = (float)(1.0 - p[m].omega);
                    plan.out[i + m] = {d.dst, gp * np, gp * m};
                }
                for (int a = 2; a < c.nmu - 3; a += c.rows) {
                    const int b = std::min(a + c.rows, c.nmu - 3);
                    v.push_back({chain_steps(a, b, c.nmu, ck.sweeps), ChainSeg{(int)packs.size(), a, b}});
                }
                packs.push_back(d);
                i += np;
            }
            // workgroups of segments of about the same length (a segment runs as
            // long as its workgroup: the row weights end kRowPadHi rows above its grid)
            std::stable_sort(v.begin(), v.end(), [](auto &x, auto &y) { return x.first > y.first; });
            const size_t per = kChainWaves / (c.wt * ck.sweeps);
            for (size_t m = 0; m < v.size();) {
                size_t n = 1;
                while (n < per && m + n < v.size() && v[m].first - v[m + n].first <= 128) ++n;
                wgs.push_back({(int)segs.size(), (int)n, c.wt, v[m].first});
                for (; n > 0; --n) segs.push_back(v[m++].second);
            }
        }
        // the longest workgroups start first
        std::stable_sort(wgs.begin(), wgs.end(), [](const ChainWg &x, const ChainWg &y) { return x.nstep > y.nstep; });
        ck.nwg = (int)wgs.size();
        int rc;
        if ((rc = stage_n(ctx, packs.data(), packs.size(), &ck.packs))) return rc;
        if ((rc = stage_n(ctx, segs.data(), segs.size(), &ck.segs))) return rc;
        if ((rc = stage_n(ctx, wgs.data(), wgs.size(), &ck.wgs))) return rc;
        plan.chunks.push_back(ck);
        staged[key] = ck;
    }
    return X2G_OK;
}

int chain_run(x2g_ctx *ctx, const ChainPlan &plan)
{
    int rc = stage_flush(ctx);
    if (rc) return rc;
    hipEvent_t ea, eb;
    if ((rc = stats_begin(ctx, &ea, &eb))) return rc;
    bool first = true;
    for (auto &c : plan.chunks) {
        if ((rc = chain_kernel(ctx, c.packs, c.segs, c.wgs, c.nwg, c.sweeps, first ? 1 : 0))) return rc;
        first = false;
    }
    return stats_end(ctx, ea, eb, plan.bytes, 1, X2G_COUNT_CHAIN, (int)plan.chunks.size());
}

}  // namespace x2g
