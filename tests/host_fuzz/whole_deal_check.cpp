// whole_deal against the rule written out: the same boundaries over random calls, in less time than the rule takes that works out anew, in
// every step of the bisection, what each workgroup has in hand and each row group sees.  (Built without sanitizers, which distort times.)
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <random>
#include <vector>

#include "hogwild_consts.h"
#include "hogwild_plan.h"

using namespace hw::host;

static void written_out(const hw_problem* p, const CallPlan& cp, const WholePlan& wp, std::vector<int>* begin) {
    const hw_plan& plan = cp.plan[0];
    const int T = plan.tiles_per_head, wgs = wp.wgs, split = wp.split, gq = p->Hq / p->Hkv;
    int nf = 0, last = 0, newest = p->F - 1;
    for (int f = 0; f < p->F; ++f)
        if (p->len[f] > 0) last = f, ++nf;
    while (newest > 0 && p->len[newest] == 0) --newest;
    const bool trimmed = p->E == 128, by_seen = trimmed ? p->W == 1 && p->len[newest] >= p->S : deal_by_seen(p, cp, wp);
    const double piece = !trimmed ? 8.0 : by_seen ? 20.0 : 12.0, open = trimmed && by_seen ? 4.0 : 2.0, tile = 1.0 + open * nf / T, per_tile = 1.0 / tile;
    auto seen = [&](int rg) {
        if (!by_seen) return T;
        return plan.tile_begin[last] + (p->len[last] - p->S + (std::min((rg + 1) * hw::PLAN_SLOT_ROWS, plan.rows) - 1) / gq + hw::TILE) / hw::TILE;
    };
    auto ahead = [&](int g) {
        int more = 0;
        for (int i = 0; i < (trimmed ? wp.whole / wgs : 0); ++i) more += seen(split + i * wgs + g) - seen(split + i * wgs);
        return more * tile;
    };
    auto deal = [&](double share) {
        int rg = 0, t = 0;
        for (int g = 0; g < wgs; ++g) {
            (*begin)[g] = rg * T + t;
            for (double room = share - ahead(g); rg < split;) {
                const int take = std::min((int)((room - piece) * per_tile), seen(rg) - t);
                if (take < std::min(4, seen(rg) - t)) break;
                room -= piece + take * tile;
                t += take;
                if (t < seen(rg)) break;
                if (!trimmed) room -= T - seen(rg);
                t = 0;
                ++rg;
            }
        }
        return rg == split;
    };
    double low = 0.0, unseen = 0.0;
    for (int rg = 0; rg < split; ++rg) {
        low += piece + seen(rg) * tile;
        unseen += trimmed ? 0 : T - seen(rg);
    }
    low /= wgs;
    double high = low + unseen / wgs + ahead(wgs - 1) + 2.0 * piece + 5 * tile;
    while (!deal(high)) high *= 2.0;
    while (high - low > 0.25) {
        const double mid = 0.5 * (low + high);
        (deal(mid) ? high : low) = mid;
    }
    deal(high);
    for (int i = wgs; i <= HW_MAX_SPLITS; ++i) (*begin)[i] = split * T;
}

int main() {
    std::mt19937 rng(11);
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    const int heads[][3] = {{28, 4, 128}, {40, 8, 128}, {32, 8, 128}, {64, 8, 128}, {40, 1, 128}, {40, 8, 64}, {16, 8, 256}, {16, 16, 128}};
    std::vector<int> want(HW_MAX_SPLITS + 1);
    int compared = 0;
    double here = 0.0, there = 0.0;
    for (int it = 0; it < 3000; ++it) {
        const int* h = heads[pick(0, 7)];
        hw_problem p{};
        p.dtype = HW_BF16;
        p.W = pick(0, 2) == 0 ? pick(2, 4) : 1;
        p.Hq = h[0]; p.Hkv = h[1];
        p.E = p.Ev = p.RotE = h[2];
        p.S = pick(100, 1500);
        std::vector<int32_t> len = {pick(0, 9000)};
        for (int w = 0; w < p.W; ++w) len.push_back(p.S + (pick(0, 3) == 0 ? pick(0, 500) : 0));
        if (pick(0, 5) == 0) len.push_back(0);
        p.F = (int)len.size();
        p.len = len.data();
        CallPlan cp;
        WholePlan wp;
        if (plan_call(&p, 256, &cp, 1) != HW_OK || !whole_size(&p, 256, cp, &wp)) continue;
        double best[2] = {1e9, 1e9};
        for (int r = 0; r < 7; ++r) {
            const auto t0 = std::chrono::steady_clock::now();
            whole_deal(&p, cp, &wp);
            const auto t1 = std::chrono::steady_clock::now();
            written_out(&p, cp, wp, &want);
            const auto t2 = std::chrono::steady_clock::now();
            best[0] = std::min(best[0], std::chrono::duration<double>(t1 - t0).count());
            best[1] = std::min(best[1], std::chrono::duration<double>(t2 - t1).count());
        }
        here += best[0];
        there += best[1];
        ++compared;
        if (!std::equal(want.begin(), want.end(), wp.runs.wg_tile_begin)) {
            std::printf("failed: other boundaries (W %d S %d, %d / %d heads, D %d)\n", p.W, p.S, p.Hq, p.Hkv, p.E);
            return 1;
        }
    }
    std::printf("%d calls, %.2f us against %.2f\n", compared, here * 1e6 / compared, there * 1e6 / compared);
    return compared > 500 && here < 0.7 * there ? 0 : 1;
}
