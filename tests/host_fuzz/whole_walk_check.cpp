// The way of every workgroup of a launch in whole row groups and runs (KH_STREAM), as the kernel goes it, over random causal chunks:
// each tile of each row group is taken once, no workgroup opens a row group that does not exist (a run may be empty: it then lies behind
// the last row group), and where unseen tiles are not taken in (head dimension 128) the workgroups' visible tiles are even.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "hogwild_consts.h"
#include "hogwild_plan.h"
#include "hogwild_walk.h"

// (The kernel's own way is hogwild_walk.h, which is compiled here: no row group is opened that does not exist, in either form of the kernel.
// The form that requests queries before it knows its tiles is that of head dimension 128, where no launch has a workgroup without tiles; at 256
// they are common, and without walk_opens they would open the row group behind the last one.)
#define CHECK(c) do { if (!(c)) { std::printf("failed: %s (S %d, %d / %d heads, D %d)\n", #c, p.S, p.Hq, p.Hkv, p.E); return 1; } } while (0)

int main() {
    const int heads[][3] = {{28, 4, 128}, {40, 8, 128}, {32, 8, 128}, {64, 8, 128}, {40, 8, 64}, {16, 16, 128}, {16, 8, 256}, {56, 56, 128}, {24, 24, 256}};
    std::mt19937 rng(5);
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    int taken = 0, empty = 0, even = 0;
    int runs = 0, guarded = 0;
    for (int it = 0; it < 20000; ++it) {
        hw_problem p{};
        const int* h = heads[pick(0, 8)];
        p.dtype = HW_BF16;
        p.W = 1;
        p.Hq = h[0]; p.Hkv = h[1];
        p.E = p.Ev = p.RotE = h[2];
        p.S = pick(1, 1500);
        std::vector<int32_t> len;
        if (pick(0, 3) > 0) len.push_back(pick(0, 8192));
        if (pick(0, 3) == 0) len.push_back(pick(0, 300));
        len.push_back(p.S + (pick(0, 4) == 0 ? pick(0, 700) : 0));
        if (pick(0, 5) == 0) len.push_back(0);
        p.F = (int)len.size();
        p.len = len.data();
        hw::host::CallPlan cp;
        hw::host::WholePlan wp;
        // the way of every workgroup of a launch: each tile of each row group once, no row group that is not there
        auto walked = [&](const hw::host::StreamPlan& runs_of, int wgs, int split, int whole_groups, int T) {
            const int all_groups = split + whole_groups, R = p.W * p.S * (p.Hq / p.Hkv);
            std::vector<char> seen_once((size_t)all_groups * T, 0);
            for (int g = 0; g < wgs; ++g) {
                const hw::Walk w = {runs_of.wg_tile_begin[g], runs_of.wg_tile_begin[g + 1], T, split, all_groups, wgs};
                bool whole = hw::walk_whole(w, g);
                int group = hw::walk_first(w, g);
                CHECK(hw::walk_opens(w, whole) || p.E == 256);
                if (!hw::walk_opens(w, whole)) {
                    guarded += group * 128 >= R;
                    continue;
                }
                for (; group >= 0; group = hw::walk_next(w, whole, group)) {
                    whole = group >= split;
                    CHECK(group < all_groups && group * 128 < R && hw::walk_from(w, whole, group) < hw::walk_to(w, whole, group));
                    for (int t = hw::walk_from(w, whole, group); t < hw::walk_to(w, whole, group); ++t) CHECK(!seen_once[(size_t)group * T + t]++);
                }
            }
            CHECK(std::count(seen_once.begin(), seen_once.end(), 1) == (long long)seen_once.size());
            return 0;
        };
        hw::host::StreamPlan alone;
        if (hw::host::plan_call(&p, 256, &cp, 1) == HW_OK && !hw::host::whole_size(&p, 256, cp, &wp) && hw::host::stream_size(&p, 256, cp, &alone)) {
            ++runs;
            hw::host::stream_deal(&p, cp, &alone);
            if (walked(alone, alone.wgs, cp.plan[0].row_groups, 0, cp.plan[0].tiles_per_head) != 0) return 1;
        }
        if (hw::host::plan_call(&p, 256, &cp, 1) != HW_OK || !hw::host::whole_size(&p, 256, cp, &wp)) continue;
        ++taken;
        hw::host::whole_deal(&p, cp, &wp);
        if (walked(wp.runs, wp.wgs, wp.split, wp.whole, cp.plan[0].tiles_per_head) != 0) return 1;
        const auto& sp = wp.runs;
        const int R = cp.plan[0].rows, T = cp.plan[0].tiles_per_head, groups = wp.split + wp.whole;
        int last = p.F - 1;
        while (last > 0 && len[last] == 0) --last;
        auto seen = [&](int rg) {
            const int token = (std::min((rg + 1) * 128, R) - 1) / (p.Hq / p.Hkv);
            return cp.plan[0].tile_begin[last] + (len[last] - p.S + token + 32) / 32;
        };
        std::vector<char> done((size_t)groups * T, 0);
        int most = 0;
        long long all = 0;
        for (int g = 0; g < wp.wgs; ++g) {
            const int begin = sp.wg_tile_begin[g], end = sp.wg_tile_begin[g + 1];
            bool whole = wp.split + g < groups;
            int rgi = whole ? wp.split + g : begin / T, mine = 0;
            bool some = whole || begin < end;
            empty += !some;
            while (some) {
                const int t0 = whole ? 0 : std::max(begin - rgi * T, 0), t1 = whole ? T : std::min(end - rgi * T, T);
                CHECK(t0 < t1 && rgi >= 0 && rgi < groups && rgi * 128 < R);
                for (int t = t0; t < t1; ++t) CHECK(!done[(size_t)rgi * T + t]++);
                mine += std::max(0, std::min(t1, seen(rgi)) - t0) + 28;
                if (!whole) ++rgi;
                else if (rgi + wp.wgs < groups) rgi += wp.wgs;
                else { whole = false; rgi = begin / T; }
                some = whole || std::max(begin, rgi * T) < end;
            }
            most = std::max(most, mine);
            all += mine;
        }
        CHECK((long long)std::count(done.begin(), done.end(), 1) == (long long)done.size());
        // with a remainder to fill up with, no workgroup has more than half again the mean (openings counted as 28 tiles)
        if (p.E == 128 && 2 * wp.split > wp.wgs && wp.whole == wp.wgs) {
            ++even;
            CHECK(2ll * most * wp.wgs <= 3 * all);
        }
    }
    std::printf("%d calls in runs, %d workgroups that would open a row group behind the last one\n", runs, guarded);
    if (runs < 1000 || guarded < 100) return 1;
    std::printf("%d calls, %d workgroups without tiles, %d of even load\n", taken, empty, even);
    return taken > 3000 && empty > 100 && even > 300 ? 0 : 1;
}
