// whole_size and whole_deal over random calls of 128-row workgroups: the row groups dealt whole and the runs cover every row group
// once, every piece of a run has a slot inside the workspace, max_pieces bounds the pieces of a row group.
#include <cstdio>
#include <random>
#include <vector>

#include "hogwild_consts.h"
#include "hogwild_plan.h"

#define CHECK(c) do { if (!(c)) { std::printf("failed: %s (Hkv %d rows %d F %d)\n", #c, p.Hkv, cp.plan[0].rows, p.F); return 1; } } while (0)

int main() {
    std::mt19937 rng(7);
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    int taken = 0, left_over = 0, taken_256 = 0;
    for (int it = 0; it < 20000; ++it) {
        hw_problem p{};
        p.dtype = pick(0, 2);
        p.F = pick(1, pick(0, 3) == 0 ? 80 : 6);
        p.W = pick(1, 8);
        p.Hkv = pick(1, 24);
        p.Hq = p.Hkv * pick(1, 10);
        p.S = pick(1, 1500);
        p.E = p.Ev = 64 << pick(0, 2);
        p.RotE = pick(0, 3) == 0 ? 32 : p.E;
        p.splits = pick(0, 9) == 0 ? 2 : 0;
        p.row_blocks = p.E == 256 && pick(0, 9) == 0 ? 1 : 0;
        std::vector<int32_t> len(p.F);
        for (auto& n : len) n = pick(0, 4) == 0 ? pick(0, 3) : pick(0, 9000);
        p.len = len.data();
        const int cus = pick(0, 5) == 0 ? pick(1, 400) : 256;
        hw::host::CallPlan cp;
        if (hw::host::plan_call(&p, cus, &cp, 1) != HW_OK) continue;
        hw::host::WholePlan wp;
        if (!hw::host::whole_size(&p, cus, cp, &wp)) continue;
        ++taken;
        hw::host::whole_deal(&p, cp, &wp);
        const hw::host::StreamPlan& sp = wp.runs;
        const bool wide_256 = p.E == 256;           // its plan is the 16-row kernel's, and may have fewer row groups than workgroups
        const int T = cp.plan[0].tiles_per_head, nrg = (cp.plan[0].rows + hw::PLAN_SLOT_ROWS - 1) / hw::PLAN_SLOT_ROWS;
        CHECK(cp.groups == 1 && p.splits == 0 && T > 0 && p.dtype != HW_F32 && p.row_blocks == 0);
        CHECK(wide_256 ? cp.plan[0].row_blocks == 1 : cp.plan[0].row_blocks == hw::WIDE_ROW_BLOCKS && cp.plan[0].row_groups == nrg && wp.whole > 0);
        taken_256 += wide_256;
        CHECK(wp.wgs >= 1 && wp.wgs <= HW_MAX_SPLITS && (long long)wp.wgs * p.Hkv <= cus);
        CHECK(wp.split >= 0 && wp.whole >= 0 && wp.whole % wp.wgs == 0 && wp.split < wp.wgs && wp.split + wp.whole == nrg);
        CHECK(sp.wg_tile_begin[0] == 0 && sp.wg_tile_begin[wp.wgs] == wp.split * T);
        std::vector<char> used(sp.slots > 0 ? sp.slots : 1, 0);
        std::vector<int> pieces(wp.split > 0 ? wp.split : 1, 0);
        for (int g = 0; g < wp.wgs; ++g) {
            const int b = sp.wg_tile_begin[g], e = sp.wg_tile_begin[g + 1];
            CHECK(b <= e);
            for (int rg = b / T; rg * T < e && b < e; ++rg) {
                CHECK(g + rg < sp.slots && !used[g + rg]);
                used[g + rg] = 1;
                ++pieces[rg];
            }
        }
        for (int rg = 0; rg < wp.split; ++rg) CHECK(pieces[rg] >= 1 && pieces[rg] <= sp.max_pieces);
        left_over += wp.split > 0;
        const size_t part = (size_t)p.Hkv * sp.slots * hw::PLAN_SLOT_ROWS * (p.Ev + 2) * 4;
        CHECK(sp.partial_bytes == part && wp.workspace_bytes >= part + (size_t)p.Hkv * cp.plan[0].rows * 8 + cp.rope_bytes && wp.workspace_bytes % 256 == 0);
    }
    std::printf("%d calls, %d with row groups left over, %d of head dimension 256\n", taken, left_over, taken_256);
    return taken > 500 && left_over > 250 && taken_256 > 100 ? 0 : 1;
}
