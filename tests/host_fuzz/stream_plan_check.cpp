// stream_plan over random calls of 128-row workgroups: the runs tile the row groups' tiles without gaps, every piece has a
// slot of its own inside the workspace, and max_pieces bounds the pieces of a row group.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "hogwild_consts.h"
#include "hogwild_plan.h"

#define CHECK(c) do { if (!(c)) { std::printf("failed: %s (Hkv %d rows %d F %d)\n", #c, p.Hkv, cp.plan[0].rows, p.F); return 1; } } while (0)

int main(int argc, char** argv) {
    const int rounds = argc > 1 ? std::atoi(argv[1]) : 20000;
    std::mt19937 rng(11);
    auto pick = [&](int lo, int hi) { return (int)(lo + rng() % (unsigned)(hi - lo + 1)); };
    int taken = 0;
    for (int it = 0; it < rounds; ++it) {
        hw_problem p{};
        p.dtype = pick(0, 3) == 0 ? HW_F16 : HW_BF16;
        p.F = pick(1, pick(0, 3) == 0 ? 64 : 6);
        p.W = pick(1, 8);
        p.Hkv = pick(1, 16);
        p.Hq = p.Hkv * pick(1, 8);
        p.S = pick(1, 1500);
        p.E = p.Ev = pick(0, 1) ? 128 : 64;
        p.RotE = pick(0, 3) == 0 ? 32 : p.E;
        std::vector<int32_t> len(p.F);
        for (auto& n : len) n = pick(0, 4) == 0 ? pick(0, 3) : pick(0, 9000);
        p.len = len.data();
        const int cus = pick(0, 5) == 0 ? pick(1, 400) : 256;
        hw::host::CallPlan cp;
        if (hw::host::plan_call(&p, cus, &cp, 1) != HW_OK) continue;
        hw::host::StreamPlan sp;
        if (!hw::host::stream_plan(&p, cus, cp, &sp)) continue;
        ++taken;
        const int T = cp.plan[0].tiles_per_head, nrg = cp.plan[0].row_groups, rows = cp.plan[0].rows;
        CHECK(sp.wgs >= 1 && sp.wgs <= HW_MAX_SPLITS && (long long)sp.wgs * p.Hkv <= (cus > p.Hkv ? cus : p.Hkv));
        CHECK(sp.wg_tile_begin[0] == 0 && sp.wg_tile_begin[sp.wgs] == nrg * T);
        std::vector<char> used(sp.slots, 0);
        std::vector<int> pieces(nrg, 0);
        for (int g = 0; g < sp.wgs; ++g) {
            const int b = sp.wg_tile_begin[g], e = sp.wg_tile_begin[g + 1];
            CHECK(b < e);
            for (int rg = b / T; rg * T < e; ++rg) {
                CHECK(g + rg < sp.slots && !used[g + rg]);
                used[g + rg] = 1;
                ++pieces[rg];
            }
        }
        for (int rg = 0; rg < nrg; ++rg) CHECK(pieces[rg] >= 1 && pieces[rg] <= sp.max_pieces);
        CHECK(sp.slots < (1 << 15));
        const size_t part = (size_t)p.Hkv * sp.slots * hw::PLAN_SLOT_ROWS * (p.Ev + 2) * 4;
        CHECK(sp.partial_bytes == part && sp.workspace_bytes >= part + (size_t)p.Hkv * rows * 8 + cp.rope_bytes && sp.workspace_bytes % 256 == 0);
    }
    std::printf("%d of %d calls in runs\n", taken, rounds);
    return taken > rounds / 20 ? 0 : 1;
}
