// whole_size and whole_deal over random calls of 128-row workgroups: the row groups dealt whole and the runs cover every row group
// once, every piece of a run has a slot inside the workspace, the merge is told of the slots that were written and of no others.  And
// the lines of the rules: which calls are dealt so, at head dimension 256 too, which by the tiles seen, which paged ones keep their tiles.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "hogwild_consts.h"
#include "hogwild_plan.h"

#define CHECK(c) do { if (!(c)) { std::printf("failed: %s (Hkv %d rows %d F %d)\n", #c, p.Hkv, cp.plan[0].rows, p.F); return 1; } } while (0)

// Is a call dealt in whole row groups of 128 rows?  (256 CUs, bf16.)
static bool whole(int D, int W, int S, int Hq, int Hkv, std::vector<int32_t> len) {
    hw_problem p{};
    p.dtype = HW_BF16;
    p.F = (int)len.size();
    p.W = W; p.S = S; p.Hq = Hq; p.Hkv = Hkv;
    p.E = p.Ev = p.RotE = D;
    p.len = len.data();
    hw::host::CallPlan cp;
    hw::host::WholePlan wp;
    return hw::host::plan_call(&p, 256, &cp, 1) == HW_OK && hw::host::whole_size(&p, 256, cp, &wp);
}

static bool wide_256(int W, int S, int Hq, int Hkv, std::vector<int32_t> len) { return whole(256, W, S, Hq, Hkv, len); }

// Decode steps keep the 16-row kernel however long the context: with one row group nothing is streamed twice.  With more, both
// launches are priced: a prompt chunk and tokens of several workers behind a long prompt go to 128-row workgroups, a step of many
// short fragments does not.
static int head_dim_256() {
    const bool ok = !wide_256(1, 1, 16, 16, {29000}) && !wide_256(1, 1, 16, 16, {120000}) && !wide_256(4, 1, 16, 16, {30000, 1, 1, 1, 1}) &&
                    !wide_256(1, 1, 32, 32, {15000}) && !wide_256(4, 4, 16, 16, {60000, 4, 4, 4, 4}) && !wide_256(2, 1, 32, 4, {120000, 1, 1}) &&
                    !wide_256(8, 1, 32, 8, {34000, 9, 9, 9, 9, 9, 9, 9, 9, 1, 1, 1, 1, 1, 1, 1, 1}) && !wide_256(4, 4, 8, 1, {60000, 4, 4, 4, 4}) &&
                    wide_256(1, 1024, 16, 8, {4096, 1024}) && wide_256(4, 8, 16, 8, {60000, 8, 8, 8, 8}) && wide_256(1, 33, 32, 32, {12000, 33});
    if (!ok) std::printf("failed: the choice of 128-row workgroups at head dimension 256\n");
    return ok ? 0 : 1;
}

// Head counts that leave CUs idle with one workgroup a CU: not where rounds would take fewer row groups one after the other.
static int rounds_instead() {
    const bool ok = !whole(128, 1, 1152, 56, 56, {1200, 1152}) && !whole(64, 1, 640, 96, 96, {4000, 640}) && !whole(64, 1, 384, 140, 140, {1200, 384}) &&
                    !whole(128, 1, 640, 96, 96, {4000, 640}) && whole(128, 1, 512, 56, 56, {1200, 512}) && whole(128, 1, 1024, 56, 56, {1200, 1024}) &&
                    whole(128, 1, 640, 56, 56, {4000, 640}) && whole(64, 1, 621, 96, 96, {150, 621}) && whole(128, 1, 1024, 40, 8, {4096, 1024}) &&
                    whole(128, 1, 1500, 32, 8, {12000, 1500}) && whole(128, 1, 1354, 36, 12, {1200, 1354});
    if (!ok) std::printf("failed: whole row groups or rounds\n");
    return ok ? 0 : 1;
}

// Are the runs of a prompt chunk of one worker dealt by the tiles that it sees?
static bool by_seen(int D, int S, int Hq, int Hkv, std::vector<int32_t> len) {
    hw_problem p{};
    p.dtype = HW_F16;
    p.F = (int)len.size();
    p.W = 1; p.S = S; p.Hq = Hq; p.Hkv = Hkv;
    p.E = p.Ev = p.RotE = D;
    p.len = len.data();
    hw::host::CallPlan cp;
    hw::host::WholePlan wp;
    return hw::host::plan_call(&p, 256, &cp, 1) == HW_OK && hw::host::whole_size(&p, 256, cp, &wp) && hw::host::deal_by_seen(&p, cp, wp);
}

// Where that was measured to pay: the share of the chunk in the tiles, the row groups left over, in one fragment as in two.
static int seen_tiles() {
    const bool ok = by_seen(128, 1400, 40, 8, {350, 1400}) && by_seen(128, 1400, 40, 8, {2700, 1400}) && by_seen(128, 1400, 40, 8, {4100}) &&
                    by_seen(128, 1024, 40, 8, {900, 1024, 0}) && by_seen(256, 1400, 16, 8, {1000, 1400}) && !by_seen(128, 1400, 40, 8, {2900, 1400}) && !by_seen(128, 1024, 40, 8, {1024, 1024}) &&
                    !by_seen(128, 1024, 40, 8, {4096, 1024}) && !by_seen(128, 1024, 40, 8, {5120}) && !by_seen(128, 830, 40, 8, {200, 830}) &&
                    !by_seen(64, 1400, 24, 8, {350, 1400}) && !by_seen(256, 950, 16, 8, {511, 950}) && !by_seen(256, 600, 16, 8, {676, 600});
    if (!ok) std::printf("failed: dealing by the tiles seen\n");
    return ok ? 0 : 1;
}

// Does a call prepare its openings ahead?
static bool ahead(int D, int W, int S, int Hq, int Hkv, std::vector<int32_t> len, bool prerotated) {
    hw_problem p{};
    p.dtype = HW_BF16;
    p.F = (int)len.size();
    p.W = W; p.S = S; p.Hq = Hq; p.Hkv = Hkv;
    p.E = p.Ev = p.RotE = D;
    p.len = len.data();
    hw::host::CallPlan cp;
    hw::host::WholePlan wp;
    hw::host::StreamPlan sp;
    if (hw::host::plan_call(&p, 256, &cp, 1) != HW_OK) return false;
    const bool whole = hw::host::whole_size(&p, 256, cp, &wp);
    return hw::host::openings_ahead(&p, cp.plan[0], prerotated, whole || hw::host::stream_size(&p, 256, cp, &sp), whole ? &wp : nullptr);
}

// Where that pays: at head dimension 128, with more than one or two openings a workgroup.
static int openings() {
    const bool ok = !ahead(64, 4, 32, 32, 8, {4781, 131, 350, 32, 1577}, true) && !ahead(64, 6, 64, 8, 2, {840, 166, 692, 1162, 64, 64, 64}, true) &&
                    !ahead(64, 1, 1400, 40, 8, {350, 1400}, false) && !ahead(256, 1, 1024, 16, 8, {4096, 1024}, false) &&
                    ahead(128, 4, 20, 64, 8, {3000, 205, 205, 205, 205}, true) && ahead(128, 1, 1024, 40, 8, {4096, 1024}, false) &&
                    ahead(128, 2, 657, 32, 8, {75, 657, 657}, false) && !ahead(128, 4, 4, 64, 8, {8192, 2048, 2048, 2048, 2048}, false) &&
                    !ahead(128, 1, 512, 64, 8, {512}, false) && !ahead(128, 1, 802, 40, 8, {479, 802}, false) && ahead(128, 1, 819, 40, 8, {5000, 819}, false) &&
                    ahead(128, 1, 528, 64, 8, {528}, false) && ahead(128, 1, 1020, 64, 8, {70, 1020}, false) && ahead(128, 1, 512, 64, 8, {512}, true) &&
                    !ahead(128, 1, 655, 28, 4, {817, 655}, false) && !ahead(128, 2, 317, 28, 4, {1202, 620, 317}, false) && ahead(128, 1, 663, 28, 4, {3204, 795}, true) &&
                    ahead(128, 8, 76, 32, 4, {1249, 76, 76, 76, 76, 76, 76, 76, 76}, false) && !ahead(128, 1, 110, 40, 8, {114, 110}, true) &&
                    ahead(128, 1, 555, 32, 8, {37, 555}, true);
    if (!ok) std::printf("failed: openings ahead\n");
    return ok ? 0 : 1;
}

// One row group in more pieces than the others does not decide how all rows are merged.
static int usual_pieces() {
    hw_problem p{};
    const int32_t len[2] = {4096, 1024};
    p.dtype = HW_BF16;
    p.F = 2; p.W = 1; p.S = 1024; p.Hq = 40; p.Hkv = 8; p.E = p.Ev = p.RotE = 128;
    p.len = len;
    hw::host::CallPlan cp;
    hw::host::WholePlan wp;
    if (hw::host::plan_call(&p, 256, &cp, 1) != HW_OK || !hw::host::whole_size(&p, 256, cp, &wp)) return 1;
    hw::host::whole_deal(&p, cp, &wp);
    const bool ok = wp.runs.max_pieces > 4 && wp.runs.usual_pieces <= 4;
    if (!ok) std::printf("failed: pieces of the row groups, %d at most, usually %d\n", wp.runs.max_pieces, wp.runs.usual_pieces);
    return ok ? 0 : 1;
}

// Paged queries of head dimension 256: K/V tiles are kept with more than two row groups of 16 a sequence, packed ones with more than
// 20 rows in the mean.
static int kept_tiles() {
    auto keep = [](int D, int W, int Hq, int Hkv, int S, int total_q) {
        static const int32_t cu = 0;
        hw_paged_problem p{};
        p.dtype = HW_BF16;
        p.F = 1; p.W = W; p.Hq = Hq; p.Hkv = Hkv; p.E = p.Ev = D; p.S = S; p.total_q = total_q;
        p.cu_seqlens_q = total_q > 0 ? &cu : nullptr;
        p.block_size = 16;
        p.max_blocks = 800;
        hw_paged_plan plan;
        return hw::host::paged_plan(&p, 256, &plan) == HW_OK && hw::host::paged_keep_in_l2(&p, plan);
    };
    const bool ok = !keep(256, 4, 16, 8, 8, 0) && !keep(256, 4, 16, 8, 12, 0) && !keep(256, 4, 16, 8, 16, 0) && keep(256, 4, 16, 8, 17, 0) &&
                    keep(256, 1, 16, 8, 128, 0) && !keep(256, 4, 16, 8, 0, 40) && keep(256, 4, 16, 8, 0, 41) && !keep(256, 32, 16, 8, 0, 31 + 128) &&
                    keep(256, 8, 64, 8, 0, 7 + 128) && !keep(128, 4, 40, 8, 64, 0) && !keep(128, 4, 40, 8, 0, 400);
    if (!ok) std::printf("failed: paged tiles kept in the L2\n");
    return ok ? 0 : 1;
}

// Decode steps of sequences of different length: any step saved is worth other shares while there is a CU for every workgroup, many have to be
// saved where there are more workgroups, and none is with several tokens or fragments then.
static int shares_save() {
    auto save = [](int D, int W, int Hq, int Hkv, int S, int F) {
        hw_paged_problem p{};
        p.dtype = HW_BF16;
        p.F = F; p.W = W; p.Hq = Hq; p.Hkv = Hkv; p.E = p.Ev = D; p.S = S;
        p.block_size = 16;
        p.max_blocks = 400;
        hw_paged_plan plan;
        return hw::host::paged_plan(&p, 256, &plan) == HW_OK && hw::host::paged_shared(&p, plan) ? hw::host::paged_shares_save(&p, plan, 256) : -2;
    };
    const bool ok = save(128, 4, 40, 8, 1, 1) == 0 && save(128, 16, 40, 8, 2, 2) == 0 && save(128, 17, 40, 8, 1, 1) == 6 && save(64, 17, 40, 8, 1, 1) == 5 &&
                    save(256, 17, 16, 8, 1, 1) == 9 && save(128, 17, 16, 8, 2, 1) == -1 && save(128, 17, 40, 8, 1, 2) == -1 && save(64, 64, 8, 2, 1, 1) == 0 &&
                    save(64, 65, 8, 2, 1, 1) == -2 && save(128, 4, 40, 8, 3, 3) == -2;
    if (!ok) std::printf("failed: steps that shares have to save\n");
    return ok ? 0 : 1;
}

// The kernel whose tiles are kept leaves the reference of the exponentials where it is, so none of its sequences may be shared out by length.
static int kept_or_shared() {
    for (int W = 2; W <= 64; W += 3)
        for (int S = 1; S <= 40; ++S)
            for (int group = 1; group <= 40; ++group) {
                hw_paged_problem p{};
                p.dtype = HW_BF16;
                p.F = 1; p.W = W; p.Hkv = 2; p.Hq = 2 * group; p.E = p.Ev = 256; p.S = S;
                p.block_size = 16;
                p.max_blocks = 400;
                for (p.row_blocks = 0; p.row_blocks <= 4; ++p.row_blocks) {
                    hw_paged_plan plan;
                    if (hw::host::paged_plan(&p, 256, &plan) == HW_OK && hw::host::paged_shared(&p, plan) && hw::host::paged_keep_in_l2(&p, plan)) {
                        std::printf("failed: kept and shared: %d sequences, %d tokens, %d heads a group\n", W, S, group);
                        return 1;
                    }
                }
            }
    return 0;
}

int main() {
    if (kept_tiles() != 0) return 1;
    if (kept_or_shared() != 0) return 1;
    if (shares_save() != 0) return 1;
    if (seen_tiles() != 0) return 1;
    if (openings() != 0) return 1;
    if (usual_pieces() != 0) return 1;
    if (rounds_instead() != 0) return 1;
    if (head_dim_256() != 0) return 1;
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
        // what is asked for is what the launch uses, or hw_plan's own where that is more; not what the runs it replaces would need
        CHECK(hw::host::call_workspace_bytes(&p, cus, cp) == std::max(cp.workspace_bytes, wp.workspace_bytes));
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
        std::vector<int> used(sp.slots > 0 ? sp.slots : 1, -1);           // row group of the piece in a slot
        std::vector<int> pieces(wp.split > 0 ? wp.split : 1, 0);
        for (int g = 0; g < wp.wgs; ++g) {
            const int b = sp.wg_tile_begin[g], e = sp.wg_tile_begin[g + 1];
            CHECK(b <= e);
            for (int rg = b / T; rg * T < e && b < e; ++rg) {
                CHECK(g + rg < sp.slots && used[g + rg] < 0);
                used[g + rg] = rg;
                ++pieces[rg];
            }
        }
        // what the merge is told (write_row_table): the workgroup with a row group's first tile counts the workgroups that begin before
        // the row group ends, and lists the slots from its own on; an empty run among them would be a slot that nobody wrote
        int most = 0;
        for (int rg = 0; rg < wp.split; ++rg) {
            int first = -1, begun = 0;
            for (int g = 0; g < wp.wgs; ++g) {
                const int b = sp.wg_tile_begin[g], e = sp.wg_tile_begin[g + 1];
                begun += b < (rg + 1) * T;
                if (std::max(b, rg * T) < std::min(e, (rg + 1) * T) && b <= rg * T) {
                    CHECK(first < 0);
                    first = g;
                }
            }
            CHECK(first >= 0 && pieces[rg] >= 1 && begun - first == pieces[rg]);
            for (int i = first; i < begun; ++i) CHECK(used[i + rg] == rg);
            most = std::max(most, pieces[rg]);
        }
        CHECK(most == sp.max_pieces);
        CHECK(sp.usual_pieces <= most && sp.usual_pieces >= (wp.split > 0));
        left_over += wp.split > 0;
        const size_t part = (size_t)p.Hkv * sp.slots * hw::PLAN_SLOT_ROWS * (p.Ev + 2) * 4;
        CHECK(sp.partial_bytes == part && wp.workspace_bytes >= part + (size_t)p.Hkv * cp.plan[0].rows * 8 + cp.rope_bytes && wp.workspace_bytes % 256 == 0);
    }
    std::printf("%d calls, %d with row groups left over, %d of head dimension 256\n", taken, left_over, taken_256);
    return taken > 500 && left_over > 250 && taken_256 > 100 ? 0 : 1;
}
