// stream_size and stream_deal over random calls of 128-row workgroups: the runs tile the row groups' tiles without gaps, every piece has a
// slot of its own inside the workspace, and max_pieces bounds the pieces of a row group; and the rule's choice for measured calls.
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "hogwild_consts.h"
#include "hogwild_plan.h"

#define CHECK(c) do { if (!(c)) { std::printf("failed: %s (Hkv %d rows %d F %d)\n", #c, p.Hkv, cp.plan[0].rows, p.F); return 1; } } while (0)

// Calls timed in rounds and in runs on an MI355X: rounds / runs.  Below 1 the runs lost time and must not be taken.
struct Measured { int W, S, Hq, Hkv, D; std::vector<int32_t> len; double gain; };
static const Measured kMeasured[] = {
    {2, 133, 40, 8, 128, {761, 133, 133}, 0.88},
    {6, 22, 64, 8, 128, {66, 2384, 28, 58, 22, 822, 162}, 0.89},
    {1, 170, 64, 8, 128, {1311, 170}, 0.89},
    {2, 707, 8, 2, 64, {0, 707, 707}, 0.90},
    {1, 1031, 12, 3, 128, {979, 1031}, 0.91},
    {1, 1286, 40, 8, 64, {0, 1286}, 0.92},
    {1, 693, 32, 8, 128, {176, 693}, 0.93},
    {6, 43, 40, 8, 128, {635, 647, 63, 260, 43, 43, 43}, 0.94},
    {1, 1433, 8, 2, 64, {459, 1433}, 0.96},
    {1, 1177, 40, 8, 64, {1177}, 0.96},
    {1, 1024, 40, 8, 128, {4096, 1024}, 1.31},
    {1, 412, 40, 8, 128, {3013, 412}, 1.28},
    {2, 576, 40, 8, 64, {3073, 576, 576}, 1.25},
    {4, 1153, 8, 2, 64, {70, 1153, 1153, 1153, 1153}, 1.46},
};

static bool stream_plan(const hw_problem* p, int cus, const hw::host::CallPlan& cp, hw::host::StreamPlan* sp) {
    if (!hw::host::stream_size(p, cus, cp, sp)) return false;
    hw::host::stream_deal(p, cp, sp);
    return true;
}

// The deal as a plain loop over row groups and fragments: the boundaries that stream_deal has to give.
static std::vector<int> plain_deal(const hw_problem* p, const hw_plan& plan, int wgs) {
    const int nrg = plan.row_groups, T = plan.tiles_per_head;
    const double kJobCost = 6.0, kOpenCost = 2.0, kMinPiece = 4.0;
    int nf = 0;
    for (int f = 0; f < p->F; ++f) nf += p->len[f] > 0;
    double left = nrg * (T + kJobCost + kOpenCost * nf), used = 0.0;
    std::vector<int> begin(1, 0);
    for (int rg = 0; rg < nrg; ++rg) {
        bool open = false;
        for (int f = 0; f < p->F; ++f) {
            const int first = plan.tile_begin[f], n = plan.tile_begin[f + 1] - first;
            for (int t = 0; t < n;) {
                const int wgs_left = wgs - (int)begin.size() + 1;
                const double target = (left + used + (wgs_left - 1) * (kJobCost + kOpenCost)) / wgs_left;
                const double opening = kOpenCost + (open ? 0.0 : kJobCost), room = target - used - opening;
                int take = (int)(room + 0.5);
                const bool cut = used > 0.0 && wgs_left > 1 && room < (open ? 1.0 : kMinPiece);
                if (cut) take = 0;
                else if (wgs_left == 1 || take > n - t) take = n - t;
                else if (take < 1) take = 1;
                if (!cut) {
                    used += opening + take;
                    left -= take + (t == 0 ? kOpenCost + (first == 0 ? kJobCost : 0.0) : 0.0);
                    open = true;
                    t += take;
                }
                if (cut || t < n) {
                    begin.push_back(rg * T + first + t);
                    used = 0.0;
                    open = false;
                }
            }
        }
    }
    begin.push_back(nrg * T);
    return begin;
}

// Planning stays small against a launch: a call sizes twice (workspace, launch) and deals once.
static int check_time() {
    std::vector<int32_t> len(60, 68);
    len.back() = 1024;
    hw_problem p{};
    p.dtype = HW_BF16;
    p.F = 60; p.W = 1; p.S = 1024; p.Hq = 40; p.Hkv = 8; p.E = p.Ev = p.RotE = 128;
    p.len = len.data();
    hw::host::CallPlan cp;
    hw::host::StreamPlan sp;
    auto best = [](auto f) {
        double t = 1e9;
        for (int b = 0; b < 20; ++b) {
            const auto t0 = std::chrono::steady_clock::now();
            for (int i = 0; i < 50; ++i) f();
            t = std::min(t, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 50);
        }
        return t;
    };
    bool taken = false;
    const double call = best([&] { hw::host::plan_call(&p, 256, &cp, 1); });
    const double runs = best([&] { hw::host::stream_size(&p, 256, cp, &sp); taken = stream_plan(&p, 256, cp, &sp); });
    std::printf("60 fragments, 40 row groups: plan_call %.2f us, runs %.2f us\n", call, runs);
    return taken && runs < 20 * call ? 0 : 1;
}

static int check_measured() {
    int wrong = 0;
    for (const Measured& m : kMeasured) {
        hw_problem p{};
        p.dtype = HW_BF16;
        p.F = (int)m.len.size(); p.W = m.W; p.S = m.S; p.Hq = m.Hq; p.Hkv = m.Hkv; p.E = p.Ev = p.RotE = m.D;
        p.len = m.len.data();
        hw::host::CallPlan cp;
        hw::host::StreamPlan sp;
        if (hw::host::plan_call(&p, 256, &cp, 1) != HW_OK || stream_plan(&p, 256, cp, &sp) != (m.gain > 1)) {
            std::printf("wrong launch: W %d S %d %d/%d D %d first length %d (measured %.2f)\n", m.W, m.S, m.Hq, m.Hkv, m.D, m.len[0], m.gain);
            ++wrong;
        }
    }
    return wrong;
}

int main(int argc, char** argv) {
    if (check_measured() != 0 || check_time() != 0) return 1;
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
        if (!hw::host::stream_size(&p, cus, cp, &sp)) continue;
        ++taken;
        const std::vector<int> plain = plain_deal(&p, cp.plan[0], sp.wgs);
        hw::host::stream_deal(&p, cp, &sp);
        CHECK((int)plain.size() == sp.wgs + 1 && std::equal(plain.begin(), plain.end(), sp.wg_tile_begin));
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
