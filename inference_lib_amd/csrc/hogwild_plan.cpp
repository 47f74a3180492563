// Argument validation and split planning of the Hogwild! attention library: pure host code that runs before any HIP
// call, so that every rejection and every plan can be tested (and fuzzed under sanitizers) on a machine without a GPU.
#include "hogwild_plan.h"

#include <algorithm>
#include <cmath>
#include <cstring>

#include "hogwild_consts.h"

namespace hw {
namespace host {

unsigned magic_of(int d) { return (unsigned)(((1ull << 32) + (unsigned long long)d - 1) / (unsigned long long)d); }

// mulhi(n, m) with m = ceil(2^32 / d) = (2^32 + e) / d, 0 <= e < d, is floor(n/d + n e / (d 2^32)): exact as long as
// n e < 2^32 (the second term then cannot carry the sum over the next integer).
bool magic_exact(unsigned long long d, unsigned long long n_max) {
    if (d <= 1) return true;
    const unsigned long long m = ((1ull << 32) + d - 1) / d;
    const unsigned long long e = m * d - (1ull << 32);
    return e == 0 || n_max < ((1ull << 32) + e - 1) / e;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

size_t elem_size(int dtype) { return dtype == HW_F32 ? 4 : 2; }

int validate(const hw_problem* p, int fused) {
    if (p == nullptr) return HW_ERR_NULL;
    if (p->dtype != HW_F32 && p->dtype != HW_F16 && p->dtype != HW_BF16) return HW_ERR_DTYPE;
    if (p->F < 1 || p->F > HW_MAX_FRAGMENTS) return HW_ERR_FRAGMENTS;
    if (p->variant != HW_VARIANT_MFMA && p->variant != HW_VARIANT_VALU_QK) return HW_ERR_UNSUPPORTED;
    if (p->W < 1 || p->Hq < 1 || p->Hkv < 1 || p->S < 1 || p->E < 1 || p->Ev < 1) return HW_ERR_SHAPE;
    if (p->Hq % p->Hkv != 0) return HW_ERR_SHAPE;
    if (!(p->scale > 0.f) || !std::isfinite(p->scale)) return HW_ERR_SHAPE;   // the row max is taken before scaling
    if (fused) {
        if (p->RotE < 0 || p->RotE > p->E || (p->RotE & 1)) return HW_ERR_SHAPE;
    }
    if (p->out == nullptr || p->q == nullptr || p->locations == nullptr) return HW_ERR_NULL;
    if (p->k == nullptr || p->v == nullptr || p->len == nullptr) return HW_ERR_NULL;
    if (fused && p->RotE > 0 && (p->cosines == nullptr || p->sines == nullptr)) return HW_ERR_NULL;
    if (p->len_dev != nullptr && (!fused || p->RotE != p->E)) return HW_ERR_UNSUPPORTED;   // fused entry, full rotary width only
    // one launch only: device-resident lengths (a captured step is one attention launch) and the VALU-logits variant
    if (p->F > HW_MAX_LAUNCH_FRAGMENTS && (p->len_dev != nullptr || p->variant != HW_VARIANT_MFMA)) return HW_ERR_UNSUPPORTED;
    long long rows = (long long)p->W * p->S * (p->Hq / p->Hkv);
    if (rows >= (1 << 20) || p->S >= (1 << 12) || p->Hq / p->Hkv >= (1 << 12)) return HW_ERR_SHAPE;
    if ((long long)p->Hkv * ((rows + 15) / 16) * HW_MAX_SPLITS >= (1 << 20)) return HW_ERR_SHAPE;   // grid size
    for (int f = 0; f < p->F; ++f) {
        if (p->len[f] < 0) return HW_ERR_SHAPE;
        if (p->cap != nullptr && p->cap[f] < p->len[f]) return HW_ERR_SHAPE;
        if (p->len[f] > 0 && (p->k[f] == nullptr || p->v[f] == nullptr)) return HW_ERR_NULL;
        if (!aligned16(p->k[f]) || !aligned16(p->v[f])) return HW_ERR_ALIGN;
        // one kv head of a fragment is addressed through a 32-bit buffer offset
        if ((long long)p->len[f] * (p->E > p->Ev ? p->E : p->Ev) * (long long)elem_size(p->dtype) >= 0x7fff0000ll) return HW_ERR_SHAPE;
    }
    if (!aligned16(p->out) || !aligned16(p->q)) return HW_ERR_ALIGN;
    if (fused && (!aligned16(p->cosines) || !aligned16(p->sines) || !aligned16(p->rq))) return HW_ERR_ALIGN;
    // kernels are instantiated for these head dims (never a silent no-op as in kernel_v21.cuh:992-995)
    if (p->E != p->Ev || (p->E != 64 && p->E != 128 && p->E != 256)) return HW_ERR_UNSUPPORTED;
    if (p->E == 256 && p->variant != HW_VARIANT_MFMA) return HW_ERR_UNSUPPORTED;
    return HW_OK;
}

int make_plan(const hw_problem* p, int num_cus, hw_plan* plan, int fused) {
    if (plan == nullptr) return HW_ERR_NULL;
    if (num_cus < 1) return HW_ERR_SHAPE;
    std::memset(plan, 0, sizeof(*plan));
    // the same limits as validate(): the planner is also reachable on its own (hw_plan_debug)
    if (p->F < 1 || p->F > HW_MAX_LAUNCH_FRAGMENTS) return HW_ERR_FRAGMENTS;
    if (p->W < 1 || p->Hq < 1 || p->Hkv < 1 || p->S < 1 || p->Ev < 1 || p->Hq % p->Hkv != 0 || p->len == nullptr) return HW_ERR_SHAPE;
    const long long rows_ll = (long long)p->W * p->S * (p->Hq / p->Hkv);
    if (rows_ll >= (1 << 20) || p->S >= (1 << 12) || p->Hq / p->Hkv >= (1 << 12)) return HW_ERR_SHAPE;
    if ((long long)p->Hkv * ((rows_ll + 15) / 16) * HW_MAX_SPLITS >= (1 << 20)) return HW_ERR_SHAPE;   // grid size
    const int rows = (int)rows_ll;
    plan->rows = rows;
    // up to 16 rows: one 16-row block per workgroup (two workgroups per CU); up to 96: two blocks, rows beyond 32 in
    // further row groups that read the same KV; more: 128-row workgroups whose waves share every K/V tile through
    // LDS (16-bit types, lengths known on the host) -- a CU can take in about 16 B/clk, so what counts is that every
    // CU reads every byte once
    const bool wide_ok = p->dtype != HW_F32 && p->len_dev == nullptr && p->variant == HW_VARIANT_MFMA && p->E <= 128;
    plan->row_blocks = rows <= 16 ? 1 : 2;
    if (wide_ok && rows > 96) plan->row_blocks = hw::WIDE_ROW_BLOCKS;   // measured crossover: 95 rows 19.2 (narrow) / 19.9 us, 120 rows 21.8 / 20.6 us
    if (p->row_blocks == 1 || p->row_blocks == 2 || (p->row_blocks == hw::WIDE_ROW_BLOCKS && wide_ok)) plan->row_blocks = p->row_blocks;
    // head dimension 256: kernels with one 16-row block only (two blocks of 256-wide accumulators do not fit the registers)
    if (p->E > 128) plan->row_blocks = 1;
    const bool wide = plan->row_blocks == hw::WIDE_ROW_BLOCKS;
    const int rows_per_wg = 16 * plan->row_blocks;
    plan->row_groups = (rows + rows_per_wg - 1) / rows_per_wg;
    plan->tile_tokens = hw::TILE;
    long long tiles = 0;
    for (int f = 0; f < p->F; ++f) {
        if (p->len[f] < 0) return HW_ERR_SHAPE;
        plan->tile_begin[f] = (int)tiles;
        tiles += ((long long)p->len[f] + hw::TILE - 1) / hw::TILE;
        if (tiles > (1ll << 30)) return HW_ERR_SHAPE;
    }
    for (int f = p->F; f <= HW_MAX_LAUNCH_FRAGMENTS; ++f) plan->tile_begin[f] = (int)tiles;
    plan->tiles_per_head = (int)tiles;

    // Split-K policy: fill every CU with its resident workgroups once, but at least one tile per wave
    // in every workgroup, and never more workgroups than tiles.
    int wgs = p->splits;
    if (wgs <= 0) {
        // the two-row-block and fp32 kernels are built for one wave per SIMD (one workgroup per CU)
        const int per_cu = (plan->row_blocks == 1 && p->dtype != HW_F32 && p->E <= 128) ? 2 : 1;
        const int target = per_cu * num_cus;
        wgs = target / (p->Hkv * plan->row_groups);
        // narrow kernels deal a workgroup's tiles to its four waves; in the wide kernel the whole workgroup takes every tile
        const int by_work = wide ? (int)((tiles + 3) / 4) : (int)((tiles + hw::NWAVES - 1) / hw::NWAVES);
        if (wgs > by_work) wgs = by_work;
        // Small problems in 16-bit types: one workgroup per kv head (and row group) holds whole rows, writes the result
        // itself and saves the merge launch (~2.4 us), which is worth more than what the split buys as long as its
        // fragments, opened one after the other, stay few: measured, single fragments of up to 16 tiles 5.8-7.0 us
        // against 8.0-8.2 us, three fragments of 6 / 8 tiles 8.4 / 8.7 against 8.9, of 15 tiles 9.4 against 7.4.  (The
        // fp32 kernel takes ~1 us per tile and loses beyond the 4 tiles that give one workgroup anyway.)
        int nonempty = 0;
        for (int f = 0; f < p->F; ++f) nonempty += p->len[f] > 0 ? 1 : 0;
        if (!wide && p->dtype != HW_F32 && tiles + 6ll * (nonempty > 0 ? nonempty - 1 : 0) <= 20) wgs = 1;
    }
    if (wgs > (int)tiles) wgs = (int)tiles;
    if (wgs > hw::MAX_SPLITS) wgs = hw::MAX_SPLITS;
    if (wgs < 1) wgs = 1;

    // Workgroup boundaries.  Opening a fragment costs a workgroup a fixed prologue (query rotation, a
    // barrier, a pipeline refill) worth about kOpenCost tiles, so boundaries balance tiles + openings
    // rather than tiles alone: a run of tiny fragments is spread over several workgroups instead of
    // serialising their prologues in one straggler.
    {
        const double kOpenCost = wide ? 2.0 : 6.0;   // in tiles of the kernel's own pace (a wide workgroup takes a tile in one step)
        int nfrag_left = 0;
        for (int f = 0; f < p->F; ++f) nfrag_left += p->len[f] > 0 ? 1 : 0;
        long long tiles_left = tiles;
        int wg = 0;
        double used = 0.0;
        plan->wg_tile_begin[0] = 0;
        for (int f = 0; f < p->F; ++f) {
            const int ft = (int)(((long long)p->len[f] + hw::TILE - 1) / hw::TILE);
            if (ft == 0) continue;
            int t = 0;
            while (t < ft) {
                const int wgs_left = wgs - wg;   // including the current one
                // fair share of what remains, counting one opening per remaining fragment and workgroup
                const double remaining = (double)tiles_left + kOpenCost * (nfrag_left + wgs_left - 1) + used;
                const double target = remaining / wgs_left;
                const double room = target - used - kOpenCost;
                if (room < 1.0 && used > 0.0 && wgs_left > 1) {   // not worth opening this fragment here
                    plan->wg_tile_begin[++wg] = plan->tile_begin[f] + t;
                    used = 0.0;
                    continue;
                }
                int take = (int)(room + 0.5);
                if (take < 1) take = 1;
                if (take > ft - t || wgs_left == 1) take = ft - t;
                used += kOpenCost + take;
                t += take;
                tiles_left -= take;
                if (t < ft) {   // the fragment continues in the next workgroup
                    plan->wg_tile_begin[++wg] = plan->tile_begin[f] + t;
                    used = 0.0;
                }
            }
            --nfrag_left;
        }
        wgs = tiles > 0 ? wg + 1 : 1;
        for (int i = wgs; i <= HW_MAX_SPLITS; ++i) plan->wg_tile_begin[i] = (int)tiles;
    }
    plan->wgs_per_head = wgs;
    plan->workgroups = wgs * p->Hkv * plan->row_groups;
    // the kernel divides with multiply-high by ceil(2^32 / d): workgroup id by row groups, (head, split) pair by
    // workgroups per head, row by GQA ratio, (worker, token) by S.  Refuse what that would get wrong.
    if (!magic_exact((unsigned long long)plan->row_groups, (unsigned long long)plan->workgroups) ||
        !magic_exact((unsigned long long)wgs, (unsigned long long)wgs * p->Hkv) ||
        !magic_exact((unsigned long long)(p->Hq / p->Hkv), (unsigned long long)rows + 32) ||
        !magic_exact((unsigned long long)p->S, (unsigned long long)p->W * p->S + 32))
        return HW_ERR_SHAPE;
    const size_t parts = (size_t)p->Hkv * wgs;
    plan->workspace_bytes = parts * rows * ((size_t)p->Ev + 2) * sizeof(float);
    plan->workspace_bytes = (plan->workspace_bytes + 255) & ~(size_t)255;
    // the attention kernel rotates in its prologue only over the full head dimension; any other rotary width
    // goes through the standalone rotation first, into the caller's rq buffer or, without one, into the workspace.
    // Pre-rotated queries (hw_sdpa) never need that: RotE means nothing there.
    if (fused && p->rq == nullptr && p->RotE != p->E && p->RotE >= 0)
        plan->workspace_bytes += ((size_t)p->F * p->W * p->Hq * p->S * p->E * elem_size(p->dtype) + 255) & ~(size_t)255;
    return HW_OK;
}

// K/V tiles are streamed past the L2 (non-temporal) where whoever reads a tile reads it at about the same time: one row group, or
// so few that all of them are under way together.  Once a CU works through row groups one after the other (more workgroups than
// half the CUs even without a split) every tile is wanted again later, and is kept: 1024 tokens behind 4096 (40 row groups, 40/8
// heads, D = 128) miss the L2 1.05 M times instead of 3.09 M (TCC_MISS), 136 -> 125 us a layer; 410 tokens behind 12 K and 16 K
// 152 -> 125 and 203 -> 167; 1500 behind 12 K at 32/8 heads 426 -> 348; 2560 rows a head behind 1.2 K ... 8 K 1.00 to 1.12 times.
// Below the line keeping costs: 256 ... 1024 rows a head of 8 heads 0.93 to 0.99, 1536 rows 0.98 to 1.06 by length.
bool keep_in_l2(const hw_problem* p, const hw_plan& plan, int num_cus) { return 2ll * plan.row_groups * p->Hkv >= num_cus; }

int plan_call(const hw_problem* p, int num_cus, CallPlan* cp, int fused) {
    if (cp == nullptr || p == nullptr) return HW_ERR_NULL;
    std::memset(cp, 0, sizeof(*cp));
    if (p->F < 1 || p->F > HW_MAX_FRAGMENTS) return HW_ERR_FRAGMENTS;
    if (p->len == nullptr) return HW_ERR_NULL;
    cp->groups = (p->F + HW_MAX_LAUNCH_FRAGMENTS - 1) / HW_MAX_LAUNCH_FRAGMENTS;
    int dummy_rq = 0;
    for (int i = 0; i < cp->groups; ++i) {
        // groups of equal size (130 fragments: 44 + 43 + 43, not 64 + 64 + 2)
        cp->first[i] = (int)(((long long)p->F * i) / cp->groups);
        cp->count[i] = (int)(((long long)p->F * (i + 1)) / cp->groups) - cp->first[i];
        hw_problem q = *p;
        q.F = cp->count[i];
        q.len = p->len + cp->first[i];
        q.cap = p->cap != nullptr ? p->cap + cp->first[i] : nullptr;
        q.rq = &dummy_rq;                      // the room for rotated queries is counted once, below
        const int st = make_plan(&q, num_cus, &cp->plan[i], fused);
        if (st != HW_OK) return st;
        cp->slot_base[i] = cp->slots;
        cp->slots += cp->plan[i].wgs_per_head;
    }
    const size_t rows = (size_t)cp->plan[0].rows;
    cp->partial_bytes = ((size_t)p->Hkv * cp->slots * rows * ((size_t)p->Ev + 2) * sizeof(float) + 255) & ~(size_t)255;
    if (fused && p->rq == nullptr && p->RotE != p->E && p->RotE >= 0)
        cp->rope_bytes = ((size_t)p->F * p->W * p->Hq * p->S * p->E * elem_size(p->dtype) + 255) & ~(size_t)255;
    cp->workspace_bytes = cp->partial_bytes + cp->rope_bytes;
    return HW_OK;
}

// Row groups of 128 rows that do not fill the CUs evenly, fewer than one for every workgroup of a head (the others are whole_size's):
// 24 row groups of 8 kv heads (600 prompt tokens at a GQA ratio of 5) are 192 workgroups, which leave 64 of 256 CUs idle.  Cut into
// equal runs across the row groups every CU gets three quarters of a row group of work instead of one.  A run that crosses into the next row group opens it anew
// (queries, partial sums), so the runs are dealt by tiles plus openings at kJobCost and kOpenCost tiles.  (Runs dealt by
// the kernel over the tiles that the locations leave visible were measured slower, 300 against 282 us for two layers of 1024
// tokens behind 4096: a row group's unseen tiles cost next to nothing as it is, and the uneven row groups give some runs a
// third one to open.)
// Where to take them: a price of each launch in tiles, rounds against runs, with kJobPrice and kOpenPrice per opening.  The
// prices and the line at kWorth were fitted to 1626 calls timed both ways, merge launches included (24 to 1500 new tokens of
// 1 to 8 workers behind 0 to 16 K, eight head layouts, D = 64 and 128; before there were whole row groups, whose calls are among
// them): the 1305 that the rule takes gain 0.994 to 1.66, 1.21 in the median (600 tokens behind 8192 at 40/8 heads, D = 128: 144 -> 124
// us a layer); the 321 that it leaves in rounds would give 0.88 to 1.17, 1.03 in the median (133 tokens of two workers behind 761:
// 28 -> 32 us).
constexpr int kMinPiece = 4;      // tiles worth opening a row group for
bool stream_size(const hw_problem* p, int num_cus, const CallPlan& cp, StreamPlan* sp) {
    const hw_plan& plan = cp.plan[0];
    if (cp.groups != 1 || p->splits > 0 || plan.row_blocks != hw::WIDE_ROW_BLOCKS || plan.row_groups < 2 || plan.tiles_per_head < 1) return false;
    constexpr double kJobPrice = 12.0, kOpenPrice = 4.0, kWorth = 1.22;   // the choice of runs
    const int nrg = plan.row_groups, T = plan.tiles_per_head;
    int nf = 0;
    for (int f = 0; f < p->F; ++f) nf += p->len[f] > 0 ? 1 : 0;
    int wgs = num_cus / p->Hkv;
    if (wgs > hw::MAX_SPLITS) wgs = hw::MAX_SPLITS;
    if ((long long)wgs * 2 * kMinPiece > (long long)nrg * T) wgs = (int)((long long)nrg * T / (2 * kMinPiece));
    if (wgs < 1 || (long long)wgs + nrg >= (1 << 15) || (long long)nrg * T >= (1ll << 30)) return false;
    const long long launched = plan.workgroups, rounds = (launched + num_cus - 1) / num_cus;
    const double cost_rounds = rounds * ((double)T / plan.wgs_per_head + kJobPrice + kOpenPrice * (1.0 + (double)(nf - 1) / plan.wgs_per_head));
    const double cost_stream = (nrg * (T + kJobPrice + kOpenPrice * nf) + (wgs - 1) * (kJobPrice + kOpenPrice)) / wgs;
    if (cost_stream * kWorth > cost_rounds) return false;
    // the kernel divides (head, workgroup) pairs by the workgroups per head: exact for every count up to wgs (see magic_exact)
    if ((unsigned long long)wgs * wgs * p->Hkv >= (1ull << 32)) return false;
    sp->wgs = wgs;
    sp->slots = wgs + nrg - 1;
    const size_t rows = (size_t)sp->slots * hw::PLAN_SLOT_ROWS;
    sp->partial_bytes = (size_t)p->Hkv * rows * ((size_t)p->Ev + 2) * sizeof(float);
    sp->workspace_bytes = ((sp->partial_bytes + (size_t)p->Hkv * plan.rows * 2 * sizeof(int) + 255) & ~(size_t)255) + cp.rope_bytes;
    return true;
}

void stream_deal(const hw_problem* p, const CallPlan& cp, StreamPlan* sp) {
    constexpr double kJobCost = 6.0, kOpenCost = 2.0;     // in tiles: a row group's prologue and epilogue; one more fragment
    const hw_plan& plan = cp.plan[0];
    const int nrg = plan.row_groups, T = plan.tiles_per_head, wgs = sp->wgs;
    // The fragments with tiles.  price[f]: tiles and openings of a row group in front of fragment f; a workgroup that holds the
    // row group and has r of its share left there takes fragments up to the first whose whole[] exceeds r + price[f].
    int nf = 0, begin[HW_MAX_LAUNCH_FRAGMENTS], tiles[HW_MAX_LAUNCH_FRAGMENTS];
    double price[HW_MAX_LAUNCH_FRAGMENTS + 1], whole[HW_MAX_LAUNCH_FRAGMENTS];
    price[0] = 0.0;
    for (int f = 0; f < p->F; ++f) {
        const int n = plan.tile_begin[f + 1] - plan.tile_begin[f];
        if (n == 0) continue;
        begin[nf] = plan.tile_begin[f];
        tiles[nf] = n;
        whole[nf] = price[nf] + kOpenCost + std::max(n - 0.5, 1.0);
        price[nf + 1] = price[nf] + kOpenCost + n;
        ++nf;
    }
    double left = nrg * (kJobCost + price[nf]);    // work not dealt yet, without the re-openings of the workgroups to come
    int wg = 0;
    double used = 0.0, target = 0.0;
    sp->wg_tile_begin[0] = 0;
    for (int rg = 0; rg < nrg; ++rg) {
        int pieces = 0;                 // of the row group, taken by the current workgroup; with the first it holds the queries
        for (int f = 0; f < nf;) {
            const int wgs_left = wgs - wg;
            if (pieces > 1) {           // whole fragments at once
                const int to = wgs_left == 1 ? nf : (int)(std::upper_bound(whole + f, whole + nf, target - used + price[f]) - whole);
                used += price[to] - price[f];
                left -= price[to] - price[f];
                f = to;
                if (f == nf) break;
            }
            for (int t = 0; t < tiles[f];) {
                const int wgs_left = wgs - wg;
                // this workgroup's fair share; what it takes of a row group that it holds already does not change that
                if (pieces < 2) target = (left + used + (wgs_left - 1) * (kJobCost + kOpenCost)) / wgs_left;
                const double opening = kOpenCost + (pieces > 0 ? 0.0 : kJobCost);
                const double room = target - used - opening;
                if (used > 0.0 && wgs_left > 1 && room < (pieces > 0 ? 1 : kMinPiece)) {      // not worth opening this here
                    sp->wg_tile_begin[++wg] = rg * T + begin[f] + t;
                    used = 0.0;
                    pieces = 0;
                    continue;
                }
                int take = (int)(room + 0.5);
                if (take < 1) take = 1;
                if (take > tiles[f] - t || wgs_left == 1) take = tiles[f] - t;
                used += opening + take;
                left -= take + (t == 0 ? kOpenCost : 0.0) + (t == 0 && f == 0 ? kJobCost : 0.0);
                ++pieces;
                t += take;
                if (t < tiles[f]) {
                    sp->wg_tile_begin[++wg] = rg * T + begin[f] + t;
                    used = 0.0;
                    pieces = 0;
                }
            }
            ++f;
        }
    }
    sp->wgs = wg + 1;
    for (int i = sp->wgs; i <= HW_MAX_SPLITS; ++i) sp->wg_tile_begin[i] = nrg * T;
    sp->max_pieces = sp->usual_pieces = 1;
    for (int rg = 0, g = 0; rg < nrg; ++rg) {
        while (sp->wg_tile_begin[g + 1] <= rg * T) ++g;
        int last = g;
        while (sp->wg_tile_begin[last + 1] < (rg + 1) * T) ++last;
        if (last - g + 1 > sp->max_pieces) sp->max_pieces = sp->usual_pieces = last - g + 1;
    }
}

// Calls with at least a row group for every workgroup of a head (one workgroup per CU; at head dimension 256 also with fewer, which
// are then all in runs).  A run across row groups writes fp32 partial sums for both of its ends, 37 MB a layer for 1024 tokens at 40/8
// heads, which the merge reads again in 11.6 us.  Here floor(row groups / workgroups) row groups go whole to each workgroup, which holds
// complete rows at the end and writes the result, and only the remainder is cut into runs (whole_deal), a fifth of the rows with 40 row
// groups on 32 workgroups.  With no remainder there is no merge launch.  The remainder are the first row groups, which see least of a
// causal chunk.
// Against runs, resp. rounds, a layer: 1024 tokens behind 4096 (40/8, D = 128) 124 -> 117 us, 2 x 574 behind 1333 88 -> 83.5, 1500
// behind nothing at 32/8 69 -> 61.5, 1500 behind 128 66.5 -> 60 (and see whole_deal).  Where the heads divide the CUs this is never
// more work a CU than rounds.  Where they do not, CUs stay idle that rounds would use, and the workgroups take nrg / wgs row groups
// one after the other against the rounds: 9 row groups of 56 heads (1119 tokens behind 1200, D = 128) 2.25 against 2, 106 against
// 101 us; 5 of 96 2.5 against 2 (D = 64: 65 against 60 behind 1200, 131 against 116 behind 4000), 3 of 140 3 against 2 (144 against
// 115).  What is saved in partial sums is worth about 16 tiles of that: 621 tokens behind 150 at 96 heads (25 tiles) 39 against 43 us.
// (Of 400 calls of 1 to 160 heads 9 took longer by 3 % or more, up to 31 %, with whole row groups throughout; 1 does with the line, 5 %.)
// Head dimension 256: the plan's kernel takes 16 rows a workgroup, so every 16 rows stream the K/V through a CU again.  Enough of
// that, counted in tiles a CU takes in, and 128-row workgroups are faster, whose openings cost more.  16/8 heads, bf16, us a layer
// before / after: 1024 tokens behind 4096 (640 tiles a CU) 296 -> 111, 1500 behind 100 168 -> 70, 2 x 200 behind 5000 154 -> 79, 2 x 300
// behind 500 (84) 75 -> 43; below the line 2 x 128 behind 1500 (55) 34 -> 36.5, 256 behind 1000 (40) 24 -> 35.5.
// With one row group nothing is streamed twice, whatever the context: 1 to 16 rows behind 4 K to 60 K at 16/8, 16/16, 32/32, 32/4 and
// 64/8 heads take 0.60 to 1.01 times as long in the 16-row kernel (81.1 against 100.6 us: 4 workers x 4 tokens behind 30 K, 16/16).
// Above that both launches are priced, in us, by fits to 1122 calls timed both ways (17 to 2000 rows of 1 to 8 workers, 2 to 17
// fragments, 1 to 32 kv heads, 10 to 400 tiles a CU): the 16-row one by the tiles of its workgroups, less where their number lets
// every kv head keep to an XCD, whose L2 its row groups then share; the 128-row one by its tiles and by the most fragments that one
// workgroup opens, into whose run short ones crowd; both by the K/V itself (+-11 % each).  Of the 845 calls above the tile count
// alone 54 lost, up to 1.49 times (a step of 17 fragments in 2 row groups).  The 736 that kWorth leaves gain 1.54 in the median, 5 of
// them lose up to 1.12 times; the 44 that would have gained more than 1.03 gain 1.13 in the median.
constexpr int kWide256Visits = 56;
static bool wide_256(const hw_problem* p, int num_cus, const CallPlan& cp) {
    const hw_plan& plan = cp.plan[0];
    if (p->E != 256 || p->dtype == HW_F32 || p->len_dev != nullptr || p->row_blocks != 0 || plan.row_groups < 2) return false;
    constexpr double kWorth = 1.12;
    const double once = (double)plan.tiles_per_head * p->Hkv / num_cus;      // tiles a CU takes in where every tile is read once
    if (plan.row_groups * once < kWide256Visits) return false;
    const int rounds = (plan.workgroups + num_cus - 1) / num_cus, nrg = (plan.rows + hw::PLAN_SLOT_ROWS - 1) / hw::PLAN_SLOT_ROWS;
    const double run16 = (double)rounds * plan.tiles_per_head / plan.wgs_per_head, run128 = (double)nrg * plan.tiles_per_head * p->Hkv / num_cus;
    int nf = 0, crowd = 0, inside = 0;           // fragments; the most of them that a run of run128 tiles touches; those of the window
    for (int f = 0, first = 0; f < p->F; ++f) {
        if (p->len[f] == 0) continue;
        ++nf;
        ++inside;
        for (; plan.tile_begin[f] - (plan.tile_begin[first + 1] - 1) >= run128 && first < f; ++first) inside -= p->len[first] > 0 ? 1 : 0;
        crowd = std::max(crowd, inside);
    }
    const double narrow = 7.7 + (plan.workgroups % 8 == 0 ? 0.48 : 0.8) * run16 + 0.6 * nf + 0.8 * once;
    const double wide = 17.4 + 1.58 * run128 + 3.6 * crowd - 0.56 * once;
    return narrow > kWorth * wide;
}

bool whole_size(const hw_problem* p, int num_cus, const CallPlan& cp, WholePlan* wp) {
    const hw_plan& plan = cp.plan[0];
    if (cp.groups != 1 || p->splits > 0 || plan.tiles_per_head < 1) return false;
    const bool few_groups = wide_256(p, num_cus, cp);        // may have fewer row groups than workgroups
    if (plan.row_blocks != hw::WIDE_ROW_BLOCKS && !few_groups) return false;
    const int nrg = (plan.rows + hw::PLAN_SLOT_ROWS - 1) / hw::PLAN_SLOT_ROWS, T = plan.tiles_per_head;
    int wgs = num_cus / p->Hkv;
    if (wgs > hw::MAX_SPLITS) wgs = hw::MAX_SPLITS;
    if (wgs < 1 || (nrg < wgs && !few_groups) || (long long)nrg * T >= (1ll << 30) || (long long)wgs + nrg >= (1 << 15)) return false;
    // the kernel divides (head, workgroup) pairs by the workgroups per head (see magic_exact)
    if ((unsigned long long)wgs * wgs * p->Hkv >= (1ull << 32)) return false;
    const int rounds = (plan.workgroups + num_cus - 1) / num_cus;
    if (!few_groups && (long long)(nrg - rounds * wgs) * T > 16ll * wgs) return false;
    wp->wgs = wgs;
    wp->split = nrg % wgs;
    wp->whole = nrg - wp->split;
    StreamPlan& sp = wp->runs;
    sp.wgs = wgs;
    sp.slots = wp->split > 0 ? wgs + wp->split - 1 : 0;
    const size_t rows = (size_t)sp.slots * hw::PLAN_SLOT_ROWS;
    sp.partial_bytes = (size_t)p->Hkv * rows * ((size_t)p->Ev + 2) * sizeof(float);
    sp.workspace_bytes = ((sp.partial_bytes + (size_t)p->Hkv * plan.rows * 2 * sizeof(int) + 255) & ~(size_t)255) + cp.rope_bytes;
    wp->workspace_bytes = sp.workspace_bytes;
    return true;
}

// One worker that brings the newest S tokens of the last fragment (a causal chunk) sees of that fragment what lies before its own
// tokens.  Dealing the remainder by the tiles seen pays where they are few enough and the remainder is large enough: plain / this, us
// a layer, 1400 tokens at 40/8 heads (23 row groups left for 32 workgroups) with the chunk 0.8, 0.5 and a third of the tiles 1.15,
// 1.05 and 1.03 times, 830 (one left) 0.94, 0.96 and 0.97, 1024 (eight left) 1.08, 0.96 to 1.06 and 1.00.  The lines are drawn through
// 623 calls of 13 head layouts.  With more than a quarter of the workgroups' number left, the chunk above a third: means of 1.00 to
// 1.14 by share, 0.97 at worst; with less left but more than one, above a half: 1.00 to 1.11, 0.98 at worst.  With one left 0.97
// whatever the share, and below a third 1.00.  Head dimension 256 with all row groups in runs: 0.75 to 1.09 with less than half the
// workgroups' number, 0.97 to 1.16 above the lines here.
bool deal_by_seen(const hw_problem* p, const CallPlan& cp, const WholePlan& wp) {
    const int T = cp.plan[0].tiles_per_head, chunk = (p->S + hw::TILE - 1) / hw::TILE;
    int last = p->F - 1;
    while (last > 0 && p->len[last] == 0) --last;
    if (p->W != 1 || p->len[last] < p->S) return false;
    if (wp.whole == 0) return 2 * wp.split > wp.wgs && (2 * chunk > T || (3 * chunk > T && 8 * wp.split > 5 * wp.wgs));
    return (2 * chunk > T && wp.split > 1) || (3 * chunk > T && 4 * wp.split > wp.wgs);
}

// One worker that brings the newest S tokens of the last fragment.
static bool causal_chunk(const hw_problem* p) {
    int last = p->F - 1;
    while (last > 0 && p->len[last] == 0) --last;
    return p->W == 1 && p->len[last] >= p->S;
}

// Whether the openings of a launch are prepared beside the tiles before them (attention_wide_kernel, AHEAD).  At head dimension 128, where
// that was measured to pay.  At 64 a tile is half the arithmetic beside the same scalar work: pre-rotated queries of 1 to 8 workers and
// 2 to 200 tokens at four head layouts took 1.00 to 1.035 times as long, 1.018 in the mean of 26 calls (4 workers x 32 tokens behind 4781
// at 32/8 heads, fp16, 22.2 -> 21.5 us a layer without), prompt chunks 1.02 to 1.06.
// With one or two openings a workgroup there is little to hide, and the opening itself is longer.  bf16, how many times as fast:
//   whole row groups, one for each workgroup and none left over: 0.954 to 0.991 below 64 tiles (512 tokens from nothing at 64/8 heads
//     17.4 against 18.1 us a layer, 802 behind 479 at 40/8 31.8 against 32.4; three of 16 calls gained, up to 1.015), 0.99 to 1.034 from
//     there on, 1.009 in the mean of 17; with a second one each 1.015 to 1.08, with a remainder to deal 0.985 to 1.55 (it is dealt for
//     this form);
//   runs alone: 0.970 to 1.038 with up to three fragments, 0.992 in the mean of 49 calls, 0.997 in the mean of 21 with four and five,
//     0.982 to 1.054 with six and more, 1.007 in the mean of 40.
// Pre-rotated queries have no rotation to wait for: 1.007 to 1.22 in whole row groups and in runs; in rounds 0.98 to 1.11 with three
// fragments or a workgroup to a row group, 1.012 in the mean of the 51 with least to do; with one opening a workgroup 0.974 to 1.03, 0.997
// in the mean of ten.
bool openings_ahead(const hw_problem* p, const hw_plan& plan, bool prerotated, bool stream_runs, const WholePlan* whole) {
    if (p->E != 128) return false;
    int nf = 0;
    for (int f = 0; f < p->F; ++f) nf += p->len[f] > 0 ? 1 : 0;
    if (prerotated) return stream_runs || nf > 2 || plan.wgs_per_head == 1;
    if (whole != nullptr) return whole->split > 0 || whole->whole > whole->wgs || plan.tiles_per_head >= 64;
    return stream_runs && nf >= 6;
}

// The remainder in runs: the smallest share (tiles, with openings) at which the workgroups, taking one after the other what fits,
// use up the row groups, found by bisection.  Dealt by the tiles seen, those behind them go with the piece in front, so that no
// workgroup opens a row group for tiles that none of its rows sees.  (Should the locations say otherwise, the launch is merely less
// even.)
// At head dimension 128 the kernel does not take unseen tiles in.  Then a causal chunk is dealt by the tiles seen whatever its share,
// and the workgroups with the later row groups, which see most, get less of the remainder or none of it.  (Taking in fewer tiles alone
// gave nothing, the last row group's workgroup having as many as before; nor did unequal shares while unseen tiles cost as much as
// others.)  us a layer: 938 tokens behind 577 at 40/8 heads 51 -> 44, 1088 behind 527 at 32/8 48 -> 40, 1112 behind 62 46 -> 41.5, 1024
// behind 4096 117 -> 115; of 86 calls of six head layouts, timed in turn with the form before, all are faster, 1.008 to 1.27 times, 1.095 in the
// mean; with the lines of deal_by_seen in front of it they would be 0.97 to 1.15 times slower, 1.022 in the mean.  The costs of a piece and
// a fragment are from the same calls: against 20 and 4 tiles 0.989 in the mean with 8 and 2 (0.86 at worst), 0.995 with 12 and 2, 0.999 with
// 16 and 4, 1.001 with 24 and 4; of several workers, dealt by all tiles, 1.015 with 8 and 2, 1.017 with 12 and 2, 1.016 with 24 and 4.
void whole_deal(const hw_problem* p, const CallPlan& cp, WholePlan* wp) {
    const hw_plan& plan = cp.plan[0];
    const int T = plan.tiles_per_head, wgs = wp->wgs, split = wp->split;
    StreamPlan& sp = wp->runs;
    if (split == 0) {
        std::fill(sp.wg_tile_begin, sp.wg_tile_begin + HW_MAX_SPLITS + 1, 0);
        sp.max_pieces = sp.usual_pieces = 0;
        return;
    }
    int nf = 0, last = 0;
    for (int f = 0; f < p->F; ++f) {
        if (p->len[f] == 0) continue;
        last = f;
        ++nf;
    }
    const bool trimmed = p->E == 128;                        // the kernel does not take unseen tiles in
    const bool by_seen = trimmed ? causal_chunk(p) : deal_by_seen(p, cp, *wp);
    // in tiles: a piece's prologue and epilogue; a row group's fragments, spread over its tiles
    const double kPieceCost = !trimmed ? 8.0 : by_seen ? 20.0 : 12.0, kOpenCost = trimmed && by_seen ? 4.0 : 2.0;
    const double tile = 1.0 + kOpenCost * nf / T;
    const int gq = p->Hq / p->Hkv;
    auto seen_tiles = [&](int rg) {                          // up to the token of the row group's last row
        if (!by_seen) return T;
        const int token = (std::min((rg + 1) * hw::PLAN_SLOT_ROWS, plan.rows) - 1) / gq;
        return plan.tile_begin[last] + (p->len[last] - p->S + token + hw::TILE) / hw::TILE;
    };
    const double per_tile = 1.0 / tile;
    // (Both once and not in every step of the bisection: their divisions were most of its time.)
    int seen_of[HW_MAX_SPLITS];                              // of the row groups to deal, fewer than there are workgroups
    double low = 0.0, unseen = 0.0;
    for (int rg = 0; rg < split; ++rg) {
        seen_of[rg] = seen_tiles(rg);
        low += kPieceCost + seen_of[rg] * tile;
        unseen += trimmed ? 0 : T - seen_of[rg];
    }
    // what workgroup g has in hand with the row groups that are its alone, above workgroup 0 (later row groups see more)
    double ahead[HW_MAX_SPLITS];
    const int own = trimmed && by_seen ? wp->whole / wgs : 0;
    std::fill(ahead, ahead + wgs, 0.0);
    for (int i = 0; i < own; ++i) {
        const int first = seen_tiles(split + i * wgs);
        for (int g = 1; g < wgs; ++g) ahead[g] += (seen_tiles(split + i * wgs + g) - first) * tile;
    }
    auto deal = [&](double share) {                          // false if something is left
        int rg = 0, t = 0;
        for (int g = 0; g < wgs; ++g) {
            sp.wg_tile_begin[g] = rg * T + t;
            for (double room = share - ahead[g]; rg < split;) {
                const int rest = seen_of[rg] - t, take = std::min((int)((room - kPieceCost) * per_tile), rest);
                if (take < std::min(kMinPiece, rest)) break;
                room -= kPieceCost + take * tile;
                t += take;
                if (take < rest) break;
                if (!trimmed) room -= T - seen_of[rg];
                t = 0;
                ++rg;
            }
        }
        return rg == split;
    };
    // Between an equal part of the tiles seen and that of all with what a workgroup opens and leaves at most besides.
    low /= wgs;
    double high = low + unseen / wgs + ahead[wgs - 1] + 2.0 * kPieceCost + (kMinPiece + 1) * tile;
    while (!deal(high)) high *= 2.0;
    while (high - low > 0.25) {
        const double mid = 0.5 * (low + high);
        (deal(mid) ? high : low) = mid;
    }
    deal(high);
    for (int i = wgs; i <= HW_MAX_SPLITS; ++i) sp.wg_tile_begin[i] = split * T;
    sp.max_pieces = 0;
    int pieces = 0;
    for (int rg = 0, g = 0; rg < split; ++rg) {
        while (sp.wg_tile_begin[g + 1] <= rg * T) ++g;
        int last = g;
        while (sp.wg_tile_begin[last + 1] < (rg + 1) * T) ++last;
        sp.max_pieces = std::max(sp.max_pieces, last - g + 1);
        pieces += last - g + 1;
    }
    sp.usual_pieces = (pieces + split / 2) / split;
}

size_t call_workspace_bytes(const hw_problem* p, int num_cus, const CallPlan& cp) {
    WholePlan wp;
    StreamPlan sp;
    if (whole_size(p, num_cus, cp, &wp)) return std::max(cp.workspace_bytes, wp.workspace_bytes);
    return stream_size(p, num_cus, cp, &sp) ? std::max(cp.workspace_bytes, sp.workspace_bytes) : cp.workspace_bytes;
}

int paged_validate(const hw_paged_problem* p) {
    if (p == nullptr) return HW_ERR_NULL;
    if (p->dtype != HW_F32 && p->dtype != HW_F16 && p->dtype != HW_BF16) return HW_ERR_DTYPE;
    if (p->F < 1 || p->F > HW_MAX_FRAGMENTS) return HW_ERR_FRAGMENTS;
    if (p->W < 1 || p->Hq < 1 || p->Hkv < 1 || p->E < 1 || p->Ev < 1) return HW_ERR_SHAPE;
    if (p->Hq % p->Hkv != 0) return HW_ERR_SHAPE;
    if (!(p->scale > 0.f) || !std::isfinite(p->scale)) return HW_ERR_SHAPE;
    const bool varlen = p->cu_seqlens_q != nullptr;
    if (varlen ? p->total_q < 0 : (p->S < 1 || p->S >= (1 << 12))) return HW_ERR_SHAPE;
    if (p->block_size < 1 || p->block_size >= (1 << 12) || p->max_blocks < 1 || p->num_blocks < 1) return HW_ERR_SHAPE;
    if ((long long)p->block_size * p->max_blocks > (1ll << 20)) return HW_ERR_SHAPE;
    if ((long long)p->num_blocks * p->Hkv * p->block_size >= (1ll << 31)) return HW_ERR_SHAPE;
    const long long tokens = varlen ? p->total_q : (long long)p->W * p->S;
    const int gq = p->Hq / p->Hkv;
    if (gq >= (1 << 12) || tokens * gq >= (1 << 20) || p->W >= (1 << 20)) return HW_ERR_SHAPE;
    if (p->out == nullptr || p->q == nullptr || p->locations == nullptr || p->fragment_lengths == nullptr) {
        if (tokens > 0) return HW_ERR_NULL;
    }
    if (p->key_cache == nullptr || p->value_cache == nullptr || p->block_table == nullptr) return HW_ERR_NULL;
    if (!aligned16(p->out) || !aligned16(p->q) || !aligned16(p->key_cache) || !aligned16(p->value_cache)) return HW_ERR_ALIGN;
    if (p->E != p->Ev || (p->E != 64 && p->E != 128 && p->E != 256)) return HW_ERR_UNSUPPORTED;
    if (p->E == 256 && p->dtype == HW_F32) return HW_ERR_UNSUPPORTED;   // the paged kernel's two fp32 K tiles per wave exceed the LDS
    return HW_OK;
}

// At head dimension 256 the paged kernel takes 16 rows a workgroup, and the row groups of a sequence read its K/V one after the
// other: with more than two of them the tiles are kept in the L2 instead of being streamed past it.  16/8 heads, bf16, us a layer: 128
// query tokens on 12 528 166 -> 114, 4 x 64 on 12 000 291 -> 203, 4 x 24 131 -> 121, 4 x 24 on 3000 39.3 -> 39.4.  Two row groups
// of a sequence are under way together: 21 to 32 rows at 8 and 16 kv heads 0.93 to 1.13 times, 0.996 in the mean of 44 calls (4 x 16 on
// 3000 27.4 -> 28.8, on 12 000 84.7 -> 81.4), and 16 rows lose 0.87 to 0.91; 33 to 48 rows 0.94 to 1.20, 1.05 in the mean.
// Packed sequences share a launch whatever they bring, and only the device knows it, so the line is their mean, and it lies lower, as
// their rows are in few long chunks: 21 to 32 rows in the mean 0.97 to 1.29, 1.08 over 14 batches (31 decoding sequences and a chunk of
// 64 on 3000 at 32/4 128 -> 99); up to 20 rows 0.91 to 1.00; from 64 on 1.01 to 1.82 (7 decoding and a chunk of 128 on 12 000 at 64/8
// 639 -> 468).  What the decoding sequences beside a chunk lose is 3 % at most of the launch (63 and a chunk of 1024 on 1500 at 16/8
// 230 -> 237).  Ten head layouts, bf16 and fp16, 1 to 64 sequences; bit-identical both ways.
// (The 128-row form for D <= 128 reads a sequence a few times at most and lost 1 to 11 % with kept tiles, except with three row groups
// a sequence and more, 1 to 6 %, which only the device knows.)
bool paged_keep_in_l2(const hw_paged_problem* p, const hw_paged_plan& plan) {
    return p->E == 256 && plan.rows > (p->cu_seqlens_q != nullptr ? 20ll : 32ll) * p->W;
}

// One row group per sequence, and what the waves go through to find a length (F * S locations) is little: a decode step, a draft of a few
// tokens.  The measurements are at paged_share in hogwild_paged.hip.  (A caller that fixes the split keeps it.)
bool paged_shared(const hw_paged_problem* p, const hw_paged_plan& plan) {
    return p->cu_seqlens_q == nullptr && p->splits <= 0 && plan.row_blocks != hw::WIDE_ROW_BLOCKS && p->W >= 2 && p->W <= 64 &&
           plan.row_groups == p->W && plan.splits >= 2 && (long long)p->F * p->S <= 8;
}

// A launch of more workgroups than CUs evens itself out, as the workgroups of short sequences make room, and shares of one size only bring
// its last round into step.  10 to 64 sequences at 4 to 16 kv heads, bf16, against equal shares: where up to six steps are saved 0.77 to
// 1.16 times as fast, 0.957 in the mean of 83 steps; with more 0.95 to 1.45, 1.14 in the mean of 61; at head dimension 256 0.88 to 1.06,
// 0.947 in the mean of six, with seven to nine, 1.10 in the mean of eight with more.  At 64, where the opening of a workgroup is shorter, 1.01
// to 1.22 with six, 0.80 to 1.18 with less, 0.979 in the mean of 45.  With several tokens or fragments looking the
// lengths up takes longer than that is worth in every round (60 sequences of 8 tokens at 8/4 heads, D = 64 17.4 -> 20.7 us).
int paged_shares_save(const hw_paged_problem* p, const hw_paged_plan& plan, int num_cus) {
    if (plan.workgroups <= num_cus) return 0;
    if ((long long)p->F * p->S > 1) return -1;
    return p->E > 128 ? 9 : p->E == 128 ? 6 : 5;
}

size_t paged_call_bytes(const hw_paged_problem* p, const hw_paged_plan& plan) {
    if (!paged_shared(p, plan)) return plan.workspace_bytes;
    const size_t bytes = (size_t)p->Hkv * plan.splits * plan.rows * ((size_t)p->Ev + 2) * sizeof(float) + (size_t)p->Hkv * plan.rows * 2 * sizeof(int);
    return std::max(plan.workspace_bytes, (bytes + 255) & ~(size_t)255);
}

int paged_plan(const hw_paged_problem* p, int num_cus, hw_paged_plan* plan) {
    if (plan == nullptr) return HW_ERR_NULL;
    if (num_cus < 1) return HW_ERR_SHAPE;
    std::memset(plan, 0, sizeof(*plan));
    const bool varlen = p->cu_seqlens_q != nullptr;
    // the same limits as paged_validate(): the planner is also reachable on its own (hw_paged_plan_debug,
    // hw_paged_workspace_bytes), and the narrowing below must not be handed anything larger
    if (p->W < 1 || p->Hq < 1 || p->Hkv < 1 || p->Ev < 1 || p->Hq % p->Hkv != 0) return HW_ERR_SHAPE;
    if (varlen ? p->total_q < 0 : (p->S < 1 || p->S >= (1 << 12))) return HW_ERR_SHAPE;
    if (p->block_size < 1 || p->block_size >= (1 << 12) || p->max_blocks < 1) return HW_ERR_SHAPE;
    if ((long long)p->block_size * p->max_blocks > (1ll << 20)) return HW_ERR_SHAPE;
    const int gq = p->Hq / p->Hkv;
    const long long tokens = varlen ? p->total_q : (long long)p->W * p->S;
    if (gq >= (1 << 12) || tokens * gq >= (1 << 20) || p->W >= (1 << 20)) return HW_ERR_SHAPE;
    plan->rows = (int)(tokens * gq);
    // rows of one worker share its KV: one 16-row block is enough for plain decoding, two when a worker brings
    // more rows (several query tokens, wide GQA groups)
    const long long rows_per_worker = varlen ? (tokens * gq + p->W - 1) / p->W : (long long)p->S * gq;
    plan->row_blocks = rows_per_worker <= 16 ? 1 : 2;
    // more than one 16-row block per sequence: workgroups of up to 128 rows whose waves share every K/V tile through LDS
    // (16-bit types; the kernel keeps a sequence's block table in LDS, up to PAGED_WIDE_MAX_BLOCKS entries).  Measured on
    // four sequences of 12 528 tokens with 3 / 6 / 12 / 19 query tokens each (15 ... 95 rows per sequence): 36.7 / 36.7 /
    // 45.9 / 69.4 us against 49.4 / 49.5 / 84.6 / 84.7 us of the 32-row workgroups, which stream a sequence's KV once per
    // 32 rows; with one token each (5 rows) the two are equal (36.0 / 36.1 us).
    const bool wide_ok = p->dtype != HW_F32 && p->max_blocks <= hw::PAGED_WIDE_MAX_BLOCKS && p->E <= 128;
    if (wide_ok && rows_per_worker > 16) plan->row_blocks = hw::WIDE_ROW_BLOCKS;
    if (p->row_blocks == 1 || p->row_blocks == 2 || (p->row_blocks == hw::WIDE_ROW_BLOCKS && wide_ok)) plan->row_blocks = p->row_blocks;
    if (p->dtype == HW_F32 || p->E > 128) plan->row_blocks = 1;   // the fp32 and the 256-wide paged kernels exist with one row block only
    const bool wide = plan->row_blocks == hw::WIDE_ROW_BLOCKS;
    const int rpw = 16 * plan->row_blocks;
    long long items;
    if (varlen) items = p->W + tokens * gq / rpw;          // sum_w ceil(rows_w / rpw) <= W + rows / rpw
    else items = (long long)p->W * (((long long)p->S * gq + rpw - 1) / rpw);
    if (items < 1) items = 1;
    plan->row_groups = (int)items;
    if (wide && varlen && p->splits <= 0 && p->W <= hw::PLAN_MAX_GROUPS && items <= hw::PLAN_MAX_GROUPS) {
        // Packed queries in 128-row workgroups: how many rows a sequence brings and how long its KV is are device data,
        // so the device deals the workgroups (every workgroup works out its own share in its prologue):
        // every kv head gets `slots` workgroup slots -- the CUs filled once, a slot per possible row group at least, not
        // more than a slot per four tiles of the longest KV the tables allow -- and each row group takes a share of them
        // in proportion to its work.  A caller that fixes the split (splits > 0) gets the unplanned launch below.
        const long long tiles = ((long long)p->block_size * p->max_blocks + hw::TILE - 1) / hw::TILE;
        const long long fill = num_cus / p->Hkv > 0 ? num_cus / p->Hkv : 1;
        const long long by_work = (long long)p->W * tiles / 4;
        long long slots = fill < by_work ? fill : by_work;
        if (slots < items) slots = items;
        // many possible row groups: the launch oversubscribes the CUs anyway, and slots beyond one per row group are
        // what lets the device cut a long sequence among many short ones
        if (2 * items > fill) slots = items + (fill < by_work ? fill : by_work);
        if (slots >= (1 << 16) || (long long)p->Hkv * slots >= (1 << 20)) return HW_ERR_SHAPE;
        plan->device_planned = 1;
        plan->row_groups = (int)slots;
        plan->splits = 1;
        plan->workgroups = (int)(p->Hkv * slots);
        const unsigned long long positions = (unsigned long long)p->block_size * p->max_blocks + hw::TILE;
        if (!magic_exact((unsigned long long)slots, (unsigned long long)p->Hkv * slots) ||
            !magic_exact((unsigned long long)gq, (unsigned long long)tokens * gq + 32) ||
            !magic_exact((unsigned long long)p->block_size, positions))
            return HW_ERR_SHAPE;
        plan->workspace_bytes = (size_t)p->Hkv * (size_t)slots * hw::PLAN_SLOT_ROWS * ((size_t)p->Ev + 2) * sizeof(float) +
                                (size_t)p->Hkv * (size_t)(plan->rows > 0 ? plan->rows : 1) * 2 * sizeof(int);
        plan->workspace_bytes = (plan->workspace_bytes + 255) & ~(size_t)255;
        return HW_OK;
    }
    int splits = p->splits;
    if (splits <= 0) {
        // The paged kernels run one workgroup per CU.  Few (kv head, row group) pairs: split until every CU has
        // one workgroup.  More pairs than half the CUs: the chip is oversubscribed anyway, and about three
        // workgroups per CU even out the tail between sequences of different length (measured best on packed
        // variable-length queries) -- there a wave keeps at least four tiles.
        const long long pairs = (long long)p->Hkv * items;
        const long long tiles = ((long long)p->block_size * p->max_blocks + hw::TILE - 1) / hw::TILE;
        long long s, by_work;
        if (wide) {
            // every wave takes every tile of its workgroup: fill the CUs once, at least four tiles per workgroup
            s = pairs < num_cus ? num_cus / pairs : 1;
            by_work = (tiles + 3) / 4;
        } else if (2 * pairs <= num_cus) {
            s = num_cus / pairs;
            by_work = (tiles + hw::NWAVES - 1) / hw::NWAVES;
        } else {
            s = (3LL * num_cus + pairs - 1) / pairs;
            by_work = tiles / (4 * hw::NWAVES);
        }
        if (s > by_work) s = by_work;
        splits = (int)s;
    }
    if (splits > 64) splits = 64;
    if (splits < 1) splits = 1;
    plan->splits = splits;
    const long long wgs = (long long)p->Hkv * items * splits;
    if (wgs >= (1 << 20)) return HW_ERR_SHAPE;
    plan->workgroups = (int)wgs;
    // the kernel divides with multiply-high by ceil(2^32 / d): workgroup id by splits, the quotient by row groups, row
    // group by row groups per worker, row by GQA ratio, token by tokens per worker, position by block size.  A large
    // divisor (many sequences) can make that inexact; such a launch is refused instead of decoding wrong indices.
    const unsigned long long positions = (unsigned long long)p->block_size * p->max_blocks + hw::TILE;
    if (!magic_exact((unsigned long long)splits, (unsigned long long)wgs) ||
        !magic_exact((unsigned long long)items, (unsigned long long)p->Hkv * items) ||
        !magic_exact((unsigned long long)(varlen ? 1 : items / p->W), (unsigned long long)items) ||
        !magic_exact((unsigned long long)gq, (unsigned long long)tokens * gq + 32) ||
        !magic_exact((unsigned long long)(varlen ? 1 : p->S), (unsigned long long)tokens + 32) ||
        !magic_exact((unsigned long long)p->block_size, positions))
        return HW_ERR_SHAPE;
    plan->workspace_bytes = (size_t)p->Hkv * splits * (size_t)(plan->rows > 0 ? plan->rows : 1) * ((size_t)p->Ev + 2) * sizeof(float);
    plan->workspace_bytes = (plan->workspace_bytes + 255) & ~(size_t)255;
    return HW_OK;
}

}  // namespace host
}  // namespace hw
