// Host-only part of the library: argument validation and split planning.  Plain C++ with no HIP dependency, so it
// builds with any host compiler (the test suite builds it with g++ -fsanitize=address,undefined and fuzzes it).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "../../include/hogwild_hip.h"

namespace hw {
namespace host {

bool aligned16(const void* p);
size_t elem_size(int dtype);

// ceil(2^32 / d) mod 2^32: the multiplier of the kernels' multiply-high division (0 stands for d == 1)
unsigned magic_of(int d);
// true if floor(n / d) == mulhi(n, magic_of(d)) for every 0 <= n <= n_max
bool magic_exact(unsigned long long d, unsigned long long n_max);

int validate(const hw_problem* p, int fused);
// fused != 0: size the workspace for hw_fused_attention (room for the rotated queries when the rotary width is not the head
// dimension and the caller passes no rq buffer); 0: for hw_sdpa
int make_plan(const hw_problem* p, int num_cus, hw_plan* plan, int fused = 1);
// Whether the launch's K/V tiles are to stay in the L2 instead of being streamed past it (hogwild_plan.cpp).
bool keep_in_l2(const hw_problem* p, const hw_plan& plan, int num_cus);
// A call's fragments in groups of at most HW_MAX_LAUNCH_FRAGMENTS, one attention launch each.  Group i takes fragments
// first[i] .. first[i] + count[i] - 1, is planned like a problem of its own (plan[i]; its workspace_bytes is not used) and
// writes its split-K partials into slots slot_base[i] .. slot_base[i] + plan[i].wgs_per_head - 1 of every kv head's
// `slots` slots.
constexpr int MAX_GROUPS = (HW_MAX_FRAGMENTS + HW_MAX_LAUNCH_FRAGMENTS - 1) / HW_MAX_LAUNCH_FRAGMENTS;
struct CallPlan {
    int groups;
    int first[MAX_GROUPS], count[MAX_GROUPS], slot_base[MAX_GROUPS];
    hw_plan plan[MAX_GROUPS];
    int slots;                 // partial slots per kv head over all groups
    size_t partial_bytes;      // part_o + part_ml of all slots
    size_t rope_bytes;         // room for the rotated queries (fused entry, rotary width != head dim, no rq buffer), else 0
    size_t workspace_bytes;    // partial_bytes + rope_bytes
};
int plan_call(const hw_problem* p, int num_cus, CallPlan* cp, int fused);
// The other way to deal a call of 128-row workgroups, for row groups that do not fill the CUs evenly (see stream_size in
// the source): one workgroup per CU takes an equal run of the sequence (row group 0: tiles 0 .. T-1, row group 1: ...) of
// its kv head, across row groups.  Piece (workgroup g, row group rg) writes its partial sums into slot g + rg.
struct StreamPlan {
    int wgs;                             // workgroups per kv head
    int slots;                           // partial slots of PLAN_SLOT_ROWS rows per kv head, not all of them used
    int max_pieces, usual_pieces;        // pieces of one row group, at most and for most of them
    int wg_tile_begin[HW_MAX_SPLITS + 1];   // first tile of each workgroup, counted through all row groups
    size_t partial_bytes;                // part_o + part_ml of all slots
    size_t workspace_bytes;              // partials, the merge's row table, and CallPlan::rope_bytes
};
// Chooses and sizes: false if the call is better served by CallPlan's launch.  Fills everything but the boundaries and
// max_pieces, with the most workgroups that the deal may come to.
bool stream_size(const hw_problem* p, int num_cus, const CallPlan& cp, StreamPlan* sp);
// Deals the runs of a call that stream_size has taken: wgs, max_pieces, wg_tile_begin.  Only the launch needs them, and they
// take a loop over row groups and workgroups (40 row groups, 32 workgroups: 1.7 us with 2 fragments, 2.6 with 60, 46 when it
// visited every fragment of every row group; sizing 0.02).
void stream_deal(const hw_problem* p, const CallPlan& cp, StreamPlan* sp);
// The same for calls with at least a row group for every workgroup, and at head dimension 256 (see whole_size in the source): as many
// row groups as go round are dealt whole -- their workgroups write the result, no partial sums -- and the others in runs.
struct WholePlan {
    int split, whole;                    // row groups 0 .. split - 1 in runs, the `whole` behind them one to a workgroup
    int wgs;                             // workgroups per kv head
    StreamPlan runs;                     // of the first (split > 0; filled by whole_deal but for the sizes)
    size_t workspace_bytes;
};
bool whole_size(const hw_problem* p, int num_cus, const CallPlan& cp, WholePlan* wp);
// Every call of the kind deals about ten times over row groups and workgroups until the share is found: 2.0 us on the host with 8 row
// groups left for 32 workgroups, 2.4 with 17 for 64, 29 with 213 for one kv head's 256 (5.2, 6.2 and 39 when what a workgroup has in
// hand and sees was worked out again in every one of them).  Sizing takes 0.02.
void whole_deal(const hw_problem* p, const CallPlan& cp, WholePlan* wp);
// Whether whole_deal counts the tiles that a causal chunk sees (hogwild_plan.cpp).
bool deal_by_seen(const hw_problem* p, const CallPlan& cp, const WholePlan& wp);
// Whether a launch of 128-row workgroups prepares its openings ahead (hogwild_plan.cpp).  `whole`: of a launch in whole row groups, else null.
bool openings_ahead(const hw_problem* p, const hw_plan& plan, bool prerotated, bool stream_runs, const WholePlan* whole);
// What a call asks for: room for CallPlan, the caller's fallback, and for the launch that is preferred to it (whole row groups
// before runs; 1024 tokens behind 4096 at 40/8 heads, D = 128: 21.3 MB, where the runs that are not taken there would need 38.1).
size_t call_workspace_bytes(const hw_problem* p, int num_cus, const CallPlan& cp);
int paged_validate(const hw_paged_problem* p);
int paged_plan(const hw_paged_problem* p, int num_cus, hw_paged_plan* plan);
// Whether the workgroups of a paged launch may be shared out by the lengths of the sequences (hogwild_plan.cpp), and what a call asks
// for: hw_paged_plan's workspace, the caller's fallback, and the merge's row table.
bool paged_shared(const hw_paged_problem* p, const hw_paged_plan& plan);
size_t paged_call_bytes(const hw_paged_problem* p, const hw_paged_plan& plan);
// How many steps of its waves the longest sequence has to need less with other than equal shares, or -1: equal ones always.
int paged_shares_save(const hw_paged_problem* p, const hw_paged_plan& plan, int num_cus);
// Whether the tiles of a paged launch are to stay in the L2 (hogwild_plan.cpp).
bool paged_keep_in_l2(const hw_paged_problem* p, const hw_paged_plan& plan);

}  // namespace host
}  // namespace hw
