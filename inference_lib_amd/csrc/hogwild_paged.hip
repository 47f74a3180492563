// Paged variants of the Hogwild! attention path for gfx950 (MI355X, CDNA4, wave64).
//
//   paged_attention_kernel ... the roles of hogwild_paged_attention_gpu_kernel21 (src/kernels/kernel_v21.cuh:318-602)
//                              and hogwild_varlen_paged_attention_gpu_kernel21 (:658-899) of the reference
//   copy_to_blocks_kernel .... copy_to_blocks_kernel (src/cache.cuh:6-49)
//
// The KV of worker (sequence) w lives in fixed-size blocks of one cache tensor, [num_blocks, Hkv, block_size, D],
// and position l of the sequence is found through block_table[w][l / block_size] (kernel_v21.cuh:405-411).
// Every "fragment" f attends the same sequence from position 0 with its own queries and its own bound
// min(fragment_lengths, location + 1) (kernel_v21.cuh:385-388).
//
// Work decomposition: a workgroup owns one kv head, one row group of one worker (up to 16 or 32 query rows, a row
// being one (token, q-head-in-group) pair of that worker) and every ns-th stripe of the sequence's 32-token
// tiles: tile t goes to wave t mod (4 * ns) of the (kv head, row group).  Nothing about the sequence lengths
// is known on the host (they are device tensors): ns is the host's nsplit, or what paged_share makes of it.  The per-tile arithmetic,
// the LDS staging and the partial/merge scheme are those of the fragment kernel; what differs is the address
// generation: each lane computes the cache row of "its" token of the tile from the block table (one table entry
// per lane and tile, prefetched two tiles ahead), the rows a lane has to fetch are picked from those with
// ds_bpermute, and K goes global -> LDS / V global -> registers with per-lane 64-bit addresses.  Tokens that no
// row of the group can see are redirected to the last visible token, so no byte outside the visible part of the
// sequence is ever read; block ids are clamped into the cache, so a corrupt table cannot fault the GPU.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "hogwild_kernels.h"
#include "hogwild_device.h"

// waves per SIMD the one-row-block 16-bit kernels are register-budgeted for (tuning knob)
#ifndef HW_PAGED_MINW
#define HW_PAGED_MINW 1
#endif

namespace hw {

// The workgroups of a kv head shared out by the lengths of the sequences (fixed-length operator, one row group per sequence; the lengths
// are device data, so every wave works the shares out for itself).  nsplit workgroups for each sequence whatever its length left the
// launch waiting for those of the longest: append and attention of five sequences of 296 to 10 543 tokens (40/8 heads, D = 128, bf16)
// 31.7 -> 22.3 us, eight of 210 to 9000 at 32/8 37 -> 24, four of 300 to 11 000 at 16/8 and D = 256 41 -> 28.6, five of 844 to 5868 23.8 -> 22.2.
// The shares are the smallest bound on the tiles of a workgroup (in steps of the four waves) at which the sequences' workgroups
// are no more than there are, found by trying one bound in every lane.  Working that out and requesting the queries again takes 0.9 us,
// a step of the four waves 1.1 to 1.2 (fit over 63 decode steps of 2 to 12 sequences, all head layouts): nsplit each wherever the longest
// sequence needs two steps at most, or no more than it would need with even shares (more workgroups than CUs: paged_shares_save).  The
// lengths are read ahead of the queries, which are requested for equal shares, as are the partial sums in the merge.
// A sequence with fewer workgroups has fewer tiles that are a wave's first, whose largest weight the storage type holds exactly: 1.04 to
// 1.09 times the error against float64 (seven ragged steps x 6 seeds, bf16 and fp16).  The reference of the exponentials therefore follows
// the tiles of such a sequence (compute_tile's FOLLOW): 0.96 to 1.00 times the error of equal shares.
struct PagedShare {
    int w, split, ns, slot0;      // sequence, which of its ns workgroups, the first one's slot
    bool found;                   // false: a slot that is left over
};
// (loc0, len0: the first location of sequence min(lane, W - 1) and the first fragment's length, requested ahead of what the workgroup
// needs besides, so that this is worked out while the rest is on its way)
__device__ __forceinline__ PagedShare paged_share(const PagedDevHeader& ph, int item, int split, int lane, int loc0, int len0) {
    const int cap = ph.block_size * ph.max_blocks, T = ph.LW * ph.LS, w = min(lane, ph.W - 1);
    // lane = sequence: the tiles that its workgroups go through
    auto tiles_to = [&](int most, int len) { return (max(min(min(len, cap), most < cap ? most + 1 : cap), 0) + TILE - 1) / TILE; };
    int most = loc0;
    for (int s = 1; s < ph.LS; ++s) most = max(most, ph.loc[w * ph.LS + s]);
    int tiles = tiles_to(most, len0);
    for (int f = 1; f < ph.F; ++f) {
        most = -1;
        for (int s = 0; s < ph.LS; ++s) most = max(most, ph.loc[f * T + w * ph.LS + s]);
        tiles += tiles_to(most, ph.frag_len[f]);
    }
    if (lane >= ph.W) tiles = 0;
    // (nothing here depends on the order of the sequences: a sequence's share, and so its result, is the same wherever it is listed)
    const PagedShare equal = {item, split, ph.nsplit, item * ph.nsplit, true};
    const int slots = ph.W * ph.nsplit, slot = item * ph.nsplit + split;
    // whether the longest sequence's workgroups would have more than `most_tiles` tiles each with equal shares
    auto more_than = [&](int most_tiles) { return __ballot(tiles > ph.nsplit * most_tiles) != 0; };
    // (on their own: sequences of one length and short steps leave here, 0.1 us sooner than behind the sum)
    if (__ballot(lane < ph.W && tiles != __builtin_amdgcn_readlane(tiles, 0)) == 0 || !more_than(2 * NWAVES)) return equal;
    const int saved = NWAVES * (ph.flags >> PH_SAVED_SHIFT);   // (in tiles, like the bounds)
    const int all = __builtin_amdgcn_readlane(wave_scan_inclusive(tiles), 63);
    const int least = max(1, (int)((float)all * __builtin_amdgcn_rcpf((float)(NWAVES * slots))));          // steps with even shares, less what is left over
    int even = NWAVES * (least + (least * NWAVES * slots < all ? 1 : 0));
    // (with many sequences the search is long; what half a workgroup of each leaves over is estimated instead)
    if (saved > 0) even = (int)((float)all * __builtin_amdgcn_rcpf((float)(slots - (ph.W >> 1)))) + saved;
    if (!more_than(even)) return equal;
    // lane = a bound on the tiles of a workgroup, multiples of the four waves: does every sequence get its workgroups?
    const float mine = (float)tiles;
    const int bound = NWAVES * (least + lane * (1 + (least >> 5)));
    const float per = __builtin_amdgcn_rcpf((float)bound);
    auto groups = [&](float t, float per_group) { return max(1, (int)__builtin_ceilf(t * per_group - 0.01f)); };
    int need = 0;
    for (int sq = 0; sq < ph.W; ++sq) need += groups(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine), sq)), per);
    const unsigned long long fits = __ballot(need <= slots);
    const int fit = fits != 0 ? __builtin_ctzll(fits) : 0;
    if (fits == 0 || !more_than(__builtin_amdgcn_readlane(bound, fit))) return equal;
    const float best = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(per), fit));
    const int n = lane < ph.W ? groups(mine, best) : 0;
    const int slot0 = wave_scan_inclusive(n) - n;
    const unsigned long long owner = __ballot(slot >= slot0 && slot < slot0 + n);
    PagedShare r;
    r.found = owner != 0;
    r.w = r.found ? __builtin_ctzll(owner) : 0;
    r.slot0 = __builtin_amdgcn_readlane(slot0, r.w);
    r.split = slot - r.slot0;
    r.ns = __builtin_amdgcn_readlane(n, r.w);
    return r;
}

// SMALL: below 4 GB the K cache is reached through one buffer descriptor, and its transfers are buffer loads.  A transfer by 64-bit address
// is a flat-encoded instruction with an LDS operand, for which the compiler waits until nothing is outstanding: it emptied the
// look-ahead at every tile (vmcnt(0) in front of each request, where 16 and 17 operations may be in flight).  Four sequences of 12 528
// tokens, append and attention 41.2 -> 39.3 us (6.0 TB/s in the attention), 2500 to 3600 tokens 18.2 -> 17.1, five of 296 to 10 543 22.3 -> 20.4;
// bit-identical.
struct CacheView {
    __amdgpu_buffer_rsrc_t k;
};
__device__ __forceinline__ CacheView make_cache_view(const PagedDevHeader& ph, int krow) {
    CacheView v;
    v.k = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(reinterpret_cast<unsigned long long>(ph.kcache)), 0,
                                            (int)((unsigned)ph.num_blocks * (unsigned)ph.Hkv * (unsigned)ph.block_size * (unsigned)krow), 0x00020000);
    return v;
}

template <int AUX>
__device__ __forceinline__ void cache_transfer(const CacheView& v, char* lds, unsigned offset) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(v.k, HW_LDS_PTR(lds), 16, offset, 0, 0, AUX);
}

template <class DT, int E, int EV, int RB, int MINW, bool SMALL, bool KEEP = false>
__global__ __launch_bounds__(NTHREADS, MINW) void paged_attention_kernel(const PagedHeader args) {
    constexpr int AUX = KEEP ? 0 : HW_KV_AUX;
    // Tiles are kept for the several row groups of a sequence, and such sequences are not shared out (paged_shared): 74.0 -> 72.9 us with
    // packed queries of 26, 24 and 42 tokens over 8464, 379 and 532 positions at 16/8 heads of 256.
    constexpr bool FOLLOW = Elem<DT>::size == 2 && !KEEP;
    typedef Geo<DT, E, EV> G;
    constexpr bool STATED = G::KL + 8 * G::NVL >= 32;      // the waits for K are stated by hand (wait_k_landed)
    constexpr int ROWS = RB * 16;
    typedef hw::Exchange<ROWS, EV> Ex;
    constexpr int SBYTES = NWAVES * G::KSTAGE;
    __shared__ __attribute__((aligned(16))) char q_lds[ROWS * G::QSTR];
    union Slot0 {
        char k[SBYTES];
        Ex ex;
    };
    __shared__ __attribute__((aligned(16))) Slot0 slot0;
    __shared__ __attribute__((aligned(16))) char slot1[SBYTES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int q = lane >> 4;
    char* const kslots[2] = {slot0.k + wv * G::KSTAGE, slot1 + wv * G::KSTAGE};

    PagedHeaderBits hb;
    paged_header_request(hb);
    // argument-independent setup while the header is in flight
    // K load i of a wave covers tile rows i*RPL .. i*RPL+RPL-1; this lane fetches a chunk of row i*RPL + lrow, and
    // which chunk follows from the bank swizzle, applied on the global side (the transfer writes LDS linearly)
    constexpr int RPL = 64 / G::CPR;
    const int lrow = lane / G::CPR, lslot = lane % G::CPR;
    auto k_chunk = [&](int i) -> unsigned {
        const int row = i * RPL + lrow;
        const int key = G::CPR >= 16 ? (row & 15) : ((row >> 1) & (G::CPR - 1));
        return (unsigned)((lslot ^ key) << 4);
    };
    WaveState<RB, G::NOC> st;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        st.m[rb] = st.top[rb] = NEG_BIG;
        st.l[rb] = 0.f;
#pragma unroll
        for (int c = 0; c < G::NOC; ++c) st.o[rb][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    st.fresh = true;
    const PagedDevHeader ph = paged_header_wait(hb);

    // logical workgroup id = ((kv head * nitems) + item) * nsplit + split; consecutive ids share an XCD
    int bid = blockIdx.x;
    if (ph.flags & PH_XCD_REMAP) bid = (bid & 7) * (ph.nwg >> 3) + (bid >> 3);
    const int hi = fast_div(bid, ph.magic_nsplit);
    const int hkv = fast_div(hi, ph.magic_nitems);
    const int GQ = ph.Hq / ph.Hkv;
    const int T = ph.LW * ph.LS;
    const int cap = ph.block_size * ph.max_blocks;
    const bool shared = (ph.flags & PH_SHARED) != 0;
    int item = hi - hkv * ph.nitems, split = bid - hi * ph.nsplit;
    int ns = ph.nsplit;                     // workgroups that share the sequence's tiles
    const int slot = item * ns + split;

    [[maybe_unused]] CacheView all;                        // the whole K cache (SMALL)
    if constexpr (SMALL) all = make_cache_view(ph, G::KROW);

    // what QueryRotation / map_row need, in the [LW, Hq, LS] layout, with the worker's row end as the row limit
    DevHeader a;
    a.q = ph.q;
    a.loc = ph.loc;
    a.cos = nullptr;
    a.sin = nullptr;
    a.rq = nullptr;
    a.part_o = ph.part_o;
    a.part_ml = ph.part_ml;
    a.len_dev = nullptr;
    a.F = ph.F; a.W = ph.LW; a.Hq = ph.Hq; a.Hkv = ph.Hkv; a.S = ph.LS;
    a.nrg = 1; a.wgs_per_head = ph.nsplit; a.nwg = ph.nwg;
    a.slot_stride = ph.nsplit; a.flags = KH_PREROTATED; a.sc = ph.sc;
    a.magic_gq = ph.magic_gq; a.magic_s = ph.magic_ls; a.magic_nrg = 0; a.magic_wg = 0;

    int w = 0, r0 = 0, rend = 0;            // sequence; first row (global numbering: token * GQ + head in group), end of its rows
    int NW = 0, gw = 0;                     // waves that share the tiles of this (kv head, row group); this one
    const HW_GLOBAL int* btw = nullptr;
    auto place = [&](int seq, int row_group, int qs, int qe) {
        w = seq;
        r0 = qs * GQ + row_group * ROWS;
        rend = qe * GQ;
        a.R = rend;
        NW = ns * NWAVES;
        gw = split * NWAVES + wv;
        btw = ph.block_table + (size_t)w * ph.max_blocks;
    };
    // block-table entry of the token this lane stands for in tile t
    auto bt_load = [&](int t) -> int {
        const int tok = min(t * TILE + (lane & 31), cap - 1);
        return btw[fast_div(tok, ph.magic_bs)];
    };
    // one batch of independent loads: queries, locations, fragment length, the table entries of two tiles
    QueryRotation<DT, E, ROWS, G::QSTR, true> qrot;
    int lm = 0, flen = 0, bt_a = 0, bt_b = 0;
    auto request = [&](int f) {
        qrot.load(a, f, hkv, r0, GQ, tid);
        lm = ph.loc[(size_t)f * T + fast_div(min(r0 + (tid & (ROWS - 1)), rend - 1), ph.magic_gq)];
        flen = ph.frag_len[ph.cu_q != nullptr ? f * ph.W + w : f];
        bt_a = bt_load(gw);
        bt_b = bt_load(gw + NW);
    };
    {
        const PagedItem it = paged_item<ROWS>(ph, item, lane, GQ);
        if (!it.found) return;              // the grid is sized for the worst case; uniform over the workgroup
        place(it.w, it.rg, it.qs, it.qe);
    }
    if (r0 >= rend) return;                 // uniform over the workgroup
    int loc0 = 0, len0 = 0, first_slot = 0;
    bool follow = false;                    // the reference of the exponentials follows the tiles: fewer workgroups than with equal shares
    if (shared) {
        loc0 = ph.loc[min(lane, ph.W - 1) * ph.LS];
        len0 = ph.frag_len[0];
    }
    request(0);
    if (shared) {
        // (what is requested holds for equal sequences: only where the share turns out another is it requested again)
        const PagedShare sh = paged_share(ph, item, split, lane, loc0, len0);
        if (!sh.found) return;              // uniform over the workgroup
        first_slot = sh.slot0;
        follow = sh.ns < ns;
        if (sh.w != item || sh.split != split || sh.ns != ns) {
            item = sh.w;
            split = sh.split;
            ns = sh.ns;
            place(item, 0, item * ph.LS, item * ph.LS + ph.LS);
            request(0);
        }
    }

    for (int f = 0; f < ph.F; ++f) {
        if (f > 0) request(f);

        // The bounds of the rows: lane l holds that of row l % ROWS.
        const int limv = (r0 + (lane & (ROWS - 1)) < rend) ? max(0, min(min(flen, cap), lm < cap ? lm + 1 : cap)) : 0x7fffffff;
        int lim[RB];
        int maxlim = 0, minlim = 0x7fffffff;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            lim[rb] = RB == 1 ? limv : __shfl(limv, rb * 16 + n, 64);
            const bool pad = r0 + rb * 16 + n >= rend;
            maxlim = max(maxlim, pad ? 0 : lim[rb]);
            minlim = min(minlim, lim[rb]);
        }
        maxlim = __builtin_amdgcn_readfirstlane(row_max16(maxlim));
        minlim = __builtin_amdgcn_readfirstlane(row_min16(minlim));

        // Issue the loads of tile t given its table entries: the same number of load instructions whether or not
        // the tile exists (a tile beyond the visible range re-reads one row that is visible, or, if nothing is
        // visible at all, some row inside the cache: a few hundred bytes that are never used).
        auto issue_tile = [&](TileRegs<DT, E, EV>& tr, char* kslot, int btv, int t) {
            const int tok_raw = t * TILE + (lane & 31);
            const int tok = min(tok_raw, cap - 1);
            const int bi = fast_div(tok, ph.magic_bs);
            const int blk = min(max(btv, 0), ph.num_blocks - 1);
            int rid = (blk * ph.Hkv + hkv) * ph.block_size + (tok - bi * ph.block_size);
            const int jstar = min(max(maxlim - 1 - t * TILE, 0), 31);
            const int rstar = __builtin_amdgcn_readlane(rid, jstar);
            rid = tok_raw < maxlim ? rid : rstar;
            asm volatile("" ::: "memory");   // the transfers keep their place between the reads of the slot (see load_tile)
#pragma unroll
            for (int i = 0; i < G::KL; ++i) {
                const int r = __shfl(rid, i * RPL + lrow, 64);
                if constexpr (SMALL) {
                    cache_transfer<AUX>(all, kslot + i * 1024, (unsigned)r * G::KROW + k_chunk(i));
                } else {
                    const HW_GLOBAL char* src = ph.kcache + (unsigned long long)(unsigned)r * G::KROW + k_chunk(i);
                    __builtin_amdgcn_global_load_lds(src, HW_LDS_PTR(kslot + i * 1024), 16, 0, AUX);
                }
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int idx = 0; idx < 8; ++idx) {
                const int r = __shfl(rid, slot_token(q, idx), 64);
                const HW_GLOBAL char* src = ph.vcache + (unsigned long long)(unsigned)r * G::VROW + n * (G::VLD * 4);
#pragma unroll
                for (int hh = 0; hh < G::NVL; ++hh) {
                    if constexpr (G::VLD == 4) {
                        const u32x4 x = AUX == 2 ? __builtin_nontemporal_load(reinterpret_cast<const HW_GLOBAL u32x4*>(src + hh * 256))
                                                        : *reinterpret_cast<const HW_GLOBAL u32x4*>(src + hh * 256);
                        tr.v[idx][hh * 4 + 0] = x.x;
                        tr.v[idx][hh * 4 + 1] = x.y;
                        tr.v[idx][hh * 4 + 2] = x.z;
                        tr.v[idx][hh * 4 + 3] = x.w;
                    } else {
                        const u32x2 x = AUX == 2 ? __builtin_nontemporal_load(reinterpret_cast<const HW_GLOBAL u32x2*>(src))
                                                        : *reinterpret_cast<const HW_GLOBAL u32x2*>(src);
                        tr.v[idx][0] = x.x;
                        tr.v[idx][1] = x.y;
                    }
                }
            }
        };

        // The first tile is requested as soon as the bounds are known, and the queries go through LDS while it is on its way (barriers
        // for LDS only: __syncthreads() would wait for it): eight sequences of 1200 tokens 17.3 -> 17.0 us with the append.
        TileRegs<DT, E, EV> tr[2];
        issue_tile(tr[0], kslots[0], bt_a, gw);
        lds_barrier();   // the previous fragment's readers are done with q_lds
        qrot.finish(a, q_lds, f, hkv, r0, GQ, false, tid);
        lds_barrier();
        constexpr bool QREG = MINW == 1;
        u32x4 qreg[QREG ? RB * G::KJ : 1];
        if constexpr (QREG) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int j = 0; j < G::KJ; ++j)
                    qreg[rb * G::KJ + j] = *reinterpret_cast<const u32x4*>(q_lds + (rb * 16 + n) * G::QSTR + (4 * j + q) * 16);
        }

        if (maxlim > 0) {   // uniform
            // Two tiles in flight per wave.  Per step: request the table entries two tiles ahead, then the K/V of
            // the next tile (its entries were requested one step earlier, ahead of the previous K/V request, so
            // they have arrived by the time the current tile's data has), then compute the current tile.
            // Two loops with one instantiation of the tile arithmetic each (see attention_kernel): pairs of tiles every
            // row of the wave sees completely, then the rest.
            int t = gw;
            if constexpr (G::SZ != 4)               // (the fp32 kernels keep one loop with both instantiations, see attention_kernel)
            for (; (t + NW + 1) * TILE <= minlim; t += 2 * NW) {
                {
                    const int bt_n = bt_load(t + 2 * NW);
                    issue_tile(tr[1], kslots[1], bt_b, t + NW);
                    if constexpr (STATED) wait_k_landed<G, 1>();   // (see wait_k_landed: the table load in between only adds to what is behind)
                    compute_tile<DT, E, EV, RB, false, QREG, false, false, FOLLOW>(tr[0], q_lds, qreg, lim, st, t * TILE, n, q, ph.sc, kslots[0], nullptr, nullptr, follow);
                    bt_a = bt_n;
                }
                {
                    const int bt_n = bt_load(t + 3 * NW);
                    issue_tile(tr[0], kslots[0], bt_a, t + 2 * NW);
                    if constexpr (STATED) wait_k_landed<G, 1>();
                    compute_tile<DT, E, EV, RB, false, QREG, false, false, FOLLOW>(tr[1], q_lds, qreg, lim, st, (t + NW) * TILE, n, q, ph.sc, kslots[1], nullptr, nullptr, follow);
                    bt_b = bt_n;
                }
            }
            for (; t * TILE < maxlim; t += 2 * NW) {
                {
                    const int bt_n = bt_load(t + 2 * NW);
                    issue_tile(tr[1], kslots[1], bt_b, t + NW);
                    if constexpr (STATED) wait_k_landed<G, 1>();
                    const int t0 = t * TILE;
                    if (G::SZ == 4 && t0 + TILE <= minlim) compute_tile<DT, E, EV, RB, false, QREG, false, false, FOLLOW>(tr[0], q_lds, qreg, lim, st, t0, n, q, ph.sc, kslots[0], nullptr, nullptr, follow);
                    else compute_tile<DT, E, EV, RB, true, QREG, false, false, FOLLOW>(tr[0], q_lds, qreg, lim, st, t0, n, q, ph.sc, kslots[0], nullptr, nullptr, follow);
                    bt_a = bt_n;
                }
                {
                    const int bt_n = bt_load(t + 3 * NW);
                    issue_tile(tr[0], kslots[0], bt_a, t + 2 * NW);
                    if constexpr (STATED) wait_k_landed<G, 1>();
                    const int t0 = (t + NW) * TILE;
                    if (G::SZ == 4 && t0 + TILE <= minlim) compute_tile<DT, E, EV, RB, false, QREG, false, false, FOLLOW>(tr[1], q_lds, qreg, lim, st, t0, n, q, ph.sc, kslots[1], nullptr, nullptr, follow);
                    else if (t0 < maxlim) compute_tile<DT, E, EV, RB, true, QREG, false, false, FOLLOW>(tr[1], q_lds, qreg, lim, st, t0, n, q, ph.sc, kslots[1], nullptr, nullptr, follow);
                    bt_b = bt_n;
                }
            }
        }
    }

    store_partials<DT, EV, RB, true>(st, slot0.ex, wv, n, q, tid, ph.part_o, ph.part_ml,
                               shared ? (size_t)(hkv * ph.nitems * ph.nsplit + slot) * (ph.LS * GQ) : (size_t)(hkv * ph.nsplit + split) * ph.R + r0,
                               min(ROWS, rend - r0));
    // where the merge finds the rows' partial sums
    if (shared && split == 0 && tid < rend - r0) {
        HW_GLOBAL int* row_tab = reinterpret_cast<HW_GLOBAL int*>(ph.part_ml + (size_t)ph.Hkv * ph.nsplit * ph.R * 2) + ((size_t)hkv * ph.R + r0) * 2;
        row_tab[2 * tid] = first_slot | (ns << 16);
        row_tab[2 * tid + 1] = tid;
    }
}

// Scatter of new K/V rows into the paged caches, one 16-byte chunk (or, for odd sizes, one element) per thread.
// A position whose block index lies outside the table, or whose table entry lies outside the cache, is skipped.
// IDX: 32 bits, unless there are more pieces than that (a division in 64 bits is a hundred instructions, and five of them stood in front
// of three dependent accesses: one token of eight sequences, 8 heads, D = 128, append and attention 18.0 -> 17.8 us, see paged_share).
template <int VEC, class IDX>   // bytes per thread
__global__ __launch_bounds__(256) void copy_to_blocks_kernel(const CopyBlocksArgs a, int sz) {
    const int ck = a.E * sz / VEC, cv = a.Ev * sz / VEC;
    const IDX rows = (IDX)a.B * a.Hkv * a.S_new;
    const IDX total = rows * (unsigned)(ck + cv);
    for (IDX idx = (IDX)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (IDX)gridDim.x * blockDim.x) {
        const IDX row = idx / (unsigned)(ck + cv);
        const int c = (int)(idx - row * (unsigned)(ck + cv));
        const IDX bh = row / (unsigned)a.S_new;
        const int t = (int)(row - bh * (unsigned)a.S_new);
        const int b = (int)(bh / (unsigned)a.Hkv);
        const int h = (int)(bh - (IDX)b * (unsigned)a.Hkv);
        const int length = a.seq_lengths[b];
        if (length < 0 && length + t < 0) continue;
        const unsigned pos = (unsigned)length + (unsigned)t;               // (two numbers below 2^31)
        const unsigned bi = pos / (unsigned)a.block_size;
        if (bi >= (unsigned)a.max_blocks) continue;
        const int blk = a.block_table[(size_t)b * a.max_blocks + bi];
        if (blk < 0 || blk >= a.num_blocks) continue;
        const int off = (int)(pos - bi * (unsigned)a.block_size);
        const size_t dst_row = ((size_t)blk * a.Hkv + h) * a.block_size + off;
        const bool is_k = c < ck;
        const char* src = is_k ? reinterpret_cast<const char*>(a.key_states) + ((long long)b * a.ks_b + (long long)h * a.ks_h + (long long)t * a.ks_s) * sz + (size_t)c * VEC
                               : reinterpret_cast<const char*>(a.value_states) + ((long long)b * a.vs_b + (long long)h * a.vs_h + (long long)t * a.vs_s) * sz + (size_t)(c - ck) * VEC;
        char* dst = is_k ? reinterpret_cast<char*>(a.kcache) + dst_row * a.E * sz + (size_t)c * VEC
                         : reinterpret_cast<char*>(a.vcache) + dst_row * a.Ev * sz + (size_t)(c - ck) * VEC;
        if constexpr (VEC == 16) *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(src);
        else if constexpr (VEC == 4) *reinterpret_cast<u32*>(dst) = *reinterpret_cast<const u32*>(src);
        else *reinterpret_cast<unsigned short*>(dst) = *reinterpret_cast<const unsigned short*>(src);
    }
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
template <class DT, int E, int EV, bool SMALL>
static hipError_t launch_paged_rb(const PagedHeader& ph, int rb, hipStream_t stream) {
    constexpr bool half = Elem<DT>::size == 2;
    // fp32 operands with two row blocks do not fit the register file; the planner never asks for them
    if constexpr (half) {
        if (rb == 2) {
            hipLaunchKernelGGL((paged_attention_kernel<DT, E, EV, 2, 1, SMALL>), dim3(ph.nwg), dim3(NTHREADS), 0, stream, ph);
            return hipGetLastError();
        }
    }
    if (rb != 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL((paged_attention_kernel<DT, E, EV, 1, half ? HW_PAGED_MINW : 1, SMALL>), dim3(ph.nwg), dim3(NTHREADS), 0, stream, ph);
    return hipGetLastError();
}

template <class DT, bool SMALL>
static hipError_t launch_paged_dt(const PagedHeader& ph, int E, int rb, hipStream_t stream) {
    if (E == 256) {     // one 16-row block per workgroup, one wave per SIMD; 16-bit types (two fp32 K tiles per wave exceed the LDS)
        if constexpr (Elem<DT>::size == 2) {
            if (rb != 1) return hipErrorInvalidValue;
            if (ph.flags & PH_KEEP) hipLaunchKernelGGL((paged_attention_kernel<DT, 256, 256, 1, 1, SMALL, true>), dim3(ph.nwg), dim3(NTHREADS), 0, stream, ph);
            else hipLaunchKernelGGL((paged_attention_kernel<DT, 256, 256, 1, 1, SMALL>), dim3(ph.nwg), dim3(NTHREADS), 0, stream, ph);
            return hipGetLastError();
        }
        return hipErrorInvalidValue;
    }
    if (E == 128) return launch_paged_rb<DT, 128, 128, SMALL>(ph, rb, stream);
    if (E != 64) return hipErrorInvalidValue;
    return launch_paged_rb<DT, 64, 64, SMALL>(ph, rb, stream);
}

template <bool SMALL>
static hipError_t launch_paged_small(const PagedHeader& ph, int dtype, int E, int rb, hipStream_t stream) {
    switch (dtype) {
        case 0: return launch_paged_dt<F32, SMALL>(ph, E, rb, stream);
        case 1: return launch_paged_dt<F16, SMALL>(ph, E, rb, stream);
        default: return launch_paged_dt<BF16, SMALL>(ph, E, rb, stream);
    }
}

hipError_t launch_paged_attention(const PagedHeader& ph, int dtype, int E, int rb, hipStream_t stream) {
    return ph.flags & PH_SMALL ? launch_paged_small<true>(ph, dtype, E, rb, stream) : launch_paged_small<false>(ph, dtype, E, rb, stream);
}

hipError_t launch_copy_to_blocks(const CopyBlocksArgs& ca, int dtype, hipStream_t stream) {
    const int sz = dtype == 0 ? 4 : 2;
    const bool vec16 = (ca.E * sz) % 16 == 0 && (ca.Ev * sz) % 16 == 0 && (ca.ks_b * sz) % 16 == 0 && (ca.ks_h * sz) % 16 == 0 &&
                       (ca.ks_s * sz) % 16 == 0 && (ca.vs_b * sz) % 16 == 0 && (ca.vs_h * sz) % 16 == 0 && (ca.vs_s * sz) % 16 == 0 &&
                       ((reinterpret_cast<uintptr_t>(ca.key_states) | reinterpret_cast<uintptr_t>(ca.value_states) |
                         reinterpret_cast<uintptr_t>(ca.kcache) | reinterpret_cast<uintptr_t>(ca.vcache)) & 15u) == 0;
    const int vec = vec16 ? 16 : sz;
    const size_t total = (size_t)ca.B * ca.Hkv * ca.S_new * (size_t)((ca.E + ca.Ev) * sz / vec);
    if (total == 0) return hipSuccess;
    size_t blocks = (total + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    auto go = [&](auto vec_tag) {
        constexpr int VEC = decltype(vec_tag)::value;
        if (total < (1ull << 31)) hipLaunchKernelGGL((copy_to_blocks_kernel<VEC, unsigned>), dim3((unsigned)blocks), dim3(256), 0, stream, ca, sz);
        else hipLaunchKernelGGL((copy_to_blocks_kernel<VEC, unsigned long long>), dim3((unsigned)blocks), dim3(256), 0, stream, ca, sz);
    };
    if (vec == 16) go(std::integral_constant<int, 16>{});
    else if (vec == 4) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 2>{});
    return hipGetLastError();
}

}  // namespace hw
