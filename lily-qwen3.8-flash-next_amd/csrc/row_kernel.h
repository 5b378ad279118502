// row_kernel.h - the row kernel: one launch serves a batch of logits rows.  Row r is scanned
// by `slices` workgroups of 256 threads (grid = slices x rows).  Each workgroup finds the exact
// top-k of its slice; with several slices the last workgroup to arrive (an atomic ticket,
// nobody waits) merges them.  That workgroup then runs the tail.
#pragma once

#include "device_common.h"
#include "select_bitmap.h"
#include "select_exhaustive.h"
#include "select_lowering.h"
#include "select_sparse.h"
#include "select_stream.h"
#include "tail.h"

namespace lily {

// ------------------------------------------------------------------ argmax

// First maximum under float comparison (NaN never wins, -0 == +0), lowest id on
// ties: elementwise.metal:145-150.  Result: the thread's best (value, id) of its share of the
// slice as a composite; id bits all zero when no element qualified.
template <int DT>
__device__ __forceinline__ uint64_t thread_argmax(const void* logits, const Geo<DT>& g) {
    constexpr int E = Geo<DT>::E;
    const uint32_t tid = threadIdx.x;
    float bv = NEG_INF;
    uint32_t bi = 0xffffffffu;
    for (uint32_t c0 = g.cb; c0 < g.ce; c0 += NT * UNROLL) {
        // Unconditional loads (chunks past the slice's end read its last chunk; `inside`
        // below discards them): a load that may be skipped is waited for as the last one issued.
        u32x4 raw[UNROLL];
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t c = min(c0 + u * NT + tid, g.ce - 1u);
            raw[u] = gload(reinterpret_cast<const u32x4*>(g.base + (size_t)c * 16));
        }
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t c = c0 + u * NT + tid;
            float v[E];
            unpack<DT>(raw[u], v);
            for (int j = 0; j < E; ++j) {
                const uint32_t id = g.id_of(c, j);
                const bool inside = c >= g.main_lo && c < g.main_hi;
                if (inside && (v[j] > bv || (v[j] == bv && id < bi))) {   // (-inf counts: == on a first one)
                    bv = v[j];
                    bi = id;
                }
            }
        }
    }
    for (int side = 0; side < 2; ++side) {
        const uint32_t lo = side == 0 ? g.id_lo : g.edge_hi_begin;
        const uint32_t hi = side == 0 ? g.edge_lo_end : g.id_hi;
        for (uint32_t id = lo + tid; id < hi; id += NT) {
            const float x = load_logit<DT>(logits, id);
            if (x > bv || (x == bv && id < bi)) {
                bv = x;
                bi = id;
            }
        }
    }
    return ((uint64_t)lilym_order_key(bv + 0.0f) << 32) | (uint32_t)(~bi);
}

// The workgroup's.
template <int DT>
__device__ __forceinline__ uint64_t slice_argmax(const RowArgs& a, const Geo<DT>& g, Shared& sh) {
    uint64_t best = wave_max_u64(thread_argmax<DT>(a.logits, g));
    if ((threadIdx.x & 63u) == 0) {
        sh.red_u[threadIdx.x >> 6] = best;
    }
    __syncthreads();
    best = sh.red_u[0];
    for (int i = 1; i < NWAVE; ++i) {
        best = sh.red_u[i] > best ? sh.red_u[i] : best;
    }
    __syncthreads();
    return best;
}

// ------------------------------------------------------------------ the row kernel

// The row's arguments are the same for every thread: read through the constant address
// space they arrive by scalar loads and stay in scalar registers.
__device__ __forceinline__ void load_row_args(RowArgs& a, const LILY_CONST RowArgs* src) {
    static_assert(sizeof(RowArgs) % 16 == 0, "RowArgs is copied in 16-byte pieces");
    const LILY_CONST u32x4* from = (const LILY_CONST u32x4*)src;
    u32x4* to = reinterpret_cast<u32x4*>(&a);
    for (unsigned i = 0; i < sizeof(RowArgs) / 16; ++i) {
        to[i] = from[i];
    }
}

// CHAIN: the kernel of launches whose rows draw in order (compiled apart from the others: what it
// adds behind the selects would cost every other launch registers).
// A workgroup barrier that orders LDS accesses only (outstanding global stores and atomics are
// not waited for).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The row and the step of a draw that leaves the choice to the device (see RowArgs::sel_row).
__device__ __forceinline__ void apply_selection(RowArgs& a) {
    if (a.sel_row != nullptr) {
        const uint32_t r = min(*(const LILY_CONST uint32_t*)a.sel_row, a.sel_rows - 1u);
        a.logits = static_cast<const char*>(a.logits) + (size_t)r * a.sel_stride;
    }
    if (a.sel_step != nullptr) {
        a.step += *(const LILY_CONST uint32_t*)a.sel_step;
    }
}

// The row's arguments once more (scalar loads, served by the scalar cache): kept in registers across
// the scan, the fields that only the merge, the tail or a second attempt at the row uses crowd the
// scan's own values out of the scalar registers.
__device__ __forceinline__ void read_again(RowArgs& a, const LILY_CONST RowArgs* src) {
    asm volatile("" : "+s"(src));
    load_row_args(a, src);
    apply_selection(a);
}

// The launch's settings once more, for the same reason.
__device__ __forceinline__ void read_again(LaunchCfg& cfg, const LILY_CONST LaunchCfg* src) {
    static_assert(sizeof(LaunchCfg) % 8 == 0, "LaunchCfg is copied in 8-byte pieces");
    asm volatile("" : "+s"(src));
    const LILY_CONST uint64_t* from = (const LILY_CONST uint64_t*)src;
    uint64_t* to = reinterpret_cast<uint64_t*>(&cfg);
    for (unsigned i = 0; i < sizeof(LaunchCfg) / 8; ++i) {
        to[i] = from[i];
    }
}

// The control block behind an acceptance of `acc` proposals (spec.metal:14-38).
__device__ __forceinline__ void write_accepted(const LaunchCfg& cfg, uint32_t acc) {
    uint32_t* ctrl = cfg.accept_ctrl;
    ctrl[0] = acc;
    ctrl[LILY_CTRL_STRIDE] = acc + 1;
    for (uint32_t i = 0; i < cfg.accept_chain; ++i) {
        const uint32_t p = cfg.accept_pos0 + acc + 1 + i;
        ctrl[(2 + 3 * i) * LILY_CTRL_STRIDE] = p;
        ctrl[(3 + 3 * i) * LILY_CTRL_STRIDE] = p / cfg.accept_ratio;
        ctrl[(4 + 3 * i) * LILY_CTRL_STRIDE] = ((p + 1) % cfg.accept_ratio == 0) ? 1u : 0u;
    }
}

// One thread of the workgroup that finished a row of a verify pass (it stored the row's draw; out_of(j):
// where row j's is): behind the last of them, the acceptance.
template <class F>
__device__ __forceinline__ void accept_behind_last_row(const LaunchCfg& cfg, F&& out_of) {
    const uint32_t m = gridDim.y;
    // (the release covers the draw, the acquire the other rows')
    if (__hip_atomic_fetch_add(cfg.chain_ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) != m - 1u) {
        return;
    }
    store_through(cfg.chain_ticket, 0u);
    uint32_t drew[LILY_MAX_VERIFY_ROWS], given[LILY_MAX_VERIFY_ROWS];
#pragma unroll
    for (uint32_t j = 0; j < LILY_MAX_VERIFY_ROWS; ++j) {
        drew[j] = load_through(out_of(min(j, m - 1u)));
        given[j] = gload(cfg.accept_ids + min(j, m - 1u));
    }
    uint32_t acc = 0;
    bool same = true;
#pragma unroll
    for (uint32_t j = 0; j + 1u < LILY_MAX_VERIFY_ROWS; ++j) {
        same = same && j + 1u < m && drew[j] == given[j + 1u];
        acc += same ? 1u : 0u;
    }
    write_accepted(cfg, acc);
}

// Rows of select_lowering(): under penalties that can only lower a value, nothing else in play.
__device__ __forceinline__ bool lowering_row(const RowArgs& a) {
    return (a.flags & F_PEN) != 0u && a.repetition >= 1.0f && a.presence >= 0.0f && a.frequency >= 0.0f &&
           a.allow == nullptr && a.n_bias == 0u;
}

// What a row of few candidates (k <= 64) that several workgroups scanned has left to do once each of
// them knows its own best: the workgroup's first wave does it all, without a barrier - the others have
// nothing left to do and are gone.  It stores its candidates, takes the row's ticket and, if it is the
// last, gathers every slice's, keeps the row's best (a candidate per lane, in order) and draws.
// (With the workgroup's four waves meeting at eight barriers from here to the draw: 7.6 us of the 13.2
// that one sampled row of 151 936 f32 logits takes in 38 slices; now 6 of 11.9.)
//
// Entries the wave gathers at most, 32 a lane.  Up to there it is the faster way for every k, dtype and kind of
// row: 4 to 100 rows of 151 936 in 5 to 38 slices, k 3 to 60: 0.77 to 1.01 of the workgroup's merge (24 f32
// rows, k = 50: 19.8 and 21.3 us), k = 64 0.76 to 0.97 (22.1 and 26.4); bf16 rows near k = 62 up to 1.04, where
// equal values at the k-th take a second sort.
constexpr uint32_t WAVE_MERGE_SLOTS = 2048;

__device__ __forceinline__ bool descending(uint64_t c) {   // lane by lane, equal only where both are 0
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)(uint32_t)c, 0x138, 0xf, 0xf, false);   // wave_shr:1
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)(uint32_t)(c >> 32), 0x138, 0xf, 0xf, false);
    return __ballot((((uint64_t)hi << 32) | lo) < c) == 0ull;
}

// The row's best entries, a lane each, in order, from the lists its slices stored at `base` (by one
// wave, all of it at work; at least the k best are among them).
// `none`: there are none.  (Asked here, branch by branch: with the call skipped instead, the kernel that holds every select compiles to
// 3 % longer launches, 64 bf16 rows of 151 936 under open masks 61.8 -> 63.8 us, 200 rows 111.4 -> 114.8.)
__device__ __forceinline__ uint64_t merge_slices_by_wave(const LaunchCfg& cfg, size_t base, uint32_t k, bool none = false) {
    const uint32_t lane = threadIdx.x & 63u, S = cfg.slices;
    uint64_t best = 0ull;   // the row's best, a lane each, in order
    if (!none && S <= WAVE_MERGE_LISTS) {
        // Few lists, each in order as a rule: one after the other into the best so far.
        uint64_t list[WAVE_MERGE_LISTS];
#pragma unroll
        for (uint32_t q = 0; q < WAVE_MERGE_LISTS; ++q) {
            const uint32_t from = min(q, S - 1u), at = min(lane, cfg.ws_k - 1u);
            list[q] = handed_load(cfg.ws_cand, (base + from) * cfg.ws_k + at);
        }
#pragma unroll
        for (uint32_t q = 0; q < WAVE_MERGE_LISTS; ++q) {
            if (q < S) {
                uint64_t c = lane < cfg.ws_k ? list[q] : 0ull;
                if (!descending(c)) {
                    c = wave_sort_desc(c);
                }
                best = q == 0u ? c : wave_merge_desc(best, c);
            }
        }
    } else if (!none && S * cfg.ws_k <= 64u) {
        // (no more entries than lanes: one sort)
        const uint64_t c = handed_load(cfg.ws_cand, base * cfg.ws_k + min(lane, S * cfg.ws_k - 1u));
        best = wave_sort_desc(lane < S * cfg.ws_k ? c : 0ull);
    } else if (!none) {
        constexpr int PER = WAVE_MERGE_SLOTS / 64, GROUP = 8;
        const uint32_t slots = S * cfg.ws_k;
        uint64_t mine[PER];
#pragma unroll
        for (int q0 = 0; q0 < PER; q0 += GROUP) {
            if ((uint32_t)q0 * 64u < slots) {
#pragma unroll
                for (int q = q0; q < q0 + GROUP; ++q) {
                    mine[q] = handed_load(cfg.ws_cand, base * cfg.ws_k + min(lane + (uint32_t)q * 64u, slots - 1u));
                }
            }
        }
        uint32_t lane_best = 0u, lane_next = 0u;   // the keys of a lane's two best
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            mine[q] = lane + (uint32_t)q * 64u < slots ? mine[q] : 0ull;
            const uint32_t key = (uint32_t)(mine[q] >> 32);
            lane_next = max(lane_next, min(lane_best, key));
            lane_best = max(lane_best, key);
        }
        // The k-th largest of the lanes' two best bounds the k-th entry: at least k entries reach it (more
        // than there are with fewer than k: all of them); what does not is dropped, the rest is listed, and
        // the list's entries are taken in 64 at a time.  Sixteen bits of the key let some three f32 entries
        // through that share the k-th's: above k = 50 a second sort in some row of a launch, 1.0 us, which
        // four more bits (0.2 us) save.
        uint32_t bound = 0u;
        auto settle = [&](int bit) {
            const uint32_t at = bound | (1u << bit);
            const uint32_t reach = (uint32_t)__popcll(__ballot(lane_best >= at)) + (uint32_t)__popcll(__ballot(lane_next >= at));
            bound = reach >= k ? at : bound;
        };
#pragma unroll
        for (int bit = 31; bit >= 16; --bit) {
            settle(bit);
        }
        if (k > 50u) {
#pragma unroll
            for (int bit = 15; bit >= 12; --bit) {
                settle(bit);
            }
        }
        uint64_t* cand = dyn_lds;
        uint32_t kept = 0;
#pragma unroll
        for (int q0 = 0; q0 < PER; q0 += GROUP) {
            if ((uint32_t)q0 * 64u < slots) {
#pragma unroll
                for (int q = q0; q < q0 + GROUP; ++q) {
                    const bool in = mine[q] != 0ull && (uint32_t)(mine[q] >> 32) >= bound;
                    const uint64_t mask = __ballot(in);
                    if (mask != 0ull) {
                        const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                            (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                        if (in) {
                            cand[kept + rank] = mine[q];
                        }
                        kept += (uint32_t)__popcll(mask);
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // (LDS of this wave: in order already)
        __builtin_amdgcn_wave_barrier();
        for (uint32_t i = 0; i < kept; i += 64u) {
            const uint64_t c = wave_sort_desc(i + lane < kept ? cand[i + lane] : 0ull);
            best = i == 0u ? c : wave_merge_desc(best, c);
        }
    }
    return best;
}

template <int DT, bool LSE, bool SPEC>
__device__ __forceinline__ bool finish_by_wave(const RowArgs& t, const LaunchCfg& cfg, uint32_t row, uint32_t s, uint32_t n,
                                               const uint64_t* found, uint32_t step, bool want_lse, Shared& sh) {
    const uint32_t lane = threadIdx.x, S = cfg.slices, vocab = cfg.vocab;
    const bool forced = (t.flags & F_FORCED) != 0u;
    const size_t slot = (size_t)row * S + s;
    // Every place is written (0 = no candidate), so the merge needs no counts.  Its lanes take every 64th
    // place, and its bound wants the row's best spread evenly over them: the slices' best begin 64 / S lanes
    // apart, each list turned within its places (LaunchCfg::turn_step).  (Unturned, lists of 64 put the same
    // rank of every slice into a lane, and the bound let 700 of 2 048 entries through; so did, less so,
    // every length near 64 or with a large factor in common with it.  Turned, those that pass are one
    // sort, rarely two.  Worked out here from S it took every row 0.1 us.)
    uint32_t turn = (s * cfg.turn_step >> 16) & 63u;
    turn = turn >= cfg.ws_k ? turn - cfg.ws_k : turn;
    for (uint32_t i = lane; !forced && i < cfg.ws_k; i += 64u) {
        const uint32_t rank = i < turn ? i + cfg.ws_k - turn : i - turn;
        handed_store(cfg.ws_cand, slot * cfg.ws_k + i, rank < n ? found[rank] : (uint64_t)0);
    }
    if (LSE && lane == 0u) {
        handed_store(cfg.ws_lse, 2 * slot, want_lse ? sh.lse_mc : 0.0);
        handed_store(cfg.ws_lse, 2 * slot + 1, want_lse ? sh.lse_s : 0.0);
    }
    const bool last = wave_last_to_arrive(&cfg.ws_ticket[row], S, cfg.relaxed_handover != 0u);
    phase(cfg, 5);
    if (!last) {
        return false;
    }
    uint32_t spec_d = 0, spec_qn = 0;
    if (SPEC && t.mode == MODE_SPEC) {
        spec_d = *t.draft;
        spec_qn = *t.q_n;
    }
    const size_t base = (size_t)row * S;
    double mt = -__builtin_huge_val(), st = 0.0;
    if (LSE && want_lse && lane < S) {
        mt = handed_load(cfg.ws_lse, 2 * (base + lane));
        st = handed_load(cfg.ws_lse, 2 * (base + lane) + 1);
    }
    const uint64_t gathered = merge_slices_by_wave(cfg, base, t.k, forced);   // the row's best, a lane each, in order
    if (LSE && want_lse) {
        const bool some = st > 0.0;
        const double m = wave_max_d(some ? mt : -__builtin_huge_val());
        const double sum = wave_sum_d(some ? st * exp2(mt - m) : 0.0);
        if (lane == 0u) {
            sh.lse_mc = m;
            sh.lse_s = sum;
        }
    }
    phase(cfg, 6);
    if (forced) {
        if (lane == 0u) {
            finish_token<DT>(t, sh, t.forced, vocab);
        }
        return true;
    }
    const uint64_t best = lane < t.k ? gathered : 0ull;
    const uint32_t have = (uint32_t)__popcll(__ballot(best != 0ull));
    if (have == 0u) {
        if (lane == 0u) {
            finish_empty(t, vocab, sh, cfg);
        }
        return true;
    }
    tail_wave<DT, SPEC>(t, vocab, step, best, have, sh, cfg, spec_d, spec_qn);
    return true;
}

// True in the workgroup that finishes the row (the last of its slices to arrive).
template <int DT, int KIND, bool LSE, bool CHAIN = false, bool SPEC = false>
__device__ __forceinline__ bool row_body(const LILY_CONST RowArgs* src, const LaunchCfg& cfg, const LILY_CONST LaunchCfg* cfg_src,
                                         Shared& sh) {
    if (cfg.served != nullptr && *(const LILY_CONST uint32_t*)(cfg.served + blockIdx.y) != 0u) {
        return false;
    }
    RowArgs a;
    load_row_args(a, src);
    apply_selection(a);
    // KIND: 0 = rows without masks, penalties or bias lists, 1 = rows with any of them (the
    // bitmap select is compiled for them), 2 = streaming rows only (no bitmap select at all).
    constexpr bool EXCL = KIND == 1;
    const uint32_t tid = threadIdx.x;
    const uint32_t s = blockIdx.x, row = blockIdx.y, S = cfg.slices;
    const uint32_t vocab = cfg.vocab;
    const uint32_t step = a.step + cfg.step_delta;
    const bool want_lse = LSE && a.out_logprob != nullptr;
    uint64_t* cand = dyn_lds;
    uint64_t* found = cand;  // where the select left the slice's candidates
    uint32_t* excl = reinterpret_cast<uint32_t*>(dyn_lds + cfg.cand_cap);

    if ((a.flags & F_FORCED) && !want_lse) {
        if (s == 0 && tid == 0) {
            emit(a, a.forced, vocab);
        }
        return s == 0;
    }

    Geo<DT> g;
    g.init(a.logits, vocab, s, S);
    phase(cfg, 0);

    const bool argmax = a.mode == MODE_ARGMAX;
    uint64_t best = 0;
    bool sorted = false;
    if (argmax) {
        best = slice_argmax<DT>(a, g, sh);
    } else {
        // A forced row with a log-probability needs the row sum only: it takes the same
        // selects (their sums are the fast ones) and its candidates are dropped below.
        bool done = false;
        uint32_t took = 2;
        if (cfg.path == 0u && (a.flags & F_STREAM)) {
            if (lowering_row(a)) {
                bool again = false;
                done = select_lowering<DT, LSE, false>(a, g, a.k, sh, cfg, again, sorted, found);
                if (!done) {
                    __syncthreads();
                }
                if (again) {
                    RowArgs f = a;
                    Geo<DT> fg = g;
                    if constexpr (LSE) {
                        read_again(f, src);
                        fg.init(f.logits, vocab, s, S);
                    }
                    done = select_lowering<DT, LSE, true>(f, fg, f.k, sh, cfg, again, sorted, found);
                    if (!done) {
                        __syncthreads();
                    }
                }
            } else {
                done = select_stream<DT, LSE, KIND != 2>(a, g, a.k, sh, cfg, sorted, found);
                if (!done) {
                    __syncthreads();
                }
            }
            took = done ? 0u : took;
        }
        // The other selects.  Launches with row sums read the arguments afresh for them: kept across
        // the streaming scan they made it spill (200 rows in three slices 46.7 -> 45.7 us).  Launches
        // without hold fewer values and keep them, and each select below asks by itself whether it is
        // still wanted: asked once around them, the merge's loads, and a wait for them, are drawn ahead of
        // every row (one sampled row 11.7 -> 11.9 us, a greedy one beside it 11.6 -> 11.7, four rows
        // under penalties 14.8 -> 14.9).
        if (!LSE || !done) {
            RowArgs f = a;
            Geo<DT> fg = g;
            if constexpr (LSE) {
                read_again(f, src);
                fg.init(f.logits, vocab, s, S);
            }
            if (KIND == 1 && !done && cfg.path == 0u && f.allow != nullptr) {
                done = select_sparse<DT, LSE>(f, fg, f.k, cand, min(cfg.dyn_slots, MERGE_CAP), sh, sorted, cfg);
                took = done ? 1u : took;
            }
            if (KIND != 2 && !done && cfg.path != 1u && cfg.bitmap_layout != 0u) {
                const bool special = f.allow != nullptr || (f.flags & F_PEN) || f.n_bias != 0;
                if (EXCL || !special) {
                    // A single pass whose running bound let too many candidates in is repeated
                    // as two passes (bound first, then collect) before the exhaustive select.
#pragma nounroll
                    for (int attempt = 0; attempt < 2 && !done; ++attempt) {
                        const bool two_pass = f.k > 64u || cfg.path == 2u || attempt == 1;
                        if (attempt == 1) {
                            __syncthreads();
                        }
                        done = select_fast<DT, EXCL, LSE>(f, fg, f.k, two_pass, cand, cfg.cand_cap, excl, sh,
                                                          cfg, sorted);
                        if (f.k > 64u || cfg.path == 2u) {
                            break;  // it was two passes already
                        }
                    }
                    took = done ? 1u : took;
                }
            }
            if (!LSE && cfg.path_stats != nullptr && tid == 0) {
                atomicAdd(&cfg.path_stats[took], 1u);
            }
            if (!done) {
                __syncthreads();
                sorted = false;
                // (in the kernels that hold the others read afresh for this select alone: of arguments that
                // those held as well, each element's evaluation reloaded up to 97 spilled lanes; 4 rows of
                // 151 936 bf16 that come here, no top_k, 692 -> 531 us.  The streaming rows' kernels spill
                // none of them: one sampled row 11.83 us without, 11.93 with)
                RowArgs e = f;
                if constexpr (KIND != 2) {
                    read_again(e, src);
                }
                select_exhaustive<DT>(e, fg.id_lo, fg.id_hi, e.k, want_lse, cand, cfg.cand_cap, sh);
            }
        }
        if (LSE && cfg.path_stats != nullptr && tid == 0) {
            atomicAdd(&cfg.path_stats[took], 1u);
        }
    }

    RowArgs t;
    read_again(t, src);
    // The settings too, in the kernels that hold every select: what only the merge and the tail read
    // was kept across the scan there and put the scan's own values into its loops as reloads (blocks
    // of dense masks with row sums: 943 lane reads in a loop that has 108 now; 200 rows
    // of them, k = 20, under penalties 140 -> 126 us).  Streaming rows' kernels have room for them.
    LaunchCfg late = cfg;
    if constexpr (KIND != 2 && !CHAIN) {
        read_again(late, cfg_src);
    }
    const bool forced = (t.flags & F_FORCED) != 0;
    // (the sparse select of a row in one slice leaves what it evaluated, which may be more than cand_cap)
    const uint32_t n_cap = KIND == 1 ? max(late.cand_cap, min(late.dyn_slots, MERGE_CAP)) : late.cand_cap;
    uint32_t n = (argmax || forced) ? 0u : min(sh.n_cand, n_cap);
    phase(late, 4);
    if (!CHAIN && S > 1 && !argmax && t.k <= 64u && late.ws_k <= 64u &&
        (S <= WAVE_MERGE_LISTS || S * late.ws_k <= WAVE_MERGE_SLOTS) &&
        (t.mode != MODE_SPEC || (SPEC && *t.q_n <= 64u))) {
        if (tid >= 64u) {
            return false;
        }
        const bool finished = finish_by_wave<DT, LSE, SPEC>(t, late, row, s, n, found, step, want_lse, sh);
        if (finished) {
            phase(late, 7);
        }
        return finished;
    }
    // What is left to rank behind the slices: every slice's candidates, or those of a row of many
    // candidates that is one slice, up to PER a thread.  (Expanded once: inside the slices' branch
    // where only that can come to it, else behind both.)
    constexpr int PER = MERGE_CAP / NT;
    uint64_t mine[PER];
    uint32_t slots = 0;
    auto rank_them = [&]() {
        sorted = false;
        if (KIND != 2 && t.k > 64u) {
            // Many candidates: every entry goes into the sort as it is.  This is the one place in a
            // kernel that holds it: with a copy behind each select as well, the kernels that can have
            // such rows spilled 30 to 60 vector registers more, and every row in them paid (the
            // constrained batch of 64 rows 37.9 -> 36.6 us; 40 f32 rows without top_k, half of them forced
            // and with log-probabilities, 70.2 -> 63.4).
            n = slots;
            sorted = wg_sort_topk(cand, mine, slots, t.k, sh, n);
        } else {
            // A bound of the k-th largest from the lanes' best entries (as in the streaming
            // select: each wave's ceil(k / NWAVE)-th largest lane maximum, the minimum over the
            // waves), then only entries at or above it are ranked.
            uint64_t best_mine = 0;
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                best_mine = mine[q] > best_mine ? mine[q] : best_mine;
            }
            const uint32_t kw = (t.k + NWAVE - 1) / NWAVE;
            const uint32_t P = kw <= 64u ? wave_kth_key16((uint32_t)(best_mine >> 48), kw) : 0u;
            if ((tid & 63u) == 0) {
                sh.red_i[tid >> 6] = P;
            }
            if (tid == 0) {
                sh.n_cand = 0;
            }
            __syncthreads();
            uint32_t bound = sh.red_i[0];
            for (int i = 1; i < NWAVE; ++i) {
                bound = min(bound, sh.red_i[i]);
            }
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                if (mine[q] != 0ull && (uint32_t)(mine[q] >> 48) >= bound) {
                    cand[atomicAdd(&sh.n_cand, 1u)] = mine[q];
                }
            }
            __syncthreads();
            n = sh.n_cand;
        }
        if (!sorted) {
            n = select_topk(cand, n, t.k, sh, sorted);
        }
        found = cand;
    };
    if (S > 1) {
        const size_t slot = (size_t)row * S + s;
        // Partials go through to memory (no dirty L2 lines to write back), the wave waits
        // for its stores, the workgroup meets, and one thread takes the row's ticket.
        if (argmax) {
            if (tid == 0) {
                handed_store(late.ws_cand, slot * late.ws_k, best);
            }
        } else {
            // Every slot is written (0 = no candidate), so the merge needs no counts.
            for (uint32_t i = tid; !forced && i < late.ws_k; i += NT) {
                handed_store(late.ws_cand, slot * late.ws_k + i, i < n ? found[i] : (uint64_t)0);
            }
            if (tid == 0) {
                handed_store(late.ws_lse, 2 * slot, want_lse ? sh.lse_mc : 0.0);
                handed_store(late.ws_lse, 2 * slot + 1, want_lse ? sh.lse_s : 0.0);
            }
        }
        // The hand-over (last_to_arrive(): a release on the ticket and an acquire behind it, or
        // the relaxed form described there).
        const bool last = last_to_arrive(&late.ws_ticket[row], S, sh.last, late.relaxed_handover != 0u);
        phase(late, 5);
        if (!last) {
            return false;
        }
        const size_t base = (size_t)row * S;
        if (argmax) {
            best = 0;
            for (uint32_t t = tid; t < S; t += NT) {
                const uint64_t c = handed_load(late.ws_cand, (base + t) * late.ws_k);
                best = c > best ? c : best;
            }
            best = wave_max_u64(best);
            if ((tid & 63u) == 0) {
                sh.red_u[tid >> 6] = best;
            }
            __syncthreads();
            best = sh.red_u[0];
            for (int i = 1; i < NWAVE; ++i) {
                best = sh.red_u[i] > best ? sh.red_u[i] : best;
            }
        } else {
            // Gather every slice's candidates (0 = no candidate) and the log-sum-exp partials
            // in one round trip.
            slots = S * late.ws_k;
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const uint32_t j = tid + (uint32_t)q * NT;
                mine[q] = (!forced && j < slots) ? handed_load(late.ws_cand, base * late.ws_k + j) : 0ull;
            }
            if (want_lse && tid < 64) {
                double mt = -__builtin_huge_val(), st = 0.0;
                if (tid < S) {
                    mt = handed_load(late.ws_lse, 2 * (base + tid));
                    st = handed_load(late.ws_lse, 2 * (base + tid) + 1);
                    if (!(st > 0.0)) {
                        mt = -__builtin_huge_val();
                    }
                }
                const double m = wave_max_d(mt);
                const double sum = wave_sum_d(st > 0.0 ? st * exp2(mt - m) : 0.0);
                if (tid == 0) {
                    sh.lse_mc = m;
                    sh.lse_s = sum;
                }
            }
            if constexpr (KIND == 2) {
                rank_them();
            }
        }
    } else if (KIND != 2 && t.k > 64u && n != 0u && !sorted) {
        slots = n;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const uint32_t j = tid + (uint32_t)q * NT;
            mine[q] = j < n ? cand[j] : 0ull;
        }
    }
    if (KIND != 2 && slots != 0u) {
        rank_them();
    }

    phase(late, 6);
    if (argmax) {
        if (tid == 0) {
            const uint32_t id = composite_id(best);
            *t.out_id = id == 0xffffffffu ? 0u : id;
        }
        return true;
    }
    if (t.flags & F_FORCED) {
        if (tid == 0) {
            finish_token<DT>(t, sh, t.forced, vocab);
        }
        return true;
    }
    if (CHAIN && late.chain_rows != 0u) {
        // Rows that draw in order.  This row's candidates - the best t.k under the counts as they
        // stood when the launch began, t.k being the draw's own count plus one for every row
        // before it - are published; the workgroup that publishes last takes the rows one after
        // the other: the ids the earlier rows drew are evaluated again (penalties that can only
        // lower took them down, so the best k_draw of the row as it stands now are still among
        // the candidates), and the tail draws from the best k_draw.
        const uint32_t rows = late.chain_rows;
        for (uint32_t i = tid; i < n; i += NT) {
            handed_store(late.chain_cand, (size_t)row * CHAIN_CAP + i, found[i]);
        }
        if (tid == 0) {
            handed_store(late.chain_n, row, n);
        }
        if (!last_to_arrive(late.chain_ticket, rows, sh.last, late.relaxed_handover != 0u)) {
            return false;
        }
        const LILY_CONST RowArgs* first = src - row;
        if (late.accept_ctrl != nullptr && tid < rows) {
            sh.proposal[tid] = gload(late.accept_ids + tid);
        }
        // Every row's first 64 candidates, their raw logits and their counts as they stand before
        // any of these rows has drawn are requested together (a wave per row, two rounds for
        // eight rows) and kept in LDS behind the tail's arrays: once the rows draw, nothing waits
        // for memory but the tail's own reads, and the counts the earlier rows left follow from
        // what they drew.  Candidates past the 64th are loaded when their row's turn comes.
        constexpr uint32_t PRE = 64;
        uint64_t* pre_c = dyn_lds + CHAIN_LDS_OFFSET / 8;                           // [rows][PRE]
        float* pre_l = reinterpret_cast<float*>(pre_c + LILY_MAX_VERIFY_ROWS * PRE);  // [rows][PRE]
        uint32_t* pre_cnt = reinterpret_cast<uint32_t*>(pre_l + LILY_MAX_VERIFY_ROWS * PRE);
        // ... and, for the rows that are speculative draws, the proposal and the first 64 entries
        // of the draft's distribution (all of it, as a rule): the tail reads them through the
        // row's pointers, which are turned to these copies.
        uint32_t* pre_qid = pre_cnt + LILY_MAX_VERIFY_ROWS * PRE;                     // [rows][PRE]
        float* pre_qp = reinterpret_cast<float*>(pre_qid + LILY_MAX_VERIFY_ROWS * PRE);
        for (uint32_t j0 = 0; j0 < rows; j0 += NWAVE) {
            const uint32_t j = j0 + (tid >> 6), lane = tid & 63u;
            if (j < rows) {
                const uint32_t nj = min(handed_load(late.chain_n, j), CHAIN_CAP);
                if (lane == 0) {
                    sh.chain_n[j] = nj;
                }
                const uint64_t c = handed_load(late.chain_cand, (size_t)j * CHAIN_CAP + lane);
                const uint32_t id = min(composite_id(c), vocab - 1u);
                pre_c[j * PRE + lane] = c;
                pre_l[j * PRE + lane] = load_logit<DT>((first + j)->logits, id);
                const LILY_CONST RowArgs* rj = first + j;
                pre_cnt[j * PRE + lane] = (rj->flags & F_PEN) ? load_through(rj->counts + id) : 0u;
                if (rj->mode == MODE_SPEC) {
                    pre_qid[j * PRE + lane] = gload(rj->q_ids + lane);
                    pre_qp[j * PRE + lane] = gload(rj->q_probs + lane);
                    if (lane == 0) {
                        sh.proposal_of[j] = gload(rj->draft);
                        sh.q_n_of[j] = gload(rj->q_n);
                    }
                }
            }
        }
        __syncthreads();
        for (uint32_t j = 0; j < rows; ++j) {
#ifdef LILY_CHAIN_TRACE
            phase(late, 8 + j);
#endif
            RowArgs r;
            {
                const LILY_CONST RowArgs* from = first + j;
                asm volatile("" : "+s"(from));
                load_row_args(r, from);
            }
            // What an earlier row drew is evaluated again, with the count it has by now.
            auto times_drawn = [&](uint32_t id) -> uint32_t {
                uint32_t times = 0;
                for (uint32_t q = 0; q < j; ++q) {
                    times += sh.drawn[q] == id ? 1u : 0u;
                }
                return times;
            };
            auto with_count = [&](uint32_t id, float l, uint32_t cnt) -> uint64_t {
                const bool allowed = r.allow == nullptr || bit_of(r.allow, id);
                return composite_of(finish_pre_temperature(r, id, l, cnt, allowed) / r.temperature, id);
            };
            const uint32_t n_now = sh.chain_n[j];
            if (tid < min(n_now, PRE)) {
                const uint64_t c = pre_c[j * PRE + tid];
                const uint32_t id = composite_id(c);
                const uint32_t times = times_drawn(id);
                cand[tid] = times == 0u ? c : with_count(id, pre_l[j * PRE + tid], pre_cnt[j * PRE + tid] + times);
            }
            if (n_now > PRE) {
                // Past what was requested ahead: the earlier rows' increments are waited for
                // (thread 0 issued them) and the counts read as they stand.
                __threadfence();
                __syncthreads();
                for (uint32_t i = tid + PRE; i < n_now; i += NT) {
                    const uint64_t c = handed_load(late.chain_cand, (size_t)j * CHAIN_CAP + i);
                    const uint32_t id = composite_id(c);
                    cand[i] = times_drawn(id) == 0u
                                  ? c
                                  : with_count(id, load_logit<DT>(r.logits, id), load_through(r.counts + id));
                }
            }
            __syncthreads();
            // The few candidates that changed are put back in order: up to a workgroup's worth
            // each thread counts the candidates that beat its own (composites are distinct).
            bool ranked = false;
            if (n_now <= NT) {
                // (read eight at a time, the slots up to the next multiple of eight cleared: a
                // loop of one dependent LDS read after the other costs a microsecond a row)
                const uint32_t n_up = (n_now + 7u) & ~7u;
                if (tid >= n_now && tid < n_up) {
                    cand[tid] = 0ull;
                }
                lds_barrier();
                const uint64_t mine = tid < n_now ? cand[tid] : ~0ull;
                uint32_t ahead = 0;
                for (uint32_t q0 = 0; q0 < n_up; q0 += 8u) {
                    uint64_t other[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        other[q] = cand[q0 + (uint32_t)q];
                    }
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        ahead += other[q] > mine ? 1u : 0u;
                    }
                }
                __syncthreads();
                if (tid < n_now) {
                    cand[ahead] = mine;
                }
                __syncthreads();
                ranked = true;
            }
            r.k = r.k_draw;
            if (r.mode == MODE_SPEC && sh.q_n_of[j] <= PRE) {
                r.draft = &sh.proposal_of[j];
                r.q_n = &sh.q_n_of[j];
                r.q_ids = pre_qid + j * PRE;
                r.q_probs = pre_qp + j * PRE;
            }
            tail<DT, KIND != 2, true>(r, vocab, r.step + late.step_delta, n_now, ranked, cand, sh, late);
            // The workgroup meets over LDS only: a barrier that also waited for thread 0's stores
            // and increments to be acknowledged by memory would cost every row a round trip
            // that nothing here depends on.
            lds_barrier();
            if (tid == 0) {
                sh.drawn[j] = sh.emitted_id;
            }
            lds_barrier();
        }
        // The scratch's largest count (and an id that holds it) follow now, once per draw.  It
        // must never understate a count: thread 0, which issued every increment (device atomics,
        // done where the reads below look), waits for them before anybody reads a count back.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid < rows && ((first + tid)->flags & F_PEN) && sh.drawn[tid] < vocab) {
            // (row tid's own scratch: the launcher hands every row of such a launch the same one,
            // but nothing here depends on that)
            const LILY_CONST RowArgs* mine = first + tid;
            const uint32_t id = sh.drawn[tid];
            const uint32_t words = (vocab + 31u) / 32u;
            const uint32_t now = load_through(mine->counts + id);
            if (atomicMax(&mine->touched[words], now) <= now) {
                mine->touched[words + 1u] = id;
            }
        }
        if (late.accept_ctrl != nullptr && tid == 0) {
            // spec_accept (spec.metal:14-38) on the draws this workgroup just made.
            uint32_t acc = 0;
            while (acc + 1 < rows && sh.drawn[acc] == sh.proposal[acc + 1]) {
                ++acc;
            }
            write_accepted(late, acc);
        }
        phase(late, 7);
        return true;
    }
    tail<DT, KIND != 2, SPEC>(t, vocab, step, n, sorted, found, sh, late);
    phase(late, 7);
    return true;
}

// Dynamic LDS: [0, cand_cap) candidates while scanning, then the bitmap.  In the tail the
// first K_CAP slots hold the sorted candidates and the three float arrays follow them
// (the launcher sizes the region for at least K_CAP * 8 + 3 * K_CAP * 4 bytes).
__device__ __forceinline__ void tail_arrays(Shared& sh) {
    float* f = reinterpret_cast<float*>(dyn_lds + K_CAP);
    sh.prob = f;
    sh.cum = f + K_CAP;
    sh.res = f + 2 * K_CAP;
}

template <int DT, int KIND, bool LSE>
__global__ __launch_bounds__(NT, KIND == 1 ? 3 : 4) void k_rows_inline(InlineRows rows, LaunchCfg cfg) {
    __shared__ Shared sh;
    // `rows` is the first kernel argument: index it in the kernel-argument segment itself
    // (indexing the by-value copy would move all of it to scratch memory).
    const LILY_CONST RowArgs* table =
        (const LILY_CONST RowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    if (threadIdx.x == 0) {
        tail_arrays(sh);
    }
    __syncthreads();
    row_body<DT, KIND, LSE>(table + blockIdx.y, cfg, (const LILY_CONST LaunchCfg*)(table + INLINE_ROWS), sh);
}

// Rows that draw in order (the verify pass under penalties): see row_body.
template <int DT, int KIND>
__global__ __launch_bounds__(NT, KIND == 1 ? 3 : 4) void k_rows_chain(InlineRows rows, LaunchCfg cfg) {
    __shared__ Shared sh;
    const LILY_CONST RowArgs* table =
        (const LILY_CONST RowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    if (threadIdx.x == 0) {
        tail_arrays(sh);
    }
    __syncthreads();
    row_body<DT, KIND, false, true>(table + blockIdx.y, cfg, (const LILY_CONST LaunchCfg*)(table + INLINE_ROWS), sh);
}

// A verify pass whose rows are independent: the one-wave form of the speculative draw is compiled in,
// and the workgroup that finishes the last row runs spec_accept (spec.metal:14-38) on the draws - a
// launch of its own behind this one took 3.9 us of a step of three rows.
template <int DT, int KIND>
__global__ __launch_bounds__(NT, KIND == 1 ? 3 : 4) void k_rows_verify(InlineRows rows, LaunchCfg cfg) {
    __shared__ Shared sh;
    const LILY_CONST RowArgs* table =
        (const LILY_CONST RowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    if (threadIdx.x == 0) {
        tail_arrays(sh);
    }
    __syncthreads();
    const bool finished = row_body<DT, KIND, false, false, true>(table + blockIdx.y, cfg, (const LILY_CONST LaunchCfg*)(table + INLINE_ROWS), sh);
    if (!finished || threadIdx.x != 0 || cfg.accept_ctrl == nullptr) {
        return;
    }
    accept_behind_last_row(cfg, [&](uint32_t j) { return (table + j)->out_id; });
}

template <int DT, int KIND, bool LSE>
__global__ __launch_bounds__(NT, KIND == 1 ? 3 : 4) void k_rows_table(LaunchCfg cfg) {
    __shared__ Shared sh;
    const LILY_CONST RowArgs* table = (const LILY_CONST RowArgs*)cfg.table;
    if (threadIdx.x == 0) {
        tail_arrays(sh);
    }
    __syncthreads();
    row_body<DT, KIND, LSE>(table + blockIdx.y, cfg, (const LILY_CONST LaunchCfg*)__builtin_amdgcn_kernarg_segment_ptr(), sh);
}

template <int DT, int KIND, bool LSE>
static hipError_t launch_variant(hipStream_t stream, uint32_t rows, const LaunchCfg& cfg,
                                 const InlineRows* inline_rows, size_t dyn_bytes) {
    const dim3 grid(cfg.slices, rows), block(NT);
    if (cfg.chain_rows != 0u) {
        if constexpr (!LSE && KIND != 0) {
            if (inline_rows != nullptr) {
                hipLaunchKernelGGL((k_rows_chain<DT, KIND>), grid, block, dyn_bytes, stream, *inline_rows, cfg);
                return hipGetLastError();
            }
        }
        return hipErrorInvalidValue;   // rows that draw in order are under penalties, travel inline, want no row sum
    }
    if (cfg.verify != 0u) {
        if constexpr (!LSE && KIND != 1) {
            if (inline_rows != nullptr) {
                hipLaunchKernelGGL((k_rows_verify<DT, KIND>), grid, block, dyn_bytes, stream, *inline_rows, cfg);
                return hipGetLastError();
            }
        }
        return hipErrorInvalidValue;   // (independent rows of a verify pass: no penalties, masks or bias lists)
    }
    if (inline_rows != nullptr) {
        hipLaunchKernelGGL((k_rows_inline<DT, KIND, LSE>), grid, block, dyn_bytes, stream,
                           *inline_rows, cfg);
    } else {
        hipLaunchKernelGGL((k_rows_table<DT, KIND, LSE>), grid, block, dyn_bytes, stream, cfg);
    }
    return hipGetLastError();
}

}  // namespace lily
