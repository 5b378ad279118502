// rows_wide.hip - rows that draw among many candidates (k > 64, up to the reference's cap of 1024,
// which is what a request without top_k gets: src/kernels/sample.rs:17, :326-331), spread over
// as many workgroups as rows of few candidates are.
//
// One launch where a slice fits its workgroup's registers and the launch the chip (k_wide_held), two otherwise
// (k_wide_bound, k_wide_draw).  Every slice's lanes take their largest values (penalised ids at their penalised
// worth), its waves name one each that r lanes reach, and from what all the row's waves named comes a lower bound of the
// row's k-th largest value that k lanes, so k values reach, and some 1.5 k in all (bound_of_keys).  The values
// that reach it are appended to the row's list - after a second look at the slice, from the L2, where there are two
// launches -; the workgroup that finishes last sorts the list, whatever the number of slices, and runs the common
// tail.  (The select of the other kernels keeps k candidates per slice and can therefore spread a row with
// k = 1024 over 4 workgroups only.)
//
// Bound: a chain of latencies.  us a launch, no top_k, two launches -> one: 4 f32 rows of 151 936 with log-probabilities
// 27.3 -> 24.4, under penalties 31.1 -> 25.2, 13 rows under penalties 39.6 -> 31.9, 26 bf16 rows under penalties 52.7 ->
// 38.8, without 37.6 -> 35.4; 40 bf16 rows in 760 workgroups 46.6 -> 41.9.  4 bf16 rows of 32 000 in 16 slices, where a block
// a slice were 4, 41.9 -> 25.9.
#include <algorithm>

#ifdef LILY_WIDE_TRACE
#define LILY_TAIL_TRACE
#endif

#include "launch.h"
#include "row_kernel.h"
#include "sort_sixteen.h"

namespace lily {

// Diagnostic stamps (LaunchCfg::phase_trace), compiled in with -DLILY_WIDE_TRACE (which also
// turns on the tail's: slots 8 to 12).  First launch: 0 start, 1 slice read, 2 maxima stored;
// second: 5 start, 6 slice read, 7 last slice in, 13 list read, 14 selected.
#ifdef LILY_WIDE_TRACE
#define WIDE_MARK(i) phase(cfg, i)
#else
#define WIDE_MARK(i)
#endif

// What the two launches share beyond LaunchCfg.
struct WideArgs {
    Handed<float> lane_max;   // [rows][slices][lanes]
    Handed<uint64_t> slice_keys;   // [rows][slices] four waves' keys (slice_keys_of())
    uint32_t lanes;       // values a slice leaves: NT, or NT / 2 (the larger of each pair of lanes)
    // k_wide_held: [rows][MAX_SLICES] slices' keys, then as many words for slices that have left their lanes' maxima
    // (0 between launches); null: two launches
    uint64_t* bounds;
    uint32_t* count;      // [rows] candidates the row's slices have left so far (0 between launches)
    WideLooks looks;
};

template <bool INLINE>
__device__ __forceinline__ const LILY_CONST RowArgs* wide_table(const LaunchCfg& cfg) {
    if (INLINE) {
        // the rows are the kernel's first argument: index the kernel-argument segment itself
        return (const LILY_CONST RowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    }
    return (const LILY_CONST RowArgs*)cfg.table;
}

// One pass over the slice's chunks, four loads in flight per thread, every load unconditional
// (a chunk number past the slice is replaced by the slice's last).  before(): called once the first loads are on their
// way; true = what it did had no registers for them, they are made again.
template <int DT, uint32_t THREADS = NT, class B, class F>
__device__ __forceinline__ void wide_scan(const Geo<DT>& g, B&& before, F&& per_chunk) {
    const uint32_t tid = threadIdx.x;
    if (g.main_hi <= g.main_lo) {
        before();
        return;
    }
    u32x4 q[4];
    auto fetch = [&](uint32_t c0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t c = min(c0 + (uint32_t)u * THREADS + tid, g.main_hi - 1u);
            q[u] = gload(reinterpret_cast<const u32x4*>(g.base + (size_t)c * 16));
        }
    };
    fetch(g.main_lo);
    if (before()) {
        fetch(g.main_lo);
    }
    for (uint32_t c0 = g.main_lo;;) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t c = c0 + (uint32_t)u * THREADS + tid;
            if (c < g.main_hi) {
                per_chunk(q[u], c);
            }
        }
        c0 += 4u * THREADS;
        if (c0 >= g.main_hi) {
            break;
        }
        fetch(c0);
    }
}

// What a raw value is worth under the row's penalties (the arithmetic of finish_pre_temperature).
__device__ __forceinline__ float wide_worth(const RowArgs& a, float x, uint32_t id) {
    if (bit_of(a.touched, id)) {
        uint32_t cnt = gload(a.counts + id);
        asm volatile("" : "+v"(cnt));   // waited for here, inside the branch
        if (cnt > 0u) {
            x = x > 0.0f ? x / a.repetition : x * a.repetition;
            x -= a.presence + a.frequency * (float)cnt;
        }
    }
    return x;
}

// Bits id0 .. id0 + E - 1 of the bitmap of penalised ids (all below the vocabulary; the word
// behind the bitmap's last is the row's largest count, so the second load stays in bounds).
template <int E>
__device__ __forceinline__ uint32_t wide_bits(const uint32_t* words, uint32_t id0) {
    const uint32_t w = id0 >> 5, sh = id0 & 31u;
    uint32_t b = gload(words + w) >> sh;
    if (sh + (uint32_t)E > 32u) {
        b |= gload(words + w + 1u) << (32u - sh);
    }
    return b & ((1u << E) - 1u);
}

// The ids of the partial 16-byte chunks at the slice's ends, one by one.
template <int DT, uint32_t THREADS = NT, class F>
__device__ __forceinline__ void wide_edges(const RowArgs& a, const Geo<DT>& g, F&& per_id) {
    for (int side = 0; side < 2; ++side) {
        const uint32_t lo = side == 0 ? g.id_lo : g.edge_hi_begin;
        const uint32_t hi = side == 0 ? g.edge_lo_end : g.id_hi;
        for (uint32_t id = lo + threadIdx.x; id < hi; id += THREADS) {
            per_id(load_logit<DT>(a.logits, id), id);
        }
    }
}

// The row's ticket: true in every thread of the workgroup that arrives last (last_to_arrive()).
__device__ __forceinline__ bool wide_last(const LaunchCfg& cfg, uint32_t row, uint32_t S, Shared& sh) {
    return last_to_arrive(&cfg.ws_ticket[row], S, sh.last, cfg.relaxed_handover != 0u);
}

// A slice's four keys of 16 bits as one word, never 0, in thread 0 (every thread calls).
__device__ __forceinline__ uint64_t slice_keys_of(float lane_max, uint32_t k, uint32_t S, Shared& sh) {
    const uint32_t tid = threadIdx.x;
    const uint32_t P = wave_kth_key16(lane_max > NEG_INF ? (lilym_order_key(lane_max) >> 16) : 0u, wide_rank(k, S));
    if ((tid & 63u) == 0u) {
        sh.hist[tid >> 6] = max(P, WIDE_LEAST_KEY);
    }
    __syncthreads();
    static_assert(NWAVE == 4, "a word of four keys");
    return tid != 0u ? 0ull : ((uint64_t)(sh.hist[3] << 16 | sh.hist[2]) << 32) | (sh.hist[1] << 16 | sh.hist[0]);
}
// ---- first launch: lane maxima, the slice's sum of exponentials

template <int DT, bool LSE, bool INLINE>
__global__ __launch_bounds__(NT, 4) void k_wide_bound(InlineRows rows_arg, LaunchCfg cfg, WideArgs w) {
    __shared__ Shared sh;
    constexpr int E = Geo<DT>::E;
    const uint32_t tid = threadIdx.x, s = blockIdx.x, row = blockIdx.y, S = cfg.slices;
    if (cfg.served != nullptr && *(const LILY_CONST uint32_t*)(cfg.served + row) != 0u) {
        return;   // drawn by an earlier launch of the same call
    }
    WIDE_MARK(0);
    RowArgs a;
    load_row_args(a, wide_table<INLINE>(cfg) + row);
    apply_selection(a);
    const bool want_lse = LSE && a.out_logprob != nullptr;
    Geo<DT> g;
    g.init(a.logits, cfg.vocab, s, S);
    const bool pen = (a.flags & F_PEN) != 0;
    float lane_max = NEG_INF;
    LseAcc lse;
    lse.init();
    wide_scan<DT>(g, []() { return false; }, [&](const u32x4& q, uint32_t c) {
        float v[E];
        unpack<DT>(q, v);
        float m;
        if (pen) {
            const uint32_t id0 = g.id_of(c, 0);
            const uint32_t bits = wide_bits<E>(a.touched, id0);
            if (bits != 0u) {
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    if ((bits >> j) & 1u) {
                        v[j] = wide_worth(a, v[j], id0 + (uint32_t)j);
                    }
                }
            }
            m = NEG_INF;
#pragma unroll
            for (int j = 0; j < E; ++j) {
                m = fmaxf(m, v[j]);   // (a NaN operand loses)
            }
        } else {
            m = chunk_max<DT>(q);   // (NaN operands lose)
        }
        lane_max = fmaxf(lane_max, m);
        if (want_lse && m > NEG_INF) {
            const float safe = lse.rebase(m, a.c2);
#pragma unroll
            for (int j = 0; j < E; ++j) {
                if (v[j] > NEG_INF) {   // (false for a NaN: worth -inf)
                    lse.term(v[j], a.c2, safe);
                }
            }
        }
    });
    wide_edges<DT>(a, g, [&](float x, uint32_t id) {
        if (pen) {
            x = wide_worth(a, x, id);
        }
        if (x > NEG_INF) {
            lane_max = fmaxf(lane_max, x);
            if (want_lse) {
                lse.add_one(x, a.c2);
            }
        }
    });
    WIDE_MARK(1);
    const size_t slot = (size_t)row * S + s;
    const float pair_max = lane_max;
    if (w.lanes == NT) {
        handed_store(w.lane_max, slot * NT + tid, lane_max);
    } else {
        // (with slices enough that half the lanes still are four times k, half the keys make
        // the select of the bound half as long)
        const int other = __builtin_amdgcn_update_dpp(0, (int)lilym_f32_bits(lane_max), 0xb1, 0xf, 0xf, true);   // quad_perm [1, 0, 3, 2]
        lane_max = fmaxf(lane_max, lilym_bits_f32((uint32_t)other));
        if ((tid & 1u) == 0u) {
            handed_store(w.lane_max, slot * (NT / 2) + tid / 2u, lane_max);
        }
    }
    // (every lane's own maximum, whatever was stored above)
    const uint64_t keys = slice_keys_of(pair_max, a.k, S, sh);
    if (tid == 0) {
        handed_store(w.slice_keys, slot, keys);
    }
    if (want_lse) {
        lse_reduce(sh, lse);
        if (tid == 0) {
            handed_store(cfg.ws_lse, 2 * slot, sh.lse_mc);
            handed_store(cfg.ws_lse, 2 * slot + 1, sh.lse_s);
        }
    }
    WIDE_MARK(2);
}

// The row's bound: the k-th largest of its S x lanes lane maxima, by a radix select on the
// leading 16 bits of their order keys, 8 bits a pass: that key with the other 16 bits clear, at
// most 2^-7 of its magnitude below the k-th largest lane maximum, which lets a few per cent more
// values through.  Every workgroup of the second launch works it out for itself, from what the
// first launch left (a row's slices all arrive at the same value; a workgroup that did it for
// all of them would have to be waited for).  A thread keeps its keys in registers (the loops
// are unrolled over MAX_SLICES in groups of eight, a group past the last is skipped by the whole
// workgroup): a pass that fetched each key from LDS, or the values from the L2 a few at a time,
// would wait out that latency over and over.  F32_LOWEST when fewer than k lanes saw a finite
// value: every value is a candidate then.
__device__ __forceinline__ float wide_bound_of(const WideArgs& w, uint32_t row, uint32_t S, uint32_t k, Shared& sh) {
    const uint32_t tid = threadIdx.x;
    static_assert(MAX_SLICES == 64, "the unrolled loops below cover 64 keys a thread");
    const uint32_t n = S * w.lanes, mine_n = (n + NT - 1u) / NT;   // keys in all, keys a thread
    float got[MAX_SLICES];
#pragma unroll
    for (int j0 = 0; j0 < (int)MAX_SLICES; j0 += 8) {
        if ((uint32_t)j0 < mine_n) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const uint32_t i = min((uint32_t)(j0 + u) * NT + tid, n - 1u);
                got[j0 + u] = handed_load(w.lane_max, (size_t)row * n + i);
            }
        }
    }
    uint32_t keys[MAX_SLICES];
#pragma unroll
    for (int j = 0; j < (int)MAX_SLICES; ++j) {
        const bool in = (uint32_t)j * NT + tid < n;   // (a group past the last was not loaded: what it holds is not read)
        keys[j] = in && got[j] > NEG_INF ? lilym_order_key(got[j]) : 0u;
    }
    uint32_t prefix = 0, pmask = 0, need = k;
    bool enough = true;
    for (int pass = 0; pass < 2 && enough; ++pass) {
        const int shift = 24 - 8 * pass;
        sh.hist[tid] = 0;
        __syncthreads();
        HistRun run;
        run.init();
#pragma unroll
        for (int j0 = 0; j0 < (int)MAX_SLICES; j0 += 8) {
            if ((uint32_t)j0 < mine_n) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t key = keys[j0 + u];
                    run.add(sh.hist, (key >> shift) & 255u, key != 0u && (key & pmask) == prefix);
                }
            }
        }
        run.flush(sh.hist);
        __syncthreads();
        find_bin(sh, need);
        if (sh.all_taken != 0u) {
            enough = false;   // fewer than k lanes saw a finite value: every value is a candidate
        } else {
            prefix |= sh.sel_bin << shift;
            pmask |= 255u << shift;
            need = sh.need;
        }
        __syncthreads();
    }
    return enough ? lower_by_slack(lilym_key_value(prefix)) : F32_LOWEST;
}

// Dynamic LDS of sixteen waves, in 64-bit slots: the sorted candidates and the tail's arrays; the sort's bins; a slice's
// candidates, then the row's by bins.
constexpr uint32_t SIXTEEN_OFF_BINS = (LILY_SAMPLE_K_CAP * 8 + 3 * LILY_SAMPLE_K_CAP * 4) / 8;
constexpr uint32_t SIXTEEN_OFF_PLACED = SIXTEEN_OFF_BINS + SIXTEEN_BINS / 2;
constexpr uint32_t SIXTEEN_LDS_BYTES = (SIXTEEN_OFF_PLACED + MERGE_CAP) * 8;

// The row's best where more of its values reach the bound than the list holds (a cluster of likely ids, ties by the
// thousand, no bound): MERGE_CAP at most of them to cand, the k best among them, in any order, by one workgroup.  Histograms of the composites'
// leading bits, twelve more each time (sixteen composites at most share all but the last four bits), until what lies at or above
// the k-th one's bin fits.  (4 bf16 rows of 248 320 under penalties, 6 000 neighbours 9 above the rest, 113 us; by the
// exhaustive select, which looks at every id nine times, 3 850.  4 rows of 50 257, 3 000 neighbours, 50 and 573.)
template <int DT, uint32_t THREADS>
__device__ __forceinline__ uint32_t wide_collect(const RowArgs& a, uint32_t vocab, float bound, uint64_t* cand, SixteenShared& six,
                                                 uint32_t& count) {
    constexpr int E = Geo<DT>::E;
    constexpr uint32_t BINS = 4096, OWN = BINS / THREADS;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const bool pen = (a.flags & F_PEN) != 0;   // (of the kind that only lowers: the host sees to it)
    uint32_t* hist = reinterpret_cast<uint32_t*>(cand);
    static_assert(BINS * 4u <= MERGE_CAP * 8u, "the histogram lies where the entries will");
    Geo<DT> g;
    g.init(a.logits, vocab, 0u, 1u);
    // fn(composite) of every id whose value reaches the bound
    auto over = [&](auto&& fn) {
        auto one = [&](float x, uint32_t id) {
            if (x >= bound) {
                x = pen ? wide_worth(a, x, id) : x;   // (never more than the raw value)
                if (x >= bound) {
                    fn(composite_of(x / a.temperature, id));
                }
            }
        };
        wide_scan<DT, THREADS>(g, []() { return false; }, [&](const u32x4& q, uint32_t c) {
            if (chunk_max<DT>(q) >= bound) {
                float v[E];
                unpack<DT>(q, v);
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    one(v[j], g.id_of(c, j));
                }
            }
        });
        wide_edges<DT, THREADS>(a, g, one);
    };
    uint64_t prefix = 0ull;
    uint32_t above = 0;   // composites above everything under the prefix
    for (int shift = 52; shift >= 4; shift -= 12) {
        __syncthreads();
        for (uint32_t i = tid; i < BINS; i += THREADS) {
            hist[i] = 0u;
        }
        __syncthreads();
        const uint64_t under = shift == 52 ? 0ull : ~0ull << (shift + 12);
        over([&](uint64_t c) {
            if ((c & under) == prefix) {
                atomicAdd(&hist[(uint32_t)(c >> shift) & (BINS - 1u)], 1u);
            }
        });
        __syncthreads();
        // from the top: thread t holds bins BINS - OWN (t + 1) .. + OWN - 1
        uint32_t h[OWN], mine = 0;
#pragma unroll
        for (uint32_t i = 0; i < OWN; ++i) {
            h[i] = hist[BINS - 1u - (tid * OWN + i)];
            mine += h[i];
        }
        const uint32_t incl = wave_scan_u32(mine);
        if (lane == 63u) {
            six.wave_u[w] = incl;
        }
        __syncthreads();
        uint32_t before = incl - mine, whole = 0;
        for (uint32_t i = 0; i < THREADS / 64u; ++i) {
            before += i < w ? six.wave_u[i] : 0u;
            whole += six.wave_u[i];
        }
        if (above + whole <= MERGE_CAP) {
            break;   // (all that lies under the prefix)
        }
#pragma unroll
        for (uint32_t i = 0; i < OWN; ++i) {
            if (above + before < a.k && above + before + h[i] >= a.k) {
                six.wave_k[0] = ((uint64_t)(BINS - 1u - (tid * OWN + i)) << 32) | (above + before);
                count = above + before + h[i];
            }
            before += h[i];
        }
        __syncthreads();
        prefix |= (six.wave_k[0] >> 32) << shift;
        above = (uint32_t)six.wave_k[0];
        if (count <= MERGE_CAP) {
            break;
        }
    }
    __syncthreads();
    if (tid == 0) {
        count = 0;
    }
    __syncthreads();
    over([&](uint64_t c) {
        if (c >= prefix) {
            const uint32_t at = atomicAdd(&count, 1u);
            if (at < MERGE_CAP) {
                cand[at] = c;
            }
        }
    });
    __syncthreads();
    return min(count, MERGE_CAP);
}

// From a slice's candidates (n_mine of them in cand) to the row's draw, in the workgroup that arrives last.
// bound: the row's; gave_up: the slice has none because it did not learn it, and looks at the whole row
// should it finish it.  HELD: of k_wide_held (the second launch of two, which are many rows, keeps the exhaustive select: with
// wide_collect() in it 128 f32 rows of 131 072 take 59 to 62 us instead of 54).
// Sixteen waves sort, and the first four draw.
template <int DT, bool LSE, uint32_t THREADS, bool HELD>
__device__ __forceinline__ void wide_finish(const LILY_CONST RowArgs* src, const LaunchCfg& cfg, const WideArgs& w, Shared& sh,
                                            uint32_t& n_mine, uint64_t* cand, uint32_t row, uint32_t S, float bound, bool gave_up,
                                            SixteenShared& six) {
    constexpr bool SIXTEEN = THREADS == SIXTEEN_THREADS;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    __syncthreads();
    WIDE_MARK(6);
    // The slice's candidates go behind those the row's other slices have left (any order: the
    // select does not care).  A row whose list would pass MERGE_CAP is counted on and not
    // written: the last workgroup sees the count and collects them itself.
    const uint32_t mine = gave_up ? MERGE_CAP + 1u : n_mine;
    if (tid == 0) {
        n_mine = __hip_atomic_fetch_add(&w.count[row], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    const uint32_t base = n_mine;
    if (base + mine <= MERGE_CAP) {
        for (uint32_t i = tid; i < mine; i += THREADS) {
            handed_store(cfg.ws_cand, (size_t)row * MERGE_CAP + base + i, cand[i]);
        }
    }
    if (!wide_last(cfg, row, S, sh)) {
        return;
    }
    if (w.bounds != nullptr && tid < S) {
        // (every slice has read them)
        store_through(w.bounds + (size_t)row * MAX_SLICES + tid, (uint64_t)0);
        store_through(w.bounds + ((size_t)gridDim.y + row) * MAX_SLICES + tid, (uint64_t)0);
    }
    WIDE_MARK(7);
    // The list's first entries are asked for together with its length: what lies behind its end is
    // dropped (the slots are the workspace's whatever they hold).
    constexpr int PER = MERGE_CAP / THREADS, FIRST = 2048 / THREADS;
    uint64_t mine_c[PER];
#pragma unroll
    for (int j = 0; j < FIRST; ++j) {
        mine_c[j] = handed_load(cfg.ws_cand, (size_t)row * MERGE_CAP + tid + (uint32_t)j * THREADS);
    }
    const uint32_t total = load_through(&w.count[row]);
    RowArgs a;
    read_again(a, src);
    const uint32_t step = a.step + cfg.step_delta;
    const bool want_lse = LSE && a.out_logprob != nullptr;
    __syncthreads();   // (everybody has read it)
    if (tid == 0) {
        store_through(&w.count[row], 0u);
    }
    uint32_t n = 0, found = total;
    bool sorted = false, exhausted = false;
    if (SIXTEEN) {
        cand = dyn_lds;
    }
    if (total > MERGE_CAP) {   // (the same in every thread)
        if constexpr (HELD) {
            found = wide_collect<DT, THREADS>(a, cfg.vocab, gave_up ? F32_LOWEST : bound, cand, six, n_mine);
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                mine_c[j] = cand[tid + (uint32_t)j * THREADS];
            }
        } else {
            __syncthreads();
            select_exhaustive<DT>(a, 0, cfg.vocab, a.k, want_lse, cand, min(cfg.dyn_slots, MERGE_CAP), sh);
            n = min(sh.n_cand, min(cfg.dyn_slots, MERGE_CAP));
            exhausted = true;
        }
        __syncthreads();
    } else if (total > (uint32_t)FIRST * THREADS) {
#pragma unroll
        for (int j = FIRST; j < PER; ++j) {
            mine_c[j] = handed_load(cfg.ws_cand, (size_t)row * MERGE_CAP + tid + (uint32_t)j * THREADS);
        }
    }
    if (!exhausted) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            if (tid + (uint32_t)j * THREADS >= found) {
                mine_c[j] = 0ull;
            }
        }
        if (want_lse && tid < 64u) {
            double mt = -__builtin_huge_val(), st = 0.0;
            if (lane < S) {
                mt = handed_load(cfg.ws_lse, 2 * ((size_t)row * S + lane));
                st = handed_load(cfg.ws_lse, 2 * ((size_t)row * S + lane) + 1);
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
        __syncthreads();
        WIDE_MARK(13);
        if constexpr (SIXTEEN) {
            n = min(found, a.k);
            sort_by_sixteen(mine_c, found, n, dyn_lds, reinterpret_cast<uint32_t*>(dyn_lds + SIXTEEN_OFF_BINS), dyn_lds + SIXTEEN_OFF_PLACED, six);
            sorted = true;
        } else {
            sorted = wg_sort_topk(cand, mine_c, found, a.k, sh, n);
            if (!sorted) {
                n = wg_select_topk(cand, found, a.k, sh);
            }
        }
    }
    WIDE_MARK(14);
    if (cfg.path_stats != nullptr && tid == 0) {
        atomicAdd(&cfg.path_stats[total > MERGE_CAP ? 2 : 1], 1u);
    }
    if (SIXTEEN && tid >= NT) {
        return;   // (the draw is four waves' work: a barrier waits for those that are left)
    }
    tail<DT, true>(a, cfg.vocab, step, n, sorted, cand, sh, cfg);
}

// ---- second launch: the values that reach the bound, then merge, select and tail

template <int DT, bool LSE, bool INLINE>
__global__ __launch_bounds__(NT, 4) void k_wide_draw(InlineRows rows_arg, LaunchCfg cfg, WideArgs w) {
    __shared__ Shared sh;
    __shared__ uint32_t n_mine;
    __shared__ float row_bound;
    __shared__ SixteenShared none;   // (four waves: not used)
    constexpr int E = Geo<DT>::E;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, s = blockIdx.x, row = blockIdx.y, S = cfg.slices;
    if (cfg.served != nullptr && *(const LILY_CONST uint32_t*)(cfg.served + row) != 0u) {
        return;
    }
    WIDE_MARK(5);
    if (tid == 0) {
        tail_arrays(sh);
        n_mine = 0;
    }
    RowArgs a;
    load_row_args(a, wide_table<INLINE>(cfg) + row);
    apply_selection(a);
    const uint32_t vocab = cfg.vocab;
    const bool pen = (a.flags & F_PEN) != 0;   // (of the kind that only lowers: the host sees to it)
    Geo<DT> g;
    g.init(a.logits, vocab, s, S);
    uint64_t* cand = dyn_lds;
    const uint32_t cap = MERGE_CAP;   // what the slice's own list holds
    const uint64_t keys = lane < S ? handed_load(w.slice_keys, (size_t)row * S + lane) : 0ull;
    float bound = F32_LOWEST;
    auto find_bound = [&]() -> bool {
        if (tid < 64u) {
            const float b = bound_of_keys(keys, a.k, S);
            if (lane == 0u) {
                row_bound = b;
            }
        }
        __syncthreads();
        bound = row_bound;
        const bool none = !(bound > F32_LOWEST);   // (the same in every wave)
        if (none) {
            bound = wide_bound_of(w, row, S, a.k, sh);
        }
        return none;
    };
    auto offer = [&](float x, uint32_t id) {
        if (!(x >= bound)) {
            return;
        }
        if (pen) {
            x = wide_worth(a, x, id);   // (never more than the raw value: the host sees to it)
            if (!(x >= bound)) {
                return;
            }
        }
        const uint32_t at = atomicAdd(&n_mine, 1u);
        if (at < cap) {
            cand[at] = composite_of(x / a.temperature, id);
        }
    };
    wide_scan<DT>(g, find_bound, [&](const u32x4& q, uint32_t c) {
        if (chunk_max<DT>(q) >= bound) {
            float v[E];
            unpack<DT>(q, v);
#pragma unroll
            for (int j = 0; j < E; ++j) {
                offer(v[j], g.id_of(c, j));
            }
        }
    });
    wide_edges<DT>(a, g, [&](float x, uint32_t id) { offer(x, id); });
    wide_finish<DT, LSE, NT, false>(wide_table<INLINE>(cfg) + row, cfg, w, sh, n_mine, cand, row, S, F32_LOWEST, false, none);
}

// ---- both in one launch, where a slice is held in registers and all of the launch's workgroups are on the chip

// What the two launches do below, without reading the slice again and without a second launch: each slice leaves its
// bound where the row's other slices look for it, and forms its sum of exponentials meanwhile.  A slice that
// does not find them all within WideArgs::looks (another stream's work holds the chip) gives up, and the row is taken by the
// exhaustive select: every wait ends.
constexpr uint32_t WIDE_HELD_GROUPS = 1024;
// Up to so many workgroups are of sixteen waves each, a piece of 16 bytes a thread, and sort with all of them (1 f32 row of
// 151 936 23.2 -> 19.8 us, under penalties 24.2 -> 20.5, 4 rows of 32 000 23.1 -> 20.8); launching four times the waves
// takes that back at 152 (4 rows 24.4 both ways, 13 rows 31.9 -> 35.9).
constexpr uint32_t WIDE_SIXTEEN_GROUPS = 128;

template <int DT, bool LSE, bool INLINE, uint32_t THREADS>
__global__ __launch_bounds__(THREADS, 4) void k_wide_held(InlineRows rows_arg, LaunchCfg cfg, WideArgs w) {
    __shared__ Shared sh;
    __shared__ uint32_t n_mine, lost;
    __shared__ float row_bound, wave_m[THREADS / 64];
    __shared__ double wave_s[THREADS / 64];
    __shared__ SixteenShared six;
    constexpr int E = Geo<DT>::E, C = (int)(NT * STREAM_UNROLL / THREADS), V = C * E;
    constexpr uint32_t EMASK = (1u << E) - 1u;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, s = blockIdx.x, row = blockIdx.y, S = cfg.slices;
    if (cfg.served != nullptr && *(const LILY_CONST uint32_t*)(cfg.served + row) != 0u) {
        return;
    }
    WIDE_MARK(0);
    if (tid == 0) {
        tail_arrays(sh);
        n_mine = 0;
        lost = 0;
    }
    RowArgs a;
    load_row_args(a, wide_table<INLINE>(cfg) + row);
    apply_selection(a);
    const bool want_lse = LSE && a.out_logprob != nullptr;
    const bool pen = (a.flags & F_PEN) != 0;
    Geo<DT> g;
    g.init(a.logits, cfg.vocab, s, S);
    const uint32_t c_last = max(g.ce, 1u) - 1u;
    auto chunk_of = [&](int u) -> uint32_t { return g.cb + (uint32_t)u * THREADS + tid; };
    auto inside = [&](int u) -> bool { return chunk_of(u) >= g.main_lo && chunk_of(u) < g.main_hi; };
    u32x4 raw[C];
#pragma unroll
    for (int u = 0; u < C; ++u) {
        raw[u] = gload(reinterpret_cast<const u32x4*>(g.base + (size_t)min(chunk_of(u), c_last) * 16));
    }
    // The chunks' bits of the bitmap of listed ids: two bytes hold a chunk's, wherever the row starts (a byte past the
    // bitmap is the scratch's own).
    struct Bits16 {
        uint16_t v;
    } __attribute__((packed));
    uint32_t todo = 0;
    static_assert(V <= 32, "a bit per value");
    if (pen) {
        uint32_t listed[C];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const uint32_t at = min(chunk_of(u), c_last) * (uint32_t)E, id = at < g.pad ? 0u : at - g.pad;
            listed[u] = ((const LILY_GLOBAL Bits16*)(reinterpret_cast<const char*>(a.touched) + (id >> 3)))->v >> (id & 7u);
        }
#pragma unroll
        for (int u = 0; u < C; ++u) {
            todo |= (inside(u) ? listed[u] & EMASK : 0u) << (u * E);
        }
    }
    float v[V];
#pragma unroll
    for (int u = 0; u < C; ++u) {
        float x[E];
        unpack<DT>(raw[u], x);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            v[u * E + j] = inside(u) && x[j] > NEG_INF ? x[j] : NEG_INF;   // (a NaN is worth -inf)
        }
    }
    // The listed ids' true values, one of every chunk at a time with their loads in flight together.
    while (__ballot(todo != 0u) != 0ull) {
        uint32_t at[C], count[C];
        float x[C];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const uint32_t m = (todo >> (u * E)) & EMASK;
            at[u] = m != 0u ? (uint32_t)__builtin_ctz(m) : 0xffu;
            todo &= ~((m & (0u - m)) << (u * E));
            const uint32_t id = m != 0u ? g.id_of(chunk_of(u), (int)at[u]) : 0u;
            x[u] = load_logit<DT>(a.logits, id);
            count[u] = gload(a.counts + id);
        }
#pragma unroll
        for (int u = 0; u < C; ++u) {
            float t = x[u];
            if (count[u] > 0u) {
                t = t > 0.0f ? t / a.repetition : t * a.repetition;
                t -= a.presence + a.frequency * (float)count[u];
            }
            t = t > NEG_INF ? t : NEG_INF;
#pragma unroll
            for (int j = 0; j < E; ++j) {
                v[u * E + j] = at[u] == (uint32_t)j ? t : v[u * E + j];
            }
        }
    }
    float cm[C], lane_max = NEG_INF;
#pragma unroll
    for (int u = 0; u < C; ++u) {
        cm[u] = v[u * E];
#pragma unroll
        for (int j = 1; j < E; ++j) {
            cm[u] = fmaxf(cm[u], v[u * E + j]);
        }
        lane_max = fmaxf(lane_max, cm[u]);
    }
    // Ids of partial chunks at the row's ends, one a thread (fewer than 16 at either end).
    uint32_t edge = 0xffffffffu;
    float ev = NEG_INF;
    if (tid < 64u) {
        edge = g.id_lo + tid < g.edge_lo_end ? g.id_lo + tid : edge;
    } else if (tid < 128u) {
        edge = g.edge_hi_begin + tid - 64u < g.id_hi ? g.edge_hi_begin + tid - 64u : edge;
    }
    if (edge != 0xffffffffu) {
        ev = load_logit<DT>(a.logits, edge);
        ev = pen ? wide_worth(a, ev, edge) : ev;
        ev = ev > NEG_INF ? ev : NEG_INF;
        lane_max = fmaxf(lane_max, ev);
    }
    if (THREADS != NT) {
        // (four threads' values are a lane's of the four waves that name keys)
        float* maxima = reinterpret_cast<float*>(dyn_lds);
        maxima[tid] = lane_max;
        __syncthreads();
        float m = NEG_INF;
        if (tid < NT) {
            for (uint32_t i = 0; i < THREADS; i += NT) {
                m = fmaxf(m, maxima[tid + i]);
            }
        }
        lane_max = m;
    }
    WIDE_MARK(1);
    // ---- the slice's keys: 0 stands for those that are not there yet
    uint64_t* bounds = w.bounds + (size_t)row * MAX_SLICES;
    const uint64_t own_keys = slice_keys_of(lane_max, a.k, S, sh);
    if (tid == 0) {
        store_through(bounds + s, own_keys);
    }
    if (want_lse) {
        LseAcc lse;
        lse.init();
#pragma unroll
        for (int u = 0; u < C; ++u) {
            if (cm[u] > NEG_INF) {
                const float safe = lse.rebase(cm[u], a.c2);
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    if (v[u * E + j] > NEG_INF) {
                        lse.term(v[u * E + j], a.c2, safe);
                    }
                }
            }
        }
        if (ev > NEG_INF) {
            lse.add_one(ev, a.c2);
        }
        // (as lse_reduce(), whatever the number of waves)
        const float m_w = wave_max_dpp(lse.mc);
        const double s_w = wave_sum_d(lse.mc > NEG_INF ? (double)lse.s * exp2((double)lse.mc - (double)m_w) : 0.0);
        if (lane == 0u) {
            wave_m[tid >> 6] = m_w;
            wave_s[tid >> 6] = s_w;
        }
        __syncthreads();
        if (tid < 64u) {
            const float m_l = lane < THREADS / 64u ? wave_m[lane] : NEG_INF;
            const float m = wave_max_dpp(m_l);
            const double all = wave_sum_d(m_l > NEG_INF ? wave_s[lane] * exp2((double)m_l - (double)m) : 0.0);
            if (lane == 0u) {
                const size_t slot = (size_t)row * S + s;
                handed_store(cfg.ws_lse, 2 * slot, (double)m);
                handed_store(cfg.ws_lse, 2 * slot + 1, all);
            }
        }
    }
    WIDE_MARK(2);
    // ---- the row's bound, once all its slices' words are there (a word is the message: nothing else is read for it)
    auto wait_for = [&](const uint64_t* words, uint32_t looks) {
        if (tid < 64u) {   // (the first wave looks)
            uint64_t keys = 0;
            for (uint32_t tries = 0;; ++tries) {
                if (tries == looks) {
                    if (lane == 0u) {
                        lost = 1u;
                    }
                    break;
                }
                keys = lane < S ? load_through(words + lane) : ~0ull;
                if (__ballot(keys == 0ull) == 0ull) {
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            const float b = bound_of_keys(lane < S ? keys : 0ull, a.k, S);
            if (lane == 0u) {
                row_bound = b;
            }
        }
        __syncthreads();
    };
    wait_for(bounds, w.looks.keys);
    float bound = row_bound;
    if (lost == 0u && !(bound > F32_LOWEST)) {
        // (the same in all the row's workgroups) Most of the row is -inf: too many waves had no value to name.  The lanes'
        // maxima change hands, and the bound is the k-th largest of those.
        if (tid < NT) {
            handed_store(w.lane_max, ((size_t)row * S + s) * NT + tid, lane_max);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        uint64_t* handed = bounds + (size_t)gridDim.y * MAX_SLICES;
        if (tid == 0) {
            __hip_atomic_store(handed + s, (uint64_t)1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
        wait_for(handed, w.looks.maxima);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        uint32_t T = 0;
        for (uint32_t t = 0x8000u; t != 0u && lost == 0u; t >>= 1) {
            if (tid == 0) {
                sh.hist[0] = 0;
            }
            __syncthreads();
            uint32_t n = 0;
            for (uint32_t j0 = 0; tid < NT && j0 < S; j0 += 8u) {
                float x[8];
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u) {
                    x[u] = handed_load(w.lane_max, ((size_t)row * S + min(j0 + u, S - 1u)) * NT + tid);
                }
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u) {
                    const bool reaches = j0 + u < S && x[u] > NEG_INF && (lilym_order_key(x[u]) >> 16) >= (T | t);
                    n += (uint32_t)__popcll(__ballot(reaches));
                }
            }
            if (lane == 0u) {
                atomicAdd(&sh.hist[0], n);
            }
            __syncthreads();
            T |= sh.hist[0] >= a.k ? t : 0u;
            __syncthreads();
        }
        bound = T > WIDE_LEAST_KEY ? lower_by_slack(lilym_key_value(T << 16)) : F32_LOWEST;
    }
    WIDE_MARK(5);
    uint64_t* cand = THREADS == NT ? dyn_lds : dyn_lds + SIXTEEN_OFF_PLACED;
    auto offer = [&](float x, uint32_t id) {
        if (x >= bound && x > NEG_INF) {
            const uint32_t at = atomicAdd(&n_mine, 1u);
            if (at < MERGE_CAP) {
                cand[at] = composite_of(x / a.temperature, id);
            }
        }
    };
#pragma unroll
    for (int u = 0; u < C; ++u) {
        if (cm[u] >= bound) {
#pragma unroll
            for (int j = 0; j < E; ++j) {
                offer(v[u * E + j], g.id_of(chunk_of(u), j));
            }
        }
    }
    offer(ev, edge);   // (-inf where there is none)
    __syncthreads();
    wide_finish<DT, LSE, THREADS, true>(wide_table<INLINE>(cfg) + row, cfg, w, sh, n_mine, cand, row, S, bound, lost != 0u, six);
}

template <int DT, bool LSE, bool INLINE>
static hipError_t launch_wide_variant(hipStream_t stream, uint32_t rows, const LaunchCfg& cfg,
                                      const InlineRows* inline_rows, const WideArgs& w) {
    const dim3 grid(cfg.slices, rows), block(NT);
    static const InlineRows none = {};
    const InlineRows& r = inline_rows != nullptr ? *inline_rows : none;
    const size_t dyn2 = (size_t)cfg.dyn_slots * 8;
    if (w.bounds != nullptr) {
        if (rows * cfg.slices <= WIDE_SIXTEEN_GROUPS) {
            hipLaunchKernelGGL((k_wide_held<DT, LSE, INLINE, SIXTEEN_THREADS>), grid, dim3(SIXTEEN_THREADS), SIXTEEN_LDS_BYTES, stream, r, cfg, w);
        } else {
            hipLaunchKernelGGL((k_wide_held<DT, LSE, INLINE, NT>), grid, block, dyn2, stream, r, cfg, w);
        }
        return hipGetLastError();
    }
    hipLaunchKernelGGL((k_wide_bound<DT, LSE, INLINE>), grid, block, 0, stream, r, cfg, w);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL((k_wide_draw<DT, LSE, INLINE>), grid, block, dyn2, stream, r, cfg, w);
    return hipGetLastError();
}

hipError_t launch_rows_wide(hipStream_t stream, int dtype, bool lse, uint32_t rows, const LaunchCfg& cfg_in,
                            const InlineRows* inline_rows, float* lane_max, uint32_t* count, uint64_t* bounds,
                            const WideLooks& looks) {
    LaunchCfg cfg = cfg_in;
    // the merging workgroup's candidates, then the tail's arrays behind the first K_CAP of them
    cfg.dyn_slots = MERGE_CAP;
    cfg.cand_cap = MERGE_CAP;
    WideArgs w;
    w.lane_max = Handed<float>{lane_max};
    w.slice_keys = Handed<uint64_t>{reinterpret_cast<uint64_t*>(lane_max + (size_t)rows * cfg.slices * NT)};   // (behind the lanes' maxima)
    w.lanes = (uint64_t)cfg.slices * (NT / 2) >= 4ull * cfg.ws_k ? NT / 2 : NT;
    w.count = count;
    w.looks = looks;
    // One launch where every slice is held in registers, wherever its row starts, and the launch's workgroups are all on
    // the chip at once (four a compute unit: they wait for each other).
    const uint32_t e = dtype == LILY_BF16 ? 8u : 4u, nch = (cfg.vocab + 2u * (e - 1u)) / e;
    const bool held = (nch + cfg.slices - 1u) / cfg.slices <= NT * STREAM_UNROLL && (uint64_t)rows * cfg.slices <= WIDE_HELD_GROUPS;
    w.bounds = held ? bounds : nullptr;
    const bool inl = inline_rows != nullptr;
#define LILY_WIDE(DT)                                                                               \
    (lse ? (inl ? launch_wide_variant<DT, true, true>(stream, rows, cfg, inline_rows, w)            \
                : launch_wide_variant<DT, true, false>(stream, rows, cfg, inline_rows, w))          \
         : (inl ? launch_wide_variant<DT, false, true>(stream, rows, cfg, inline_rows, w)           \
                : launch_wide_variant<DT, false, false>(stream, rows, cfg, inline_rows, w)))
    return dtype == LILY_BF16 ? LILY_WIDE(LILY_BF16) : LILY_WIDE(LILY_F32);
#undef LILY_WIDE
}

}  // namespace lily
