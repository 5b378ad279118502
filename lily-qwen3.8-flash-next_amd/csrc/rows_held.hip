// rows_held.hip - rows of few candidates (k <= 64) in slices that a workgroup holds in registers.
// Compiled once per (logits type, blocks a slice): -DLILY_DT=0|1 -DLILY_BLOCKS=1|2.
//
// The streaming selects (select_stream.h, select_lowering.h) are made for slices of many blocks: a
// bound that moves, chunks queued by their raw values, listed ids and sums settled behind the scan,
// a check of the whole at the end.  A slice of one or two blocks is over before any of that pays.
// Here each thread keeps its 16 to 64 values, turns the few that bias list, mask or penalties touch
// into their true ones where they lie, and from there on every row is a plain one: the bound is one of
// true values, what reaches it is listed once, and nothing can fail but the list's place (ties by
// the thousand), where the exhaustive select takes over.  Ids that are admitted, or likely, in clusters
// fill some waves and leave others nothing: the bound then comes from the chunks of 16 bytes (64 bf16 rows of 50 257, k = 50,
// 30 % admitted in runs of 128: 27 us, 85 streamed; 4 rows under penalties, 1 000 neighbours 9 above the rest, 18.5 and 90.
// With the waves' bounds alone such slices were given up: 333 and 98).
#include <type_traits>

#include "launch.h"
#include "row_kernel.h"

#if !defined(LILY_DT) || !defined(LILY_BLOCKS)
#error "compile with -DLILY_DT=<lily_dtype> -DLILY_BLOCKS=<1|2>"
#endif

namespace lily {

namespace {

constexpr uint32_t HELD_SEG = 512;                  // values a wave lists
constexpr uint32_t HELD_CAP = HELD_SEG * NWAVE;
// Dynamic LDS: the listed (value, id) pairs, then the ranked candidates; the merge of a row's slices
// and the tail begin at the front again.
constexpr uint32_t HELD_LDS_BYTES = LILY_SAMPLE_K_CAP * 8 + 3 * LILY_SAMPLE_K_CAP * 4;
static_assert(HELD_MERGE_SLOTS == WAVE_MERGE_SLOTS, "held rows: what one wave merges");
static_assert(HELD_LDS_BYTES >= (HELD_CAP + 64 + NT + NT / 4) * 8 && HELD_LDS_BYTES >= WAVE_MERGE_SLOTS * 8, "held rows: LDS layout");

// Workgroups a compute unit shall hold: by the registers that the values take.
template <int DT, int NB>
constexpr int HELD_RESIDENT = NB * Geo<DT>::E <= 8 ? 4 : 3;

// Bias lists of a launch's rows, and which of a thread's values they touch.
struct HeldBias {
    uint32_t id[STREAM_BIAS_CAP];
    float delta[STREAM_BIAS_CAP];
    uint32_t of_thread[NT][2];
};

// EXTRA: rows with a mask or a bias list are among the launch's.  True in the wave that finished the row.
template <int DT, int NB, bool LSE, bool EXTRA, bool SPEC>
__device__ __forceinline__ bool held_row(const LILY_CONST RowArgs* src, const LaunchCfg& cfg, Shared& sh, HeldBias* bias_lds) {
    if (cfg.served != nullptr && *(const LILY_CONST uint32_t*)(cfg.served + blockIdx.y) != 0u) {
        return false;
    }
    constexpr int E = Geo<DT>::E, C = NB * (int)STREAM_UNROLL, V = C * E;
    using Mask = std::conditional_t<(V > 32), uint64_t, uint32_t>;   // a bit per value
    constexpr uint32_t EMASK = (1u << E) - 1u;
    RowArgs a;
    load_row_args(a, src);
    apply_selection(a);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t s = blockIdx.x, row = blockIdx.y, S = cfg.slices, vocab = cfg.vocab;
    const uint32_t step = a.step + cfg.step_delta;
    const bool want_lse = LSE && a.out_logprob != nullptr;
    const bool forced = (a.flags & F_FORCED) != 0u;
    if (forced && !want_lse) {
        if (s == 0 && tid == 0) {
            emit(a, a.forced, vocab);
        }
        return s == 0 && w == 0;
    }
    // (a draft's distribution may be longer than the one-wave draw takes: the workgroup stays then)
    const bool by_workgroup = SPEC && a.mode == MODE_SPEC && *a.q_n > 64u;
    Geo<DT> g;
    g.init(a.logits, vocab, s, S);
    phase(cfg, 0);

    // ---- everything the slice is made of, asked for at once
    const uint32_t c_last = g.ce - 1u;
    auto chunk_of = [&](int u) -> uint32_t { return g.cb + (uint32_t)u * NT + tid; };
    u32x4 raw[C];
#pragma unroll
    for (int u = 0; u < C; ++u) {
        raw[u] = gload(reinterpret_cast<const u32x4*>(g.base + (min(chunk_of(u), c_last) << 4)));   // (rows are below 4 GiB)
    }
    // Ids of partial chunks at the row's ends, one a thread (fewer than 16 at either end).
    uint32_t edge = 0xffffffffu;
    if (tid < 64u) {
        edge = g.id_lo + tid < g.edge_lo_end ? g.id_lo + tid : edge;
    } else if (tid < 128u) {
        edge = g.edge_hi_begin + tid - 64u < g.id_hi ? g.edge_hi_begin + tid - 64u : edge;
    }
    float ev = load_logit<DT>(a.logits, edge != 0xffffffffu ? edge : 0u);
    // The chunks' bits of the bitmap of listed ids: two bytes hold a chunk's, wherever the row starts
    // (a byte past the bitmap is the scratch's own; a chunk before the row's first id is no streamed one).
    const bool pen = (a.flags & F_PEN) != 0u;
    uint32_t listed_raw[C];
    struct Bits16 {
        uint16_t v;
    } __attribute__((packed));
    auto first_id = [&](int u) -> uint32_t {
        const uint32_t at = min(chunk_of(u), c_last) * (uint32_t)E;
        return at < g.pad ? 0u : at - g.pad;
    };
    if (pen) {
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const uint32_t id = first_id(u);
            listed_raw[u] = ((const LILY_GLOBAL Bits16*)(reinterpret_cast<const char*>(a.touched) + (id >> 3)))->v >> (id & 7u);
        }
    }
    const bool masked = EXTRA && a.allow != nullptr;
    const uint32_t row_words = (vocab + 31u) / 32u;
    uint32_t allow_lo[EXTRA ? C : 1], allow_hi[EXTRA ? C : 1];
    if (masked) {
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const uint32_t wi = first_id(u) >> 5;
            allow_lo[EXTRA ? u : 0] = gload(a.allow + min(wi, row_words - 1u));
            allow_hi[EXTRA ? u : 0] = gload(a.allow + min(wi + 1u, row_words - 1u));
        }
    }
    const uint32_t n_bias = EXTRA ? min(a.n_bias, STREAM_BIAS_CAP) : 0u;
    if (EXTRA && n_bias != 0u) {
        bias_lds->of_thread[tid][0] = 0u;
        bias_lds->of_thread[tid][1] = 0u;
        uint32_t id = 0xffffffffu;
        if (tid < n_bias) {
            id = gload(&a.bias[tid].id);
            bias_lds->id[tid] = id;
            bias_lds->delta[tid] = gload(&a.bias[tid].delta);
        }
        __syncthreads();
        if (tid < n_bias && id < vocab) {
            const uint32_t c = (id + g.pad) / (uint32_t)E;
            if (c >= g.main_lo && c < g.main_hi) {
                const uint32_t bit = (c - g.cb) / NT * (uint32_t)E + (id + g.pad) % (uint32_t)E;
                atomicOr(&bias_lds->of_thread[(c - g.cb) % NT][bit >> 5], 1u << (bit & 31u));
            }
        }
        __syncthreads();
    }
    // The oracle's map of a raw value: the bias list in its order, the penalties of `count` emissions.
    auto true_value = [&](uint32_t id, float x, bool biased, uint32_t count) -> float {
        if (EXTRA && biased) {
            for (uint32_t j = 0; j < n_bias; ++j) {
                if (bias_lds->id[j] == id) {
                    x += bias_lds->delta[j];
                }
            }
        }
        if (count > 0u) {
            x = x > 0.0f ? x / a.repetition : x * a.repetition;
            x -= a.presence + a.frequency * (float)count;
        }
        return x;
    };
    phase(cfg, 1);

    // ---- the values
    const bool whole = g.cb >= g.main_lo && g.cb + C * NT <= g.main_hi;   // every chunk is streamed
    auto inside = [&](int u) -> bool { return chunk_of(u) >= g.main_lo && chunk_of(u) < g.main_hi; };
    float v[V];
#pragma unroll
    for (int u = 0; u < C; ++u) {
        float x[E];
        if (!whole && !inside(u)) {
            const uint32_t ninf = DT == LILY_BF16 ? 0xff80ff80u : 0xff800000u;
            raw[u] = u32x4{ninf, ninf, ninf, ninf};
        }
        unpack<DT>(raw[u], x);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            v[u * E + j] = x[j];
        }
    }
    Mask todo = 0, allowed = ~(Mask)0, biased = 0;
    if (pen) {
#pragma unroll
        for (int u = 0; u < C; ++u) {
            todo |= (Mask)(whole || inside(u) ? listed_raw[u] & EMASK : 0u) << (u * E);
        }
    }
    if (EXTRA && n_bias != 0u) {
        biased = (Mask)bias_lds->of_thread[tid][0];
        if (V > 32) {
            biased |= (Mask)((uint64_t)bias_lds->of_thread[tid][1] << 32);
        }
        todo |= biased;
    }
    if (masked) {
        allowed = 0;
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const uint64_t two = ((uint64_t)allow_hi[EXTRA ? u : 0] << 32) | allow_lo[EXTRA ? u : 0];
            allowed |= (Mask)((uint32_t)(two >> (first_id(u) & 31u)) & EMASK) << (u * E);
        }
        todo &= allowed;
    }
    // The values that something touches, one of every chunk at a time with all their loads in flight
    // together (the raw value comes once more: it is nearer there than a register whose number is not
    // known).  A chunk rarely holds a second one.
    while (__ballot(todo != 0) != 0ull) {
        uint32_t at[C], id[C], count[C];
        float x[C];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const uint32_t m = (uint32_t)(todo >> (u * E)) & EMASK;
            at[u] = m != 0u ? (uint32_t)__builtin_ctz(m) : 0xffu;
            todo &= ~((Mask)(m & (0u - m)) << (u * E));
            id[u] = m != 0u ? chunk_of(u) * (uint32_t)E + at[u] - g.pad : 0u;
            x[u] = load_logit<DT>(a.logits, id[u]);
            count[u] = pen ? gload(a.counts + id[u]) : 0u;
        }
#pragma unroll
        for (int u = 0; u < C; ++u) {
            if (__ballot(at[u] != 0xffu) != 0ull) {
                const float t = true_value(id[u], x[u], EXTRA && ((biased >> (u * E + (int)(at[u] % (uint32_t)E))) & 1) != 0, count[u]);
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    v[u * E + j] = at[u] == (uint32_t)j ? t : v[u * E + j];
                }
            }
        }
    }
    if (masked) {
#pragma unroll
        for (int j = 0; j < V; ++j) {
            v[j] = ((allowed >> j) & 1) != 0 ? v[j] : NEG_INF;
        }
    }
    if (edge != 0xffffffffu) {
        ev = true_value(edge, ev, n_bias != 0u, pen ? gload(a.counts + edge) : 0u);
        ev = !masked || bit_of(a.allow, edge) ? ev : NEG_INF;
    } else {
        ev = NEG_INF;
    }

    // ---- the bound: k values reach the least of the waves' ceil(k / NWAVE)-th largest lane maxima
    float cm[C], lane_max = ev > NEG_INF ? ev : NEG_INF;
#pragma unroll
    for (int u = 0; u < C; ++u) {
        cm[u] = max2_raw(max3_raw(v[u * E], v[u * E + 1], v[u * E + 2]), v[u * E + 3]);
        if (E == 8) {
            cm[u] = max2_raw(max3_raw(cm[u], v[u * E + 4 % E], v[u * E + 5 % E]), max2_raw(v[u * E + 6 % E], v[u * E + 7 % E]));
        }
        lane_max = max2_raw(lane_max, cm[u]);
    }
    const uint32_t kw = (min(a.k, 64u * NWAVE) + NWAVE - 1u) / NWAVE;
    const uint32_t P = wave_kth_key16(lane_max > NEG_INF ? (lilym_order_key(lane_max) >> 16) : 0u, kw);
    const float wave_top = LSE && want_lse ? wave_max_dpp(lane_max) : 0.0f;
    if (lane == 0u) {
        sh.bound[0][w] = P != 0u ? lilym_key_value(P << 16) : F32_LOWEST;
        sh.wmax[0][w] = wave_top;
    }
    __syncthreads();
    float T = sh.bound[0][0], top = sh.wmax[0][0];
    for (int i = 1; i < NWAVE; ++i) {
        T = fminf(T, sh.bound[0][i]);
        top = fmaxf(top, sh.wmax[0][i]);
    }
    // The k-th largest of the chunks' largest values, of all the waves' (which all call) or of this one's; F32_LOWEST where
    // fewer than k have one.
    auto chunks_bound = [&](bool all) -> float {
        uint32_t key[C], found = 0;
#pragma unroll
        for (int u = 0; u < C; ++u) {
            key[u] = cm[u] > NEG_INF ? lilym_order_key(cm[u]) >> 16 : 0u;
        }
        // (the first look: whether k have any)
#pragma unroll 1
        for (int bit = 16; bit >= 0; --bit) {
            const uint32_t at = bit == 16 ? 1u : found | (1u << bit);
            uint32_t reach = 0;
#pragma unroll
            for (int u = 0; u < C; ++u) {
                reach += (uint32_t)__popcll(__ballot(key[u] >= at));
            }
            if (all) {
                uint32_t* counts = sh.hist + (bit & 1) * NWAVE;   // (a barrier lies between a place's readers and its next writer)
                if (lane == 0u) {
                    counts[w] = reach;
                }
                __syncthreads();
                reach = counts[0];
                for (int i = 1; i < NWAVE; ++i) {
                    reach += counts[i];
                }
            }
            if (bit == 16) {
                if (reach < a.k) {
                    break;
                }
            } else {
                found = reach >= a.k ? at : found;
            }
        }
        return found != 0u ? lilym_key_value(found << 16) : F32_LOWEST;
    };
    if (__builtin_expect(T == F32_LOWEST && !forced, 0)) {   // (what is rare lies behind the rest: 9.95 -> 9.86 us for one row)
        // Masks, rows that are mostly -inf: a wave with fewer values than its share.
        T = chunks_bound(true);
    }
    // (values a little below the bound may share its quotient by the temperature)
    T = forced ? __builtin_huge_valf() : lower_by_slack(T);
    // Where the bound of the poorest wave lets clusters through whole: the k-th largest of a wave's own chunks is a bound too,
    // which k of them reach, ties aside, and that much has its place.
    uint32_t reaching = 0;
#pragma unroll
    for (int u = 0; u < C; ++u) {
        reaching += (uint32_t)__popcll(__ballot(cm[u] >= T));
    }
    if (__builtin_expect(reaching > 64u, 0)) {
        T = fmaxf(T, lower_by_slack(chunks_bound(false)));   // (this wave's from here on)
    }
    phase(cfg, 2);

    // ---- what reaches it is listed, the rest goes into the sum
    // Finite and far from overflow: every term is formed as 2^(x * c2 - ref).
    const float ref = top > NEG_INF ? fminf(fmaxf(top * a.c2, -1.0e30f), 1.0e30f) : 0.0f;
    uint64_t* pairs = dyn_lds;             // [NWAVE][HELD_SEG]: value's bits << 32 | id
    uint64_t* ranked = dyn_lds + HELD_CAP;
    uint32_t fill = 0;                     // this wave's
    auto list = [&](bool pass, float x, uint32_t id) {
        const uint64_t mask = __ballot(pass);
        if (mask != 0ull) {
            const uint32_t at = fill + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            if (pass && at < HELD_SEG) {
                pairs[w * HELD_SEG + at] = ((uint64_t)lilym_f32_bits(x) << 32) | id;
            }
            fill += (uint32_t)__popcll(mask);
        }
    };
    // A chunk's terms in f32, the chunks' sums in double.
    auto power = [&](float x) -> float { return __builtin_amdgcn_exp2f(__builtin_fmaf(x, a.c2, -ref)); };
    auto chunk_sum = [&](int u, auto&& keep) -> float {
        float e[E];
#pragma unroll
        for (int j = 0; j < E; ++j) {
            e[j] = power(keep(v[u * E + j]) ? v[u * E + j] : NEG_INF);
        }
        const float low = (e[0] + e[1]) + (e[2] + e[3]);
        return E == 8 ? low + ((e[4 % E] + e[5 % E]) + (e[6 % E] + e[7 % E])) : low;
    };
    double sum = 0.0;
#pragma unroll
    for (int u = 0; u < C; ++u) {
        const bool some = __ballot(cm[u] >= T) != 0ull;
        if (some) {
#pragma unroll
            for (int j = 0; j < E; ++j) {
                list(v[u * E + j] >= T, v[u * E + j], chunk_of(u) * (uint32_t)E + (uint32_t)j - g.pad);
            }
        }
        if (LSE && want_lse) {
            sum += (double)(some ? chunk_sum(u, [&](float x) { return !(x >= T); }) : chunk_sum(u, [](float) { return true; }));
        }
    }
    if (__ballot(edge != 0xffffffffu) != 0ull) {
        list(ev >= T, ev, edge);
        if (LSE && want_lse) {
            sum += (double)power(ev >= T ? NEG_INF : ev);
        }
    }
    if (LSE && want_lse) {
        if (__ballot(sum != sum) != 0ull) {
            // (a NaN counts as -inf)
            sum = 0.0;
#pragma unroll
            for (int u = 0; u < C; ++u) {
                sum += (double)chunk_sum(u, [&](float x) { return x < T; });
            }
            sum += (double)power(ev < T ? ev : NEG_INF);
        }
        const double all = wave_sum_d(sum);
        if (lane == 0u) {
            sh.red_d[w] = all;
        }
    }
    if (lane == 0u) {
        sh.qfill[w] = fill;
    }
    __syncthreads();
    phase(cfg, 8);
    uint32_t n = 0;
    bool overflow = false;
    uint32_t ends[NWAVE];   // of the waves' segments, as one list
    for (int i = 0; i < NWAVE; ++i) {
        n += sh.qfill[i];
        ends[i] = n;
        overflow = overflow || sh.qfill[i] > HELD_SEG;
    }
    if (cfg.path_stats != nullptr && tid == 0u) {
        atomicAdd(&cfg.path_stats[overflow ? 2 : 0], 1u);
    }
    auto pair_at = [&](uint32_t i) -> uint64_t {
        const uint32_t seg = (i >= ends[0] ? 1u : 0u) + (i >= ends[1] ? 1u : 0u) + (i >= ends[2] ? 1u : 0u);
        const uint32_t from = seg == 0u ? 0u : seg == 1u ? ends[0] : seg == 2u ? ends[1] : ends[2];
        return pairs[seg * HELD_SEG + i - from];
    };
    const double c2d = (double)a.c2;
    // (a listed value's term, in double: these carry most of the sum)
    auto term = [&](float x) -> double {
        const double d = __builtin_fma((double)x, c2d, -(double)ref);
        return d > -1000.0 ? pow2_d(d < 900.0 ? d : 900.0) : 0.0;
    };
    double listed_sum = 0.0;
    // The slice's whole sum, by the first wave.
    auto keep_sum = [&]() {
        if (LSE && want_lse) {
            for (int i = 0; i < NWAVE; ++i) {
                listed_sum += sh.red_d[i];
            }
            if (lane == 0u) {
                sh.lse_mc = (double)ref;
                sh.lse_s = listed_sum;
            }
        }
    };
    uint64_t c = 0ull;      // a candidate per lane of the first wave, in order
    if (!overflow && n <= 64u) {
        if (w != 0u && !by_workgroup) {
            return false;
        }
        if (w == 0u) {
            const uint64_t p = lane < n ? pair_at(lane) : 0ull;
            const float x = lilym_bits_f32((uint32_t)(p >> 32));
            c = lane < n ? composite_of(x / a.temperature, (uint32_t)p) : 0ull;
            c = wave_sort_desc(c);
            if (LSE && want_lse) {
                listed_sum = wave_sum_d(lane < n ? term(x) : 0.0);
            }
        }
    } else if (!overflow && n <= NT) {
        // Up to four waves' worth (k from 40 on, masks): up to two waves' two threads an entry, each counts what it has ahead
        // of it in one half of the list, sixteen at a time; else a thread an entry.
        const bool two = n <= NT / 2u;
        const uint32_t entry = two ? tid & (NT / 2u - 1u) : tid, half = two ? tid / (NT / 2u) : 0u;
        const uint64_t p = entry < n ? pair_at(entry) : 0ull;
        const float x = lilym_bits_f32((uint32_t)(p >> 32));
        const uint64_t mine = entry < n ? composite_of(x / a.temperature, (uint32_t)p) : 0ull;
        uint64_t* all = ranked + 64;   // [NT], then each entry's count in the upper half
        uint32_t* upper = reinterpret_cast<uint32_t*>(all + NT);
        if (half == 0u) {
            all[entry] = mine;
        }
        if (w == 3u) {
            ranked[lane] = 0ull;
        }
        if (LSE && want_lse) {
            listed_sum = wave_sum_d(half == 0u && entry < n ? term(x) : 0.0);
            if (lane == 0u) {
                sh.red3[0][w] = listed_sum;
            }
        }
        __syncthreads();
        uint32_t ahead = 0;
        const uint32_t to = two ? min(n, half * 64u + 64u) : n;
        for (uint32_t i = half * 64u; i < to; i += 16u) {
            uint64_t other[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                other[q] = all[i + (uint32_t)q];
            }
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                ahead += other[q] > mine ? 1u : 0u;
            }
        }
        if (half == 1u) {
            upper[entry] = ahead;
        }
        __syncthreads();
        if (half == 0u && mine != 0ull) {
            ahead += two ? upper[entry] : 0u;
            if (ahead < 64u) {
                ranked[ahead] = mine;
            }
        }
        __syncthreads();
        if (w != 0u && !by_workgroup) {
            return false;
        }
        c = w == 0u ? ranked[lane] : 0ull;
        if (LSE && want_lse) {
            listed_sum = 0.0;
            for (int i = 0; i < NWAVE; ++i) {
                listed_sum += sh.red3[0][i];
            }
        }
    } else {
        // More than that: masks that leave whole waves without a value, ties.
        if (!overflow) {
            constexpr int PER = HELD_CAP / NT;
            uint64_t mine[PER];
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const uint32_t i = tid + (uint32_t)q * NT;
                const uint64_t p = i < n ? pair_at(i) : 0ull;
                const float x = lilym_bits_f32((uint32_t)(p >> 32));
                mine[q] = i < n ? composite_of(x / a.temperature, (uint32_t)p) : 0ull;
                if (LSE && want_lse && i < n) {
                    listed_sum += term(x);
                }
            }
            if (LSE && want_lse) {
                listed_sum = wave_sum_d(listed_sum);
                if (lane == 0u) {
                    sh.red3[0][w] = listed_sum;
                }
            }
            __syncthreads();   // (the pairs have been read)
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                if (tid + (uint32_t)q * NT < n) {
                    pairs[tid + (uint32_t)q * NT] = mine[q];
                }
            }
            __syncthreads();
        } else {
            // Ties by the thousand.  (From the row itself: by now the values' registers are free.)
            select_exhaustive<DT>(a, g.id_lo, g.id_hi, a.k, want_lse, pairs, 64u, sh);
            n = min(sh.n_cand, 64u);
        }
        bool sorted = false;
        n = select_topk(pairs, n, a.k, sh, sorted);
        __syncthreads();
        if (w != 0u && !by_workgroup) {
            return false;
        }
        if (w == 0u) {
            c = wave_sort_desc(lane < n ? pairs[lane] : 0ull);
        }
        if (LSE && want_lse) {
            listed_sum = 0.0;
            for (int i = 0; i < NWAVE; ++i) {
                listed_sum += sh.red3[0][i];
            }
        }
    }
    c = lane < a.k ? c : 0ull;
    n = (uint32_t)__popcll(__ballot(c != 0ull));
    if (w == 0u && !overflow) {
        keep_sum();
    }
    phase(cfg, 4);

    // ---- the row
    if (SPEC && by_workgroup) {
        const size_t base = (size_t)row * S;
        if (S > 1u) {
            if (tid < cfg.ws_k) {   // (at most 64: the first wave)
                handed_store(cfg.ws_cand, (base + s) * cfg.ws_k + tid, c);
            }
            if (!last_to_arrive(&cfg.ws_ticket[row], S, sh.last, cfg.relaxed_handover != 0u)) {
                return false;
            }
            c = w == 0u ? merge_slices_by_wave(cfg, base, a.k) : 0ull;
            c = lane < a.k ? c : 0ull;
        }
        __syncthreads();
        if (tid == 0u) {
            tail_arrays(sh);
        }
        if (w == 0u) {
            dyn_lds[lane] = c;
            n = (uint32_t)__popcll(__ballot(c != 0ull));
            if (lane == 0u) {
                sh.n_cand = n;
            }
        }
        __syncthreads();
        tail<DT, false, true>(a, vocab, step, sh.n_cand, true, dyn_lds, sh, cfg);
        return w == 0u;
    }
    if (S > 1u) {
        ranked[lane] = c;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // (LDS of this wave: in order already)
        __builtin_amdgcn_wave_barrier();
        const bool finished = finish_by_wave<DT, LSE, SPEC>(a, cfg, row, s, n, ranked, step, want_lse, sh);
        if (finished) {
            phase(cfg, 7);
        }
        return finished;
    }
    if (forced) {
        if (lane == 0u) {
            finish_token<DT>(a, sh, a.forced, vocab);
        }
    } else if (n == 0u) {
        if (lane == 0u) {
            finish_empty(a, vocab, sh, cfg);
        }
    } else {
        uint32_t spec_d = 0, spec_qn = 0;
        if (SPEC && a.mode == MODE_SPEC) {
            spec_d = *a.draft;
            spec_qn = *a.q_n;
        }
        tail_wave<DT, SPEC>(a, vocab, step, c, n, sh, cfg, spec_d, spec_qn);
    }
    phase(cfg, 7);
    return true;
}

template <int DT, int NB, bool LSE, bool EXTRA>
__global__ __launch_bounds__(NT, (HELD_RESIDENT<DT, NB>)) void k_held_inline(InlineRows rows, LaunchCfg cfg) {
    __shared__ Shared sh;
    __shared__ HeldBias bias[1];
    const LILY_CONST RowArgs* table = (const LILY_CONST RowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    held_row<DT, NB, LSE, EXTRA, false>(table + blockIdx.y, cfg, sh, EXTRA ? bias : nullptr);
}

template <int DT, int NB, bool LSE, bool EXTRA>
__global__ __launch_bounds__(NT, (HELD_RESIDENT<DT, NB>)) void k_held_table(LaunchCfg cfg) {
    __shared__ Shared sh;
    __shared__ HeldBias bias[1];
    held_row<DT, NB, LSE, EXTRA, false>((const LILY_CONST RowArgs*)cfg.table + blockIdx.y, cfg, sh, EXTRA ? bias : nullptr);
}

// A verify pass whose rows are independent (see k_rows_verify).
template <int DT, int NB>
__global__ __launch_bounds__(NT, (HELD_RESIDENT<DT, NB>)) void k_held_verify(InlineRows rows, LaunchCfg cfg) {
    __shared__ Shared sh;
    const LILY_CONST RowArgs* table = (const LILY_CONST RowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    const bool finished = held_row<DT, NB, false, false, true>(table + blockIdx.y, cfg, sh, nullptr);
    if (!finished || threadIdx.x != 0u || cfg.accept_ctrl == nullptr) {
        return;
    }
    accept_behind_last_row(cfg, [&](uint32_t j) { return (table + j)->out_id; });
}

template <int DT, int NB, bool LSE, bool EXTRA>
hipError_t launch_held(hipStream_t stream, uint32_t rows, const LaunchCfg& cfg, const InlineRows* inline_rows) {
    const dim3 grid(cfg.slices, rows), block(NT);
    if (inline_rows != nullptr) {
        hipLaunchKernelGGL((k_held_inline<DT, NB, LSE, EXTRA>), grid, block, HELD_LDS_BYTES, stream, *inline_rows, cfg);
    } else {
        hipLaunchKernelGGL((k_held_table<DT, NB, LSE, EXTRA>), grid, block, HELD_LDS_BYTES, stream, cfg);
    }
    return hipGetLastError();
}

}  // namespace

#define LILY_CAT_(a, b, c, d) a##b##c##d
#define LILY_CAT(a, b, c, d) LILY_CAT_(a, b, c, d)

hipError_t LILY_CAT(launch_rows_held_dt, LILY_DT, _blocks, LILY_BLOCKS)(hipStream_t stream, bool lse, bool extra, uint32_t rows,
                                                                       const LaunchCfg& cfg, const InlineRows* inline_rows) {
    if (cfg.verify != 0u) {
        if (inline_rows == nullptr || lse || extra) {
            return hipErrorInvalidValue;   // (independent rows of a verify pass travel inline, plain ones)
        }
        hipLaunchKernelGGL((k_held_verify<LILY_DT, LILY_BLOCKS>), dim3(cfg.slices, rows), dim3(NT), HELD_LDS_BYTES, stream,
                           *inline_rows, cfg);
        return hipGetLastError();
    }
    if (lse) {
        return extra ? launch_held<LILY_DT, LILY_BLOCKS, true, true>(stream, rows, cfg, inline_rows)
                     : launch_held<LILY_DT, LILY_BLOCKS, true, false>(stream, rows, cfg, inline_rows);
    }
    return extra ? launch_held<LILY_DT, LILY_BLOCKS, false, true>(stream, rows, cfg, inline_rows)
                 : launch_held<LILY_DT, LILY_BLOCKS, false, false>(stream, rows, cfg, inline_rows);
}

}  // namespace lily
