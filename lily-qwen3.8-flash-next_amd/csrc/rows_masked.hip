// rows_masked.hip - rows under an allow-mask, a workgroup of 1 024 threads a row.  Compiled once per logits
// type: -DLILY_DT=0|1.
//
// A grammar admits some per cent of the vocabulary, or nearly all of it, and such rows name no top_k as a rule: 3 000
// ids to evaluate, 1 024 of them to sort.  That is a chain of latencies, not work to be spread: cut into
// four slices of 256 threads each row paid for a hand-over, a second gathering and a sort by one wave a
// SIMD (64 rows of 151 936 bf16, 2 % admitted: slices done 16 us, ticket 18, sorted 27, drawn 36).  Here
// sixteen waves read the mask, evaluate what it admits, sort in LDS, and the first four waves draw.
//
//   * Ids that lie scattered, up to 16 384: listed one by one, evaluated a lane each, sorted from the registers that
//     hold them.  (2 % admitted one by one, by words instead: 62 us for one row, 63 for 64; by ids 20 and 21.)
//   * Ids in clusters (12 and more to a word that admits any): the words are listed, 32 lanes a word; a run of ids is one
//     request, and nobody lists them (runs of up to 64: 23 us, by ids 26).  Each thread's words lie 1 024 apart, or a
//     cluster would be one thread's work.
//   * Clusters of more ids than the sort holds (8 192), in few words: histograms over the composites' leading bits, every value
//     evaluated anew for each, until what reaches the k-th one's bin fits.
//   * More: the row is streamed once, each piece's largest value kept in LDS (16 bits of it); from the threads' maxima
//     comes a bound as rows_wide.hip takes it, and the pieces that reach it are looked at again.  Where more reach it
//     than the sort holds (ties by the thousand), the histograms.
//
// us a launch, bf16, 151 936 ids, no top_k, 1 row / 64, the slices' kernels -> this one.  One by one: 0.2 % admitted 21.7 / 26.5 -> 13.2 / 14.5,
// 2 % 25.3 / 29.7 -> 20.0 / 21.1, 5 % 32.9 / 36.4 -> 27.9 / 30.8, 10 % 37.2 / 41.1 -> 42.0 / 42.8, 20 % 69.5 / 81.3 -> 48.4 / 50.4, all
// 73.2 / 85.6 -> 50.7 / 52.4.  In runs of up to 64: 0.2 % 22.3 / 26.2 -> 13.5 / 14.5, 2 % 26.4 / 33.1 -> 20.9 / 22.6, 10 % 41 / 473 -> 47.6 /
// 48.8, 20 % 68.8 / 80.9 -> 50.1 / 57.5.  One row in four under a mask of 97 %, the others of 2 %, 64 rows: 77 -> 52.
#include <type_traits>

#include "launch.h"
#include "row_kernel.h"
#include "sort_sixteen.h"

#if !defined(LILY_DT)
#error "compile with -DLILY_DT=<lily_dtype>"
#endif

namespace lily {

namespace {

constexpr uint32_t MT = SIXTEEN_THREADS, MWAVE = SIXTEEN_WAVES;
constexpr uint32_t MASKED_WORDS = MASKED_MAX_VOCAB / 32u, WORDS_PER = MASKED_WORDS / MT;
constexpr uint32_t MASKED_CAP = 8192;      // values that are sorted
constexpr uint32_t MASKED_LISTED = 2 * MASKED_CAP;   // ids that are listed
constexpr uint32_t MASKED_CLUSTERED = 12;  // ids a word of a mask in clusters, on average
// Words in clusters of more ids than the sort holds: so many are histogrammed, where that is the faster way (20 us and 0.03 a
// word; the row streamed 25 and 0.2 for every 1 000 ids of the vocabulary).
__device__ __forceinline__ uint32_t masked_few_words(uint32_t vocab) { return 350u + vocab / 170u; }
constexpr uint32_t MBINS = SIXTEEN_BINS;   // of the sort
constexpr uint32_t HBINS = 4096;           // of the histograms, 12 bits
// Dynamic LDS in 64-bit slots: the sorted candidates and the tail's arrays; the sort's bins; the values as they
// come (the histograms, before there are any); the words that admit anything (bits, number), and where those are
// done with the values by bins.  (A list of ids lies where the words would.)
constexpr uint32_t OFF_BINS = (LILY_SAMPLE_K_CAP * 8 + 3 * LILY_SAMPLE_K_CAP * 4) / 8;
constexpr uint32_t OFF_MIXED = OFF_BINS + MBINS / 2;
constexpr uint32_t OFF_PLACED = OFF_MIXED + MASKED_CAP;
constexpr uint32_t MASKED_LDS_BYTES = (OFF_PLACED + MASKED_CAP) * 8;
static_assert(MASKED_WORDS * 6 <= MASKED_CAP * 8 && HBINS * 4 <= MASKED_CAP * 8 && MASKED_MAX_VOCAB / 4 * 2 <= MASKED_CAP * 16 &&
                  MASKED_CAP * 2 <= OFF_BINS * 8, "masked rows: LDS layout");

struct MaskedShared {
    SixteenShared six;
    float wave_f[MWAVE];
    double wave_d[MWAVE];
    uint32_t n, bin, above, need, pieces;
    uint32_t bias_id[STREAM_BIAS_CAP];
    float bias_delta[STREAM_BIAS_CAP];
    uint32_t biased[MASKED_WORDS / 32];    // bit w: some pair names an id of word w
};

// A thread's sum of exponentials, as LseAcc with the sum in double: a thread adds up to 256 values one by one, and where one of them
// carries the row the others are each near half a step of it (a row of 248 320 whose best is worth 16.4 more than the rest:
// 1.0e-5 off in f32, in double 2e-8).
struct MaskedSum {
    float mc;
    double s;
    __device__ __forceinline__ void init() {
        mc = NEG_INF;
        s = 0.0;
    }
    __device__ __forceinline__ float rebase(float cm, float c) {
        const float mcn = fmaxf(mc, cm * c), safe = fmaxf(mcn, F32_LOWEST);
        s *= (double)__builtin_amdgcn_exp2f(mc - safe);
        mc = mcn;
        return safe;
    }
    __device__ __forceinline__ void term(float v, float c, float safe) { s += (double)__builtin_amdgcn_exp2f(__builtin_fmaf(v, c, -safe)); }
    __device__ __forceinline__ void add_one(float v, float c) {
        if (v > NEG_INF) {
            const float safe = rebase(v, c);
            term(v, c, safe);
        }
    }
};

template <int DT, bool LSE>
__device__ __forceinline__ void masked_row(const LILY_CONST RowArgs* src, const LaunchCfg& cfg, Shared& sh, MaskedShared& ms) {
    RowArgs a;
    load_row_args(a, src);
    apply_selection(a);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t vocab = cfg.vocab, words = (vocab + 31u) / 32u;
    const bool want_lse = LSE && a.out_logprob != nullptr;
    const bool forced = (a.flags & F_FORCED) != 0u, pen = (a.flags & F_PEN) != 0u;
    if (forced && !want_lse) {
        if (tid == 0) {
            emit(a, a.forced, vocab);
        }
        return;
    }
    phase(cfg, 0);
    uint64_t* mixed = dyn_lds + OFF_MIXED;
    uint64_t* placed = dyn_lds + OFF_PLACED;
    uint32_t* bins = reinterpret_cast<uint32_t*>(dyn_lds + OFF_BINS);
    uint32_t* hist = reinterpret_cast<uint32_t*>(mixed);
    uint32_t* word_bits = reinterpret_cast<uint32_t*>(placed);
    uint16_t* word_at = reinterpret_cast<uint16_t*>(word_bits + MASKED_WORDS);
    uint32_t* id_list = reinterpret_cast<uint32_t*>(placed);

    // ---- what the mask admits: its words, or its ids
    uint32_t bits[WORDS_PER], some = 0, admitted = 0;
    auto fetch_words = [&]() {
#pragma unroll
        for (uint32_t i = 0; i < WORDS_PER; ++i) {
            bits[i] = gload(a.allow + min(i * MT + tid, words - 1u));
        }
    };
    auto count_words = [&]() {
        some = 0;
        admitted = 0;
#pragma unroll
        for (uint32_t i = 0; i < WORDS_PER; ++i) {
            const uint32_t at = i * MT + tid;
            bits[i] = at < words ? bits[i] & range32_at(0u, vocab, (int64_t)at * 32) : 0u;
            some += bits[i] != 0u ? 1u : 0u;
            admitted += (uint32_t)__popc(bits[i]);
        }
    };
    auto list_words = [&](uint32_t place) {
#pragma unroll
        for (uint32_t i = 0; i < WORDS_PER; ++i) {
            if (bits[i] != 0u) {
                word_bits[place] = bits[i];
                word_at[place] = (uint16_t)(i * MT + tid);
                ++place;
            }
        }
    };
    fetch_words();
    if (tid == 0) {
        tail_arrays(sh);
        ms.n = 0u;
        ms.pieces = 0u;
        ms.bin = 0u;
    }
    const uint32_t n_bias = min(a.n_bias, STREAM_BIAS_CAP);
    if (tid < MASKED_WORDS / 32u) {
        ms.biased[tid] = 0u;
    }
    if (tid < n_bias) {
        ms.bias_id[tid] = gload(&a.bias[tid].id);
        ms.bias_delta[tid] = gload(&a.bias[tid].delta);
    }
    count_words();
    uint32_t n_words, total;
    const uint32_t place = scan_all(some, ms.six, n_words) - some;
    const uint32_t id_place = scan_all(admitted, ms.six, total) - admitted;
    if (tid < n_bias && ms.bias_id[tid] < vocab) {
        const uint32_t at = ms.bias_id[tid] >> 5;
        atomicOr(&ms.biased[at >> 5], 1u << (at & 31u));
    }
    const bool scattered = total < n_words * MASKED_CLUSTERED, listed = scattered && total <= MASKED_LISTED;
    const bool by_words = !scattered && (total <= MASKED_CAP || n_words <= masked_few_words(vocab));
    if (listed) {
        uint32_t to = id_place;
#pragma unroll
        for (uint32_t i = 0; i < WORDS_PER; ++i) {
            for (uint32_t left = bits[i]; left != 0u; left &= left - 1u) {
                id_list[to++] = (i * MT + tid) * 32u + (uint32_t)__builtin_ctz(left);
            }
        }
    } else if (by_words) {
        list_words(place);
    }
    __syncthreads();
    phase(cfg, 1);

    // An admitted value before the temperature.
    auto worth = [&](const RowArgs& a, float u, uint32_t id, bool biased, uint32_t count) -> float {
        if (__ballot(biased) != 0ull) {
            for (uint32_t j = 0; j < n_bias; ++j) {   // (pairs of one id in the list's order)
                u = ms.bias_id[j] == id ? u + ms.bias_delta[j] : u;
            }
        }
        if (count > 0u) {
            u = u > 0.0f ? u / a.repetition : u * a.repetition;
            u -= a.presence + a.frequency * (float)count;
        }
        return u;
    };
    auto has_bias = [&](uint32_t word) -> bool { return n_bias != 0u && ((ms.biased[word >> 5] >> (word & 31u)) & 1u) != 0u; };
    // fn(that value, id, whether there is one) over every admitted id: 32 lanes a word,
    // eight words' loads in flight.
    auto over_admitted = [&](auto&& fn) {
        constexpr uint32_t R = 8;
        for (uint32_t i0 = 0; i0 < n_words; i0 += R * (MT / 32u)) {
            uint32_t id[R], count[R];
            float x[R];
            bool in[R], biased[R];
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                const uint32_t i = i0 + r * (MT / 32u) + (tid >> 5);
                const uint32_t at = word_at[min(i, n_words - 1u)];
                in[r] = i < n_words && ((word_bits[min(i, n_words - 1u)] >> (tid & 31u)) & 1u) != 0u;
                id[r] = min(at * 32u + (tid & 31u), vocab - 1u);
                biased[r] = has_bias(at);
                x[r] = load_logit<DT>(a.logits, id[r]);
                count[r] = pen ? gload(a.counts + id[r]) : 0u;
            }
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                if (i0 + r * (MT / 32u) >= n_words) {
                    break;
                }
                fn(worth(a, x[r], id[r], biased[r], count[r]), id[r], in[r]);
            }
        }
    };
    // The same over the listed ids from `from` on, a lane each, all their loads in flight.
    auto over_listed = [&](uint32_t from, auto&& fn) {
        constexpr uint32_t R = MASKED_CAP / MT;
        uint32_t id[R], count[R];
        float x[R];
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
            id[r] = id_list[min(from + r * MT + tid, total - 1u)];
            x[r] = load_logit<DT>(a.logits, id[r]);
            count[r] = pen ? gload(a.counts + id[r]) : 0u;
        }
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
            if (from + r * MT < total) {
                fn(r, worth(a, x[r], id[r], has_bias(id[r] >> 5), count[r]), id[r], from + r * MT + tid < total);
            }
        }
    };
    MaskedSum lse;
    lse.init();
    auto collect = [&](uint64_t least, bool sum) {
        over_admitted([&](float u, uint32_t id, bool in) {
            if (sum && in) {
                lse.add_one(u, a.c2);
            }
            const uint64_t c = in ? composite_of(u / a.temperature, id) : 0ull;
            const uint64_t mask = __ballot(c != 0ull && c >= least);
            if (mask != 0ull && !forced) {
                uint32_t base = 0;
                if (lane == 0u) {
                    base = atomicAdd(&ms.n, (uint32_t)__popcll(mask));
                }
                base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                const uint32_t at = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                if (c != 0ull && c >= least && at < MASKED_CAP) {
                    mixed[at] = c;
                }
            }
        });
    };
    // The row streamed, sixteen bytes a thread and request: false where the bound lets more through than the sort holds.
    auto streamed = [&]() -> bool {
        constexpr int E = Geo<DT>::E, C = 4, V = C * E;
        constexpr uint32_t EMASK = (1u << E) - 1u;
        RowArgs a;   // (kept across the other ways, the arguments would be spilled there)
        read_again(a, src);
        Geo<DT> g;
        g.init(a.logits, vocab, 0u, 1u);
        const uint32_t n_pieces = g.main_hi - g.main_lo;   // (at most 65 536)
        uint16_t* piece_key = reinterpret_cast<uint16_t*>(mixed);
        uint16_t* piece_list = reinterpret_cast<uint16_t*>(dyn_lds);
        struct Bits16 {
            uint16_t v;
        } __attribute__((packed));
        // fn(u, piece, its first id, its true values from v[u * E] on) of pieces number(0) .. number(C - 1) (n_pieces: none).
        float v[V];
        auto pieces = [&](auto&& number, auto&& fn) {
            u32x4 raw[C];
            uint32_t piece[C], first[C], lo[C], hi[C], listed_raw[C];
#pragma unroll
            for (int u = 0; u < C; ++u) {
                piece[u] = number(u);
                const uint32_t c = g.main_lo + min(piece[u], n_pieces - 1u);
                first[u] = c * (uint32_t)E - g.pad;
                raw[u] = gload(reinterpret_cast<const u32x4*>(g.base + (size_t)c * 16));
                lo[u] = gload(a.allow + (first[u] >> 5));
                hi[u] = g.pad != 0u ? gload(a.allow + min((first[u] >> 5) + 1u, words - 1u)) : 0u;
                // (two bytes of the bitmap of listed ids hold a piece's bits, wherever the row starts)
                listed_raw[u] = pen ? ((const LILY_GLOBAL Bits16*)(reinterpret_cast<const char*>(a.touched) + (first[u] >> 3)))->v : 0u;
            }
            uint32_t todo = 0u, biased = 0u;
#pragma unroll
            for (int u = 0; u < C; ++u) {
                const uint64_t two = ((uint64_t)hi[u] << 32) | lo[u];
                const uint32_t allowed = piece[u] < n_pieces ? (uint32_t)(two >> (first[u] & 31u)) & EMASK : 0u;
                float x[E];
                unpack<DT>(raw[u], x);
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    v[u * E + j] = ((allowed >> j) & 1u) != 0u && x[j] > NEG_INF ? x[j] : NEG_INF;   // (a NaN is worth -inf)
                }
                uint32_t touched = (listed_raw[u] >> (first[u] & 7u)) & EMASK;
                const uint32_t word = first[u] >> 5;
                if (__ballot(has_bias(word) || (g.pad != 0u && has_bias(min(word + 1u, words - 1u)))) != 0ull) {
                    uint32_t some_biased = 0u;
                    for (uint32_t j = 0; j < n_bias; ++j) {
                        const uint32_t at = ms.bias_id[j] - first[u];
                        some_biased |= at < (uint32_t)E ? 1u << at : 0u;
                    }
                    touched |= some_biased;
                    biased |= some_biased << (u * E);
                }
                todo |= (touched & allowed) << (u * E);
            }
            // The values that something touches, one of every piece at a time with their loads in flight together.
            while (__ballot(todo != 0u) != 0ull) {
                uint32_t at[C], count[C];
                float x[C];
#pragma unroll
                for (int u = 0; u < C; ++u) {
                    const uint32_t m = (todo >> (u * E)) & EMASK;
                    at[u] = m != 0u ? (uint32_t)__builtin_ctz(m) : 0xffu;
                    todo &= ~((m & (0u - m)) << (u * E));
                    const uint32_t id = m != 0u ? first[u] + at[u] : 0u;
                    x[u] = load_logit<DT>(a.logits, id);
                    count[u] = pen ? gload(a.counts + id) : 0u;
                }
#pragma unroll
                for (int u = 0; u < C; ++u) {
                    const uint32_t j0 = at[u] & (uint32_t)(E - 1);
                    float t = worth(a, x[u], first[u] + j0, at[u] != 0xffu && ((biased >> (u * E + (int)j0)) & 1u) != 0u, count[u]);
                    t = t > NEG_INF ? t : NEG_INF;
#pragma unroll
                    for (int j = 0; j < E; ++j) {
                        v[u * E + j] = at[u] == (uint32_t)j ? t : v[u * E + j];
                    }
                }
            }
            static_assert(C == 4, "a call for each");
            fn(std::integral_constant<int, 0>{}, piece[0]);
            fn(std::integral_constant<int, 1>{}, piece[1]);
            fn(std::integral_constant<int, 2>{}, piece[2]);
            fn(std::integral_constant<int, 3>{}, piece[3]);
        };
        // Ids of partial pieces at the row's ends, one a thread (fewer than 16 at either end).
        uint32_t edge = 0xffffffffu;
        if (tid < 64u) {
            edge = g.id_lo + tid < g.edge_lo_end ? g.id_lo + tid : edge;
        } else if (tid < 128u) {
            edge = g.edge_hi_begin + tid - 64u < g.id_hi ? g.edge_hi_begin + tid - 64u : edge;
        }
        float ev = NEG_INF;
        if (edge != 0xffffffffu && bit_of(a.allow, edge)) {
            ev = worth(a, load_logit<DT>(a.logits, edge), edge, has_bias(edge >> 5), pen ? gload(a.counts + edge) : 0u);
            ev = ev > NEG_INF ? ev : NEG_INF;
        }
        lse.add_one(ev, a.c2);
        float top[C] = {ev, NEG_INF, NEG_INF, NEG_INF};
        for (uint32_t p0 = 0; p0 < n_pieces; p0 += C * MT) {
            pieces([&](int u) { return p0 + (uint32_t)u * MT + tid; },
                   [&](auto at, uint32_t piece) {
                       constexpr int u = decltype(at)::value;
                       float m = v[u * E];
#pragma unroll
                       for (int j = 1; j < E; ++j) {
                           m = fmaxf(m, v[u * E + j]);
                       }
                       top[u] = fmaxf(top[u], m);
                       if (piece < n_pieces) {
                           piece_key[piece] = (uint16_t)(m > NEG_INF ? lilym_order_key(m) >> 16 : 0u);
                       }
                       if (LSE && want_lse && m > NEG_INF) {
                           const float safe = lse.rebase(m, a.c2);
#pragma unroll
                           for (int j = 0; j < E; ++j) {
                               lse.term(v[u * E + j], a.c2, safe);   // (2^-inf is 0)
                           }
                       }
                   });
        }
        if (forced) {
            return true;
        }
        // The bound: each wave's lanes are four sets of maxima.
        uint32_t top_key[C];
        uint64_t keys = 0ull;
#pragma unroll
        for (int u = 0; u < C; ++u) {
            top_key[u] = top[u] > NEG_INF ? lilym_order_key(top[u]) >> 16 : 0u;
            keys |= (uint64_t)max(wave_kth_key16(top_key[u], wide_rank(a.k, MWAVE)), WIDE_LEAST_KEY) << (16 * u);
        }
        if (lane == 0u) {
            ms.six.wave_k[w] = keys;
        }
        __syncthreads();
        static_assert(C == NWAVE && MWAVE <= 64, "a word of four keys a wave, a lane each");
        float bound = bound_of_keys(lane < MWAVE ? ms.six.wave_k[lane] : 0ull, a.k, MWAVE);
        // The pieces that reach it.  Clusters leave sets without a value, or with few: where too many have none to name, or
        // five eighths as many maxima again as k reach what they name (on Gaussian rows some two fifths do), the bound is the k-th
        // largest of all the maxima.
        uint32_t n_reach = 0;
        for (bool exact = !(bound > F32_LOWEST);; exact = true) {   // (the same in every wave)
            if (exact) {
                uint32_t T = 0;
                for (uint32_t t = 0x8000u; t != 0u; t >>= 1) {
                    if (tid == 0) {
                        ms.bin = 0u;
                        ms.pieces = 0u;
                    }
                    __syncthreads();
                    uint32_t reach = 0;
#pragma unroll
                    for (int u = 0; u < C; ++u) {
                        reach += (uint32_t)__popcll(__ballot(top_key[u] >= (T | t)));
                    }
                    if (lane == 0u) {
                        atomicAdd(&ms.bin, reach);
                    }
                    __syncthreads();
                    T |= ms.bin >= a.k ? t : 0u;
                    __syncthreads();
                }
                if (T <= WIDE_LEAST_KEY) {
                    return false;
                }
                bound = lower_by_slack(lilym_key_value(T << 16));
            }
            const uint32_t least = lilym_order_key(bound) >> 16;
            uint32_t maxima = 0;
#pragma unroll
            for (int u = 0; u < C; ++u) {
                maxima += (uint32_t)__popcll(__ballot(top_key[u] >= least));
            }
            if (!exact && lane == 0u) {
                atomicAdd(&ms.bin, maxima);
            }
            for (uint32_t p0 = 0; p0 < n_pieces; p0 += MT) {
                const uint32_t p = p0 + tid;
                const bool reaches = p < n_pieces && piece_key[min(p, n_pieces - 1u)] >= least;
                const uint64_t mask = __ballot(reaches);
                if (mask != 0ull) {
                    uint32_t base = 0;
                    if (lane == 0u) {
                        base = atomicAdd(&ms.pieces, (uint32_t)__popcll(mask));
                    }
                    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                    const uint32_t at = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                    if (reaches && at < MASKED_CAP) {
                        piece_list[at] = (uint16_t)p;
                    }
                }
            }
            __syncthreads();
            n_reach = ms.pieces;
            if (exact || ms.bin <= a.k + a.k * 5u / 8u) {
                break;
            }
            __syncthreads();   // (everybody has read it)
        }
        if (n_reach > MASKED_CAP) {
            return false;
        }
        auto offer = [&](float x, uint32_t id) {
            const uint64_t mask = __ballot(x >= bound);
            if (mask != 0ull) {
                uint32_t base = 0;
                if (lane == 0u) {
                    base = atomicAdd(&ms.n, (uint32_t)__popcll(mask));
                }
                base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                const uint32_t at = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                if (x >= bound && at < MASKED_CAP) {
                    mixed[at] = composite_of(x / a.temperature, id);
                }
            }
        };
        for (uint32_t i0 = 0; i0 < n_reach; i0 += C * MT) {
            pieces(
                [&](int u) {
                    const uint32_t i = i0 + (uint32_t)u * MT + tid;
                    return i < n_reach ? (uint32_t)piece_list[i] : n_pieces;
                },
                [&](auto at, uint32_t piece) {
                    constexpr int u = decltype(at)::value;
                    if (i0 + (uint32_t)u * MT < n_reach) {
#pragma unroll
                        for (int j = 0; j < E; ++j) {
                            offer(v[u * E + j], (g.main_lo + piece) * (uint32_t)E - g.pad + (uint32_t)j);
                        }
                    }
                });
        }
        offer(ev, edge);   // (-inf where there is none)
        __syncthreads();
        return ms.n <= MASKED_CAP;
    };
    uint32_t took = 1, n = 0;
    bool sorted = false;
    // Listed ids stay where they are evaluated, HALVES * MASKED_CAP / MT of them a thread, until they are sorted.
    auto sort_listed = [&](auto halves) {
        constexpr uint32_t HALVES = decltype(halves)::value, R = MASKED_CAP / MT;
        uint64_t mine[HALVES * R] = {};
        uint32_t here = 0;
#pragma unroll
        for (uint32_t h = 0; h < HALVES; ++h) {
            over_listed(h * MASKED_CAP, [&](uint32_t r, float u, uint32_t id, bool in) {
                if (LSE && want_lse && in) {
                    lse.add_one(u, a.c2);
                }
                mine[h * R + r] = in ? composite_of(u / a.temperature, id) : 0ull;
                here += mine[h * R + r] != 0ull ? 1u : 0u;
            });
        }
        if (!forced) {
            scan_all(here, ms.six, n);   // (and every thread has read its ids)
            sort_by_sixteen(mine, n, min(a.k, n), dyn_lds, bins, mixed, ms.six);
            sorted = true;
        }
    };
    if (listed && total != 0u) {   // (the same in every thread)
        if (total <= MASKED_CAP) {
            sort_listed(std::integral_constant<uint32_t, 1>{});
        } else {
            sort_listed(std::integral_constant<uint32_t, 2>{});
        }
    } else if (by_words && (total <= MASKED_CAP || forced)) {
        collect(0ull, LSE && want_lse);
    } else if (by_words || !streamed()) {
        bool first = by_words;   // (the sum is there otherwise)
        if (!by_words) {
            // Ties by the thousand, values that rise all along the row.
            took = 2;
            __syncthreads();
            if (tid == 0) {
                ms.n = 0u;
            }
            fetch_words();
            count_words();
            const uint32_t again = scan_all(some, ms.six, n_words) - some;
            list_words(again);
            __syncthreads();
        }
        // The bin of the k-th composite, twelve bits at a time from the top, until what lies at or above it fits.
        uint64_t prefix = 0ull;
        uint32_t above = 0;   // composites above everything under the prefix
        for (int shift = 52;; shift -= 12) {   // (sixteen composites at most share all but the last four bits)
            for (uint32_t i = tid; i < HBINS; i += MT) {
                hist[i] = 0u;
            }
            __syncthreads();
            const uint64_t under = shift >= 52 ? 0ull : ~0ull << (shift + 12);
            HistRun run;
            run.init();
            over_admitted([&](float u, uint32_t id, bool in) {
                if (LSE && want_lse && first && in) {
                    lse.add_one(u, a.c2);
                }
                const uint64_t c = in ? composite_of(u / a.temperature, id) : 0ull;
                run.add(hist, (uint32_t)(c >> shift) & (HBINS - 1u), c != 0ull && (c & under) == prefix);
            });
            run.flush(hist);
            __syncthreads();
            // from the top: thread t holds bins HBINS - 4 (t + 1) .. + 3
            uint32_t h[HBINS / MT], mine = 0, whole;
#pragma unroll
            for (uint32_t i = 0; i < HBINS / MT; ++i) {
                h[i] = hist[HBINS - 1u - (tid * (HBINS / MT) + i)];
                mine += h[i];
            }
            uint32_t before = scan_all(mine, ms.six, whole) - mine;
            if (above + whole <= a.k) {
                // fewer values than are asked for: all of them
                break;
            }
#pragma unroll
            for (uint32_t i = 0; i < HBINS / MT; ++i) {
                if (above + before < a.k && above + before + h[i] >= a.k) {
                    ms.bin = HBINS - 1u - (tid * (HBINS / MT) + i);
                    ms.above = above + before;
                    ms.need = above + before + h[i];
                }
                before += h[i];
            }
            __syncthreads();
            prefix |= (uint64_t)ms.bin << shift;
            above = ms.above;
            first = false;
            if (ms.need <= MASKED_CAP) {
                break;
            }
        }
        __syncthreads();
        collect(prefix, false);
    }
    phase(cfg, 2);
    if (LSE && want_lse) {
        const float m_w = wave_max_dpp(lse.mc);
        __syncthreads();
        if (lane == 0u) {
            ms.wave_f[w] = m_w;
        }
        __syncthreads();
        float m = ms.wave_f[0];
        for (uint32_t i = 1; i < MWAVE; ++i) {
            m = fmaxf(m, ms.wave_f[i]);
        }
        const double s = wave_sum_d(lse.mc > NEG_INF ? lse.s * exp2((double)lse.mc - (double)m) : 0.0);
        if (lane == 0u) {
            ms.wave_d[w] = s;
        }
        __syncthreads();
        if (tid == 0) {
            double t = 0.0;
            for (uint32_t i = 0; i < MWAVE; ++i) {
                t += ms.wave_d[i];
            }
            sh.lse_mc = (double)m;
            sh.lse_s = t;
        }
    }
    __syncthreads();
    if (cfg.path_stats != nullptr && tid == 0) {
        atomicAdd(&cfg.path_stats[took], 1u);
    }
    RowArgs t;
    read_again(t, src);
    if (forced) {
        if (tid == 0) {
            finish_token<DT>(t, sh, t.forced, vocab);
        }
        return;
    }

    // ---- the k best in order
    if (!sorted) {
        n = min(ms.n, MASKED_CAP);
        constexpr uint32_t PER = MASKED_CAP / MT;
        uint64_t mine[PER];
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            mine[j] = tid + j * MT < n ? mixed[tid + j * MT] : 0ull;
        }
        sort_by_sixteen(mine, n, min(t.k, n), dyn_lds, bins, placed, ms.six);
    }
    const uint32_t k = min(t.k, n);
    phase(cfg, 6);
    if (tid >= NT) {
        return;   // (the draw is four waves' work: a barrier waits for those that are left)
    }
    tail<DT, true, false>(t, vocab, t.step + cfg.step_delta, k, true, dyn_lds, sh, cfg);
    phase(cfg, 7);
}

template <int DT, bool LSE>
__global__ __launch_bounds__(MT) void k_masked_inline(InlineRows rows, LaunchCfg cfg) {
    __shared__ Shared sh;
    __shared__ MaskedShared ms;
    const LILY_CONST RowArgs* table = (const LILY_CONST RowArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    masked_row<DT, LSE>(table + blockIdx.y, cfg, sh, ms);
}

template <int DT, bool LSE>
__global__ __launch_bounds__(MT) void k_masked_table(LaunchCfg cfg) {
    __shared__ Shared sh;
    __shared__ MaskedShared ms;
    masked_row<DT, LSE>((const LILY_CONST RowArgs*)cfg.table + blockIdx.y, cfg, sh, ms);
}

template <int DT, bool LSE>
hipError_t launch_masked(hipStream_t stream, uint32_t rows, const LaunchCfg& cfg, const InlineRows* inline_rows) {
    static LdsAllowed allowed_inline, allowed_table;
    if (inline_rows != nullptr) {
        const hipError_t e = allowed_inline.say(reinterpret_cast<const void*>(k_masked_inline<DT, LSE>), MASKED_LDS_BYTES);
        if (e != hipSuccess) {
            return e;
        }
        hipLaunchKernelGGL((k_masked_inline<DT, LSE>), dim3(1, rows), dim3(MT), MASKED_LDS_BYTES, stream, *inline_rows, cfg);
    } else {
        const hipError_t e = allowed_table.say(reinterpret_cast<const void*>(k_masked_table<DT, LSE>), MASKED_LDS_BYTES);
        if (e != hipSuccess) {
            return e;
        }
        hipLaunchKernelGGL((k_masked_table<DT, LSE>), dim3(1, rows), dim3(MT), MASKED_LDS_BYTES, stream, cfg);
    }
    return hipGetLastError();
}

}  // namespace

#define LILY_CAT_(a, b) a##b
#define LILY_CAT(a, b) LILY_CAT_(a, b)

hipError_t LILY_CAT(launch_rows_masked_dt, LILY_DT)(hipStream_t stream, bool lse, uint32_t rows, const LaunchCfg& cfg,
                                                    const InlineRows* inline_rows) {
    return lse ? launch_masked<LILY_DT, true>(stream, rows, cfg, inline_rows)
               : launch_masked<LILY_DT, false>(stream, rows, cfg, inline_rows);
}

}  // namespace lily
