// rows_masked.hip - rows under an allow-mask, a workgroup of 1 024 threads a row.  Compiled once per logits
// type: -DLILY_DT=0|1.
//
// A grammar admits some per cent of the vocabulary, and such rows name no top_k as a rule: 3 000
// ids to evaluate, 1 024 of them to sort.  That is a chain of latencies, not work to be spread: cut into
// four slices of 256 threads each row paid for a hand-over, a second gathering and a sort by one wave a
// SIMD (64 rows of 151 936 bf16, 2 % admitted: slices done 16 us, ticket 18, sorted 27, drawn 36).  Here
// sixteen waves read the mask, evaluate what it admits, sort in LDS, and the first four waves draw.
//
// Ids that lie scattered are listed one by one and evaluated a lane each.  Where they lie in clusters (12 and more to
// a word that admits any) the words are listed, 32 lanes a word: a run of ids is one request, and nobody lists them.
// (us a launch, bf16, 151 936 ids, 2 % admitted, by words -> by ids: one by one 1 row 62 -> 23, 64 rows 63 -> 24, in runs of up to 4 / 16
// ids 41 -> 23 / 28 -> 26, of up to 64 23 -> 26.  Each thread's words lie 1 024 apart, or a cluster would be one
// thread's to list.)
//
// A mask that admits more ids than the sort holds (8 192), in clusters, is taken by the same kernel: histograms over the
// composites' leading bits, every value evaluated anew for each, until what reaches the k-th one's bin fits.  Others, and
// those of more words than that pays for, are left to the launch behind, which streams the row (us, this way / left /
// by that launch alone: 64 rows of 151 936 bf16 in runs of up to 64, 10 % 50 / 74 / 68, 20 % 74 / 91 / 81; all of 49 152 ids
// 70 / 65 / 59, of 32 000 54 / 61 / 55).
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
constexpr uint32_t MASKED_CLUSTERED = 12;  // ids a word of a mask in clusters, on average
// Words that may admit ids where there are more than the sort holds: 0.031 us each, against some 46 us and 0.2 for every
// 1 000 ids of the row by the launch behind (one row to 64).
__device__ __forceinline__ uint32_t masked_most_words(uint32_t vocab) { return 800u + vocab / 150u; }
constexpr uint32_t MBINS = SIXTEEN_BINS;   // of the sort
constexpr uint32_t HBINS = 4096;           // of the histograms, 12 bits
// Dynamic LDS in 64-bit slots: the sorted candidates and the tail's arrays; the sort's bins; the values as they
// come (the histograms, before there are any); the words that admit anything (bits, number), and where those are
// done with the values by bins.  (A list of ids lies where the words would.)
constexpr uint32_t OFF_BINS = (LILY_SAMPLE_K_CAP * 8 + 3 * LILY_SAMPLE_K_CAP * 4) / 8;
constexpr uint32_t OFF_MIXED = OFF_BINS + MBINS / 2;
constexpr uint32_t OFF_PLACED = OFF_MIXED + MASKED_CAP;
constexpr uint32_t MASKED_LDS_BYTES = (OFF_PLACED + MASKED_CAP) * 8;
static_assert(MASKED_WORDS * 6 <= MASKED_CAP * 8 && HBINS * 4 <= MASKED_CAP * 8, "masked rows: LDS layout");

struct MaskedShared {
    SixteenShared six;
    float wave_f[MWAVE];
    double wave_d[MWAVE];
    uint32_t n, bin, above, need;
    uint32_t bias_id[STREAM_BIAS_CAP];
    float bias_delta[STREAM_BIAS_CAP];
    uint32_t biased[MASKED_WORDS / 32];    // bit w: some pair names an id of word w
};

template <int DT, bool LSE>
__device__ __forceinline__ void masked_row(const LILY_CONST RowArgs* src, const LaunchCfg& cfg, Shared& sh, MaskedShared& ms) {
    RowArgs a;
    load_row_args(a, src);
    apply_selection(a);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t vocab = cfg.vocab, words = (vocab + 31u) / 32u;
    const uint32_t step = a.step + cfg.step_delta;
    const bool want_lse = LSE && a.out_logprob != nullptr;
    const bool forced = (a.flags & F_FORCED) != 0u, pen = (a.flags & F_PEN) != 0u;
    if (forced && !want_lse) {
        if (tid == 0) {
            cfg.masked_served[blockIdx.y] = 1u;
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
#pragma unroll
    for (uint32_t i = 0; i < WORDS_PER; ++i) {
        bits[i] = gload(a.allow + min(i * MT + tid, words - 1u));
    }
    if (tid == 0) {
        tail_arrays(sh);
        ms.n = 0u;
    }
    const uint32_t n_bias = min(a.n_bias, STREAM_BIAS_CAP);
    if (tid < MASKED_WORDS / 32u) {
        ms.biased[tid] = 0u;
    }
    if (tid < n_bias) {
        ms.bias_id[tid] = gload(&a.bias[tid].id);
        ms.bias_delta[tid] = gload(&a.bias[tid].delta);
    }
#pragma unroll
    for (uint32_t i = 0; i < WORDS_PER; ++i) {
        const uint32_t at = i * MT + tid;
        bits[i] = at < words ? bits[i] & range32_at(0u, vocab, (int64_t)at * 32) : 0u;
        some += bits[i] != 0u ? 1u : 0u;
        admitted += (uint32_t)__popc(bits[i]);
    }
    uint32_t n_words, total;
    uint32_t place = scan_all(some, ms.six, n_words) - some;
    const uint32_t id_place = scan_all(admitted, ms.six, total) - admitted;
    if (tid < n_bias && ms.bias_id[tid] < vocab) {
        const uint32_t at = ms.bias_id[tid] >> 5;
        atomicOr(&ms.biased[at >> 5], 1u << (at & 31u));
    }
    const bool scattered = total < n_words * MASKED_CLUSTERED, listed = scattered && total <= MASKED_CAP;
    if (listed) {
        uint32_t to = id_place;
#pragma unroll
        for (uint32_t i = 0; i < WORDS_PER; ++i) {
            for (uint32_t left = bits[i]; left != 0u; left &= left - 1u) {
                id_list[to++] = (i * MT + tid) * 32u + (uint32_t)__builtin_ctz(left);
            }
        }
    } else {
#pragma unroll
        for (uint32_t i = 0; i < WORDS_PER; ++i) {
            if (bits[i] != 0u) {
                word_bits[place] = bits[i];
                word_at[place] = (uint16_t)(i * MT + tid);
                ++place;
            }
        }
    }
    __syncthreads();
    // Dense masks are better streamed by many workgroups.
    const bool served = total <= MASKED_CAP || (!scattered && n_words <= masked_most_words(vocab));
    if (tid == 0) {
        cfg.masked_served[blockIdx.y] = served ? 1u : 0u;
    }
    if (!served) {
        return;
    }
    phase(cfg, 1);

    // An admitted value before the temperature.
    auto worth = [&](float u, uint32_t id, bool biased, uint32_t count) -> float {
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
                fn(worth(x[r], id[r], biased[r], count[r]), id[r], in[r]);
            }
        }
    };
    // The same over the listed ids, a lane each, all their loads in flight.
    auto over_listed = [&](auto&& fn) {
        constexpr uint32_t R = MASKED_CAP / MT;
        uint32_t id[R], count[R];
        float x[R];
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
            id[r] = id_list[min(r * MT + tid, total - 1u)];
            x[r] = load_logit<DT>(a.logits, id[r]);
            count[r] = pen ? gload(a.counts + id[r]) : 0u;
        }
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
            if (r * MT >= total) {
                break;
            }
            fn(worth(x[r], id[r], has_bias(id[r] >> 5), count[r]), id[r], r * MT + tid < total);
        }
    };
    LseAcc lse;
    lse.init();
    auto collect = [&](auto&& over, uint64_t least, bool sum) {
        over([&](float u, uint32_t id, bool in) {
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
    if (listed) {
        if (total != 0u) {   // (the same in every thread)
            collect(over_listed, 0ull, LSE && want_lse);
        }
    } else if (total <= MASKED_CAP || forced) {
        collect(over_admitted, 0ull, LSE && want_lse);
    } else {
        // The bin of the k-th composite, twelve bits at a time from the top, until what lies at or above it fits.
        uint64_t prefix = 0ull;
        uint32_t above = 0;   // composites above everything under the prefix
        bool first = true;
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
        collect(over_admitted, prefix, false);
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
        const double s = wave_sum_d(lse.mc > NEG_INF ? (double)lse.s * exp2((double)lse.mc - (double)m) : 0.0);
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
        atomicAdd(&cfg.path_stats[1], 1u);
    }
    if (forced) {
        if (tid == 0) {
            finish_token<DT>(a, sh, a.forced, vocab);
        }
        return;
    }

    // ---- the k best in order
    const uint32_t n = min(ms.n, MASKED_CAP), k = min(a.k, n);
    constexpr uint32_t PER = MASKED_CAP / MT;
    uint64_t mine[PER];
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        mine[j] = tid + j * MT < n ? mixed[tid + j * MT] : 0ull;
    }
    sort_by_sixteen(mine, n, k, dyn_lds, bins, placed, ms.six);
    phase(cfg, 6);
    if (tid >= NT) {
        return;   // (the draw is four waves' work: a barrier waits for those that are left)
    }
    tail<DT, true, false>(a, vocab, step, k, true, dyn_lds, sh, cfg);
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
