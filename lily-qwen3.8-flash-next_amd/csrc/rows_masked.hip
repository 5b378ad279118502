// rows_masked.hip - rows under an allow-mask, a workgroup of 1 024 threads a row.  Compiled once per logits
// type: -DLILY_DT=0|1.
//
// A grammar admits some per cent of the vocabulary, in clusters, and such rows name no top_k as a rule: 3 000
// ids to evaluate, 1 024 of them to sort.  That is a chain of latencies, not work to be spread: cut into
// four slices of 256 threads each row paid for a hand-over, a second gathering and a sort by one wave a
// SIMD (64 rows of 151 936 bf16, 2 % admitted: slices done 16 us, ticket 18, sorted 27, drawn 36).  Here
// sixteen waves list the mask's words that admit anything, evaluate them a word for every 32 lanes (a run of
// ids is one request), sort in LDS, and the first four waves draw.
//
// A mask that admits more ids than the sort holds (8 192) is taken by the same kernel: histograms over the
// composites' leading bits, every value evaluated anew for each, until what reaches the k-th one's bin fits.  One that
// admits a third of the vocabulary is left to the launch behind, which streams the row.
#include "launch.h"
#include "row_kernel.h"

#if !defined(LILY_DT)
#error "compile with -DLILY_DT=<lily_dtype>"
#endif

namespace lily {

namespace {

constexpr uint32_t MT = 1024, MWAVE = MT / 64;
constexpr uint32_t MASKED_WORDS = MASKED_MAX_VOCAB / 32u, WORDS_PER = MASKED_WORDS / MT;
constexpr uint32_t MASKED_CAP = 8192;      // values that are sorted
constexpr uint32_t MASKED_DENSE = 49152;   // ids a mask may admit
constexpr uint32_t MBINS = 2048;           // of the sort
constexpr uint32_t HBINS = 4096;           // of the histograms, 12 bits
// Dynamic LDS in 64-bit slots: the sorted candidates and the tail's arrays; the sort's bins; the values as they
// come (the histograms, before there are any); the words that admit anything (bits, number), and where those are
// done with the values by bins.
constexpr uint32_t OFF_BINS = (LILY_SAMPLE_K_CAP * 8 + 3 * LILY_SAMPLE_K_CAP * 4) / 8;
constexpr uint32_t OFF_MIXED = OFF_BINS + MBINS / 2;
constexpr uint32_t OFF_PLACED = OFF_MIXED + MASKED_CAP;
constexpr uint32_t MASKED_LDS_BYTES = (OFF_PLACED + MASKED_CAP) * 8;
static_assert(MASKED_WORDS * 6 <= MASKED_CAP * 8 && HBINS * 4 <= MASKED_CAP * 8, "masked rows: LDS layout");

struct MaskedShared {
    uint32_t wave_u[MWAVE];
    uint64_t wave_k[MWAVE];
    float wave_f[MWAVE];
    double wave_d[MWAVE];
    uint32_t n, bin, above, need;
    uint32_t bias_id[STREAM_BIAS_CAP];
    float bias_delta[STREAM_BIAS_CAP];
    uint32_t biased[MASKED_WORDS / 32];    // bit w: some pair names an id of word w
};

// The threads' values summed up to and including each, over the whole workgroup; `all`: all of them.
__device__ __forceinline__ uint32_t scan_all(uint32_t x, MaskedShared& ms, uint32_t& all) {
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t incl = wave_scan_u32(x);
    __syncthreads();   // (what the last call left has been read)
    if (lane == 63u) {
        ms.wave_u[w] = incl;
    }
    __syncthreads();
    uint32_t before = 0;
    all = 0;
    for (uint32_t i = 0; i < MWAVE; ++i) {
        const uint32_t t = ms.wave_u[i];
        before += i < w ? t : 0u;
        all += t;
    }
    return before + incl;
}

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

    // ---- the words that admit anything, in order
    uint32_t bits[WORDS_PER], some = 0, admitted = 0;
#pragma unroll
    for (uint32_t i = 0; i < WORDS_PER; ++i) {
        bits[i] = gload(a.allow + min(tid * WORDS_PER + i, words - 1u));
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
        const uint32_t at = tid * WORDS_PER + i;
        bits[i] = at < words ? bits[i] & range32_at(0u, vocab, (int64_t)at * 32) : 0u;
        some += bits[i] != 0u ? 1u : 0u;
        admitted += (uint32_t)__popc(bits[i]);
    }
    uint32_t n_words, total;
    uint32_t place = scan_all(some, ms, n_words) - some;
    scan_all(admitted, ms, total);
    if (tid < n_bias && ms.bias_id[tid] < vocab) {
        const uint32_t at = ms.bias_id[tid] >> 5;
        atomicOr(&ms.biased[at >> 5], 1u << (at & 31u));
    }
#pragma unroll
    for (uint32_t i = 0; i < WORDS_PER; ++i) {
        if (bits[i] != 0u) {
            word_bits[place] = bits[i];
            word_at[place] = (uint16_t)(tid * WORDS_PER + i);
            ++place;
        }
    }
    __syncthreads();
    // Dense masks are better streamed by many workgroups: the launch behind this one takes those rows.
    const bool served = total <= MASKED_DENSE;
    if (tid == 0) {
        cfg.masked_served[blockIdx.y] = served ? 1u : 0u;
    }
    if (!served) {
        return;
    }
    phase(cfg, 1);

    // fn(value before the temperature, id, whether there is one) over every admitted id: 32 lanes a word,
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
                biased[r] = n_bias != 0u && ((ms.biased[at >> 5] >> (at & 31u)) & 1u) != 0u;
                x[r] = load_logit<DT>(a.logits, id[r]);
                count[r] = pen ? gload(a.counts + id[r]) : 0u;
            }
#pragma unroll
            for (uint32_t r = 0; r < R; ++r) {
                if (i0 + r * (MT / 32u) >= n_words) {
                    break;
                }
                float u = x[r];
                if (__ballot(biased[r]) != 0ull) {
                    for (uint32_t j = 0; j < n_bias; ++j) {   // (pairs of one id in the list's order)
                        u = ms.bias_id[j] == id[r] ? u + ms.bias_delta[j] : u;
                    }
                }
                if (count[r] > 0u) {
                    u = u > 0.0f ? u / a.repetition : u * a.repetition;
                    u -= a.presence + a.frequency * (float)count[r];
                }
                fn(u, id[r], in[r]);
            }
        }
    };
    LseAcc lse;
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
    if (total <= MASKED_CAP || forced) {
        collect(0ull, LSE && want_lse);
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
            uint32_t before = scan_all(mine, ms, whole) - mine;
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

    // ---- the k best in order: a counting sort (see wg_sort_topk), eight values a thread
    const uint32_t n = min(ms.n, MASKED_CAP), k = min(a.k, n);
    constexpr uint32_t PER = MASKED_CAP / MT;
    uint64_t mine[PER];
    uint32_t hi = 0u, lo = 0xffffffffu;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        mine[j] = tid + j * MT < n ? mixed[tid + j * MT] : 0ull;
        const uint32_t key = (uint32_t)(mine[j] >> 32);
        hi = max(hi, key);
        lo = mine[j] != 0ull ? min(lo, key) : lo;
    }
    hi = wave_max_u32(hi);
    lo = wave_min_u32(lo);
    if (lane == 0u) {
        ms.wave_k[w] = ((uint64_t)hi << 32) | lo;
    }
#pragma unroll
    for (uint32_t i = 0; i < MBINS / MT; ++i) {
        bins[tid + i * MT] = 0u;
    }
    __syncthreads();
    hi = 0u;
    lo = 0xffffffffu;
    for (uint32_t i = 0; i < MWAVE; ++i) {
        hi = max(hi, (uint32_t)(ms.wave_k[i] >> 32));
        lo = min(lo, (uint32_t)ms.wave_k[i]);
    }
    uint32_t longest = 0;
    if (n != 0u) {
        const bool crosses = hi >= 0x80000000u && lo < 0x80000000u;
        const float top = lilym_key_value(hi);
        const float range = crosses ? top - lilym_key_value(lo) : (float)(hi - lo) + 1.0f;
        const float scale = (float)MBINS / range * 0.9999f;
        const bool spread = scale > 0.0f && range < 3.0e38f && scale <= 3.0e38f;
        auto bin_of = [&](uint64_t c) -> uint32_t {   // never decreases as c does
            const uint32_t key = (uint32_t)(c >> 32);
            const float d = crosses ? top - lilym_key_value(key) : (float)(hi - key);
            return spread ? (uint32_t)fminf(d * scale, (float)(MBINS - 1u)) : 0u;
        };
        uint32_t at_of[PER];   // bin, and place in it from bit 16 on
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            at_of[j] = 0u;
            if (mine[j] != 0ull) {
                const uint32_t b = bin_of(mine[j]);
                at_of[j] = b | (atomicAdd(&bins[b], 1u) << 16);
            }
        }
        __syncthreads();
        const uint32_t h0 = bins[2u * tid], h1 = bins[2u * tid + 1u];
        static_assert(MBINS == 2 * MT, "two bins a thread");
        uint32_t whole;
        const uint32_t from = scan_all(h0 + h1, ms, whole) - h0 - h1;
        longest = max(from < k ? h0 : 0u, from + h0 < k ? h1 : 0u);
        longest = wave_max_u32(longest);
        __syncthreads();
        bins[2u * tid] = from;
        bins[2u * tid + 1u] = from + h0;
        if (lane == 0u) {
            ms.wave_u[w] = longest;
        }
        __syncthreads();
        longest = 0;
        for (uint32_t i = 0; i < MWAVE; ++i) {
            longest = max(longest, ms.wave_u[i]);
        }
        if (longest <= SORT_BIN_MAX) {
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                if (mine[j] != 0ull) {
                    placed[bins[at_of[j] & 0xffffu] + (at_of[j] >> 16)] = mine[j];
                }
            }
            __syncthreads();
            // The few that share a bin are ranked against each other.
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                if (mine[j] != 0ull) {
                    const uint32_t b = at_of[j] & 0xffffu, begin = bins[b], end = b + 1u < MBINS ? bins[b + 1u] : n;
                    if (begin < k) {
                        uint32_t rank = begin;
                        for (uint32_t i = begin; i < end; ++i) {
                            rank += placed[i] > mine[j] ? 1u : 0u;
                        }
                        if (rank < k) {
                            dyn_lds[rank] = mine[j];
                        }
                    }
                }
            }
            __syncthreads();
        } else {
            // Ties by the hundred, an outlier that stretches the steps: bitonic, all of them.
            uint32_t p = 128;
            while (p < n) {
                p <<= 1;
            }
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                placed[tid + j * MT] = mine[j];
            }
            __syncthreads();
            for (uint32_t size = 2; size <= p; size <<= 1) {
                for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                    for (uint32_t i = tid; i < (p >> 1); i += MT) {
                        const uint32_t pos = (i / stride) * (stride << 1) + (i % stride), partner = pos + stride;
                        const bool desc = (pos & size) == 0u;
                        const uint64_t x = placed[pos], y = placed[partner];
                        if (desc ? x < y : x > y) {
                            placed[pos] = y;
                            placed[partner] = x;
                        }
                    }
                    __syncthreads();
                }
            }
            if (tid < k) {
                dyn_lds[tid] = placed[tid];
            }
            __syncthreads();
        }
    }
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
