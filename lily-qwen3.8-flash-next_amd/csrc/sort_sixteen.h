// sort_sixteen.h - the k best of a workgroup's entries in order, by sixteen waves.
#pragma once

#include "device_common.h"

namespace lily {

constexpr uint32_t SIXTEEN_THREADS = 1024, SIXTEEN_WAVES = SIXTEEN_THREADS / 64;
constexpr uint32_t SIXTEEN_BINS = 2048;

struct SixteenShared {
    uint32_t wave_u[SIXTEEN_WAVES];
    uint64_t wave_k[SIXTEEN_WAVES];
};

// The threads' values summed up to and including each, over the whole workgroup; `all`: all of them.
__device__ __forceinline__ uint32_t scan_all(uint32_t x, SixteenShared& ms, uint32_t& all) {
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t incl = wave_scan_u32(x);
    __syncthreads();   // (what the last call left has been read)
    if (lane == 63u) {
        ms.wave_u[w] = incl;
    }
    __syncthreads();
    uint32_t before = 0;
    all = 0;
    for (uint32_t i = 0; i < SIXTEEN_WAVES; ++i) {
        const uint32_t t = ms.wave_u[i];
        before += i < w ? t : 0u;
        all += t;
    }
    return before + incl;
}

// The k best of n entries, PER a thread (`mine`; 0 where there is none), in order to sorted[0 .. k): a counting sort as
// wg_sort_topk's, whose four waves take 5.4 us for 1 024 of 1 200 entries.  bins: SIXTEEN_BINS words; placed: PER *
// SIXTEEN_THREADS entries; k <= n.  All threads call.
template <uint32_t PER>
__device__ __forceinline__ void sort_by_sixteen(const uint64_t (&mine)[PER], uint32_t n, uint32_t k, uint64_t* sorted, uint32_t* bins,
                                                uint64_t* placed, SixteenShared& ms) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    uint32_t hi = 0u, lo = 0xffffffffu;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
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
    for (uint32_t i = 0; i < SIXTEEN_BINS / SIXTEEN_THREADS; ++i) {
        bins[tid + i * SIXTEEN_THREADS] = 0u;
    }
    __syncthreads();
    hi = 0u;
    lo = 0xffffffffu;
    for (uint32_t i = 0; i < SIXTEEN_WAVES; ++i) {
        hi = max(hi, (uint32_t)(ms.wave_k[i] >> 32));
        lo = min(lo, (uint32_t)ms.wave_k[i]);
    }
    if (n != 0u) {
        // Steps of the key where the values are of one sign; around zero, where the exponents run away, steps of the
        // value up to 1 and of the key of 1 and the value beyond.  (Steps of the value alone put what a few
        // outliers leave into a few bins: 9 bf16 rows of 248 320 under masks of 2 %, a heavy tail, 44.4 us, now 29.7.)
        const bool crosses = hi >= 0x80000000u && lo < 0x80000000u;
        auto around_zero = [&](uint32_t key) -> int32_t {   // never decreases as the key does not
            const float x = lilym_key_value(key);
            const int32_t m = (int32_t)(lilym_f32_bits(fabsf(x) + 1.0f) - 0x3f800000u);
            return x < 0.0f ? -m : m;
        };
        const int32_t top = crosses ? around_zero(hi) : 0;
        const uint32_t range = crosses ? (uint32_t)top - (uint32_t)around_zero(lo) : hi - lo;
        const float scale = (float)SIXTEEN_BINS / ((float)range + 1.0f) * 0.9999f;
        auto bin_of = [&](uint64_t c) -> uint32_t {   // never decreases as c does
            const uint32_t key = (uint32_t)(c >> 32);
            const uint32_t d = crosses ? (uint32_t)top - (uint32_t)around_zero(key) : hi - key;
            return (uint32_t)fminf((float)d * scale, (float)(SIXTEEN_BINS - 1u));
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
        static_assert(SIXTEEN_BINS == 2 * SIXTEEN_THREADS, "two bins a thread");
        uint32_t whole;
        const uint32_t from = scan_all(h0 + h1, ms, whole) - h0 - h1;
        uint32_t longest = max(from < k ? h0 : 0u, from + h0 < k ? h1 : 0u);   // of the bins that matter
        uint32_t matter = from + h0 < k ? from + h0 + h1 : from < k ? from + h0 : 0u;   // ... whose entries are the first so many
        longest = wave_max_u32(longest);
        matter = wave_max_u32(matter);
        __syncthreads();
        bins[2u * tid] = from;
        bins[2u * tid + 1u] = from + h0;
        if (lane == 0u) {
            ms.wave_k[w] = ((uint64_t)longest << 32) | matter;
        }
        __syncthreads();
        longest = 0;
        matter = 0;
        for (uint32_t i = 0; i < SIXTEEN_WAVES; ++i) {
            longest = max(longest, (uint32_t)(ms.wave_k[i] >> 32));
            matter = max(matter, (uint32_t)ms.wave_k[i]);
        }
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            if (mine[j] != 0ull) {
                placed[bins[at_of[j] & 0xffffu] + (at_of[j] >> 16)] = mine[j];
            }
        }
        if (longest <= SORT_BIN_MAX) {
            __syncthreads();
            // The few that share a bin are ranked against each other.
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                if (mine[j] != 0ull) {
                    const uint32_t b = at_of[j] & 0xffffu, begin = bins[b], end = b + 1u < SIXTEEN_BINS ? bins[b + 1u] : whole;
                    if (begin < k) {
                        uint32_t rank = begin;
                        for (uint32_t i = begin; i < end; ++i) {
                            rank += placed[i] > mine[j] ? 1u : 0u;
                        }
                        if (rank < k) {
                            sorted[rank] = mine[j];
                        }
                    }
                }
            }
            __syncthreads();
        } else {
            // Ties by the hundred, outliers among values near zero: bitonic, all that matter (what lies behind them up
            // to a power of two may be sorted with them).
            uint32_t p = 128;
            while (p < matter) {
                p <<= 1;
            }
            for (uint32_t i = whole + tid; i < p; i += SIXTEEN_THREADS) {
                placed[i] = 0ull;
            }
            __syncthreads();
            for (uint32_t size = 2; size <= p; size <<= 1) {
                for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                    for (uint32_t i = tid; i < (p >> 1); i += SIXTEEN_THREADS) {
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
                sorted[tid] = placed[tid];
            }
            __syncthreads();
        }
    }
}

}  // namespace lily
