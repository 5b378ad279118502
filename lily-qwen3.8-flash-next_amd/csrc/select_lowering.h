// select_lowering.h - the streaming select of rows under penalties that can only lower a value
// (repetition >= 1, presence and frequency >= 0), without a mask or a bias list.
#pragma once

#include "select_stream.h"

namespace lily {

// ------------------------------------------------------------------ rows under lowering penalties
//
// The pass of select_stream() (blocks, lane maxima, a bound that moves, queued chunks), for rows
// that hold ids whose true value lies below the raw one: the "listed" ids, bits of the scratch's
// bitmap.  A decoded sequence keeps coming back to its likely tokens, so the largest raw values of
// a row are listed ids as a rule, and their counts grow with the sequence:
//
//   * The lane maxima that the bound comes from leave out every chunk that may hold a listed id.
//     What is left has its true value, so the bound is one of true values: k of them reach it,
//     however many of the raw maxima the penalties take down.  (A bound of raw values with a slack
//     of k / 8 + 2 was good until a row had drawn more than that many of its leading ids; every
//     such row then went through the exhaustive select: 1 306 us a step instead of 140 for 200 rows
//     of 248 320 bf16 logits over a decode of 4 000 steps; now 79 on a fresh history and 88 then.)
//     Which chunks those are comes from a bit per eight ids that the scratch keeps beside its
//     bitmap: 0.8 % of a bf16 row's bytes, eight lanes' load a block, and the 64 chunks of a wave's
//     load are one 64-bit lane mask.  (With the bitmap itself beside the chunks - 6 % more bytes,
//     a byte moved to every lane - the scan of 1 024 rows took 58.6 us instead of 53.3; now 52.)
//   * The largest of those maxima bounds the row's largest true value from below, and with it the
//     cut below which nothing is summed.  The largest raw value under the penalty of the largest
//     count, which used to bound it alone, is worthless once some id was drawn a hundred times
//     (1 024 rows of 151 936 bf16 logits went from 75 to 180 us over 2 000 steps; now 74 and 74).
//     It still counts where it is the better one, as does the true value of the id counted most often.
//   * Chunks are queued by their raw maxima and evaluated exactly behind the scan, chunks above
//     the cut alone are noted (a number in LDS) and their terms formed behind the scan.
//   * A flat row - most of its chunks lie above the cut - is not noted: from the first block on
//     (or from the block on that finds the notes filling up) the chunks come with their bits of the
//     bitmap, listed elements are taken out as they arrive, the others are summed on the spot, and
//     the chunks that held a listed id are noted; behind the scan those are looked at again and
//     their listed ids evaluated.  Where the notes overflow the workgroup walks the bitmap instead.
//     The hand-over has to come before the notes overflow (a slice that lost notes is taken again
//     from its start), so it goes by where the fullest segment is headed: 1 024 rows of 151 936
//     bf16 logits N(0, 2^2) with 4, 33 and 82 % of their elements above the cut (T 0.2, 0.3, 0.4)
//     175 -> 150, 194 -> 165 and 149 -> 137 us against a hand-over at three quarters of the place,
//     which came too late for every rate between 45 and 100 % of the chunks.  Dropping the notes of
//     up to three blocks is the cheaper way there (kept: 172 and 158 us at T 0.3 and 0.4).
//     The same form takes a slice again whose queue overflowed or whose candidates did not stand
//     (FLAT), there with a walk ahead of the scan too, whose true values enter the bound: listed ids
//     by the thousand above everything else cost it that walk and nothing more.

template <int DT>
__device__ __forceinline__ float listed_value(const RowArgs& a, float raw, uint32_t count) {
    float t = raw;
    if (count > 0u) {
        t = t > 0.0f ? t / a.repetition : t * a.repetition;
        t -= a.presence + a.frequency * (float)count;
    }
    return t;
}

// FLAT: the second form from the first block on.  `again`: set where that is worth a second call.
template <int DT, bool LSE, bool FLAT>
__device__ __forceinline__ bool select_lowering(const RowArgs& a, const Geo<DT>& g, uint32_t k, Shared& sh,
                                                const LaunchCfg& cfg, bool& again, bool& sorted, uint64_t*& out) {
    bool flat = FLAT;   // the same in every thread
    constexpr int E = Geo<DT>::E;
    constexpr int U = STREAM_UNROLL;
    constexpr uint32_t BLOCK = NT * U;
    constexpr uint32_t QSEG = Q_CAP / NWAVE;
    constexpr uint32_t SSEG = S_CAP / NWAVE;
    constexpr uint32_t EMASK = (1u << E) - 1u;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t nchunks = g.ce - g.cb;
    const uint32_t nblocks = (nchunks + BLOCK - 1) / BLOCK;
    const bool want_lse = LSE && a.out_logprob != nullptr;
    const float c2 = a.c2;
    const uint32_t row_words = (g.vocab + 31u) / 32u;
    again = false;
    if (nblocks > MAX_BLOCKS) {
        return stream_fail(cfg, 1u);
    }
    StreamLds L;
    L.init();

    // Every load of a block is issued whatever its chunk (see select_stream()).
    const uint32_t c_last = g.ce - 1u;
    auto fetch_row = [&](u32x4 (&dst)[U], uint32_t b) {
        const uint32_t c0 = g.cb + b * BLOCK + tid;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t c = min(c0 + (uint32_t)u * NT, c_last);
            dst[u] = gload(reinterpret_cast<const u32x4*>(g.base + (c << 4)));  // rows are below 4 GiB
        }
    };
    const char* touched_bytes = reinterpret_cast<const char*>(a.touched);
    struct Bits8 {
        uint32_t lo, hi;
    } __attribute__((packed));
    struct Bits {
        uint32_t lo, hi;
    };
    auto fetch_bits = [&](Bits& d, int32_t at) {
        const LILY_GLOBAL Bits8* from = (const LILY_GLOBAL Bits8*)(touched_bytes + at);
        d.lo = from->lo;
        d.hi = from->hi;
    };
    const int32_t bit0 = (int32_t)(g.cb * (uint32_t)E) - (int32_t)g.pad;   // the slice's first chunk's first id
    const uint32_t bit_sh = (uint32_t)bit0 & 7u;
    // The coarse map (a bit per eight ids, four words behind the bitmap): the 64 chunks of a wave's
    // load are CW consecutive words of it, read from any bit on, so the lanes of a wave bring the
    // words of its four loads and the one behind each: lane u * CW + q (and every LANES-th from
    // there on) word q of load u.  A chunk of a row that does not start on a multiple of eight ids
    // lies in two groups of eight: its own bit and the next one.  Words past the map's end are its
    // last (of chunks that are not streamed).
    constexpr uint32_t CW = 64u * (uint32_t)E / 256u, CLANES = (uint32_t)U * CW;
    const int32_t cbit0 = bit0 >> 3;
    const uint32_t cbit_sh = (uint32_t)cbit0 & 31u, cbit_sh2 = cbit_sh + (DT == LILY_BF16 && g.pad != 0u ? 1u : 0u);
    // (from the scratch's counts on, whose last words lie before the bitmap: offsets stay positive)
    const char* maps = reinterpret_cast<const char*>(a.touched) - 16;
    const uint32_t coarse_at = 16u + (row_words + LISTED_SPARE) * 4u;
    const uint32_t coarse_last = coarse_at + (g.vocab + 255u) / 256u * 4u;
    const uint32_t coarse_lane =
        coarse_at + (uint32_t)((cbit0 >> 5) + (int32_t)((lane % CLANES / CW * NWAVE + w) * CW + lane % CW)) * 4u;
    auto fetch_coarse = [&](u32x4 (&dst)[U], Bits& d, uint32_t b) {
        const LILY_GLOBAL Bits8* from =
            (const LILY_GLOBAL Bits8*)(maps + min(coarse_lane + b * (NWAVE * U * CW * 4u), coarse_last));
        d.lo = from->lo;
        d.hi = from->hi;
        fetch_row(dst, b);
    };
    // Whether this lane's chunk of load u may hold a listed id, from the block's coarse words.
    auto coarse_word = [&](const Bits& d) -> Bits {
        Bits r;
        if (DT == LILY_BF16) {
            r.lo = __builtin_amdgcn_alignbit(d.hi, d.lo, cbit_sh) |
                   __builtin_amdgcn_alignbit(d.hi, cbit_sh2 == 32u ? d.hi : d.lo, cbit_sh2 & 31u);
            r.hi = 0u;
        } else {
            const uint64_t v = (((uint64_t)d.hi << 32) | d.lo) >> cbit_sh;
            r.lo = (uint32_t)v;
            r.hi = (uint32_t)(v >> 32);
        }
        return r;
    };
    auto coarse_hit = [&](const Bits& d, int u) -> bool {
        if (DT == LILY_BF16) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)d.lo, 2 * u);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)d.lo, 2 * u + 1);
            return __builtin_amdgcn_inverse_ballot_w64(((uint64_t)hi << 32) | lo);
        }
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)d.lo, u);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)d.hi, u);
        const uint64_t v = ((uint64_t)hi << 32) | lo;
        return (((v >> ((bit_sh + 4u * lane) >> 3)) | (v >> ((bit_sh + 4u * lane + 3u) >> 3))) & 1ull) != 0ull;
    };
    // The bitmap itself (flat rows): load u of a block brings the wave 64 consecutive chunks, whose
    // bits are WPP consecutive words - of a bitmap read from any byte on, the rest of the row's
    // misalignment shifted out.  Lane u * WPP + q brings word q of piece u, and the lanes take
    // theirs from one another by four moves through the LDS crossbar.  (Four 16-bit loads a lane
    // instead cost 12 registers more, which this kernel spills.)  The byte before the bitmap that a
    // row with a partial first chunk starts in is the scratch's own (its counts lie there), as are
    // the words behind it: their bits stand for ids outside the row, whose chunks are not streamed.
    constexpr uint32_t WPP = 64u * E / 32u;
    const int32_t byte0 = (bit0 >> 3) + (int32_t)((min(lane / WPP, 3u) * NT + w * 64u) * (uint32_t)E / 8u + (lane % WPP) * 4u);
    const int32_t byte_last = (int32_t)(row_words * 4u + 8u);
    auto fetch_exact = [&](u32x4 (&dst)[U], Bits& d, uint32_t b) {
        fetch_bits(d, min(byte0 + (int32_t)(b * (BLOCK * (uint32_t)E / 8u)), byte_last));
        fetch_row(dst, b);
    };
    // A byte per chunk of the block, bit j = element j is a listed id.
    auto exact_bits = [&](const Bits& bits) -> uint32_t {
        const int word = (int)__builtin_amdgcn_alignbit(bits.hi, bits.lo, bit_sh);
        const uint32_t sh_l = (lane % (32u / (uint32_t)E)) * (uint32_t)E;
        uint32_t all = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t from = ((uint32_t)u * WPP + lane / (32u / (uint32_t)E)) * 4u;
            const uint32_t v = (uint32_t)__builtin_amdgcn_ds_bpermute((int)from, word);
            all |= ((v >> sh_l) & EMASK) << (8 * u);
        }
        return all;
    };
    // The chunks of block 0 that are streamed.  (Opaque: formed where it is asked for, not ahead of the
    // scan, whose scalar registers it would hold.)
    auto first_chunks = [&]() -> uint32_t {
        uint32_t cb = g.cb;
        asm volatile("" : "+s"(cb));
        const uint32_t lo = max(g.main_lo, cb), hi = min(g.main_hi, cb + BLOCK);
        return hi > lo ? hi - lo : 0u;
    };
    auto full_block = [&](uint32_t b) -> bool {
        const uint32_t c0 = g.cb + b * BLOCK;
        return c0 >= g.main_lo && c0 + BLOCK <= g.main_hi;
    };
    // Nothing is in flight here on any path that is taken; said outright, because the compiler
    // cannot tell and would otherwise drain the blocks requested ahead at every wait of the scan.
    __builtin_amdgcn_s_waitcnt(0);
    u32x4 buf_a[U], buf_b[U], buf_c[U];
    Bits bits_a, bits_b, bits_c;
    if (nblocks > 0) {
        if (FLAT) {
            fetch_exact(buf_a, bits_a, 0);
        } else {
            fetch_coarse(buf_a, bits_a, 0);
        }
    }
    if (tid == 0) {
        sh.n_fc = 0;
        sh.fail = 0;
        sh.n_pairs = 0;
    }
    __syncthreads();
    phase(cfg, 13);
    // The largest count any id of the scratch ever had (kept in the first spare word behind
    // the bitmap) bounds how far penalties can lower a value.
    const uint32_t max_count = *(const LILY_CONST uint32_t*)(a.touched + row_words);
    // What a raw value is worth at least: as an id with the scratch's largest count.
    // (A product with a reciprocal a little below the exact one: a bound needs no division.)
    const float low_scale = 1.0f / a.repetition * 0.9999995f;
    const float low_off = a.presence + a.frequency * (float)max(max_count, 1u);
    auto lowered = [&](float m) -> float { return (m > 0.0f ? m * low_scale : m * a.repetition) - low_off; };
    // Any id's true value bounds the row's largest from below.  One is worth the look: the id the
    // scratch counted most often, whose true value no other bound here describes well.  It comes
    // by scalar loads, which are waited for apart from the block requested above.
    float row_floor = NEG_INF;
    if (want_lse && max_count != 0u) {
        const uint32_t heavy = *(const LILY_CONST uint32_t*)(a.touched + row_words + 1u);
        if (heavy < g.vocab) {
            const uint32_t cnt = *(const LILY_CONST uint32_t*)(a.counts + heavy);
            float raw;
            if (DT == LILY_BF16) {
                const uintptr_t at = reinterpret_cast<uintptr_t>(a.logits) + (uintptr_t)heavy * 2u;
                const uint32_t word = *(const LILY_CONST uint32_t*)(at & ~(uintptr_t)3u);
                raw = lilym_bits_f32(((at & 2u) ? word >> 16 : word & 0xffffu) << 16);
            } else {
                raw = lilym_bits_f32(*(const LILY_CONST uint32_t*)(static_cast<const uint32_t*>(a.logits) + heavy));
            }
            const float t = listed_value<DT>(a, raw, cnt);
            row_floor = t > NEG_INF ? t : NEG_INF;   // (a NaN bounds nothing)
        }
    }
    phase(cfg, 1);

    // ---- scan
    StreamPriority prio;
    prio.init(nblocks);
    const uint32_t kw = (min(k, 64u * NWAVE) + NWAVE - 1) / NWAVE;
    float lane_max = NEG_INF;   // over chunks without listed ids (flat: over ids that are not listed)
    float lane_raw = NEG_INF;   // over all ids
    float T = F32_LOWEST;       // the block's bound, the same in every thread
    float ref_s = 0.0f;         // reference of acc_t
    float row_max = NEG_INF;    // lower bound of the row's largest true value, as of the last refresh
    float own_max = NEG_INF;    // ... as this wave's own lanes know it
    float skip_b = NEG_INF;     // the block's cut: nothing at or below it is summed
    uint32_t wq = 0;            // this wave's queue fill
    uint32_t sfill = 0;         // this wave's noted chunks
    uint32_t note_max = 0;      // the fullest segment of noted chunks, as of the last refresh
    uint32_t flat_from = 0;     // flat rows: the first block without its listed ids
    bool give_up = false;       // a wave's queue or notes overflowed (the same in every thread)
    WaveLse wl;
    wl.init();
    double acc_t = 0.0;
    constexpr int UP_UNSET = StreamSums::UP_UNSET;
    int up = UP_UNSET;          // this thread's acc_t is relative to ref_s + up
    uint32_t parity = 0;
    double base = -1.0e300;     // ref_s + up; far below anything while up is unset
    const double c2d = (double)c2;
    // One term of acc_t: the thread's own reference starts at its first term and moves up (its sum
    // scaled down by the same power of two) when a term lies beyond 2^900 of it.
    auto term_d = [&](float v) -> double {
        double d = __builtin_fma((double)v, c2d, -base);
        if (d > 900.0) {
            double e = (double)v * c2d - (double)ref_s;
            e = e < 1.0e9 ? (e > -1.0e9 ? e : -1.0e9) : 1.0e9;
            const int now = (int)__builtin_floor(e);
            if (up != UP_UNSET) {
                acc_t = __builtin_ldexp(acc_t, up - now);
            }
            up = now;
            base = (double)ref_s + (double)up;
            d = e - (double)up;
        }
        if (!(d > -1000.0)) {
            return 0.0;  // -inf, NaN, or nothing against what the thread already holds
        }
        return pow2_d(d);
    };
    const float lse_cut = (log2f((float)g.vocab) + 21.0f) * (a.temperature * 0.6931471805599453f);

    // Brings T up to date with everything the lanes have seen, the current block included.  `count`:
    // what the wave publishes beside it (its notes); returns the waves' sum of it.
    auto refresh_bound = [&](bool first, bool maxima, uint32_t count) -> uint32_t {
        const uint32_t key16 = lane_max > NEG_INF ? (lilym_order_key(lane_max) >> 16) : 0u;
        const uint32_t P = wave_kth_key16(key16, kw);
        const float mine = P != 0u ? lilym_key_value(P << 16) : F32_LOWEST;
        const float wm = maxima ? wave_max_dpp(fmaxf(lane_max, lowered(lane_raw))) : 0.0f;
        if (lane == 0) {
            sh.bound[parity][w] = mine;
            sh.wfill[parity][w] = wq > QSEG || (!flat && sfill > SSEG) ? 1u : 0u;
            sh.wnote[parity][w] = count;
            if (maxima) {
                sh.wmax[parity][w] = wm;
            }
        }
        __syncthreads();
        float t = sh.bound[parity][0];
        for (int i = 1; i < NWAVE; ++i) {
            t = fminf(t, sh.bound[parity][i]);
        }
        T = fmaxf(T, lower_by_slack(t));
        uint32_t sum = 0;
        note_max = 0;
        for (int i = 0; i < NWAVE; ++i) {
            give_up = give_up || sh.wfill[parity][i] != 0u;
            note_max = max(note_max, sh.wnote[parity][i]);
            sum += sh.wnote[parity][i];
        }
        if (maxima) {
            float m = sh.wmax[parity][0];
            for (int i = 1; i < NWAVE; ++i) {
                m = fmaxf(m, sh.wmax[parity][i]);
            }
            row_max = fmaxf(m, row_floor);
            if (first) {
                // Finite and far from overflow: every term is formed as 2^(v*c2 - ref_s).
                ref_s = m > NEG_INF ? fminf(fmaxf(m * c2, -1.0e30f), 1.0e30f) : 0.0f;
            }
        }
        parity ^= 1u;
        return sum;
    };

    // Appends a chunk's number (within the slice) for the lanes of `mask` to the wave's notes.
    auto note_chunk = [&](uint32_t number, bool mine, uint64_t mask) {
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
            (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
        const uint32_t at = sfill + rank;
        if (mine && at < SSEG) {
            L.noted[w * SSEG + at] = (uint16_t)number;
        }
        sfill += (uint32_t)__popcll(mask);
    };
    // The scan is compiled twice: with the listed ids left in the chunks, and without (a flat row).
    auto scan = [&](auto apart, uint32_t b_first) {
        constexpr bool APART = decltype(apart)::value;
        auto work = [&](u32x4 (&cur)[U], const Bits& bits, uint32_t b) {
            if (give_up || (!APART && flat) || b >= nblocks) {
                return;
            }
            prio.set(b);
            uint32_t hits = APART ? exact_bits(bits) : 0u;
            auto hit = [&](int u) -> uint32_t { return (hits >> (8 * u)) & 0xffu; };
            if (!full_block(b)) {
                const uint32_t ninf = DT == LILY_BF16 ? 0xff80ff80u : 0xff800000u;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint32_t c = g.cb + (b * U + u) * NT + tid;
                    if (c < g.main_lo || c >= g.main_hi) {
                        cur[u] = u32x4{ninf, ninf, ninf, ninf};
                        hits &= ~(0xffu << (8 * u));
                    }
                }
            }
            const float T_prev = T;
            // Once the bound is positive only chunks with a positive element can matter to it: their
            // maximum comes from the cheaper form, which reports +0 for all others.
            const bool nonneg = DT == LILY_BF16 && __builtin_amdgcn_readfirstlane((int)(T_prev > 0.0f)) != 0;
            float m8[U];
            float block_max = NEG_INF;
            bool nan_seen = false;
            if (nonneg) {
                int bm = 0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    m8[u] = chunk_max_nonneg<DT>(cur[u]);
                    bm = max(bm, (int)lilym_f32_bits(m8[u]));
                }
                // (a positive NaN's pattern lies above +inf's: the maxima are taken again, ignoring it)
                nan_seen = __ballot(bm > 0x7f800000) != 0ull;
                block_max = lilym_bits_f32((uint32_t)bm);
            }
            if (!nonneg || nan_seen) {
                block_max = NEG_INF;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    m8[u] = chunk_max<DT>(cur[u]);
                    block_max = max2_raw(block_max, m8[u]);
                }
            }
            if (APART) {
                // Listed elements leave the chunks in which something could be summed or reach the bound.
                const float low = LSE && want_lse ? fminf(skip_b, T_prev) : T_prev;
                block_max = NEG_INF;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool need = hit(u) != 0u && !(m8[u] < low);
                    const uint64_t nmask = __ballot(need);
                    if (nmask != 0ull) {
                        cur[u] = chunk_without<DT>(cur[u], need ? hit(u) : 0u);
                        m8[u] = chunk_max<DT>(cur[u]);
                        note_chunk((b * U + (uint32_t)u) * NT + tid, need, nmask);
                    }
                    block_max = max2_raw(block_max, m8[u]);
                }
            }
            if (APART) {
                lane_max = max2_raw(lane_max, block_max);
            } else {
                const Bits words = coarse_word(bits);
#pragma unroll
                for (int u = 0; u < U; u += 2) {
                    lane_max = max3_raw(lane_max, coarse_hit(words, u) ? NEG_INF : m8[u],
                                        coarse_hit(words, u + 1) ? NEG_INF : m8[u + 1]);
                }
            }
            lane_raw = max2_raw(lane_raw, block_max);
            bool some = false;
            if (LSE && want_lse) {
                // A term 2^(v*c2) below 2^-21 / vocab of the largest one cannot move the row sum by
                // more than 2^-21 of it, even with every element of the row at that level.
                skip_b = fmaxf(row_max, own_max) - lse_cut;
                some = __ballot(block_max > skip_b) != 0ull;
                if (!APART && some) {
                    // Between two refreshes the wave's own lanes may have seen more than the row knew.
                    own_max = wave_max_dpp(fmaxf(lane_max, lowered(lane_raw)));
                    skip_b = fmaxf(row_max, own_max) - lse_cut;
                    some = __ballot(block_max > skip_b) != 0ull;
                }
                wl.skip_below = skip_b;
                if (APART && some) {
                    wl.prepare(block_max < T_prev ? block_max : T_prev, c2);  // nothing above T_prev is added
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        wl.template add_prepared<DT>(cur[u], m8[u], c2, !(m8[u] >= T_prev));
                    }
                }
            }
            if (b < 4u || (b & 3u) == 0u) {
                const uint32_t noted = note_max;
                uint32_t count = sfill;
                if (LSE && !APART && want_lse && b == 0u) {
                    // (nothing is noted yet) chunks above the cut as this wave alone would place it:
                    // no fewer than lie above the row's
                    const float cut = wave_max_dpp(fmaxf(lane_max, lowered(lane_raw))) - lse_cut;
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        count += (uint32_t)__popcll(__ballot(m8[u] > cut));
                    }
                }
                const uint32_t counted =
                    refresh_bound(b == 0u, b == 0u || (LSE && want_lse && (b < 4u || (b & 7u) == 0u)), count);
                if (LSE && want_lse) {
                    skip_b = fmaxf(row_max, own_max) - lse_cut;
                    wl.skip_below = skip_b;
                    some = some && __ballot(block_max > skip_b) != 0ull;
                    note_max = b == 0u ? 0u : note_max;
                    if (!APART && b == 0u && counted * 8u >= first_chunks() * 7u) {
                        // Flat from the start?  Every wave counts its elements above the cut (where
                        // seven eighths of the block's chunks lie above): 31 of 32 of them, or seven
                        // eighths and, for every 256, a chunk with a value in the upper quarter of the
                        // way from the cut to the largest value.  A row with a heavy tail whose large values
                        // all come later holds seven eighths above its first block's cut one time in
                        // two thousand, but a dozen values in that quarter where a flat row holds
                        // more than forty; taken for a flat one it is the last of its launch by 12 us
                        // (one launch in eight for 200 rows in three slices, 44.1 -> 45.7 us on average).
                        const float high = skip_b + 0.75f * lse_cut;
                        // (Counted by the lanes: sums of ballots took scalar registers from the scan.)
                        uint32_t above = 0;   // (and the chunks of the upper quarter in the upper half)
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            float v[E];
                            unpack<DT>(cur[u], v);
#pragma unroll
                            for (int j = 0; j < E; ++j) {
                                above += v[j] > skip_b ? 1u : 0u;
                            }
                            above += m8[u] > high ? 0x10000u : 0u;
                        }
                        // (red_i: what is written behind the scan could overtake a wave that still
                        // reads here - a slice of one block has no barrier in between)
                        above = wave_scan_u32(above);
                        if (lane == 63u) {
                            sh.red_i[w] = above;
                        }
                        __syncthreads();
                        uint32_t all = 0;
                        for (int i = 0; i < NWAVE; ++i) {
                            all += sh.red_i[i];
                        }
                        const uint32_t held = first_chunks() * (uint32_t)E, low = all & 0xffffu;
                        if (low * 32u >= held * 31u || (low * 8u >= held * 7u && (all >> 16) * 256u >= held)) {
                            // (nothing of the block has been queued or noted: it is scanned again)
                            flat = true;
                            flat_from = 0u;
                            return;
                        }
                    } else if (!APART && b != 0u) {
                        // Would the fullest segment overflow before the next refresh, at a quarter
                        // more than the rate it grew at since the last one?  Then this block (not
                        // queued or noted yet) and those to come are scanned the other way; within
                        // the first four the few notes are dropped and the row is scanned again.
                        const uint32_t since = b <= 4u ? 1u : 4u, ahead = min(b < 4u ? 1u : 4u, nblocks - b);
                        if ((note_max - noted) * ahead * 5u > (SSEG - min(note_max, SSEG)) * since * 4u) {
                            flat = true;
                            flat_from = b < 4u ? 0u : b;
                            wq = b < 4u ? 0u : wq;
                            sfill = b < 4u ? 0u : sfill;
                            return;
                        }
                    }
                }
            }
            const bool any_late = LSE && want_lse && APART && T != T_prev &&
                                  __ballot(block_max >= T_prev && block_max > skip_b) != 0ull;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool pass = m8[u] >= T;
                const uint64_t mask = __ballot(pass);
                if (mask != 0ull) {
                    const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                    const uint32_t at = wq + rank;
                    if (pass && at < QSEG) {
                        L.qraw[w * QSEG + at] = cur[u];
                        L.qidx[w * QSEG + at] = g.cb + (b * U + u) * NT + tid;
                    }
                    wq += (uint32_t)__popcll(mask);
                }
                if (any_late) {
                    // At or above the previous bound but below the new one: not queued after all.
                    const bool late = m8[u] >= T_prev && !pass;
                    if (__ballot(late) != 0ull) {
                        wl.prepare(late ? m8[u] : NEG_INF, c2);
                        wl.template add_prepared<DT>(cur[u], m8[u], c2, late);
                    }
                }
                if (LSE && !APART && some) {
                    // Above the cut alone: the chunk's number is noted, its terms are formed behind the
                    // scan, against the final cut.
                    const bool note = !pass && m8[u] > skip_b;
                    const uint64_t nmask = __ballot(note);
                    if (nmask != 0ull) {
                        note_chunk((b * U + (uint32_t)u) * NT + tid, note, nmask);
                    }
                }
            }
        };
        // A request past the last block asks for the last block again: with the same loads in
        // flight on every path the wait for a block's data leaves the blocks requested after it in
        // flight (see select_stream()).
        auto request = [&](u32x4 (&dst)[U], Bits& d, uint32_t b) {
            if (APART) {
                fetch_exact(dst, d, min(b, nblocks - 1u));
            } else {
                fetch_coarse(dst, d, min(b, nblocks - 1u));
            }
        };
        if (APART && !FLAT) {
            request(buf_a, bits_a, b_first);
        }   // (otherwise block 0 was requested at the very start)
        request(buf_b, bits_b, b_first + 1u);
        for (uint32_t b = b_first; b < nblocks && !give_up && (APART || !flat); b += 3) {
            request(buf_c, bits_c, b + 2u);
            work(buf_a, bits_a, b);
            if (b + 1 < nblocks) {
                request(buf_a, bits_a, b + 3u);
                work(buf_b, bits_b, b + 1);
                if (b + 2 < nblocks) {
                    request(buf_b, bits_b, b + 4u);
                    work(buf_c, bits_c, b + 2);
                }
            }
        }
    };
    // fn(true value, id) for every listed id of the streamed chunks from first_c on: 2 048 words of the
    // bitmap a round (eight a thread, requested together); their ids are listed in LDS, in the notes'
    // place, and evaluated four a thread with all loads in flight.
    auto walk_listed = [&](uint32_t first_c, auto&& fn) {
        constexpr uint32_t PER = 8, LIST = S_CAP / 2;
        uint32_t* list = reinterpret_cast<uint32_t*>(L.noted);
        const uint32_t lo = first_c < g.main_hi ? g.id_of(first_c, 0) : 0u;
        const uint32_t hi = first_c < g.main_hi ? g.id_of(g.main_hi, 0) : 0u;
        const uint32_t w_end = (hi + 31u) >> 5;
        for (uint32_t w0 = lo >> 5; w0 < w_end; w0 += NT * PER) {
            uint32_t word[PER], mine = 0;
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i) {
                word[i] = gload(a.touched + min(w0 + i * NT + tid, row_words - 1u));
            }
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i) {
                word[i] &= range32_at(lo, hi, (int64_t)(w0 + i * NT + tid) * 32);
                mine += (uint32_t)__popc(word[i]);
            }
            const uint32_t incl = wave_scan_u32(mine);
            if (lane == 63u) {
                sh.red_i[w] = incl;
            }
            __syncthreads();   // (also: the list's place has been read by everybody)
            uint32_t at0 = incl - mine, total = 0;
            for (uint32_t i = 0; i < (uint32_t)NWAVE; ++i) {
                at0 += i < w ? sh.red_i[i] : 0u;
                total += sh.red_i[i];
            }
            __syncthreads();   // (the next round writes red_i again)
            for (uint32_t p0 = 0; p0 < total; p0 += LIST) {
                uint32_t at = at0;
#pragma unroll
                for (uint32_t i = 0; i < PER; ++i) {
                    for (uint32_t m = word[i]; m != 0u; m &= m - 1u, ++at) {
                        if (at - p0 < LIST) {
                            list[at - p0] = ((w0 + i * NT + tid) << 5) + (uint32_t)__builtin_ctz(m);
                        }
                    }
                }
                __syncthreads();
                const uint32_t n = min(total - p0, LIST);
                for (uint32_t e0 = tid; e0 < n; e0 += 4u * NT) {
                    uint32_t id[4], cnt[4];
                    float raw[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        id[q] = list[min(e0 + (uint32_t)q * NT, n - 1u)];
                        raw[q] = load_logit<DT>(a.logits, id[q]);
                        cnt[q] = gload(a.counts + id[q]);
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (e0 + (uint32_t)q * NT < n) {
                            fn(listed_value<DT>(a, raw[q], cnt[q]), id[q]);
                        }
                    }
                }
                __syncthreads();
            }
        }
    };
    if (nblocks == 0) {
        refresh_bound(true, true, 0u);  // the same barriers in every workgroup
    } else {
        if constexpr (FLAT) {
            // Where a slice comes here because its leading ids are listed ones by the hundred, what
            // is not listed says little about its k-th value: the listed ids' true values enter the
            // lanes' maxima ahead of the scan (each is an element of its own, like any other).
            walk_listed(g.main_lo, [&](float x, uint32_t) { lane_max = max2_raw(lane_max, x); });
        }
        if constexpr (!FLAT) {
            scan(std::false_type{}, 0u);
        }
        if ((FLAT || LSE) && flat && flat_from < nblocks && !give_up) {
            scan(std::true_type{}, flat_from);
        }
    }
    phase(cfg, 2);

    // ---- behind the scan
    const float wave_top = LSE && want_lse ? wave_max_dpp(fmaxf(lane_max, lowered(lane_raw))) : 0.0f;
    if (lane == 0) {
        sh.qfill[w] = !flat && sfill > SSEG ? QSEG + 1u : wq;
        sh.nfill[w] = sfill;
        sh.wmax[parity][w] = wave_top;
    }
    __syncthreads();
    phase(cfg, 14);
    const float filt = T;
    QueueOrder order, notes;
    order.init(sh.qfill);
    bool walk = false;   // flat rows with more chunks of listed ids than notes
    {
        uint32_t fill[NWAVE];
        bool overflow = give_up;
#pragma unroll
        for (int i = 0; i < NWAVE; ++i) {
            overflow = overflow || sh.qfill[i] > QSEG;
            walk = walk || sh.nfill[i] > SSEG;
            fill[i] = min(sh.nfill[i], SSEG);
        }
        notes.init(fill);
        if (overflow) {
            again = true;
            return stream_fail(cfg, 4u);
        }
    }
    // The terms formed from here on are relative to the largest value that is known to be there
    // (a term 2^900 above it - a listed id that the penalties leave far above everything else -
    // goes the way of the moving references).
    double ref_p = 0.0, acc_p = 0.0;
    bool simple_p = false;   // the same in every thread
    if (LSE && want_lse) {
        float m = sh.wmax[parity][0];
        for (int i = 1; i < NWAVE; ++i) {
            m = fmaxf(m, sh.wmax[parity][i]);
        }
        m = fmaxf(m, row_floor);
        skip_b = fmaxf(skip_b, m - lse_cut);
        simple_p = m > NEG_INF;
        ref_p = simple_p ? (double)m * c2d : 0.0;
        ref_p = ref_p < 1.0e30 ? (ref_p > -1.0e30 ? ref_p : -1.0e30) : 1.0e30;
    }
    auto add_term = [&](float x) {
        if (LSE && want_lse && x > skip_b) {
            const double d = __builtin_fma((double)x, c2d, -ref_p);
            if (simple_p && d <= 900.0) {
                acc_p += d > -1000.0 ? pow2_d(d) : 0.0;
            } else {
                acc_t += term_d(x);
            }
        }
    };
    auto offer = [&](float u, uint32_t id) {
        if (u >= filt && u > NEG_INF) {
            const uint32_t at = atomicAdd(&sh.n_fc, 1u);
            if (at < FC_CAP) {
                L.fc[at] = composite_of(u / a.temperature, id);
            }
        }
    };
    const uint32_t flat_chunk = flat ? g.cb + flat_from * BLOCK : 0xffffffffu;   // the first chunk without its listed ids
    // The noted chunks: their 16 bytes and their bits are asked for first, four chunks a thread,
    // and looked at behind the queue's listing below, which touches LDS only.
    uint32_t n_cc[4] = {0u, 0u, 0u, 0u}, n_dm[4] = {0u, 0u, 0u, 0u};
    u32x4 n_q[4] = {};
    bool n_ok[4] = {false, false, false, false};
    auto noted_request = [&](uint32_t e0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t e = e0 + (uint32_t)i * NT;
            const uint32_t c = g.cb + (uint32_t)L.noted[notes.template slot<SSEG>(min(e, notes.total - 1u))];
            // (A chunk outside the slice was scanned as -inf throughout, and is noted where
            // chunk maxima are the kind that reports +0 for it.)
            n_ok[i] = e < notes.total && c >= g.main_lo && c < g.main_hi && !(walk && c >= flat_chunk);
            n_cc[i] = min(c, c_last);
            n_q[i] = gload(reinterpret_cast<const u32x4*>(g.base + (n_cc[i] << 4)));
            n_dm[i] = bits32_at(a.touched, row_words, (int64_t)g.id_of(n_cc[i], 0)) & EMASK;
        }
    };
    // Elements above the final cut (or bound) count with their true values; of a flat row's chunks
    // only the listed ones (the others were summed and queued as they came).  The four chunks' first
    // counts are requested together: a chunk rarely holds a second listed id.
    auto noted_consume = [&]() {
        const float low = LSE && want_lse ? fminf(skip_b, filt) : filt;
        uint32_t todo[4], cnt0[4], j0[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            todo[i] = 0;
            float v[E];
            unpack<DT>(n_q[i], v);
#pragma unroll
            for (int j = 0; j < E; ++j) {
                todo[i] |= v[j] >= low && v[j] > NEG_INF ? 1u << j : 0u;
            }
            todo[i] &= n_ok[i] ? (n_cc[i] >= flat_chunk ? n_dm[i] : EMASK) : 0u;
            const uint32_t listed = todo[i] & n_dm[i];
            j0[i] = listed != 0u ? (uint32_t)__builtin_ctz(listed) : 0u;
            cnt0[i] = gload(a.counts + min(g.id_of(n_cc[i], (int)j0[i]), g.vocab - 1u));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll 1
            for (uint32_t m = todo[i]; m != 0u; m &= m - 1u) {
                const uint32_t j = (uint32_t)__builtin_ctz(m);
                const uint32_t id = g.id_of(n_cc[i], (int)j);
                float x = chunk_elem<DT>(n_q[i], j);
                if ((n_dm[i] >> j) & 1u) {
                    x = listed_value<DT>(a, x, j == j0[i] ? cnt0[i] : gload(a.counts + id));
                }
                add_term(x);
                offer(x, id);   // (nothing of a chunk that was noted for its sum reaches the bound)
            }
        }
    };
    constexpr bool NOTES = LSE || FLAT;
    if (NOTES && notes.total != 0u) {
        noted_request(tid);
    }
    if (!FLAT && (!flat || flat_from != 0u)) {
        stream_pairs_list<DT>(L, g, order, filt, LSE && want_lse ? skip_b : __builtin_huge_valf(), sh,
                              [&](uint32_t c) { return c < flat_chunk; }, [](uint32_t) { return false; });
    }
    __syncthreads();
    const bool paired = sh.n_pairs <= FC_CAP;
    if (!FLAT && paired && (!flat || flat_from != 0u)) {
        stream_pairs_take(L, a, filt, sh, add_term);
    }
    // Chunks without their listed ids (flat rows), and all of them where the pairs outgrew their
    // place: one thread per queued chunk.
    if (flat || !paired) {
        for (uint32_t ch = tid; ch < order.total; ch += NT) {
            const uint32_t slot = order.template slot<QSEG>(ch);
            const uint32_t c = L.qidx[slot];
            const bool bare = c >= flat_chunk;
            if (!bare && paired) {
                continue;
            }
            const u32x4 q = L.qraw[slot];
            const uint32_t dm = bare ? 0u : bits32_at(a.touched, row_words, (int64_t)g.id_of(c, 0)) & EMASK;
#pragma unroll 1
            for (uint32_t j = 0; j < (uint32_t)E; ++j) {
                float x = chunk_elem<DT>(q, j);
                if (!(x >= filt) && !(LSE && want_lse && x > skip_b)) {
                    continue;
                }
                const uint32_t id = g.id_of(c, (int)j);
                if ((dm >> j) & 1u) {
                    x = listed_value<DT>(a, x, gload(a.counts + id));
                }
                add_term(x);
                offer(x, id);
            }
        }
    }
    if (NOTES && notes.total != 0u) {
        for (uint32_t e0 = tid;; ) {
            noted_consume();
            e0 += 4u * NT;
            if (e0 - tid >= notes.total) {   // (the same trips in every thread)
                break;
            }
            noted_request(e0);
        }
    }
    phase(cfg, 8);
    if (NOTES && walk) {
        walk_listed(max(flat_chunk, g.main_lo), [&](float x, uint32_t id) {
            add_term(x);
            offer(x, id);
        });
    }
    // Ids of partial 16-byte chunks at the row's ends were not streamed: exact, one by one.
    for (int side = 0; side < 2; ++side) {
        const uint32_t lo = side == 0 ? g.id_lo : g.edge_hi_begin;
        const uint32_t hi = side == 0 ? g.edge_lo_end : g.id_hi;
        for (uint32_t id = lo + tid; id < hi; id += NT) {
            const float x = listed_value<DT>(a, load_logit<DT>(a.logits, id), gload(a.counts + id));
            add_term(x);
            offer(x, id);
        }
    }
    phase(cfg, 9);
    if (LSE && want_lse) {
        StreamSums sums;
        sums.ref_s = ref_s;
        sums.up = up;
        sums.acc_t = acc_t;
        sums.acc_r = 0.0;
        sums.ref_p = ref_p;
        sums.acc_p = acc_p;
        sums.simple_p = simple_p;
        stream_row_sum<DT>(a, g, sums, wl, sh, cfg);
    }
    __syncthreads();
    const bool stands = stream_accept(L, filt, a.temperature, k, sh, cfg, sorted, out);
    again = !stands;
    return stands;
}

}  // namespace lily
