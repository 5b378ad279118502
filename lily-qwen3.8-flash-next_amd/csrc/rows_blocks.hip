// rows_blocks.hip - rows of few candidates (k <= 64) in slices of several blocks, a block at a time in
// registers.  Compiled once per logits type: -DLILY_DT=0|1.
//
// The way of rows_held.hip for batches whose slices are longer: a thread holds 16 (f32) or 32 (bf16) values of
// a block while the next one is on its way.  Listed ids leave their chunks as they pass and are noted
// where their raw value might matter; a wave evaluates its notes four a lane at a time.  So the bound is one of
// true values, the row's sum takes every value once as it passes, what reaches the bound as it stands is listed
// with its value, and at the end those that still reach it are ranked; nothing is looked at twice.
//
// A block of a dense history (an eighth of the ids and more) lists more than a wave's notes hold: the wave then evaluates
// them straight from their bits, where nothing else gives a bound once for that and once more for the list and the
// sum.  us a launch, 200 bf16 rows of 151 936, N(0, 2^2), 13 / 25 / 60 % of the ids listed 59 / 72 / 103 (the flat form of
// select_lowering.h 107 / 136 / 285; given up to the exhaustive select, as such slices once were, 670 to 680), half of the first
// tenth listed 52 (79).
//
// Clusters of likely ids fill some waves and leave others what lies behind; the bound is the poorest wave's, and all of a
// cluster reaches it.  A wave whose list might run over goes on behind a bound of its own, from its chunks and its list, which
// it makes short.  (600 bf16 rows of 151 936, k = 20, 1 000 neighbours 9 above the rest: 54 us, the streaming select 49;
// 2 480 when such slices were given up.  3 000 inside the row: 49, 43 and 2 480.  For rows without clusters the look costs 0.3 to 0.6 us.)
//
// Bound: the vector unit where the row's sum takes most values (200 rows of 248 320 bf16, N(0, 2^2), under penalties:
// 50 us a launch for 99 MB, 25 vector instructions a value, which keep the unit busy two thirds of the time; 74 through
// the flat form of select_lowering.h, whose scan spends fewer but behind whose scan the noted chunks are looked at again), the memory
// where it does not (1 000 rows of 151 936, k = 64, without log-probabilities 50 us, 6.1 TB/s; 1 024 rows 62 through
// select_stream.h).  Rows with a heavy tail, whose sum takes a few chunks, are no faster this way than through
// select_lowering.h (200 rows of 151 936, 0.5 / 5 / 10 % listed 33.1 / 35.8 / 37.2 us, 32.8 / 34.8 / 36.8 there; 13 % 39, 77 there; 200 rows of
// 248 320 39.5 / 43.7 / 46.3, 38.1 / 39.3 / 90 there).
// A chunk with values for the list offers them one by one: a wave-wide test each, most of them for nothing, takes
// fewer instructions than finding the ones there are (53.0 -> 50.8 us for the 200 rows of 248 320).
// Tried: listed ids evaluated as their chunks pass (a round trip a block: 82 us for 1 024 rows with a heavy tail,
// 74 this way), all of them ahead of the blocks (138 us: their gathers read more than the row), three copies
// of the loop for two blocks on their way (leaves the instruction cache: 3 to 10 % longer).
#include <type_traits>

#include "launch.h"
#include "row_kernel.h"

#if !defined(LILY_DT)
#error "compile with -DLILY_DT=<lily_dtype>"
#endif

namespace lily {

namespace {

constexpr uint32_t LIST_SEG = 640;                   // values a wave lists: 64 chunks', and 64 candidates with their ties
constexpr uint32_t LIST_CAP = LIST_SEG * NWAVE;
constexpr uint32_t FINAL_CAP = 512;                  // ... of which so many reach the last bound
constexpr uint32_t NOTE_SEG = 512;                   // listed ids a wave notes before it evaluates them
// Dynamic LDS: the listed (value, id) pairs, the final candidates, the ranked ones.
constexpr uint32_t OFF_FINAL = LIST_CAP, OFF_RANKED = OFF_FINAL + FINAL_CAP, OFF_UPPER = OFF_RANKED + 64;
constexpr uint32_t OFF_NOTES = OFF_UPPER + 64;
constexpr uint32_t BLOCKS_LDS_BYTES = OFF_NOTES * 8 + NOTE_SEG * NWAVE * 4;
static_assert(BLOCKS_LDS_BYTES >= WAVE_MERGE_SLOTS * 8, "one wave's merge works at the front");

// PEN: rows under penalties are among the launch's.  True in the wave that finished the row.
template <int DT, bool LSE, bool PEN>
__device__ __forceinline__ bool blocks_row(const LILY_CONST RowArgs* src, const LaunchCfg& cfg, Shared& sh) {
    if (cfg.served != nullptr && *(const LILY_CONST uint32_t*)(cfg.served + blockIdx.y) != 0u) {
        return false;
    }
    constexpr int E = Geo<DT>::E, U = (int)STREAM_UNROLL;
    constexpr uint32_t EMASK = (1u << E) - 1u, BLOCK = NT * U;
    RowArgs a;
    load_row_args(a, src);
    apply_selection(a);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t s = blockIdx.x, row = blockIdx.y, S = cfg.slices, vocab = cfg.vocab;
    const bool want_lse = LSE && a.out_logprob != nullptr;
    const bool forced = (a.flags & F_FORCED) != 0u;
    if (forced && !want_lse) {
        if (s == 0 && tid == 0) {
            emit(a, a.forced, vocab);
        }
        return s == 0 && w == 0;
    }
    Geo<DT> g;
    g.init(a.logits, vocab, s, S);
    phase(cfg, 0);
    const uint32_t nblocks = (g.ce - g.cb + BLOCK - 1u) / BLOCK;
    const uint32_t c_last = g.ce - 1u;
    const bool pen = PEN && (a.flags & F_PEN) != 0u;
    struct Bits16 {
        uint16_t v;
    } __attribute__((packed));
    auto chunk_of = [&](uint32_t b, int u) -> uint32_t { return g.cb + (b * U + (uint32_t)u) * NT + tid; };
    struct Block {
        u32x4 raw[U];
        uint32_t bits[U];
    } next;
    // (a row without penalties asks for bits all the same, of its logits: as many loads on every path, or a
    // wait for one block would wait for those behind it)
    const char* listed = pen ? reinterpret_cast<const char*>(a.touched) : g.base;
    // Every load is issued whatever its chunk: chunks past the slice's end are its last one, blocks past its
    // last one that.
    auto fetch = [&](uint32_t b_asked) {
        const uint32_t b = min(b_asked, max(nblocks, 1u) - 1u);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            next.raw[u] = gload(reinterpret_cast<const u32x4*>(g.base + (min(chunk_of(b, u), c_last) << 4)));   // (rows are below 4 GiB)
        }
        if (PEN) {
            // (two bytes of the bitmap of listed ids hold a chunk's bits, wherever the row starts)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int32_t first = (int32_t)(min(chunk_of(b, u), c_last) * (uint32_t)E) - (int32_t)g.pad;
                next.bits[u] = ((const LILY_GLOBAL Bits16*)(listed + (max(first, 0) >> 3)))->v;
            }
        }
    };
    fetch(0u);
    auto true_value = [&](float x, uint32_t count) -> float {
        if (count > 0u) {
            x = x > 0.0f ? x / a.repetition : x * a.repetition;
            x -= a.presence + a.frequency * (float)count;
        }
        return x;
    };
    // Ids of partial chunks at the row's ends, one a thread (fewer than 16 at either end).
    uint32_t edge = 0xffffffffu;
    if (tid < 64u) {
        edge = g.id_lo + tid < g.edge_lo_end ? g.id_lo + tid : edge;
    } else if (tid < 128u) {
        edge = g.edge_hi_begin + tid - 64u < g.id_hi ? g.edge_hi_begin + tid - 64u : edge;
    }
    float ev = NEG_INF;
    if (edge != 0xffffffffu) {
        ev = true_value(load_logit<DT>(a.logits, edge), pen ? gload(a.counts + edge) : 0u);
        ev = ev > NEG_INF ? ev : NEG_INF;
    }
    phase(cfg, 1);

    // ---- the blocks
    const uint32_t kw = (min(a.k, 64u * NWAVE) + NWAVE - 1u) / NWAVE;
    // A term below 2^-21 / vocab of the largest one cannot move the row's sum by more than 2^-21 of it.
    const float lse_cut = (log2f((float)vocab) + 21.0f) * (a.temperature * 0.6931471805599453f);
    float lane_max = ev;        // of true values
    float T = F32_LOWEST;       // the bound, the same in every thread of a wave
    float skip = NEG_INF;       // chunks at or below it are left out of the sum
    float ref = F32_LOWEST;     // the wave's reference: terms are 2^(x * c2 - ref)
    double sum = 0.0;
    uint32_t fill = 0;          // this wave's listed values
    uint32_t noted = 0;         // ... and noted ids
    uint32_t* notes = reinterpret_cast<uint32_t*>(dyn_lds + OFF_NOTES) + w * NOTE_SEG;
    const bool raising = pen && !(a.repetition >= 1.0f && a.presence >= 0.0f && a.frequency >= 0.0f);
    uint32_t parity = 0;
    uint64_t* pairs = dyn_lds;  // [NWAVE][LIST_SEG]: value's bits << 32 | id
    auto list = [&](bool pass, float x, uint32_t id) {
        const uint64_t mask = __ballot(pass);
        if (mask != 0ull) {
            const uint32_t at = fill + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            if (pass && at < LIST_SEG) {
                pairs[w * LIST_SEG + at] = ((uint64_t)lilym_f32_bits(x) << 32) | id;
            }
            fill += (uint32_t)__popcll(mask);
        }
    };
    auto power = [&](float x) -> float { return __builtin_amdgcn_exp2f(__builtin_fmaf(x, a.c2, -ref)); };
    // k values reach the least of the waves' ceil(k / NWAVE)-th largest lane maxima.
    auto refresh = [&]() {
        const uint32_t P = wave_kth_key16(lane_max > NEG_INF ? (lilym_order_key(lane_max) >> 16) : 0u, kw);
        const float wave_top = LSE && want_lse ? wave_max_dpp(lane_max) : 0.0f;
        if (lane == 0u) {
            sh.bound[parity][w] = P != 0u ? lilym_key_value(P << 16) : F32_LOWEST;
            sh.wmax[parity][w] = wave_top;
        }
        __syncthreads();
        float t = sh.bound[parity][0], top = sh.wmax[parity][0];
        for (int i = 1; i < NWAVE; ++i) {
            t = fminf(t, sh.bound[parity][i]);
            top = fmaxf(top, sh.wmax[parity][i]);
        }
        // (values a little below the bound may share its quotient by the temperature)
        T = forced ? __builtin_huge_valf() : fmaxf(T, lower_by_slack(t));
        skip = LSE && want_lse ? top - lse_cut : skip;
        parity ^= 1u;
    };
    // Terms would dwarf the wave's reference: it moves up to the wave's largest.
    auto raise = [&](float largest) {
        if (__ballot(__builtin_fmaf(largest, a.c2, -ref) > LSE_RAISE) != 0ull) {
            const float now = fminf(fmaxf(wave_max_dpp(largest) * a.c2, -1.0e30f), 1.0e30f);
            sum *= (double)__builtin_amdgcn_exp2f(ref - now);
            ref = now;
        }
    };
    // A listed id's true value, t (NEG_INF in lanes without one), once there is a bound.
    auto take = [&](float t, uint32_t id) {
        const bool in = t >= T;
        list(in, t, id);
        if (LSE && want_lse) {
            raise(t);
            const double d = __builtin_fma((double)t, (double)a.c2, -(double)ref);
            sum += !in && d > -1000.0 ? pow2_d(d) : 0.0;
        }
    };
    // The wave's list made short: the k-th largest value on it is a bound (this wave's from here on, a little below it as
    // ever), what does not reach it goes into the sum.  (Ties stay; with too many of them the list overflows.)
    // (It is rare, and read from LDS over and over: what it would hold in registers the blocks need.)
    auto compact = [&]() {
        const uint32_t n = min(fill, LIST_SEG);
        uint32_t found = 0u;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // (LDS of this wave: in order already)
        __builtin_amdgcn_wave_barrier();
        const uint32_t* values = reinterpret_cast<const uint32_t*>(pairs + w * LIST_SEG) + 1;   // (the upper halves)
        auto key_of = [&](uint32_t i0) -> uint32_t {   // 0 past the last
            const uint32_t key = lilym_order_key(lilym_bits_f32(values[2u * min(i0 + lane, LIST_SEG - 1u)]));
            return i0 + lane < n ? key : 0u;
        };
        uint32_t hi = 0u, lo = 0xffffffffu;
#pragma unroll 5
        for (uint32_t i0 = 0; i0 < LIST_SEG; i0 += 64u) {
            const uint32_t key = key_of(i0);
            hi = max(hi, key);
            lo = key != 0u ? min(lo, key) : lo;
        }
        hi = wave_max_u32(hi);
        lo = wave_min_u32(lo);
        if (n < a.k) {
            return;
        }
        // (from the first bit in which the values differ to where just k reach)
        const int bits = hi != lo ? 32 - __builtin_clz(hi ^ lo) : 0;
        found = bits < 32 ? hi >> bits << bits : 0u;
#pragma unroll 1
        for (int bit = bits - 1; bit >= 0; --bit) {
            const uint32_t at = found | (1u << bit);
            uint32_t reach = 0;
#pragma unroll 5
            for (uint32_t i0 = 0; i0 < LIST_SEG; i0 += 64u) {
                reach += (uint32_t)__popcll(__ballot(key_of(i0) >= at));
            }
            found = reach >= a.k ? at : found;
            if (reach == a.k) {
                break;
            }
        }
        T = fmaxf(T, lower_by_slack(lilym_key_value(found)));
        fill = 0u;
#pragma unroll 1
        for (uint32_t i0 = 0; i0 < n; i0 += 64u) {   // (what stays moves to places that have been read)
            const uint64_t p = pairs[w * LIST_SEG + min(i0 + lane, n - 1u)];
            __builtin_amdgcn_wave_barrier();
            const float x = lilym_bits_f32((uint32_t)(p >> 32));
            const bool there = i0 + lane < n, stays = there && x >= T;
            list(stays, x, (uint32_t)p);
            __builtin_amdgcn_wave_barrier();
            if (LSE && want_lse) {
                raise(there && !stays ? x : NEG_INF);
                const double d = __builtin_fma((double)x, (double)a.c2, -(double)ref);
                sum += there && !stays && d > -1000.0 ? pow2_d(d) : 0.0;
            }
        }
    };
    // The noted ids, by the wave that noted them, four a lane with all loads in flight.
    auto drain = [&]() {
        const uint32_t n = noted;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // (LDS of this wave: in order already)
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (uint32_t e0 = 0; e0 < n; e0 += 256u) {
            if (fill > LIST_SEG - 256u && fill <= LIST_SEG) {
                compact();
            }
            uint32_t id[4], count[4];
            float x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                id[q] = min(notes[min(e0 + (uint32_t)q * 64u + lane, n - 1u)], vocab - 1u);
                x[q] = load_logit<DT>(a.logits, id[q]);
                count[q] = gload(a.counts + id[q]);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (e0 + (uint32_t)q * 64u < n) {
                    float t = e0 + (uint32_t)q * 64u + lane < n ? true_value(x[q], count[q]) : NEG_INF;
                    t = t > NEG_INF ? t : NEG_INF;
                    lane_max = fmaxf(lane_max, t);
                    take(t, id[q]);
                }
            }
        }
        noted = 0u;
    };
    // A block's listed ids straight from their bits (E a chunk), where the notes have no room for them; `bounded`: taken,
    // else looked at for the bound.
    auto settle = [&](uint32_t b, uint32_t left, bool bounded) {
#pragma unroll 1
        while (__ballot(left != 0u) != 0ull) {
            if (bounded && fill > LIST_SEG - 256u && fill <= LIST_SEG) {
                compact();
            }
            uint32_t id[4], count[4];
            float x[4];
            bool in[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                in[q] = left != 0u;
                const uint32_t at = in[q] ? (uint32_t)__builtin_ctz(left) : 0u;
                left &= left - 1u;
                id[q] = in[q] ? chunk_of(b, (int)(at / (uint32_t)E)) * (uint32_t)E + at % (uint32_t)E - g.pad : 0u;
                x[q] = load_logit<DT>(a.logits, id[q]);
                count[q] = gload(a.counts + id[q]);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float t = in[q] ? true_value(x[q], count[q]) : NEG_INF;
                t = t > NEG_INF ? t : NEG_INF;
                lane_max = fmaxf(lane_max, t);
                if (bounded) {
                    take(t, id[q]);
                }
            }
        }
    };
    // (One copy of the loop's code, each block's registers handed over by moves: three copies, for two blocks on
    // their way, left the instruction cache and were the slower way at every size.)
    StreamPriority prio;
    prio.init(nblocks);
#pragma unroll 1
    for (uint32_t b = 0; b < nblocks; ++b) {
        prio.set(b);
        u32x4 cur[U];
        uint32_t away[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            cur[u] = next.raw[u];
            away[u] = PEN && pen ? (next.bits[u] >> ((chunk_of(b, u) * (uint32_t)E - g.pad) & 7u)) & EMASK : 0u;
        }
        if (!(g.cb + b * BLOCK >= g.main_lo && g.cb + (b + 1u) * BLOCK <= g.main_hi)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t c = chunk_of(b, u);
                if (c < g.main_lo || c >= g.main_hi) {
                    const uint32_t ninf = DT == LILY_BF16 ? 0xff80ff80u : 0xff800000u;
                    cur[u] = u32x4{ninf, ninf, ninf, ninf};
                    away[u] = 0u;   // (what the bits there stand for lies outside the row)
                }
            }
        }
        fetch(b + 1u);
        // Once the bound and the cut are positive a chunk without a positive value cannot matter to either: the
        // cheaper maximum, +0 for all such chunks.
        const float low = LSE && want_lse ? fminf(T, skip) : T;
        const bool positive = DT == LILY_BF16 && __builtin_amdgcn_readfirstlane((int)(low > 0.0f)) != 0;
        float cm[U], block_max = NEG_INF;
        bool nan_seen = false;
        if (positive) {
            int top = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                cm[u] = chunk_max_nonneg<DT>(cur[u]);
                top = max(top, (int)lilym_f32_bits(cm[u]));
            }
            // (a positive NaN's pattern lies above +inf's: the maxima are taken again, ignoring it)
            nan_seen = __ballot(top > 0x7f800000) != 0ull;
        }
        if (!positive || nan_seen) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                cm[u] = chunk_max<DT>(cur[u]);
            }
        }
        // Listed ids leave the chunks whose raw values might matter (their true ones lie no higher, where
        // penalties only lower) and are noted, to be evaluated by the hundred.  In the other chunks, which
        // reach neither the bound nor the cut, they may stay.  The first block's are noted when it has given a bound
        // (before, all of them were: 200 rows with a heavy tail, 10 % listed, 43.7 -> 40.3 us).
        const uint32_t noted_before = noted;
        auto note = [&](int u, uint64_t mask) {
            uint32_t left = away[u];
            do {
                const uint32_t at = noted + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                if (left != 0u && at < NOTE_SEG) {
                    notes[at] = chunk_of(b, u) * (uint32_t)E + (uint32_t)__builtin_ctz(left) - g.pad;
                }
                noted += (uint32_t)__popcll(mask);
                left &= left - 1u;
                mask = __ballot(left != 0u);
            } while (mask != 0ull);
        };
        auto bits = [&]() -> uint32_t {
            uint32_t all = 0u;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                all |= away[u] << (u * E);
            }
            return all;
        };
        if (PEN && pen && b != 0u) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                away[u] = raising || cm[u] >= low ? away[u] : 0u;
                const uint64_t mask = __ballot(away[u] != 0u);
                if (mask != 0ull) {
                    cur[u] = chunk_without<DT>(cur[u], away[u]);
                    cm[u] = chunk_max<DT>(cur[u]);
                    note(u, mask);
                }
            }
        }
        if (PEN && pen && b == 0u) {
            float raw_max[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                raw_max[u] = cm[u];
                cur[u] = chunk_without<DT>(cur[u], away[u]);
                cm[u] = chunk_max<DT>(cur[u]);
                lane_max = max2_raw(lane_max, cm[u]);
            }
            refresh();
            if (T == F32_LOWEST) {   // (the same in every thread as yet: what is not listed does not suffice for a bound)
                settle(b, bits(), false);
                refresh();
            }
            const float low_now = LSE && want_lse ? fminf(T, skip) : T;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                away[u] = raising || raw_max[u] >= low_now ? away[u] : 0u;
                const uint64_t mask = __ballot(away[u] != 0u);
                if (mask != 0ull) {
                    note(u, mask);
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                block_max = max2_raw(block_max, cm[u]);
            }
            lane_max = max2_raw(lane_max, block_max);
            // (the last block's comes behind its notes, which it takes in; one a block for four blocks: 400 rows, k = 64, with
            // log-probabilities 45.4 -> 44.8 us without the third's)
            if (PEN ? (b < 2u || (b & 3u) == 3u) && b + 1u < nblocks : b < 2u || (b & 3u) == 3u || b + 1u == nblocks) {
                refresh();
            }
        }
        if (PEN) {
            if (pen) {
                const bool crowd = noted > NOTE_SEG;   // (a dense history: the wave goes by the block's bits)
                noted = crowd ? noted_before : noted;
                if (noted > NOTE_SEG / 2u || b + 1u == nblocks) {
                    drain();
                }
                if (crowd) {
                    settle(b, bits(), true);
                }
            }
            if (b + 1u == nblocks) {
                refresh();
            }
        }
        // Values that might not all find a place: a cluster of likely ids, of which the other waves have few, whose
        // bounds are the least.  Behind the k-th largest of the block's chunks no more than k have any, and a list of k is there.
        uint64_t reaches[U];
        uint32_t reaching = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            reaches[u] = __ballot(cm[u] >= T);
            reaching += (uint32_t)__popcll(reaches[u]);
        }
        if (fill + (uint32_t)E * reaching > LIST_SEG && fill <= LIST_SEG) {
            uint32_t key[U], found = 0u;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                key[u] = cm[u] > NEG_INF ? lilym_order_key(cm[u]) >> 16 : 0u;
            }
#pragma unroll 1
            for (uint32_t bit = 0x8000u; bit != 0u; bit >>= 1) {
                uint32_t reach = 0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    reach += (uint32_t)__popcll(__ballot(key[u] >= (found | bit)));
                }
                found = reach >= a.k ? found | bit : found;
            }
            T = found != 0u ? fmaxf(T, lower_by_slack(lilym_key_value(found << 16))) : T;
            compact();
#pragma unroll
            for (int u = 0; u < U; ++u) {
                reaches[u] = __ballot(cm[u] >= T);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool some = reaches[u] != 0ull;
            const bool summed = LSE && want_lse && __ballot(cm[u] > skip) != 0ull;
            if (!some && !summed) {
                continue;
            }
            float v[E];
            unpack<DT>(cur[u], v);
            if (some) {
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    list(v[j] >= T, v[j], chunk_of(b, u) * (uint32_t)E + (uint32_t)j - g.pad);
                    if (LSE) {
                        v[j] = v[j] >= T ? NEG_INF : v[j];   // (their terms are formed with the list's)
                    }
                }
            }
            if (summed) {
                raise(cm[u]);
                float all;
                for (;;) {
                    float e[E];
#pragma unroll
                    for (int j = 0; j < E; ++j) {
                        e[j] = power(v[j]);
                    }
                    const float four = (e[0] + e[1]) + (e[2] + e[3]);
                    all = E == 8 ? four + ((e[4 % E] + e[5 % E]) + (e[6 % E] + e[7 % E])) : four;
                    if (__ballot(all != all) == 0ull) {
                        break;
                    }
                    // (a NaN counts as -inf)
#pragma unroll
                    for (int j = 0; j < E; ++j) {
                        v[j] = v[j] == v[j] ? v[j] : NEG_INF;
                    }
                }
                sum += (double)all;
            }
        }
    }
    if (nblocks == 0u) {
        refresh();
    }
    if (fill > FINAL_CAP / NWAVE && fill <= LIST_SEG) {
        // (what all waves list is to be ranked in one piece)
        uint32_t reach = 0;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (uint32_t i0 = 0; i0 < fill; i0 += 64u) {
            const float x = lilym_bits_f32((uint32_t)(pairs[w * LIST_SEG + min(i0 + lane, fill - 1u)] >> 32));
            reach += (uint32_t)__popcll(__ballot(i0 + lane < fill && x >= T));
        }
        if (reach > FINAL_CAP / NWAVE) {
            compact();
        }
    }
    if (__ballot(edge != 0xffffffffu) != 0ull) {
        list(ev >= T && ev > NEG_INF, ev, edge);
        if (LSE && want_lse) {
            raise(ev);
            sum += (double)power(ev >= T ? NEG_INF : ev);
        }
    }
    phase(cfg, 2);

    // ---- behind the blocks: what still reaches the bound
    if (LSE && want_lse) {
        const double all = wave_sum_d(sum);
        if (lane == 0u) {
            sh.red_d[w] = all;
            sh.wthr[w] = ref;
        }
    }
    if (lane == 0u) {
        sh.qfill[w] = fill;
        sh.bound[parity][w] = T;
    }
    if (tid == 0u) {
        sh.n_fc = 0u;
    }
    uint64_t* final = dyn_lds + OFF_FINAL;
    uint64_t* ranked = dyn_lds + OFF_RANKED;
    uint32_t* upper = reinterpret_cast<uint32_t*>(dyn_lds + OFF_UPPER);   // [128]
    if (tid < 64u) {
        ranked[tid] = 0ull;
    }
    __syncthreads();
    uint32_t total = 0;
    bool overflow = false;
    uint32_t ends[NWAVE];   // of the waves' segments, as one list
    for (int i = 0; i < NWAVE; ++i) {
        total += sh.qfill[i];
        ends[i] = total;
        overflow = overflow || sh.qfill[i] > LIST_SEG;
        T = fmaxf(T, sh.bound[parity][i]);   // (any wave's)
    }
    double mc = 0.0, rest = 0.0;   // the reference of the slice's sum, and the sum of what was not listed
    if (LSE && want_lse) {
        float top = sh.wthr[0];
        for (int i = 1; i < NWAVE; ++i) {
            top = fmaxf(top, sh.wthr[i]);
        }
        mc = top > F32_LOWEST ? (double)top : 0.0;
        for (int i = 0; i < NWAVE; ++i) {
            const double d = (double)sh.wthr[i] - mc;
            rest += d > -1000.0 ? sh.red_d[i] * pow2_d(d) : 0.0;
        }
    }
    double listed_sum = 0.0;
    if (!overflow) {
        const uint32_t rounds = (total + NT - 1u) / NT;
        for (uint32_t q = 0; q < rounds; ++q) {
            const uint32_t i = q * NT + tid;
            const uint32_t seg = (i >= ends[0] ? 1u : 0u) + (i >= ends[1] ? 1u : 0u) + (i >= ends[2] ? 1u : 0u);
            const uint32_t from = seg == 0u ? 0u : seg == 1u ? ends[0] : seg == 2u ? ends[1] : ends[2];
            const uint64_t p = i < total ? pairs[seg * LIST_SEG + i - from] : 0ull;
            const float x = lilym_bits_f32((uint32_t)(p >> 32));
            if (LSE && want_lse && i < total) {
                // (in double: these carry most of the sum)
                const double d = __builtin_fma((double)x, (double)a.c2, -mc);
                listed_sum += d > -1000.0 ? pow2_d(d < 900.0 ? d : 900.0) : 0.0;
            }
            const bool stays = i < total && x >= T;
            const uint64_t mask = __ballot(stays);
            if (mask != 0ull) {
                uint32_t base = 0;
                if (lane == 0u) {
                    base = atomicAdd(&sh.n_fc, (uint32_t)__popcll(mask));
                }
                base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                const uint32_t at = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                if (stays && at < FINAL_CAP) {
                    final[at] = composite_of(x / a.temperature, (uint32_t)p);
                }
            }
        }
        if (LSE && want_lse) {
            listed_sum = wave_sum_d(listed_sum);
            if (lane == 0u) {
                sh.red3[0][w] = listed_sum;
            }
        }
    }
    __syncthreads();
    phase(cfg, 8);
    uint32_t n = sh.n_fc;
    overflow = overflow || n > FINAL_CAP;
    if (cfg.path_stats != nullptr && tid == 0u) {
        atomicAdd(&cfg.path_stats[overflow ? 2 : 0], 1u);
    }
    if (LSE && want_lse && !overflow && tid == 0u) {
        double all = rest;
        for (int i = 0; i < NWAVE; ++i) {
            all += sh.red3[0][i];
        }
        sh.lse_mc = mc;
        sh.lse_s = all;
    }
    uint64_t c = 0ull;      // a candidate per lane of the first wave, in order
    if (!overflow && n <= 64u) {
        if (w != 0u) {
            return false;
        }
        c = wave_sort_desc(lane < n ? final[lane] : 0ull);
    } else {
        if (overflow) {
            // Ties by the thousand, or values that rise all along the slice.
            __syncthreads();   // (n_fc has been read)
            select_exhaustive<DT>(a, g.id_lo, g.id_hi, a.k, want_lse, final, 64u, sh);
            n = min(sh.n_cand, 64u);
        }
        // Two threads an entry, each counts what it has ahead of it in one half of the list, sixteen at a time.
        const uint32_t half_n = (n + 31u) / 32u * 16u;   // (of a list filled up with zeros)
        for (uint32_t i = n + tid; i < 2u * half_n; i += NT) {
            final[i] = 0ull;
        }
        __syncthreads();
        for (uint32_t e0 = 0; e0 < n; e0 += 128u) {
            const uint32_t entry = e0 + (tid & 127u), half = tid >> 7;
            const uint64_t mine = entry < n ? final[entry] : ~0ull;
            uint32_t ahead = 0;
            for (uint32_t i = half * half_n; i < half * half_n + half_n; i += 16u) {
                uint64_t other[16];
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    other[q] = final[i + (uint32_t)q];
                }
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    ahead += other[q] > mine ? 1u : 0u;
                }
            }
            if (half == 1u) {
                upper[tid & 127u] = ahead;
            }
            __syncthreads();
            if (half == 0u && entry < n && mine != 0ull) {
                ahead += upper[tid];
                if (ahead < 64u) {
                    ranked[ahead] = mine;
                }
            }
            __syncthreads();
        }
        if (w != 0u) {
            return false;
        }
        c = ranked[lane];
    }
    phase(cfg, 3);
    RowArgs t;
    read_again(t, src);
    c = lane < t.k ? c : 0ull;
    n = (uint32_t)__popcll(__ballot(c != 0ull));
    const uint32_t step = t.step + cfg.step_delta;
    phase(cfg, 4);

    // ---- the row
    if (S > 1u) {
        ranked[lane] = c;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // (LDS of this wave: in order already)
        __builtin_amdgcn_wave_barrier();
        const bool finished = finish_by_wave<DT, LSE, false>(t, cfg, row, s, n, ranked, step, want_lse, sh);
        if (finished) {
            phase(cfg, 7);
        }
        return finished;
    }
    if (forced) {
        if (lane == 0u) {
            finish_token<DT>(t, sh, t.forced, vocab);
        }
    } else if (n == 0u) {
        if (lane == 0u) {
            finish_empty(t, vocab, sh, cfg);
        }
    } else {
        tail_wave<DT, false>(t, vocab, step, c, n, sh, cfg, 0u, 0u);
    }
    phase(cfg, 7);
    return true;
}

template <int DT, bool LSE, bool PEN>
__global__ __launch_bounds__(NT, 4) void k_blocks_table(LaunchCfg cfg) {
    __shared__ Shared sh;
    blocks_row<DT, LSE, PEN>((const LILY_CONST RowArgs*)cfg.table + blockIdx.y, cfg, sh);
}

template <int DT, bool LSE, bool PEN>
hipError_t launch_blocks(hipStream_t stream, uint32_t rows, const LaunchCfg& cfg) {
    if (cfg.slices > WAVE_MERGE_LISTS && cfg.slices * cfg.ws_k > WAVE_MERGE_SLOTS) {
        return hipErrorInvalidValue;   // (more than finish_by_wave() looks at)
    }
    hipLaunchKernelGGL((k_blocks_table<DT, LSE, PEN>), dim3(cfg.slices, rows), dim3(NT), BLOCKS_LDS_BYTES, stream, cfg);
    return hipGetLastError();
}

}  // namespace

#define LILY_CAT_(a, b) a##b
#define LILY_CAT(a, b) LILY_CAT_(a, b)

hipError_t LILY_CAT(launch_rows_blocks_dt, LILY_DT)(hipStream_t stream, bool lse, bool pen, uint32_t rows, const LaunchCfg& cfg) {
    if (pen) {
        return lse ? launch_blocks<LILY_DT, true, true>(stream, rows, cfg) : launch_blocks<LILY_DT, false, true>(stream, rows, cfg);
    }
    return lse ? launch_blocks<LILY_DT, true, false>(stream, rows, cfg) : launch_blocks<LILY_DT, false, false>(stream, rows, cfg);
}

}  // namespace lily
