// lm_head_codes.hip - the language-model head over the reference's affine codes for a decode
// step: up to 16 hidden rows against 4- or 8-bit weights, read once at the speed of memory.
//
// The reference's form for few rows (gemv_q4_bf16_f32out / gemv_q8_bf16_f32out,
// src/kernels/metal/quant.metal:8-60 and 130-176): the codes are never turned into weights; a
// group's part of a logit is  scale * sum(q * x) + bias * sum(x)  with f32 sums.  Here sum(q * x)
// and sum(x) of a group of 64 come out of the matrix cores - the codes as bf16 integers (exact),
// a block of ones beside them - and the scale and bias meet the sums once per group and column.
#include <hip/hip_runtime.h>

#include "launch.h"
#include "lm_head_epilogue.h"

namespace lily {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t w32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t w32x2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int CB = LILY_TILE_COLS / 32;   // blocks of 16 columns a wave multiplies: half a tile's
constexpr int THREADS = 512;              // eight waves: two halves of the columns x four shares of d
constexpr int AHEAD = 4;                  // stages asked from memory ahead of the one being multiplied
constexpr int NBUF = 2;                   // stages of codes in LDS: one multiplied, one being written
constexpr int STAGE_BYTES = LILY_TILE_COLS * 128;   // 128 bytes (one line of memory) of every row
constexpr int PART_CB = 4 * 64 + 16;      // floats of one block's partial sums (padded: two blocks
                                          // read side by side then lie in different banks)
constexpr int PART_SHARE = 2 * CB * PART_CB;   // one share of d: all 128 columns
constexpr int RING_BYTES = NBUF * STAGE_BYTES;
constexpr int PART_BYTES = 4 * PART_SHARE * 4;
constexpr int RED_BYTES = 80 * 4;         // the waves' maxima, then their sums, the rows' exponent scales
constexpr uint32_t GROUPS_MAX = 252;      // groups of a row
constexpr uint32_t COMPUTE_UNITS = 256;

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __builtin_bit_cast(float, b << 16); }

// The product instruction: 16 x 16 outputs over 32 values of d.  Lane l gives row (or column)
// l % 16, the 8 values of d from 8 * (l / 16) on; it receives column l % 16, rows 4 * (l / 16) + v.
__device__ __forceinline__ f32x4 product(const w32x4& a, const w32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
}

// Words from one column's scales and biases to the next's: one more than there are groups (an even
// number: an odd distance spreads the 16 columns a product reads at once over the banks without a
// computed turn).  Two workgroups a compute unit up to 94 groups, with and without that word.
__host__ __device__ constexpr uint32_t scale_pitch(uint32_t groups) {
    return groups + 1u;
}
// Bytes of LDS a launch needs: the stages, then every scale and bias of the tile's 128 columns (the partial
// sums take their place at a tile's end, while the next one's are in registers), the reductions.
inline uint32_t codes_lds_bytes(uint32_t groups) {
    const uint32_t sz = (uint32_t)LILY_TILE_COLS * scale_pitch(groups) * 4u;
    return (uint32_t)RING_BYTES + (sz > (uint32_t)PART_BYTES ? sz : (uint32_t)PART_BYTES) + (uint32_t)RED_BYTES;
}

static_assert(RING_BYTES + LILY_TILE_COLS * scale_pitch(GROUPS_MAX) * 4 + RED_BYTES <= CU_LDS_BYTES, "the scales' place");

}  // namespace

// A workgroup of eight waves per 128 columns (one summary) at a time, tile after tile in steps of the grid: as
// many workgroups as the chip holds at once.  The codes pass through LDS as they lie in memory: a stage is 128
// bytes - one line - of each of the 128 rows, brought by 16 loads of 1 KB (two a wave, eight whole lines each),
// AHEAD stages on their way in registers, written to LDS one pass before they are multiplied.  (A lane's own
// operand would be 8 bytes of each of 16 rows: the 64 lines such a load touches, not its bytes, bounded an earlier
// form at a seventh of the memory's speed.  Loads that write LDS themselves keep only what LDS holds in
// flight, which is too little here.)  The stage's 256 (4-bit) or 128 (8-bit) values of d are split among four
// waves, the 128 columns between two; the four partial tiles are added through LDS at the end.
//
// The requests run on from one tile into the next: AHEAD stages of the next one are on their way while the partial
// sums are added, the summary is formed and the next scales are brought (whole lines: asked for with the stages,
// two groups at a time, they were twice the requests of the codes).  A tile's ends were a third of a workgroup's
// time.  V = 151 936, head and draws in one call, us, a workgroup a tile -> staying: 4 bits d = 4096 4 rows 90 -> 81,
// 12 rows 104 -> 93, d = 2560 64 -> 56, d = 1280 7 rows 53 -> 43; 8 bits d = 4096 147 -> 140, d = 2560 98 -> 91; d = 3328, whose
// rows of scales are no multiple of 16 bytes, 4 bits 12 rows 103 -> 85, 8 bits 8 rows 129 -> 115.  Bound: the memory; 512
// tiles more are 30 us (5.1 TB/s) with 4 bits, 52 (5.5) with 8, a third of a round a third of that.  Tried: the
// scales a trip earlier, in registers (83), as many workgroups as give each the same number of tiles (396 of
// three: 91), two and four stages asked for at once (83, 89), six on their way (89), no turn of d's start (8 bits 141 ->
// 146), one instruction less a block (83).
//
// 4-bit codes become bf16 without arithmetic: 0x4300 | q is the bf16 128 + q, two codes a
// register by one and-or ((word >> 4p) & 0x000f000f | 0x43004300: codes p and p + 4, so the
// hidden values are put in that order too), and the 128 is taken off with the bias (bias - 128
// * scale meets the same sum of x).  8-bit codes go through the byte-to-f32 conversion, whose
// upper half is the bf16.
template <int WBITS>
__global__ void __launch_bounds__(THREADS, 4)   // (four waves a SIMD: two workgroups a compute unit)
k_lm_head_codes(const RowScales scales_arg, const uint16_t* __restrict__ hidden, uint64_t hidden_stride, const uint32_t* __restrict__ codes,
                uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                float* __restrict__ logits, uint64_t logits_stride,
                float* __restrict__ tile_max, float* __restrict__ tile_sum, uint32_t tiles_per_row,
                const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases, uint32_t group_shift) {
    const float* __restrict__ c2_of_row = scales_of(scales_arg);
    carry(scales_arg, gridDim.x - 1u);   // (one with no more tiles than any other)
    constexpr int STEPS = WBITS == 4 ? 2 : 1;          // products over 32 values a wave makes per stage and block
    constexpr uint32_t STAGE_K = 128u * 8u / WBITS;    // values of d in a stage
    constexpr uint32_t WAVE_K = STAGE_K / 4u;          // ... of which a wave multiplies these
    extern __shared__ __align__(16) char lds[];
    uint32_t* sz = reinterpret_cast<uint32_t*>(lds + RING_BYTES);   // scales and biases
    float* part = reinterpret_cast<float*>(lds + RING_BYTES);       // [4 shares][2 * CB][4 v x 64 lanes, padded], at a tile's end
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t share = wave & 3u, half = wave >> 2;
    const uint32_t c = lane & 15u, kq = lane >> 4;
    const uint32_t nstages = d / STAGE_K, groups = d >> group_shift, pitch = scale_pitch(groups);
    const uint32_t trips = (nstages + AHEAD - 1u) / AHEAD;   // of AHEAD stages a tile
    float* red = reinterpret_cast<float*>(lds + RING_BYTES + max((uint32_t)PART_BYTES, (uint32_t)LILY_TILE_COLS * pitch * 4u));

    // Where the requests are: trip `s0 / AHEAD` of a tile.  Each tile walks d from a place of its own (rot) and
    // wraps round: rows lie a power of two apart for the usual d, and tiles that all start at column
    // 0 and advance in step queue up at one memory channel after the other.
    struct Cursor {
        uint32_t tile, s0, rot;
    };
    auto at_tile = [&](uint32_t tile) -> Cursor { return Cursor{tile, 0u, (tile * 5u) % nstages}; };
    // (behind the last tile: that one's last stage again and again)
    auto behind = [&](const Cursor& p) -> Cursor {
        if (p.s0 + AHEAD < trips * AHEAD) {
            return Cursor{p.tile, p.s0 + AHEAD, p.rot};
        }
        return p.tile + gridDim.x < tiles_per_row ? at_tile(p.tile + gridDim.x) : p;
    };
    auto place = [&](const Cursor& p, uint32_t j) -> uint32_t {
        const uint32_t at = min(p.s0 + j, nstages - 1u) + p.rot;
        return at >= nstages ? at - nstages : at;
    };

    // ---- who brings what.  Load i of a wave is the 1 KB block 2 * wave + i of a stage: the
    // lines of 8 columns, lane l the 16 bytes that belong at l * 16 - piece (l % 8) ^ (l / 8) of
    // column l / 8 (the pieces of a line change places by the column's number: 16 columns'
    // operands are then read out of all banks).
    const uint32_t piece = (lane & 7u) ^ (lane >> 3);
    // A lane's hidden values: row c (the last one again past `rows`), the wave's share of the
    // stage, 8 values a product from 8 * kq on (two neighbouring eights for 4-bit codes).
    const char* from_a = reinterpret_cast<const char*>(hidden) + (uint64_t)min(c, rows - 1u) * hidden_stride * 2u +
                         (share * WAVE_K + kq * 8u * STEPS) * 2u;
    // (every load unconditional, past the end of d the last stage again: the compiler then
    // counts the loads in flight and waits for the oldest only)
    auto fetch_codes = [&](w32x4 (&l)[2], const Cursor& p, uint32_t j) {
        const uint32_t at = place(p, j);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t col = p.tile * LILY_TILE_COLS + 8u * (2u * wave + (uint32_t)i) + (lane >> 3);
            l[i] = *reinterpret_cast<const w32x4*>(reinterpret_cast<const char*>(codes) +
                                                   (uint64_t)min(col, vocab - 1u) * (weight_stride * 4u) + at * 128u + piece * 16u);
        }
    };
    auto fetch_hidden = [&](w32x4 (&l)[STEPS], const Cursor& p, uint32_t j) {
        const char* from = from_a + (uint64_t)place(p, j) * (STAGE_K * 2u);
#pragma unroll
        for (int t = 0; t < STEPS; ++t) {
            l[t] = *reinterpret_cast<const w32x4*>(from + 16 * t);
        }
    };
    auto stage = [&](const w32x4 (&l)[2], uint32_t buf) {
        char* base = lds + buf * STAGE_BYTES + wave * 2048u + lane * 16u;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<w32x4*>(base + i * 1024) = l[i];
        }
    };
    // ---- a tile's scales and biases: group g of column col as one word (scale, bias) at
    // sz[col * pitch + g].  Eight neighbouring threads a column, 16 bytes - eight groups - a load (rows of an
    // even number of groups begin at multiples of 4 bytes, which is what such a load asks for).
    const bool wide = groups >= 8u && ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) == 0u;
    struct Piece {
        w32x4 v;
    } __attribute__((packed, aligned(4)));
    struct Scales {
        w32x4 scale[2], bias[2];
    };
    // (What a tile's ends need beside the loop is computed there: opaque, or the compiler keeps it in registers
    // that the loop has no room for.)
    auto here = [&]() -> uint32_t {
        uint32_t t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    auto begin_tile = [&](uint32_t tile) {
        const uint32_t t = here();
        auto col_of = [&](int u) -> uint32_t { return (t >> 3) + 64u * (uint32_t)u; };
        auto from_of = [&](int u) -> uint64_t { return (uint64_t)min(tile * LILY_TILE_COLS + col_of(u), vocab - 1u) * groups; };
        if (!wide) {
            for (uint32_t g = t & 7u; g < groups; g += 8u) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const uint64_t at = from_of(u) + g;
                    sz[col_of(u) * pitch + g] = (uint32_t)scales[at] | ((uint32_t)biases[at] << 16);
                }
            }
            return;
        }
        // (a row's last groups may be brought by several: the same values)
        auto group_of = [&](uint32_t g0) -> uint32_t { return min(g0 + (t & 7u) * 8u, groups - 8u); };
        auto fetch = [&](Scales& l, uint32_t g0) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const uint64_t at = from_of(u) + group_of(g0);
                l.scale[u] = reinterpret_cast<const Piece*>(scales + at)->v;
                l.bias[u] = reinterpret_cast<const Piece*>(biases + at)->v;
            }
        };
        auto put = [&](const Scales& l, uint32_t g0) {
            auto half_of = [](const w32x4& v, int e) -> uint32_t { return (v[e >> 1] >> (16 * (e & 1))) & 0xffffu; };
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    sz[col_of(u) * pitch + group_of(g0) + (uint32_t)e] = half_of(l.scale[u], e) | (half_of(l.bias[u], e) << 16);
                }
            }
        };
        for (uint32_t g0 = 0; g0 < groups; g0 += 128u) {
            Scales some, more;
            fetch(some, g0);
            if (g0 + 64u < groups) {
                fetch(more, g0 + 64u);
                put(more, g0 + 64u);
            }
            put(some, g0);
        }
    };
    // where a lane's codes lie in a stage (block cb: column 64 * half + 16 * cb + c; the wave's
    // share of the line is its pieces 2 * share and the next, 8 bytes a lane) and its scales in sz
    const uint32_t col_of_lane = 64u * half + c;
    const uint32_t code_at = (col_of_lane >> 3) * 1024u + ((c & 7u) * 8u + ((2u * share + (kq >> 1)) ^ (c & 7u))) * 16u + (kq & 1u) * 8u;
    const uint32_t scale_at = col_of_lane * pitch;

    f32x4 total[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        total[cb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const w32x4 ONES = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    const f32x4 ZERO = {0.0f, 0.0f, 0.0f, 0.0f};

    auto multiply = [&](const w32x4 (&hid)[STEPS], uint32_t at, uint32_t buf) {
        w32x4 a[STEPS];
#pragma unroll
        for (int t = 0; t < STEPS; ++t) {
            const w32x4 h = hid[t];
            if constexpr (WBITS == 4) {
                // values 0..7 in the order 0 4 1 5 2 6 3 7 of the codes' registers
                a[t].x = __builtin_amdgcn_perm(h.z, h.x, 0x05040100u);
                a[t].y = __builtin_amdgcn_perm(h.z, h.x, 0x07060302u);
                a[t].z = __builtin_amdgcn_perm(h.w, h.y, 0x05040100u);
                a[t].w = __builtin_amdgcn_perm(h.w, h.y, 0x07060302u);
            } else {
                a[t] = h;
            }
        }
        // the sums of the hidden values themselves, where the products' sums will lie
        f32x4 xs = product(a[0], ONES, ZERO);
        if constexpr (STEPS == 2) {
            xs = product(a[1], ONES, xs);
        }
        // the wave's values of this stage lie in one group (64 values, or 32 of one)
        const uint32_t g = (at * STAGE_K + share * WAVE_K) >> group_shift;
        const char* codes_in = lds + buf * STAGE_BYTES;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const w32x2 raw = *reinterpret_cast<const w32x2*>(codes_in + code_at + cb * 2048);
            w32x4 b[STEPS];
            if constexpr (WBITS == 4) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const uint32_t word = raw[t];
                    b[t].x = (word & 0x000f000fu) | 0x43004300u;
                    b[t].y = ((word >> 4) & 0x000f000fu) | 0x43004300u;
                    b[t].z = ((word >> 8) & 0x000f000fu) | 0x43004300u;
                    b[t].w = ((word >> 12) & 0x000f000fu) | 0x43004300u;
                }
            } else {
                uint32_t out[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const uint32_t word = raw[p >> 1];
                    const float lo = (float)((word >> (16 * (p & 1))) & 0xffu);
                    const float hi = (float)((word >> (16 * (p & 1) + 8)) & 0xffu);
                    out[p] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo),
                                                   0x07060302u);
                }
                b[0] = w32x4{out[0], out[1], out[2], out[3]};
            }
            f32x4 qx = product(a[0], b[0], ZERO);
            if constexpr (STEPS == 2) {
                qx = product(a[1], b[1], qx);
            }
            const uint32_t word = sz[scale_at + g + (uint32_t)cb * 16u * pitch];
            const float s = bf16_bits_to_f32(word);   // (the shift drops the bias)
            float z = __builtin_bit_cast(float, word & 0xffff0000u);
            if constexpr (WBITS == 4) {
                z = __builtin_fmaf(-128.0f, s, z);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                total[cb][v] = __builtin_fmaf(s, qx[v], __builtin_fmaf(z, xs[v], total[cb][v]));
            }
        }
    };

    // The tile's end: the four partial tiles are added, the logits stored, the summary formed.  Thread t then holds
    // column t % 128 of the rows 4 * (t / 128) .. + 3, the same for a wave's lanes.
    auto end_tile = [&](uint32_t tile, auto&& between) {
        const uint32_t tid = here(), lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
        const uint32_t share = wave & 3u, half = wave >> 2, rq = wave >> 1;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                part[share * PART_SHARE + (half * CB + cb) * PART_CB + v * 64 + lane] = total[cb][v];
            }
            total[cb] = ZERO;
        }
        __syncthreads();
        const uint32_t col_in = tid & 127u, col = tile * LILY_TILE_COLS + col_in;
        const float NEG = -__builtin_huge_valf();
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t r = 4u * rq + (uint32_t)j;
            const uint32_t at = (col_in >> 4) * PART_CB + (uint32_t)j * 64u + rq * 16u + (col_in & 15u);
            x[j] = (part[at] + part[PART_SHARE + at]) + (part[2 * PART_SHARE + at] + part[3 * PART_SHARE + at]);
            if (r < rows && col < vocab) {
                logits[(uint64_t)r * logits_stride + col] = x[j];
            }
            // what a stored value counts for: a NaN and a column outside the vocabulary count as -inf
            x[j] = (col < vocab && x[j] == x[j]) ? x[j] : NEG;
        }
        // each row's largest value and sum of exponentials over the 128 columns (two waves a row).
        // Four values over the 64 lanes, halved with them: the two halves of the wave, then the two rows
        // of 16 lanes of a half, change places for two values at a time; then lanes 8, 4, 2 and 1 apart.
        // Lane 16 * j ends with value j.  (A butterfly for each value took 24 moves through the LDS
        // crossbar.)
        auto across = [&](const float (&v)[4], auto op) -> float {
            auto bits = [](float f) { return __builtin_bit_cast(uint32_t, f); };
            float y[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const auto both = __builtin_amdgcn_permlane32_swap(bits(v[i]), bits(v[i + 2]), false, false);
                y[i] = op(__builtin_bit_cast(float, (uint32_t)both[0]), __builtin_bit_cast(float, (uint32_t)both[1]));
            }
            const auto both = __builtin_amdgcn_permlane16_swap(bits(y[0]), bits(y[1]), false, false);
            float z = op(__builtin_bit_cast(float, (uint32_t)both[0]), __builtin_bit_cast(float, (uint32_t)both[1]));
            z = op(z, moved<0x128>(z));      // (rotated by 8)
            z = op(z, moved<0x141>(z));      // (eight lanes mirrored)
            z = op(z, moved<0x4e>(z));       // (quads: 2 3 0 1)
            return op(z, moved<0xb1>(z));    // (quads: 1 0 3 2)
        };
        // (red: [8 waves][4] maxima, then the same of sums; rows 4 * rq on are the waves 2 * rq and the next)
        const float top4 = across(x, [](float p, float q) { return fmaxf(p, q); });
        if ((lane & 15u) == 0u) {
            red[wave * 4u + (lane >> 4)] = top4;
        }
        __syncthreads();
        between();   // (the partial sums have been read)
        float e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float c2 = red[64u + 4u * rq + (uint32_t)j];
            const float top = fmaxf(red[8u * rq + (uint32_t)j], red[8u * rq + 4u + (uint32_t)j]) * c2;
            e[j] = x[j] > NEG ? __builtin_amdgcn_exp2f(__builtin_fmaf(x[j], c2, -top)) : 0.0f;
        }
        const float sum4 = across(e, [](float p, float q) { return p + q; });
        if ((lane & 15u) == 0u) {
            red[32u + wave * 4u + (lane >> 4)] = sum4;
        }
        __syncthreads();
        if (tid < 16u && tid < rows) {
            const uint32_t at0 = 8u * (tid >> 2) + (tid & 3u);
            const float top = fmaxf(red[at0], red[at0 + 4u]), sum = red[32u + at0] + red[32u + at0 + 4u];
            const size_t at = (size_t)tid * tiles_per_row + tile;
            tile_max[at] = top;
            tile_sum[at] = top > NEG ? sum : 0.0f;
        }
    };

    // ---- the stages.  Two rings of registers hold the loads on their way, AHEAD stages deep:
    // in pass s codes[j] holds the codes of stage s + 1 and hid[j] the hidden values of stage s.
    // Every pass multiplies the stage that lies in one half of LDS, writes the next one's codes
    // into the other half (nobody reads it: the barrier that closed the pass before saw to
    // that), asks for the codes and the hidden values AHEAD further on into the registers just
    // freed, and meets the other waves.
    w32x4 codes_ring[AHEAD][2], hid[AHEAD][STEPS];
    Cursor now = at_tile(blockIdx.x), next = behind(now);
    const float c2_mine = c2_of_row[min(tid, rows - 1u)];
    __builtin_amdgcn_sched_barrier(0);
    fetch_codes(codes_ring[AHEAD - 1], now, 0u);   // (these registers' own stage is asked for behind it)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
        fetch_hidden(hid[j], now, (uint32_t)j);
        if (j + 1 < AHEAD) {
            fetch_codes(codes_ring[j], now, (uint32_t)(j + 1));
        }
        __builtin_amdgcn_sched_barrier(0);   // (in this order: the loop waits for the oldest only)
    }
    if (tid < 16u) {
        red[64u + tid] = c2_mine;
    }
    stage(codes_ring[AHEAD - 1], 0u);
    fetch_codes(codes_ring[AHEAD - 1], next, 0u);
    __builtin_amdgcn_sched_barrier(0);
    begin_tile(now.tile);
    __syncthreads();   // (the scales and stage 0 are written)
    static_assert(AHEAD % 2 == 0, "the halves of LDS alternate within a trip");
    const uint32_t my_tiles = (tiles_per_row - blockIdx.x + gridDim.x - 1u) / gridDim.x;
    for (uint32_t t = 0; t < my_tiles * trips; ++t) {
        const Cursor after = behind(next);
        const bool ends = now.s0 + AHEAD >= trips * AHEAD;
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            const uint32_t buf = (uint32_t)j & 1u;
            if (now.s0 + (uint32_t)j < nstages) {
                multiply(hid[j], place(now, (uint32_t)j), buf);
            }
            stage(codes_ring[j], buf ^ 1u);
            // (nor may the compiler move the requests down to where their values are used)
            __builtin_amdgcn_sched_barrier(0);
            fetch_hidden(hid[j], next, (uint32_t)j);
            fetch_codes(codes_ring[j], j + 1 < AHEAD ? next : after, (uint32_t)(j + 1) % AHEAD);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        }
        if (ends) {
            const bool more = next.tile != now.tile;
            end_tile(now.tile, [&]() {
                if (more) {
                    begin_tile(next.tile);
                }
            });
        }
        now = next;
        next = after;
    }
}

template <int WBITS>
static hipError_t launch_codes(hipStream_t stream, const void* hidden, uint64_t hidden_stride, const void* weight,
                               uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                               const RowScales& c2_of_row, void* logits, uint64_t logits_stride, float* tile_max,
                               float* tile_sum, const HeadWeights& wq) {
    const uint32_t tiles_per_row = (vocab + LILY_TILE_COLS - 1u) / LILY_TILE_COLS;
    const uint32_t lds = codes_lds_bytes(d >> wq.group_shift);
    // (what does not fit the chip at once would only start later)
    const uint32_t places = COMPUTE_UNITS * (2u * lds <= CU_LDS_BYTES ? 2u : 1u);
    static LdsAllowed allowed;
    const hipError_t e = allowed.say(reinterpret_cast<const void*>(k_lm_head_codes<WBITS>));
    if (e != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL((k_lm_head_codes<WBITS>), dim3(tiles_per_row < places ? tiles_per_row : places), dim3(THREADS), lds, stream, c2_of_row,
                       static_cast<const uint16_t*>(hidden), hidden_stride, static_cast<const uint32_t*>(weight),
                       weight_stride, rows, d, vocab, static_cast<float*>(logits), logits_stride,
                       tile_max, tile_sum, tiles_per_row, static_cast<const uint16_t*>(wq.scales),
                       static_cast<const uint16_t*>(wq.biases), wq.group_shift);
    return hipGetLastError();
}

bool lm_head_codes_serves(uint32_t rows, uint32_t d, uint32_t vocab, uint64_t hidden_stride, uint64_t weight_stride,
                          const HeadWeights& wq) {
    if ((wq.bits != 4u && wq.bits != 8u) || rows < 1u || rows > 16u || wq.group_shift < 6u) {
        return false;
    }
    // whole stages (128 bytes of codes a row), all the tile's scales in LDS beside the stages, and an
    // even number of groups a row: nothing here needs that, but heads with an odd one have always
    // been multiplied by the weights in bf16, and their logits stay what they are
    const uint32_t stage_k = 128u * 8u / wq.bits, groups = d >> wq.group_shift;
    return d >= stage_k && d % stage_k == 0u && groups % 2u == 0u && (groups << wq.group_shift) == d &&
           groups <= GROUPS_MAX;
}

hipError_t launch_lm_head_codes(hipStream_t stream, const void* hidden, uint64_t hidden_stride, const void* weight,
                                uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                                const RowScales& c2_of_row, void* logits, uint64_t logits_stride, float* tile_max,
                                float* tile_sum, const HeadWeights& wq) {
    if (!lm_head_codes_serves(rows, d, vocab, hidden_stride, weight_stride, wq)) {
        return hipErrorInvalidValue;
    }
    const auto launch = wq.bits == 8u ? launch_codes<8> : launch_codes<4>;
    return launch(stream, hidden, hidden_stride, weight, weight_stride, rows, d, vocab, c2_of_row, logits, logits_stride,
                  tile_max, tile_sum, wq);
}

}  // namespace lily
