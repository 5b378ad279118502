// lm_head_codes_rows.hip - the language-model head over affine codes for 17 rows and more: the
// weights are the bf16 values dequant_q4_bf16 / dequant_q8_bf16 make of the codes
// (src/kernels/metal/quant.metal:179-233), as in a batch of the reference, but they never exist in
// memory: every code is read once, turned into its weight in the register that the matrix
// instruction takes it from, and multiplied with all rows of the tile.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "launch.h"
#include "lm_head_epilogue.h"

namespace lily {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t w32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int STEP_K = 64;                               // values of d between two barriers
constexpr int CODE_BYTES = LILY_TILE_COLS * 128;         // a stage of codes: one line of every column
constexpr int AHEAD = 2;                                 // stages of codes on their way in registers

inline uint32_t rows_lds_bytes(int mi, uint32_t groups) {
    return 2u * (uint32_t)mi * 32u * STEP_K * 2u + CODE_BYTES + LILY_TILE_COLS * groups * 4u;
}

}  // namespace

// One workgroup of four waves per MI * 32 rows x 128 columns; a wave multiplies 32 columns with all
// the rows, so no code is turned into a weight twice within a tile.
//
// Codes: a stage is 128 bytes - one line of memory, 128 or 256 values of d - of each of a wave's
// 32 columns, four loads of eight whole lines, AHEAD stages on their way in registers.  They pass
// through 4 KB of LDS that only this wave touches (no barrier), which turns "eight lanes a column"
// into "a lane its own column": a lane then holds 16 bytes of codes in a row and dequantises eight
// at a time.  Which values of d a product takes together is free, as long as the hidden values
// are read in the same places: m-th product of a step, upper half of the lanes h:
//   8 bits: values 32 * (m / 2) + 16 * h + 8 * (m % 2) on;   4 bits: 32 * h + 8 * m on.
// Hidden values: 64 of d a step for all rows, two halves of LDS, a barrier a step, loads
// HIDDEN_AHEAD steps ahead (the L2 holds them).  The loads in flight come back in order, so the codes'
// effective lead is HIDDEN_AHEAD steps.
// Scales and biases: the tile's, brought once as whole lines, a word (scale, bias) per group.
//
// LDS: 2 x MI * 4 KB + 16 KB + 512 bytes a group.  Of a compute unit's 160 KB, three workgroups of
// 32 rows fit up to 58 groups, two up to 112; of 64 rows three up to 42, two up to 96; of 128 rows
// two up to 64 groups (d = 4096 in groups of 64).  One alone has nothing to cover its barriers: 512
// rows of 4 bits take 1.21 times as long per value of d at d = 8192 as at 4096, and larger batches
// go another way from fewer rows on (sampler_api.cpp, HEAD_LIBRARY_ROWS_CODE_LINES_ALONE).
//
// Before it, tiles that brought 4 or 8 bytes of codes and two 2-byte scales a thread and load (the
// requests, not the bytes, were their bound) and turned each code into LDS.  V = 151 936, f32
// logits, before and now: d = 4096, 8 bits, 20 rows 256 -> 146 us, 50 rows 428 -> 169, 100 rows
// 502 -> 237, 200 rows 795 -> 422; 4 bits 357 -> 123, 258 -> 165, 439 -> 224, 723 -> 398.
// With 4 bits and few rows the vector unit bounds it (20 rows: 67 % of the cycles; in a first form
// that took 124 us the launch without turning codes into weights took 91, without its products
// 124): 23 instructions for eight 4-bit codes.  With 8 bits and 50 rows at d = 2560 nothing is
// saturated (vector unit 47 %, products 23 %): 1 187 workgroups over 768 places are 1.55
// generations, and each step of 64 has a barrier.  Tried on the first form and no faster: the conversion of two 8-bit floats an instruction
// in place of four byte conversions (124 -> 122), codes as the denormal halves of a mixed-precision
// FMA (124 -> 118, none for 8 bits, and it overflows for scales from 2^104 on), codes read out of
// LDS a step ahead (none).
template <int WBITS, int MI>
__global__ void __launch_bounds__(256, MI == 4 ? 2 : 3)
k_lm_head_codes_rows(const RowScales scales_arg, const uint16_t* __restrict__ hidden, uint64_t hidden_stride, const uint32_t* __restrict__ codes,
                     uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                     float* __restrict__ logits, uint64_t logits_stride,
                     float* __restrict__ tile_max, float* __restrict__ tile_sum, uint32_t tiles_per_row,
                     uint32_t m_tiles, const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases,
                     uint32_t group_shift) {
    const float* __restrict__ c2_of_row = scales_of(scales_arg);
    carry(scales_arg, 0u);
    constexpr int BM = MI * 32;
    constexpr int STAGE_K = 1024 / WBITS, STEPS = STAGE_K / STEP_K;   // steps of 64 in a stage: 2 or 4
    constexpr int HIDDEN_AHEAD = MI == 4 ? 2 : 4;
    constexpr uint32_t HIDDEN_BYTES = BM * STEP_K * 2;
    extern __shared__ __align__(16) char lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, c = lane & 31u, h = lane >> 5;
    // Consecutive workgroups go to consecutive XCDs: those that multiply the same columns with
    // different rows run side by side on one XCD, and the codes come out of its L2 after the first.
    const uint32_t slot = blockIdx.x >> 3;
    const uint32_t m_tile = slot % m_tiles, n_tile = (slot / m_tiles) * 8u + (blockIdx.x & 7u);
    if (n_tile >= tiles_per_row) {
        return;
    }
    const uint32_t m0 = m_tile * BM, n0 = n_tile * LILY_TILE_COLS;
    const uint32_t nstages = d / STAGE_K, nsteps = nstages * STEPS, groups = d >> group_shift;
    // (each tile walks d from a place of its own: rows lie a power of two apart for the usual d)
    const uint32_t rot = (n_tile * 5u) % nstages;
    auto place = [&](uint32_t stage_no) -> uint32_t {
        const uint32_t at = min(stage_no, nstages - 1u) + rot;
        return at >= nstages ? at - nstages : at;
    };
    char* own_codes = lds + 2u * HIDDEN_BYTES + wave * 4096u;
    uint32_t* sz = reinterpret_cast<uint32_t*>(lds + 2u * HIDDEN_BYTES + CODE_BYTES);

    // ---- codes: load i of a wave is the lines of its columns 8 * i ... + 7, lane l the 16 bytes that
    // belong at l * 16: of column 8 * i + l / 8 the piece (l % 8) ^ (column / 2) % 8 (pieces change
    // places by the column's number: two lines fill the banks, so the 16 columns whose pieces are
    // read at once hit 16 different groups of them)
    const char* from_c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t col = n0 + 32u * wave + 8u * (uint32_t)i + (lane >> 3), q = (lane & 7u) ^ ((4u * (uint32_t)i + (lane >> 4)) & 7u);
        from_c[i] = reinterpret_cast<const char*>(codes) + (uint64_t)min(col, vocab - 1u) * weight_stride * 4u + q * 16u;
    }
    auto fetch_codes = [&](w32x4 (&r)[4], uint32_t stage_no) {
        const uint32_t at = place(stage_no) * 128u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            r[i] = *reinterpret_cast<const w32x4*>(from_c[i] + at);
        }
    };
    // ---- hidden values: piece i of thread t is 16 bytes (t % 8) of row 32 * i + t / 8, at the place
    // (t % 8) ^ (row / 2) % 8 of the row's 128 bytes
    const char* from_h[MI];
    const uint32_t hidden_at = (tid >> 3) * 128u + ((tid & 7u) ^ ((tid >> 4) & 7u)) * 16u;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const uint32_t r = m0 + 32u * (uint32_t)i + (tid >> 3);
        from_h[i] = reinterpret_cast<const char*>(hidden) + (uint64_t)min(r, rows - 1u) * hidden_stride * 2u + (tid & 7u) * 16u;
    }
    auto fetch_hidden = [&](w32x4 (&r)[MI], uint32_t step) {
        const uint32_t t = min(step, nsteps - 1u);
        const uint32_t at = place(t / STEPS) * (STAGE_K * 2u) + (t % STEPS) * (STEP_K * 2u);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            r[i] = *reinterpret_cast<const w32x4*>(from_h[i] + at);
        }
    };
    auto stage_hidden = [&](const w32x4 (&r)[MI], uint32_t buf) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            *reinterpret_cast<w32x4*>(lds + buf * HIDDEN_BYTES + (uint32_t)i * 4096u + hidden_at) = r[i];
        }
    };

    // (everything below asks memory unconditionally, past the end the last stage again: the
    // compiler then counts the loads in flight and waits for the oldest only)
    w32x4 ring_c[AHEAD][4], ring_h[HIDDEN_AHEAD][MI];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
        fetch_codes(ring_c[j], (uint32_t)j);
    }
#pragma unroll
    for (int j = 0; j < HIDDEN_AHEAD; ++j) {
        fetch_hidden(ring_h[j], (uint32_t)j);
    }
    // ---- scales and biases: group g of column c at sz[c * groups + (g + c) % groups] (32 columns
    // read one group at once: turned by the column's number, they lie in different banks)
    {
        // (eight neighbouring threads a column; no division but one a column)
        const uint32_t col0 = tid >> 3, lane8 = tid & 7u;
        auto put = [&](uint32_t at0, uint32_t turn, uint32_t g, uint32_t scale, uint32_t bias) {
            const uint32_t at = g + turn;
            sz[at0 + (at >= groups ? at - groups : at)] = scale | (bias << 16);
        };
        uint32_t turn[4];
        uint64_t from[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            turn[u] = (col0 + 32u * (uint32_t)u) % groups;
            from[u] = (uint64_t)min(n0 + col0 + 32u * (uint32_t)u, vocab - 1u) * groups;
        }
        if (groups % 8u == 0u &&
            ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 15u) == 0u) {
            for (uint32_t g0 = 0; g0 < groups; g0 += 64u) {   // 16 bytes, eight groups, a load
                const uint32_t g = min(g0 + lane8 * 8u, groups - 8u);   // (the last ones by several: the same values)
                w32x4 s[4], b[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    s[u] = *reinterpret_cast<const w32x4*>(scales + from[u] + g);
                    b[u] = *reinterpret_cast<const w32x4*>(biases + from[u] + g);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        put((col0 + 32u * (uint32_t)u) * groups, turn[u], g + (uint32_t)e,
                            (s[u][e >> 1] >> (16 * (e & 1))) & 0xffffu, (b[u][e >> 1] >> (16 * (e & 1))) & 0xffffu);
                    }
                }
            }
        } else {
            for (uint32_t g = lane8; g < groups; g += 8u) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    put((col0 + 32u * (uint32_t)u) * groups, turn[u], g, scales[from[u] + g], biases[from[u] + g]);
                }
            }
        }
    }
    stage_hidden(ring_h[0], 0u);
    fetch_hidden(ring_h[0], (uint32_t)HIDDEN_AHEAD);
    __syncthreads();

    f32x16 acc[MI][1];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            acc[mi][0][v] = 0.0f;
        }
    }
    const uint32_t col_in = 32u * wave + c, scales_at = col_in * groups, turn = col_in % groups;
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    // the weight of a code: q * scale + bias as one fused f32 operation, rounded to nearest even
    auto weights_of = [&](const w32x4& raw, int m, float scale, float bias) -> bf16x8 {
        // eight codes as the bytes of two words (4 bits: the even codes, then the odd ones)
        uint32_t lo, hi;
        if constexpr (WBITS == 8) {
            lo = raw[2 * (m & 1)];
            hi = raw[2 * (m & 1) + 1];
        } else {
            lo = raw[m] & 0x0f0f0f0fu;
            hi = (raw[m] >> 4) & 0x0f0f0f0fu;
        }
        w32x4 out;
        if constexpr (WBITS == 8) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t word = p < 2 ? lo : hi;
                const f32x2 f = {__builtin_fmaf((float)((word >> (16 * (p & 1))) & 0xffu), scale, bias),
                                 __builtin_fmaf((float)((word >> (16 * (p & 1) + 8)) & 0xffu), scale, bias)};
                out[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
            }
        } else {
            // (opaque here: the compiler would turn the bytes back into an extraction a code)
            asm("" : "+v"(lo), "+v"(hi));
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const f32x2 f = {__builtin_fmaf((float)((lo >> (8 * p)) & 0xffu), scale, bias),
                                 __builtin_fmaf((float)((hi >> (8 * p)) & 0xffu), scale, bias)};
                out[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
            }
        }
        return __builtin_bit_cast(bf16x8, out);
    };
    // stage s with its codes in ring_c[j]; MORE: another one follows, and loads are asked ahead of it
    auto stage = [&](auto j_const, uint32_t s, auto more) {
        constexpr int j = decltype(j_const)::value;
        constexpr bool MORE = decltype(more)::value;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *reinterpret_cast<w32x4*>(own_codes + (uint32_t)i * 1024u + lane * 16u) = ring_c[j][i];
        }
        __builtin_amdgcn_wave_barrier();
        if constexpr (MORE) {
            fetch_codes(ring_c[j], s + AHEAD);
            __builtin_amdgcn_sched_barrier(0);   // (asked here, not where they are used)
        }
        const uint32_t first_k = place(s) * STAGE_K;
#pragma unroll
        for (int u = 0; u < STEPS; ++u) {
            constexpr int PIECES = WBITS == 8 ? 2 : 1;   // 16-byte pieces of codes a lane takes per step
            const uint32_t buf = (uint32_t)(j * STEPS + u) & 1u;
            w32x4 raw[PIECES];
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                const uint32_t piece = 2u * (uint32_t)(u * PIECES + i) + h;
                raw[i] = *reinterpret_cast<const w32x4*>(own_codes + c * 128u + (piece ^ ((c >> 1) & 7u)) * 16u);
            }
            const uint32_t g = (first_k + (uint32_t)u * STEP_K) >> group_shift;
            const uint32_t at = g + turn;
            const uint32_t word = sz[scales_at + (at >= groups ? at - groups : at)];
            const float scale = __builtin_bit_cast(float, word << 16);
            const float bias = __builtin_bit_cast(float, word & 0xffff0000u);
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const uint32_t piece = WBITS == 8 ? 4u * (uint32_t)(m >> 1) + 2u * h + (uint32_t)(m & 1) : 4u * h + (uint32_t)m;
                const char* a_at = lds + buf * HIDDEN_BYTES + c * 128u + (piece ^ ((c >> 1) & 7u)) * 16u;
                const bf16x8 w = weights_of(raw[WBITS == 8 ? m >> 1 : 0], m, scale, bias);
#pragma unroll
                for (int mi = 0; mi < MI; ++mi) {
                    const bf16x8 a = *reinterpret_cast<const bf16x8*>(a_at + mi * 4096);
                    acc[mi][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w, acc[mi][0], 0, 0, 0);
                }
            }
            // the next step's hidden values into the other half (its readers passed the last barrier)
            constexpr int STEP0 = j * STEPS;
            const int next = (STEP0 + u + 1) % HIDDEN_AHEAD;
            stage_hidden(ring_h[next], buf ^ 1u);
            if (MORE || u + 1 + HIDDEN_AHEAD < STEPS) {   // (known when this is compiled)
                __builtin_amdgcn_sched_barrier(0);
                fetch_hidden(ring_h[next], s * STEPS + (uint32_t)u + 1u + HIDDEN_AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
        }
        __builtin_amdgcn_wave_barrier();
    };
    static_assert(AHEAD == 2 && (2 * STEPS) % HIDDEN_AHEAD == 0, "two stages a trip, the rings' places fixed in it");
    typedef std::integral_constant<int, 0> Even;
    typedef std::integral_constant<int, 1> Odd;
    uint32_t s = 0;
    for (; s + 2u <= nstages; s += 2u) {
        stage(Even{}, s, std::true_type{});
        stage(Odd{}, s + 1u, std::true_type{});
    }
    if (s < nstages) {
        stage(Even{}, s, std::false_type{});
    }
    head_epilogue<1, MI, 1, true>(acc, lds, 0u, wave, m0, n_tile, rows, vocab, c2_of_row, logits, logits_stride, tile_max,
                                  tile_sum, tiles_per_row);
}

template <int WBITS, int MI>
static hipError_t launch_codes_rows(hipStream_t stream, const void* hidden, uint64_t hidden_stride, const void* weight,
                                    uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                                    const RowScales& c2_of_row, void* logits, uint64_t logits_stride, float* tile_max,
                                    float* tile_sum, const HeadWeights& wq) {
    const uint32_t tiles_per_row = (vocab + LILY_TILE_COLS - 1u) / LILY_TILE_COLS, m_tiles = (rows + MI * 32u - 1u) / (MI * 32u);
    const uint32_t lds = rows_lds_bytes(MI, d >> wq.group_shift);
    static LdsAllowed allowed;
    const hipError_t e = allowed.say(reinterpret_cast<const void*>(k_lm_head_codes_rows<WBITS, MI>));
    if (e != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL((k_lm_head_codes_rows<WBITS, MI>), dim3((tiles_per_row + 7u) / 8u * 8u * m_tiles), dim3(256), lds,
                       stream, c2_of_row, static_cast<const uint16_t*>(hidden), hidden_stride, static_cast<const uint32_t*>(weight),
                       weight_stride, rows, d, vocab, static_cast<float*>(logits), logits_stride, tile_max,
                       tile_sum, tiles_per_row, m_tiles, static_cast<const uint16_t*>(wq.scales),
                       static_cast<const uint16_t*>(wq.biases), wq.group_shift);
    return hipGetLastError();
}

bool lm_head_codes_rows_serves(uint32_t d, const HeadWeights& wq) {
    if ((wq.bits != 4u && wq.bits != 8u) || wq.group_shift < 6u) {
        return false;   // (a step of 64 values has one scale a column)
    }
    // whole stages, and all the tile's scales in LDS beside the stages
    const uint32_t groups = d >> wq.group_shift;
    return d != 0u && d % (1024u / wq.bits) == 0u && groups >= 1u && (groups << wq.group_shift) == d &&
           rows_lds_bytes(4, groups) <= CU_LDS_BYTES;
}

uint32_t lm_head_codes_rows_resident(uint32_t d, const HeadWeights& wq) {
    return CU_LDS_BYTES / rows_lds_bytes(4, d >> wq.group_shift);
}

hipError_t launch_lm_head_codes_rows(hipStream_t stream, const void* hidden, uint64_t hidden_stride, const void* weight,
                                     uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                                     const RowScales& c2_of_row, void* logits, uint64_t logits_stride, float* tile_max,
                                     float* tile_sum, const HeadWeights& wq) {
    if (!lm_head_codes_rows_serves(d, wq)) {
        return hipErrorInvalidValue;
    }
#define LILY_CODES_ROWS(MI)                                                                                          \
    (wq.bits == 4u ? launch_codes_rows<4, MI>(stream, hidden, hidden_stride, weight, weight_stride, rows, d, vocab,  \
                                              c2_of_row, logits, logits_stride, tile_max, tile_sum, wq)              \
                   : launch_codes_rows<8, MI>(stream, hidden, hidden_stride, weight, weight_stride, rows, d, vocab,  \
                                              c2_of_row, logits, logits_stride, tile_max, tile_sum, wq))
    if (rows <= 32u) {
        return LILY_CODES_ROWS(1);
    }
    if (rows <= 64u) {
        return LILY_CODES_ROWS(2);
    }
    return LILY_CODES_ROWS(4);
#undef LILY_CODES_ROWS
}

}  // namespace lily
