// lm_head_epilogue.h - what every tile of the head does with its sums: the logits as they are
// stored, and the largest value and the sum of exponentials of each row's 128 columns.
#pragma once

#include <hip/hip_runtime.h>

#include "row_args.h"

namespace lily {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// x as the lane CTRL names holds it (DPP controls: 0x120 + n = rotate right by n within each
// row of 16 lanes).
template <int CTRL>
__device__ __forceinline__ float rotated(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}

// acc: the sums of a wave's MI x NI products of 32 x 32; four waves, WAVES_M x (4 / WAVES_M), this
// one at (wm, wn), hold WAVES_M * MI * 32 rows from m0 on by the 128 columns of tile n_tile.  `lds`
// is free for reuse, (4 / WAVES_M + 2) floats a row; every thread of the workgroup calls.
template <int WAVES_M, int MI, int NI, bool OUT_F32>
__device__ __forceinline__ void head_epilogue(f32x16 (&acc)[MI][NI], char* lds, uint32_t wm, uint32_t wn, uint32_t m0,
                                              uint32_t n_tile, uint32_t rows, uint32_t vocab,
                                              const float* __restrict__ c2_of_row, void* __restrict__ logits_out,
                                              uint64_t logits_stride, float* __restrict__ tile_max,
                                              float* __restrict__ tile_sum, uint32_t tiles_per_row) {
    constexpr int WAVES_N = 4 / WAVES_M, BM = WAVES_M * MI * 32;
    static_assert(WAVES_N * NI * 32 == LILY_TILE_COLS, "a workgroup's columns are one summary");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n0 = n_tile * LILY_TILE_COLS;
    // Element v of a lane's 16 sits in row 8 * (v / 4) + 4 * (lane / 32) + v % 4
    // of its 32 x 32 product, column lane % 32.  Values are rounded to bf16 first, in place: the
    // maximum and the sum describe the logits as they are stored.
    float* red = reinterpret_cast<float*>(lds);              // [WAVES_N][BM] by column group
    float* row_max = red + WAVES_N * BM;                  // [BM]
    float* row_c2 = row_max + BM;                            // [BM]
    if (tid < (uint32_t)BM) {
        row_c2[tid] = c2_of_row[min(m0 + tid, rows - 1u)];
    }
    const float NEG = -__builtin_huge_valf();
    bool in_vocab[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
        in_vocab[ni] = n0 + wn * (NI * 32u) + (uint32_t)ni * 32u + (lane & 31u) < vocab;
    }
    if constexpr (!OUT_F32) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float f = acc[mi][ni][v];   // (a bit_cast of the element itself reads element 0)
                    const uint32_t u = __builtin_bit_cast(uint32_t, f);
                    // round to nearest even; a NaN stays one (quiet)
                    const uint32_t r = (u & 0x7fffffffu) > 0x7f800000u ? ((u >> 16) | 0x40u)
                                                                       : ((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
                    acc[mi][ni][v] = __builtin_bit_cast(float, r << 16);
                }
            }
        }
    }
    // what a stored value counts for: a NaN and a column outside the vocabulary count as -inf
    auto worth = [&](int mi, int ni, int v) -> float {
        const float x = acc[mi][ni][v];
        return (in_vocab[ni] && x == x) ? x : NEG;
    };
    // A reduction over the 32 lanes that hold one row's columns: rotations by 8, 4, 2 and 1 within
    // each row of 16 lanes (DPP operands of the arithmetic itself), then one exchange between the
    // two rows.  (Five exchanges through the LDS crossbar per value, as __shfl_xor compiles, made
    // the epilogue as long as the products at 1024 rows.)
    auto across32 = [&](float x, auto op) -> float {
        x = op(x, rotated<0x128>(x));
        x = op(x, rotated<0x124>(x));
        x = op(x, rotated<0x122>(x));
        x = op(x, rotated<0x121>(x));
        return op(x, __shfl_xor(x, 16));
    };
    auto row_of = [&](int mi, int v) -> uint32_t {
        return wm * (MI * 32u) + (uint32_t)mi * 32u + 8u * (uint32_t)(v >> 2) + 4u * (lane >> 5) +
               (uint32_t)(v & 3);
    };
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            float m = NEG;
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                m = fmaxf(m, worth(mi, ni, v));
            }
            m = across32(m, [](float p, float q) { return fmaxf(p, q); });
            if ((lane & 31u) == 0u) {
                red[wn * BM + row_of(mi, v)] = m;
            }
        }
    }
    __syncthreads();
    if (tid < (uint32_t)BM) {
        float m = red[tid];
#pragma unroll
        for (int g = 1; g < WAVES_N; ++g) {
            m = fmaxf(m, red[g * BM + tid]);
        }
        row_max[tid] = m;
    }
    __syncthreads();
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t r = row_of(mi, v);
            const float c = row_c2[r], top = row_max[r] * c;
            float e = 0.0f;
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                const float x = worth(mi, ni, v);
                e += x > NEG ? __builtin_amdgcn_exp2f(__builtin_fmaf(x, c, -top)) : 0.0f;
            }
            e = across32(e, [](float p, float q) { return p + q; });
            if ((lane & 31u) == 0u) {
                red[wn * BM + r] = e;
            }
        }
    }
    __syncthreads();
    if (tid < (uint32_t)BM && m0 + tid < rows) {
        const size_t at = (size_t)(m0 + tid) * tiles_per_row + n_tile;
        float e = red[tid];
#pragma unroll
        for (int g = 1; g < WAVES_N; ++g) {
            e += red[g * BM + tid];
        }
        tile_max[at] = row_max[tid];
        tile_sum[at] = row_max[tid] > NEG ? e : 0.0f;
    }
    // the logits themselves
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
            const uint32_t col = n0 + wn * (NI * 32u) + (uint32_t)ni * 32u + (lane & 31u);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t r = m0 + row_of(mi, v);
                if (r < rows && col < vocab) {
                    const float f = acc[mi][ni][v];
                    if constexpr (OUT_F32) {
                        static_cast<float*>(logits_out)[(uint64_t)r * logits_stride + col] = f;
                    } else {
                        static_cast<uint16_t*>(logits_out)[(uint64_t)r * logits_stride + col] =
                            (uint16_t)(__builtin_bit_cast(uint32_t, f) >> 16);
                    }
                }
            }
        }
    }
}

}  // namespace lily
