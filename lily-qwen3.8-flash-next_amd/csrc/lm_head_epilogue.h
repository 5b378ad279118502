// lm_head_epilogue.h - what every tile of the head does with its sums: the logits as they are
// stored, and the largest value and the sum of exponentials of each row's 128 columns.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <type_traits>

#include "launch.h"
#include "row_args.h"

namespace lily {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// x as the lane that the DPP control CTRL names holds it.
template <int CTRL>
__device__ __forceinline__ float moved(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

// (For kernels whose first argument the scales are.  Those that travel with the launch are read from where the
// arguments lie.)
__device__ __forceinline__ const float* scales_of(const RowScales& c2) {
    const char* args = (const char*)(const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
    return c2.p != nullptr ? c2.p : reinterpret_cast<const float*>(args + offsetof(RowScales, few));
}

// What the launch carries to the device (RowScales), by workgroup `who`.  (A kernel of its own ahead of the head was a
// trip across the bus with nothing beside it: 50 rows over 8-bit codes, d = 2560, 127.5 -> 123.7 us a call, 100 bf16 rows
// 214 -> 211, 16 rows over 8-bit codes of 40 000, d = 2048, 41.0 -> 38.6.)
__device__ __forceinline__ void carry(const RowScales& c2, uint32_t who) {
    if (blockIdx.x == who) {
        const uint4* src = static_cast<const uint4*>(c2.src);
        for (uint32_t i = threadIdx.x; i < c2.pieces; i += blockDim.x) {
            static_cast<uint4*>(c2.dst)[i] = src[i];
        }
    }
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
    // A reduction of a lane's 16 values over the 32 lanes that hold the same rows: the values are
    // halved with the lanes.  First the two rows of 16 lanes change halves (one instruction for two
    // values: the even row then holds value v of both, the odd row value v + 8), then lanes 8, 4, 2
    // and 1 apart.  The lane ends with the value (lane / 2) % 16: 38 instructions for 16 values where
    // a butterfly for each value took 96 and a place in LDS for each of 16 writes.
    auto across32 = [&](float (&x)[16], auto op) -> float {
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const auto both = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x[v]),
                                                               __builtin_bit_cast(uint32_t, x[v + 8]), false, false);
            x[v] = op(__builtin_bit_cast(float, (uint32_t)both[0]), __builtin_bit_cast(float, (uint32_t)both[1]));
        }
        auto halve = [&](int n, bool upper, auto ctrl) {
#pragma unroll
            for (int v = 0; v < n; ++v) {
                const float keep = upper ? x[v + n] : x[v], give = upper ? x[v] : x[v + n];
                x[v] = op(keep, moved<decltype(ctrl)::value>(give));
            }
        };
        halve(4, (lane & 8u) != 0u, std::integral_constant<int, 0x128>{});   // (rotated by 8)
        halve(2, (lane & 4u) != 0u, std::integral_constant<int, 0x141>{});   // (eight lanes mirrored)
        halve(1, (lane & 2u) != 0u, std::integral_constant<int, 0x4e>{});    // (quads: 2 3 0 1)
        return op(x[0], moved<0xb1>(x[0]));                                  // (quads: 1 0 3 2)
    };
    auto row_of = [&](int mi, int v) -> uint32_t {
        return wm * (MI * 32u) + (uint32_t)mi * 32u + 8u * (uint32_t)(v >> 2) + 4u * (lane >> 5) +
               (uint32_t)(v & 3);
    };
    const uint32_t own_v = (lane >> 1) & 15u;   // the value a lane ends with, and its row
    const uint32_t own_row = wm * (MI * 32u) + 8u * (own_v >> 2) + 4u * (lane >> 5) + (own_v & 3u);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
        float m[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            m[v] = NEG;
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                m[v] = fmaxf(m[v], worth(mi, ni, v));
            }
        }
        const float top = across32(m, [](float p, float q) { return fmaxf(p, q); });
        if ((lane & 1u) == 0u) {
            red[wn * BM + own_row + (uint32_t)mi * 32u] = top;
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
        float e[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t r = row_of(mi, v);
            const float c = row_c2[r], top = row_max[r] * c;
            e[v] = 0.0f;
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                const float x = worth(mi, ni, v);
                e[v] += x > NEG ? __builtin_amdgcn_exp2f(__builtin_fmaf(x, c, -top)) : 0.0f;
            }
        }
        const float sum = across32(e, [](float p, float q) { return p + q; });
        if ((lane & 1u) == 0u) {
            red[wn * BM + own_row + (uint32_t)mi * 32u] = sum;
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
    // the logits themselves (a lane's place once, the rows' distances the same for all lanes)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
        const uint32_t col = n0 + wn * (NI * 32u) + (uint32_t)ni * 32u + (lane & 31u);
        uint64_t at = (uint64_t)(m0 + row_of(0, 0)) * logits_stride + col;
        const uint64_t jump = 5u * logits_stride;   // (from row 3 of four to the next four)
        if (col < vocab) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    if (m0 + row_of(mi, v) < rows) {
                        const float f = acc[mi][ni][v];
                        if constexpr (OUT_F32) {
                            static_cast<float*>(logits_out)[at] = f;
                        } else {
                            static_cast<uint16_t*>(logits_out)[at] = (uint16_t)(__builtin_bit_cast(uint32_t, f) >> 16);
                        }
                    }
                    at += (v & 3) == 3 ? jump : logits_stride;
                }
            }
        }
    }
}

}  // namespace lily
