// launch.h - host-callable launchers defined in sampler_kernels.hip.
#pragma once

#include <hip/hip_runtime_api.h>

#include <atomic>

#include "row_args.h"

namespace lily {

constexpr uint32_t CU_LDS_BYTES = 160u * 1024u;   // a compute unit's

// A launch may have 64 KB of LDS without asking.  One of these beside a kernel asks for all of a
// compute unit's, once per device; any number of threads launch it with any sizes meanwhile.  (A
// table of the size each launch needed let a thread with a small one lower what another had just
// raised.)
struct LdsAllowed {
    std::atomic<bool> said[64] = {};
    // `bytes`: always the same for one kernel (a kernel with LDS of its own cannot have all of it)
    hipError_t say(const void* kernel, uint32_t bytes = CU_LDS_BYTES) {
        int device = 0;
        hipError_t e = hipGetDevice(&device);
        const bool known = e == hipSuccess && device >= 0 && device < 64;
        if (e != hipSuccess || (known && said[device].load(std::memory_order_acquire))) {
            return e;
        }
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e == hipSuccess && known) {
            said[device].store(true, std::memory_order_release);
        }
        return e;
    }
};

// `kind`: 0 = no row has a mask, penalties or a bias list, 1 = some row has, 2 = every sampled
// row takes the streaming select; `lse`: some row wants a log-probability.
// `dyn_bytes`: dynamic LDS (see shape_of in sampler_api.cpp).
hipError_t launch_rows(hipStream_t stream, int dtype, int kind, bool lse, uint32_t rows,
                       const LaunchCfg& cfg, const InlineRows* inline_rows, size_t dyn_bytes);
hipError_t launch_fill_u32(hipStream_t stream, uint32_t* p, uint32_t n, uint32_t v);
hipError_t launch_add_history(hipStream_t stream, const ScratchView& sc, const uint32_t* ids,
                              uint32_t n);
hipError_t launch_uncount(hipStream_t stream, const ScratchView& sc, uint32_t token);
hipError_t launch_uncount_after(hipStream_t stream, const ScratchView& sc, const uint32_t* draws,
                                uint32_t m, const uint32_t* accepted, uint32_t cap);
// touched = the ids with a non-zero count.
hipError_t launch_rebuild_listed(hipStream_t stream, const ScratchView& sc);
hipError_t launch_spec_accept(hipStream_t stream, const uint32_t* draws, const uint32_t* ids,
                              uint32_t* ctrl, uint32_t m, uint32_t pos0, uint32_t ratio,
                              uint32_t chain);
// logits[rows, vocab] = hidden[rows, d] x weight[vocab, d]^T (bf16, strides in elements, d a
// multiple of 64), with the largest value and the sum of 2^((x - largest) * c2_of_row[row]) of
// every LILY_TILE_COLS columns in tile_max / tile_sum [rows, ceil(vocab / LILY_TILE_COLS)].
// out_f32: the logits are f32 [rows, logits_stride] instead of bf16.  wq.bits 4 / 8: `weight` points
// at the reference's affine codes (u32 words, weight_stride words a row), wq.scales / wq.biases at
// bf16 [vocab, d >> wq.group_shift]; f32 logits only.
// The rows' exponent scales: in device memory, or (p null, at most SCALES_INLINE rows) with the launch itself.  A launch that
// has them with it may also carry something to the device while it runs, for the launches behind it: `pieces` of
// 16 bytes from src (pinned host memory, mapped into the device) to dst.
constexpr uint32_t SCALES_INLINE = 128;
struct RowScales {
    const float* p = nullptr;
    float few[SCALES_INLINE] = {};
    const void* src = nullptr;
    void* dst = nullptr;
    uint32_t pieces = 0;
    RowScales() = default;
    RowScales(const float* from) : p(from) {}
};
struct HeadWeights {
    uint32_t bits = 0;          // 0 = bf16 weights
    const void* scales = nullptr;
    const void* biases = nullptr;
    uint32_t group_shift = 6;   // log2 of the group size
    // batches of at least this many rows go through the vendor's GEMM library where it is present
    // and takes the shape, followed by the pass that forms the summaries (0: never)
    uint32_t library_rows = 0;
    unsigned long long* library_calls = nullptr;   // counts the calls that went that way
};
hipError_t launch_lm_head_bf16(hipStream_t stream, const void* hidden, uint64_t hidden_stride,
                               const void* weight, uint64_t weight_stride, uint32_t rows, uint32_t d,
                               uint32_t vocab, const RowScales& c2_of_row, void* logits,
                               uint64_t logits_stride, float* tile_max, float* tile_sum, bool out_f32,
                               const HeadWeights& wq);
// The same over codes for up to 16 rows in the reference's form for few rows (the codes are not
// turned into weights: scale * sum(q * x) + bias * sum(x) per group, f32 logits); `serves` says
// whether a shape can take it (groups of 64 or more, operands within 4 GB).
bool lm_head_codes_serves(uint32_t rows, uint32_t d, uint32_t vocab, uint64_t hidden_stride, uint64_t weight_stride,
                          const HeadWeights& wq);
hipError_t launch_lm_head_codes(hipStream_t stream, const void* hidden, uint64_t hidden_stride, const void* weight,
                                uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                                const RowScales& c2_of_row, void* logits, uint64_t logits_stride, float* tile_max,
                                float* tile_sum, const HeadWeights& wq);
// The same for any number of rows with the weights in bf16, as dequant_q4/q8_bf16 make them of the
// codes (groups of 64 or more, whole lines of codes).
bool lm_head_codes_rows_serves(uint32_t d, const HeadWeights& wq);
// Workgroups of its 128-row tile that fit a compute unit's LDS (d and groups that it serves).
uint32_t lm_head_codes_rows_resident(uint32_t d, const HeadWeights& wq);
hipError_t launch_lm_head_codes_rows(hipStream_t stream, const void* hidden, uint64_t hidden_stride, const void* weight,
                                     uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab,
                                     const RowScales& c2_of_row, void* logits, uint64_t logits_stride, float* tile_max,
                                     float* tile_sum, const HeadWeights& wq);
// The batch form through the vendor's GEMM library, opened by name at run time: the product alone
// (codes are turned into bf16 weights first, in memory this call keeps per device and stream);
// hipErrorNotSupported where the library is absent or has no algorithm for the shape - the
// caller then runs its own kernel.  launch_head_summaries: tile_max / tile_sum of stored logits.
constexpr uint32_t HEAD_LIBRARY_MAX_TILES = 2048;   // summaries a row that launch_head_summaries takes
bool head_library_present();
hipError_t launch_head_library(hipStream_t stream, const void* hidden, uint64_t hidden_stride, const void* weight,
                               uint64_t weight_stride, uint32_t rows, uint32_t d, uint32_t vocab, void* logits,
                               uint64_t logits_stride, bool out_f32, const HeadWeights& wq);
hipError_t launch_head_summaries(hipStream_t stream, const void* logits, uint64_t logits_stride, uint32_t rows,
                                 uint32_t vocab, const float* c2_of_row, float* tile_max, float* tile_sum,
                                 bool f32);
// The same of at most INLINE_ROWS rows that travel with the launch, each with its row of the summaries in
// RowArgs::pad; none under penalties or a mask.
hipError_t launch_rows_tiles_inline(hipStream_t stream, int dtype, bool lse, bool extra, uint32_t rows, const LaunchCfg& cfg,
                                    const InlineRows& inline_rows, const float* tile_max, const float* tile_sum,
                                    uint32_t tiles);
// The draw of `rows` rows of cfg.table from the summaries ([.., tiles] each) and the few tiles of
// the logits (bf16 or f32) that matter; tile_row[r] = the summaries' row of table row r; served[r] is set
// for rows under penalties or a mask (1 = drawn, 0 = declined: the row is better read whole).
// `extra`: some row carries a bias list or a mask.
hipError_t launch_rows_tiles(hipStream_t stream, int dtype, bool lse, bool extra, uint32_t rows,
                             const LaunchCfg& cfg, const float* tile_max, const float* tile_sum,
                             uint32_t tiles, const uint32_t* tile_row, uint32_t* served);
// Rows that are all greedy (MODE_ARGMAX), given inline or as cfg.table; cfg.accept_ctrl (inline rows): a
// verify pass, whose acceptance runs behind the last row.
hipError_t launch_rows_argmax(hipStream_t stream, int dtype, uint32_t rows, const LaunchCfg& cfg,
                              const InlineRows* inline_rows);
// Sampled rows of the streaming kind (F_STREAM), given inline or as cfg.table, whose slices hold at most `blocks`
// (1 or 2) times 256 x STREAM_UNROLL pieces of 16 bytes and k <= 64 candidates each, at most
// HELD_MERGE_SLOTS a row in more than three slices.  `extra`: some row carries a mask or a bias list;
// cfg.verify: a verify pass of independent plain rows (inline).
constexpr uint32_t HELD_MERGE_SLOTS = 2048;
hipError_t launch_rows_held(hipStream_t stream, int dtype, uint32_t blocks, bool lse, bool extra, uint32_t rows,
                            const LaunchCfg& cfg, const InlineRows* inline_rows);
// The same rows of cfg.table (no mask, no bias list, plain draws) in slices of any length, a block at a time.
hipError_t launch_rows_blocks(hipStream_t stream, int dtype, bool lse, bool pen, uint32_t rows, const LaunchCfg& cfg);
// Plain draws under an allow-mask with at most STREAM_BIAS_CAP bias pairs, given inline or as cfg.table: a workgroup a
// row whatever cfg.slices says, vocabularies up to MASKED_MAX_VOCAB.
constexpr uint32_t MASKED_MAX_VOCAB = 262144;
hipError_t launch_rows_masked(hipStream_t stream, int dtype, bool lse, uint32_t rows, const LaunchCfg& cfg,
                              const InlineRows* inline_rows);
// Rows that draw among many candidates (k > 64), spread over cfg.slices workgroups a row: two
// launches (the row's bound, then the values that reach it, merge, select, tail).
// lane_max [rows][slices][256]; count [rows] and bounds [2][rows][MAX_SLICES], both 0 between launches (bounds: for the
// one launch that small batches take instead).
// `looks`: how often a slice of that launch looks for the words of its row's other slices, in either of its waits,
// before it leaves the row to the exhaustive select.
struct WideLooks {
    uint32_t keys = 1u << 13, maxima = 1u << 13;
};
hipError_t launch_rows_wide(hipStream_t stream, int dtype, bool lse, uint32_t rows, const LaunchCfg& cfg,
                            const InlineRows* inline_rows, float* lane_max, uint32_t* count, uint64_t* bounds,
                            const WideLooks& looks);
// `bytes` (a multiple of 16) from pinned host memory, mapped into the device at src, to dst.
hipError_t launch_copy_pieces(hipStream_t stream, const void* src, void* dst, size_t bytes);
// The same of up to sizeof(PlacedPieces) bytes from any host memory, through the launch's arguments.
constexpr unsigned PLACED_PIECES = 128;
struct alignas(16) PlacedPieces {
    char b[PLACED_PIECES * 16];
};
hipError_t launch_place_pieces(hipStream_t stream, const void* src, void* dst, size_t bytes);
hipError_t launch_probe_read(hipStream_t stream, const void* base, uint32_t rows, uint64_t row_bytes,
                             uint64_t stride_bytes, uint32_t* out);
hipError_t launch_copy_row(hipStream_t stream, const uint32_t* src, uint32_t* dst, uint32_t words,
                           uint32_t rows, const uint32_t* row_dev);

}  // namespace lily
