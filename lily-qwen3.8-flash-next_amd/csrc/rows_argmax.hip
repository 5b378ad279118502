// rows_argmax.hip - launches whose rows are all greedy (temperature 0, nothing else asked): the exact
// first maximum of every row (elementwise.metal:145-150).
//
// The shortest call there is: its time is a chain of latencies - the launch, the arguments, one pass
// over the slice, the ticket's round trip, the partials' -, so the kernel holds nothing else: no
// select, 32 bytes of LDS, a row's arguments in 40 bytes, and from the slice's best on one wave works
// alone, without a barrier.  One row of 151 936 f32 logits in 38 slices: 6.25 us through the row
// kernel, 5.0 here.
#include "launch.h"
#include "row_kernel.h"

namespace lily {

namespace {

struct ArgmaxRow {
    const void* logits;
    uint32_t* out_id;
    const uint32_t* sel_row;   // see RowArgs
    uint64_t sel_stride;
    uint32_t sel_rows;
    uint32_t pad;
};
struct ArgmaxRows {
    ArgmaxRow r[INLINE_ROWS];
};

template <int DT, class ROW>
__device__ __forceinline__ bool argmax_row(const LILY_CONST ROW* r, const LaunchCfg& cfg) {
    __shared__ uint64_t best_of[NWAVE];
    const uint32_t tid = threadIdx.x, s = blockIdx.x, row = blockIdx.y, S = cfg.slices;
    const void* logits = r->logits;
    if (r->sel_row != nullptr) {
        const uint32_t at = min(*(const LILY_CONST uint32_t*)r->sel_row, r->sel_rows - 1u);
        logits = static_cast<const char*>(logits) + (size_t)at * r->sel_stride;
    }
    phase(cfg, 0);
    Geo<DT> g;
    g.init(logits, cfg.vocab, s, S);
    uint64_t best = wave_max_u64(thread_argmax<DT>(logits, g));
    if ((tid & 63u) == 0u) {
        best_of[tid >> 6] = best;
    }
    __syncthreads();
    if (tid >= 64u) {
        return false;
    }
#pragma unroll
    for (int i = 0; i < NWAVE; ++i) {
        best = best_of[i] > best ? best_of[i] : best;
    }
    phase(cfg, 4);
    if (S > 1u) {
        if (tid == 0u) {
            handed_store(cfg.ws_cand, ((size_t)row * S + s) * cfg.ws_k, best);
        }
        if (!wave_last_to_arrive(&cfg.ws_ticket[row], S, cfg.relaxed_handover != 0u)) {
            return false;
        }
        phase(cfg, 5);
        static_assert(MAX_SLICES <= 64u, "a slice a lane");
        best = wave_max_u64(tid < S ? handed_load(cfg.ws_cand, ((size_t)row * S + tid) * cfg.ws_k) : 0ull);
    }
    if (tid == 0u) {
        const uint32_t id = composite_id(best);
        *r->out_id = id == 0xffffffffu ? 0u : id;
    }
    phase(cfg, 7);
    return true;
}

template <int DT>
__global__ __launch_bounds__(NT) void k_argmax_inline(ArgmaxRows rows, LaunchCfg cfg) {
    const LILY_CONST ArgmaxRow* table = (const LILY_CONST ArgmaxRow*)__builtin_amdgcn_kernarg_segment_ptr();
    const bool finished = argmax_row<DT>(table + blockIdx.y, cfg);
    if (finished && threadIdx.x == 0u && cfg.accept_ctrl != nullptr) {
        accept_behind_last_row(cfg, [&](uint32_t j) { return (table + j)->out_id; });
    }
}

template <int DT>
__global__ __launch_bounds__(NT) void k_argmax_table(LaunchCfg cfg) {
    if (cfg.served != nullptr && *(const LILY_CONST uint32_t*)(cfg.served + blockIdx.y) != 0u) {
        return;
    }
    argmax_row<DT>((const LILY_CONST RowArgs*)cfg.table + blockIdx.y, cfg);
}

}  // namespace

hipError_t launch_rows_argmax(hipStream_t stream, int dtype, uint32_t rows, const LaunchCfg& cfg,
                              const InlineRows* inline_rows) {
    const dim3 grid(cfg.slices, rows), block(NT);
    if (inline_rows != nullptr) {
        ArgmaxRows few = {};
        for (uint32_t j = 0; j < rows && j < (uint32_t)INLINE_ROWS; ++j) {
            const RowArgs& r = inline_rows->r[j];
            few.r[j] = ArgmaxRow{r.logits, r.out_id, r.sel_row, r.sel_stride, r.sel_rows, 0u};
        }
        if (dtype == LILY_BF16) {
            hipLaunchKernelGGL((k_argmax_inline<LILY_BF16>), grid, block, 0, stream, few, cfg);
        } else {
            hipLaunchKernelGGL((k_argmax_inline<LILY_F32>), grid, block, 0, stream, few, cfg);
        }
    } else if (dtype == LILY_BF16) {
        hipLaunchKernelGGL((k_argmax_table<LILY_BF16>), grid, block, 0, stream, cfg);
    } else {
        hipLaunchKernelGGL((k_argmax_table<LILY_F32>), grid, block, 0, stream, cfg);
    }
    return hipGetLastError();
}

}  // namespace lily
