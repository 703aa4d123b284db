// q4_gemm_launch.hpp -- launches of the GEMM's fast kernel for one group size.
// Each group size is a translation unit of its own, so that they compile in
// parallel.
#pragma once

#include "q4_gemm_kernel.hpp"

namespace sltx {

void launch_gemm_fast_g32(const GemmParams& p, bool bf16, bool silu, bool split, int wm, int kg, long grid,
                          hipStream_t st);
void launch_gemm_fast_g64(const GemmParams& p, bool bf16, bool silu, bool split, int wm, int kg, long grid,
                          hipStream_t st);
void launch_gemm_fast_g128(const GemmParams& p, bool bf16, bool silu, bool split, int wm, int kg, long grid,
                           hipStream_t st);

// p.K % 128 == 0 (GS = 2: % 256), group size 32 << GS, 4-byte aligned scales
// and biases.  grid: blocks of the launch plan.
template <int GS, int WM, bool BF16, bool SILU>
void launch_gemm_fast_k(const GemmParams& p, bool split, int kg, long grid, hipStream_t st) {
    const dim3 t(kThreads);
    if constexpr (WM == 2) {
        // 128-row weight tiles: a single round (the plan's choice)
        if (kg == 2) {
            if (split)
                hipLaunchKernelGGL((q4_gemm_kernel<WM, BF16, SILU, false, true, false, false, GS, 2>), dim3(grid), t, 0, st, p);
            else
                hipLaunchKernelGGL((q4_gemm_kernel<WM, BF16, SILU, false, false, false, false, GS, 2>), dim3(grid), t, 0, st, p);
            return;
        }
    }
    if (split) {
        hipLaunchKernelGGL((q4_gemm_kernel<WM, BF16, SILU, false, true, false, false, GS>), dim3(grid), t, 0, st, p);
    } else if (p.K % (4 * BK) == 0 && (long)p.tiles_m * p.tiles_n > kCUs) {
        // More tiles than one block per CU: one persistent block per CU walks
        // them (the ring's stage parity restarts with each tile: K % 256 == 0).
        hipLaunchKernelGGL((q4_gemm_kernel<WM, BF16, SILU, false, false, false, true, GS>), dim3(kCUs), t, 0, st, p);
    } else {
        hipLaunchKernelGGL((q4_gemm_kernel<WM, BF16, SILU, false, false, false, false, GS>), dim3(grid), t, 0, st, p);
    }
}

// The gated pairs take fp16 activations only.
template <int GS>
void launch_gemm_fast(const GemmParams& p, bool bf16, bool silu, bool split, int wm, int kg, long grid,
                      hipStream_t st) {
    auto by_height = [&](auto b, auto s) {
        if (wm == 2) launch_gemm_fast_k<GS, 2, decltype(b)::value, decltype(s)::value>(p, split, kg, grid, st);
        else launch_gemm_fast_k<GS, 3, decltype(b)::value, decltype(s)::value>(p, split, kg, grid, st);
    };
    if (bf16) by_height(std::true_type{}, std::false_type{});
    else if (silu) by_height(std::false_type{}, std::true_type{});
    else by_height(std::false_type{}, std::false_type{});
}

}  // namespace sltx
