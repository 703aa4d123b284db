// q4_gemm_g64.hip -- the fast GEMM kernels of group size 64.
#include "q4_gemm_launch.hpp"

namespace sltx {

void launch_gemm_fast_g64(const GemmParams& p, bool bf16, bool silu, bool split, int wm, int kg, long grid,
                          hipStream_t st) {
    launch_gemm_fast<1>(p, bf16, silu, split, wm, kg, grid, st);
}

}  // namespace sltx
