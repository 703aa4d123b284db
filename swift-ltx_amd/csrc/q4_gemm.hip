// q4_gemm.hip -- host side of the 4-bit dequant GEMM (q4_gemm_kernel.hpp):
// launch plan (tile height, K splits), the generic kernel's launches, and the
// passes that add split-K partial sums.
#include "q4_gemm_launch.hpp"

namespace sltx {

// Split-K reduction: out[m, n] = epilogue(sum over splits of the partials),
// summed in split order (deterministic).  SILU reduces gate and up
// separately before silu(gate) * up.  S > 0 is the split count, known at
// compile time: every split's loads are issued before the first add, so the
// pass pays one memory latency instead of one per split (the adds keep the
// split order, so the sums are the same bit for bit).  S == 0: any count.
template <bool SILU, int S>
__global__ __launch_bounds__(256) void q4_splitk_reduce_kernel(GemmParams p) {
    // each thread: 8 consecutive outputs of one row
    const int nb8 = (p.N + 7) / 8;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)p.M * nb8) return;
    const size_t m = idx / nb8;
    const int n0 = (int)(idx % nb8) * 8;
    const size_t nw = SILU ? 2 * (size_t)p.N : (size_t)p.N;
    const size_t stride = (size_t)p.M * nw;
    const float* src = p.ws + m * nw;
    const bool vin = (p.N & 7) == 0;   // 16-byte aligned workspace rows and no tail
    float a[8], u[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = u[e] = 0.0f;
    if constexpr (S > 0) {
        f32x4 q[S][2], r[SILU ? S : 1][2];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const f32x4* g = reinterpret_cast<const f32x4*>(src + s * stride + n0);
            q[s][0] = g[0];
            q[s][1] = g[1];
            if (SILU) {
                const f32x4* h = reinterpret_cast<const f32x4*>(src + s * stride + p.N + n0);
                r[s][0] = h[0];
                r[s][1] = h[1];
            }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                a[e] += q[s][0][e];
                a[4 + e] += q[s][1][e];
                if (SILU) {
                    u[e] += r[s][0][e];
                    u[4 + e] += r[s][1][e];
                }
            }
        }
    } else {
    for (int s = 0; s < p.splits; ++s, src += stride) {
        if (vin) {
            const f32x4* q = reinterpret_cast<const f32x4*>(src + n0);
            const f32x4 q0 = q[0], q1 = q[1];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                a[e] += q0[e];
                a[4 + e] += q1[e];
            }
            if (SILU) {
                const f32x4* r = reinterpret_cast<const f32x4*>(src + p.N + n0);
                const f32x4 r0 = r[0], r1 = r[1];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    u[e] += r0[e];
                    u[4 + e] += r1[e];
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (n0 + e < p.N) {
                    a[e] += src[n0 + e];
                    if (SILU) u[e] += src[p.N + n0 + e];
                }
            }
        }
    }
    }
    const bool vec = out_vec_ok(p);
    if (SILU) {
        const bool gelu = p.epilogue == kEpiGeluMul;
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = glu_f32(gelu, a[e], u[e]);
        store_out8(p, m * p.N, n0, a, vec);
    } else {
        epi_store8(p, m * p.N, n0, a, vec);
    }
}

// Split-K reduction fused with the residual add and the RMSNorm of each
// output row (one block of 256 threads per row, N % 8 == 0):
//   o = half(sum over splits, in split order)        the projection (linear)
//   t = float(residual) + float(o);  r = half(t)     elemAdd / residualRmsNorm
//   rms = rsqrt(mean(q^2) + eps), q = t (sum_rounded == 0, residualRmsNorm,
//         Kernels.swift:238-290) or q = float(r) (sum_rounded == 1: elemAdd then
//         rmsNorm of the stored fp16 stream, Kernels.swift:40-86, 121-128)
//   out = half(float(r) * rms * w)
// The partial sums follow q4_splitk_reduce_kernel and the row sum of squares
// follows rms_norm_vec_kernel (thread t: pieces t, t + 256, ... of 8 values;
// wave trees, then the four waves in order), so the results equal the unfused
// GEMM + reduce + norm sequence bit for bit.  S > 0 is the split count,
// known at compile time: a piece's loads of every split are issued before its
// first add (same order of adds).
template <int VPT, int S>
__global__ __launch_bounds__(256) void q4_splitk_residual_rms_norm_kernel(
    GemmParams p, const float* w, float eps, uint16_t* res_out, uint16_t* out, int sum_rounded) {
    __shared__ float red[4];
    const int nv = p.N / 8;
    const size_t m = blockIdx.x;
    const size_t stride = (size_t)p.M * p.N;
    const f16x8* R = reinterpret_cast<const f16x8*>(p.residual + m * p.N);
    f16x8 r[VPT];
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
        const int v = threadIdx.x + 256 * u;
        if (v >= nv) continue;
        float a[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = 0.0f;
        const float* q = p.ws + m * p.N + (size_t)v * 8;
        if constexpr (S > 0) {
            f32x4 qs[S][2];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                qs[s][0] = reinterpret_cast<const f32x4*>(q + s * stride)[0];
                qs[s][1] = reinterpret_cast<const f32x4*>(q + s * stride)[1];
            }
#pragma unroll
            for (int s = 0; s < S; ++s) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a[e] += qs[s][0][e];
                    a[4 + e] += qs[s][1][e];
                }
            }
        } else {
            for (int s = 0; s < p.splits; ++s, q += stride) {
                const f32x4 q0 = reinterpret_cast<const f32x4*>(q)[0];
                const f32x4 q1 = reinterpret_cast<const f32x4*>(q)[1];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a[e] += q0[e];
                    a[4 + e] += q1[e];
                }
            }
        }
        const f16x8 h = R[v];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float t = (float)h[e] + h2f(f2h(a[e]));
            r[u][e] = (f16)t;
            const float sq = sum_rounded ? (float)r[u][e] : t;
            ss += sq * sq;
        }
        reinterpret_cast<f16x8*>(res_out + m * p.N)[v] = r[u];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float rms = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)p.N + eps);
    const f32x4* W = reinterpret_cast<const f32x4*>(w);
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
        const int v = threadIdx.x + 256 * u;
        if (v >= nv) continue;
        const f32x4 w0 = W[2 * v], w1 = W[2 * v + 1];
        f16x8 o8;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o8[e] = (f16)((float)r[u][e] * rms * w0[e]);
            o8[4 + e] = (f16)((float)r[u][4 + e] * rms * w1[e]);
        }
        reinterpret_cast<f16x8*>(out + m * p.N)[v] = o8;
    }
}

// The fixed-count kernel needs whole 128-k super-stages, and for group size
// 128 whole pairs of them (scales and biases move as dword pairs of groups, so
// their arrays must also be 4-byte aligned; 2-byte aligned ones take the
// generic kernel, which reads them as 16-bit values), and 32-bit offsets
// within a tile's rows.
static bool fast_gemm(const GemmParams& p) {
    const uintptr_t sb_addr = reinterpret_cast<uintptr_t>(p.s0) | reinterpret_cast<uintptr_t>(p.b0) |
                              reinterpret_cast<uintptr_t>(p.s1) | reinterpret_cast<uintptr_t>(p.b1);
    return !p.a_f32 && p.K <= (1 << 22) && p.K % (p.gshift == 2 ? 4 * BK : 2 * BK) == 0 && (sb_addr & 3) == 0;
}

// Launch plan: block-tile height WM (BM = 64*WM) and K splits, chosen by
// estimated time on 256 CUs: rounds of blocks x (k-tiles per block x the
// measured time of one k-tile -- 1.37 us at BM = 192, 0.95 us at BM = 128,
// a 256-row W tile -- plus ~8 us of prologue and epilogue, which every round
// repeats) + ~2 us per launch, plus, when split, writing the fp32 partials
// (~6 TB/s) and the reduce pass reading them back (~4 TB/s, its own launch).
// Measured at M = 750 (lm_head, N = 128256): 664 us at BM = 192 vs 730 us at
// BM = 128; DiT up (M = 6144, bf16): 318 vs 356 us.  Tiles of 128 x 128
// (kg = 2, the fast kernel) are for single rounds where 256-row weight tiles
// would leave CUs idle or split K.  Measured, kg = 2 against the best kg = 1
// plan: q|k|v at M = 750 (240 blocks against 120 in two splits) 33.5 / 42.4 us,
// gate/up at M = 200 32.0 / 40.9, 2048 x 2048 at M = 1537 23.0 / 30.9, 4096 x
// 4096 at M = 1000 47.5 / 52.7; long K turns it round: down at M = 750 64 / 55,
// 2048 x 8192 at M = 1537 76 / 71, the T5 GeGLU pair at M = 128 45.5 / 42.2.
// Its 0.62 us per k-tile (0.55 measured) puts the line between those.  Splits cover an even
// number of k-tiles (packed weights move two k-tiles at a time).
struct GemmPlan {
    int wm, kg, tiles_m, tiles_n, splits, split_tiles;
    size_t ws_bytes;
};

static GemmPlan plan_gemm(const GemmParams& p, bool allow_split) {
    const bool silu = p.epilogue == kEpiSiluMul || p.epilogue == kEpiGeluMul;
    const int nk = (p.K + BK - 1) / BK;
    const size_t nw = silu ? 2 * (size_t)p.N : (size_t)p.N;
    GemmPlan best = {2, 1, 0, 0, 1, nk, 0};
    double best_us = 1e30;
    const bool fast = fast_gemm(p);
    static const struct { int wm, kg; double kt_us; } kTiles[] = {{2, 1, 0.95}, {3, 1, 1.37}, {2, 2, 0.62}};
    for (const auto& t : kTiles) {
        // fp32 activations hold a k-tile of A in registers: the 192-row tile
        // would spill, so they take the 128-row tile only
        if ((p.a_f32 && t.wm > 2) || (t.kg > 1 && !fast)) continue;
        const int wm = t.wm, bm = 64 * wm, bn_out = BN / t.kg / (silu ? 2 : 1);
        const long tiles_n = ((long)p.N + bn_out - 1) / bn_out;
        const long tiles_m = (p.M + bm - 1) / bm;
        const long tiles = tiles_m * tiles_n;
        const double kt_us = t.kt_us;
        const int smax = allow_split ? 8 : 1;
        for (int s = 1; s <= smax; ++s) {
            if (s > 1 && nk < 8 * s) break;
            int chunk = (nk + s - 1) / s;
            chunk = s > 1 ? (chunk + 1) / 2 * 2 : chunk;
            const int s_eff = (nk + chunk - 1) / chunk;
            if (s > 1 && s_eff != s) continue;
            const long blocks = tiles * s_eff;
            if (t.kg > 1 && blocks > kCUs) break;
            const long rounds = (blocks + kCUs - 1) / kCUs;
            double us = (double)rounds * (chunk * kt_us + 8.0) + 2.0;
            const bool ws = s_eff > 1;
            if (ws) {
                const double part = (double)s_eff * p.M * nw * 4.0;
                us += part / 6.0e6 + 3.0 + (part + (double)p.M * p.N * 2.0) / 4.0e6;
            }
            if (us < best_us) {
                best_us = us;
                best = {wm, t.kg, (int)tiles_m, (int)tiles_n, s_eff, chunk,
                        ws ? (size_t)s_eff * p.M * nw * sizeof(float) : 0};
            }
        }
    }
    return best;
}

size_t gemm_workspace_bytes(const GemmParams& p) { return plan_gemm(p, true).ws_bytes; }
int gemm_splits(const GemmParams& p) { return plan_gemm(p, true).splits; }
void gemm_tile(const GemmParams& p, int* rows, int* wrows) {
    const GemmPlan pl = plan_gemm(p, true);
    *rows = 64 * pl.wm;
    *wrows = BN / pl.kg;
}
size_t gemm_partials_workspace_bytes(const GemmParams& p) {
    return (size_t)gemm_splits(p) * p.M * p.N * sizeof(float);
}

// The fast kernel's launcher of each group size, one translation unit each
// (q4_gemm_g32.hip, q4_gemm_g64.hip, q4_gemm_g128.hip).
template <int WM, bool BF16, bool SPLIT>
static void launch_wm(const GemmParams& p, bool silu, int kg, long grid, hipStream_t st) {
    if constexpr (WM == 2) {
        if (p.a_f32) {
            hipLaunchKernelGGL((q4_gemm_kernel<2, false, false, true, SPLIT, true>), dim3(grid),
                               dim3(kThreads), 0, st, p);
            return;
        }
    }
    if (fast_gemm(p)) {
        if (p.gshift == 0) launch_gemm_fast_g32(p, BF16, silu, SPLIT, WM, kg, grid, st);
        else if (p.gshift == 1) launch_gemm_fast_g64(p, BF16, silu, SPLIT, WM, kg, grid, st);
        else launch_gemm_fast_g128(p, BF16, silu, SPLIT, WM, kg, grid, st);
        return;
    }
    if (silu)
        hipLaunchKernelGGL((q4_gemm_kernel<WM, BF16, true, true, SPLIT>), dim3(grid), dim3(kThreads), 0, st, p);
    else
        hipLaunchKernelGGL((q4_gemm_kernel<WM, BF16, false, true, SPLIT>), dim3(grid), dim3(kThreads), 0, st, p);
}

template <bool SPLIT>
static void launch_dtype(const GemmParams& p, bool a_bf16, bool silu, long grid, const GemmPlan& pl,
                         hipStream_t st) {
    if (a_bf16) {
        if (pl.wm == 2) launch_wm<2, true, SPLIT>(p, silu, pl.kg, grid, st);
        else launch_wm<3, true, SPLIT>(p, silu, pl.kg, grid, st);
    } else {
        if (pl.wm == 2) launch_wm<2, false, SPLIT>(p, silu, pl.kg, grid, st);
        else launch_wm<3, false, SPLIT>(p, silu, pl.kg, grid, st);
    }
}

template <bool SILU>
void launch_reduce_s(const GemmParams& p, dim3 g, hipStream_t st) {
    // the loads-first form needs whole 16-byte rows (N % 8 == 0)
    const int s = (p.N & 7) == 0 ? p.splits : 0;
    switch (s) {
    case 2: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 2>), g, dim3(256), 0, st, p); break;
    case 3: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 3>), g, dim3(256), 0, st, p); break;
    case 4: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 4>), g, dim3(256), 0, st, p); break;
    case 5: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 5>), g, dim3(256), 0, st, p); break;
    case 6: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 6>), g, dim3(256), 0, st, p); break;
    case 7: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 7>), g, dim3(256), 0, st, p); break;
    case 8: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 8>), g, dim3(256), 0, st, p); break;
    default: hipLaunchKernelGGL((q4_splitk_reduce_kernel<SILU, 0>), g, dim3(256), 0, st, p); break;
    }
}

hipError_t launch_splitk_reduce(const GemmParams& p, hipStream_t st) {
    const bool silu = p.epilogue == kEpiSiluMul || p.epilogue == kEpiGeluMul;
    const size_t total = (size_t)p.M * ((p.N + 7) / 8);
    const dim3 rgrid((unsigned)((total + 255) / 256));
    if (silu)
        launch_reduce_s<true>(p, rgrid, st);
    else
        launch_reduce_s<false>(p, rgrid, st);
    return hipGetLastError();
}

hipError_t launch_gemm(GemmParams p, bool a_bf16, hipStream_t st) {
    const bool silu = p.epilogue == kEpiSiluMul || p.epilogue == kEpiGeluMul;
    GemmPlan plan = plan_gemm(p, p.ws != nullptr);
    p.nib_mask = 0x0F0F0F0Fu;
    p.tiles_m = plan.tiles_m;
    p.tiles_n = plan.tiles_n;
    p.splits = plan.splits;
    p.split_tiles = plan.split_tiles;
    const long ntiles = (long)p.tiles_m * p.tiles_n;
    if (ntiles <= 0) return hipSuccess;
    const long blocks = ntiles * p.splits;
    const long grid = (blocks + 7) / 8 * 8;
    if (grid > 0x7fffffffL) return hipErrorInvalidValue;
    if (p.splits > 1) {
        launch_dtype<true>(p, a_bf16, silu, grid, plan, st);
        (void)launch_splitk_reduce(p, st);
    } else {
        launch_dtype<false>(p, a_bf16, silu, grid, plan, st);
    }
    return hipGetLastError();
}

template <int VPT>
void launch_rrn_s(const GemmParams& p, const float* norm_w, float eps, uint16_t* res_out,
                  uint16_t* norm_out, int sr, hipStream_t st) {
    const dim3 g(p.M), t(256);
    switch (p.splits) {
    case 2: hipLaunchKernelGGL((q4_splitk_residual_rms_norm_kernel<VPT, 2>), g, t, 0, st, p, norm_w, eps, res_out, norm_out, sr); break;
    case 3: hipLaunchKernelGGL((q4_splitk_residual_rms_norm_kernel<VPT, 3>), g, t, 0, st, p, norm_w, eps, res_out, norm_out, sr); break;
    case 4: hipLaunchKernelGGL((q4_splitk_residual_rms_norm_kernel<VPT, 4>), g, t, 0, st, p, norm_w, eps, res_out, norm_out, sr); break;
    default: hipLaunchKernelGGL((q4_splitk_residual_rms_norm_kernel<VPT, 0>), g, t, 0, st, p, norm_w, eps, res_out, norm_out, sr); break;
    }
}

// GEMM into fp32 partials (gemm_splits(p) > 1; p.ws holds
// gemm_partials_workspace_bytes(p)), then the fused reduce + residual +
// RMSNorm pass.  Requires N % 8 == 0, N <= 16384 and 16-byte aligned rows.
hipError_t launch_gemm_residual_rms_norm(GemmParams p, bool a_bf16, const float* norm_w, float eps,
                                         uint16_t* res_out, uint16_t* norm_out, bool sum_rounded,
                                         hipStream_t st) {
    if (p.M <= 0 || p.N <= 0) return hipSuccess;
    if (p.N % 8 != 0 || p.N / 8 > 8 * 256 || !p.ws || !p.residual) return hipErrorInvalidValue;
    if ((long)p.M * 256 > 0xffffffffL) return hipErrorInvalidValue;   // one 256-thread block per row
    const GemmPlan plan = plan_gemm(p, true);
    if (plan.splits < 2) return hipErrorInvalidValue;
    p.nib_mask = 0x0F0F0F0Fu;
    p.tiles_m = plan.tiles_m;
    p.tiles_n = plan.tiles_n;
    p.splits = plan.splits;
    p.split_tiles = plan.split_tiles;
    const long blocks = (long)p.tiles_m * p.tiles_n * p.splits;
    const long grid = (blocks + 7) / 8 * 8;
    if (grid > 0x7fffffffL) return hipErrorInvalidValue;
    launch_dtype<true>(p, a_bf16, false, grid, plan, st);
    const int vpt = (p.N / 8 + 255) / 256;
    const int sr = sum_rounded ? 1 : 0;
    if (vpt == 1)
        launch_rrn_s<1>(p, norm_w, eps, res_out, norm_out, sr, st);
    else if (vpt == 2)
        launch_rrn_s<2>(p, norm_w, eps, res_out, norm_out, sr, st);
    else if (vpt <= 4)
        launch_rrn_s<4>(p, norm_w, eps, res_out, norm_out, sr, st);
    else
        launch_rrn_s<8>(p, norm_w, eps, res_out, norm_out, sr, st);
    return hipGetLastError();
}

}  // namespace sltx
