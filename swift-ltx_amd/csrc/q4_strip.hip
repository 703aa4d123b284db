// q4_strip.hip -- 4-bit dequant matmul for few output columns of many fp32
// activation rows: a diffusion transformer's output projection
// (DiTLinear.applyF32in's q4 branch, DiTModel.swift:102-125) on CDNA4 MFMA.
//
// Same product as q4_gemm_kernel.hpp, Y[M,N] = X[M,K] . dequant(W)[N,K]^T with
// fp32 accumulation, x cast as cast_f32_to_f16 does, half(clamp(x, -65504,
// 65504)) (Kernels.swift:816-822).
// With few columns X is nearly all of the traffic (M = 6144, K = 2048, N =
// 128: 50 MB of fp32 against 0.14 MB of weights), so the launch is bound by
// streaming X from HBM once.  The GEMM's 128 x 256 tiles gave it 48 blocks,
// half of each padding, four K splits and a reduce pass.
//  * Block: 32 or 64 activation rows x 128 weight rows, all of K, 512 threads:
//    the lower height that covers the launch in one round of blocks.  Column blocks of the same rows follow
//    each other on one XCD, so rows past the first column block come from its
//    L2.
//  * The 8 waves split K as in q4_wide.hip: in a round of 128 k, wave g takes
//    the 16-k MFMA step g and all of the block's 32 x 32 tiles
//    (v_mfma_f32_32x32x16_f16), so no element of X or W is read from LDS
//    by two waves, each packed word is dequantized once per block, and X is cast
//    in registers on its way to the MFMA.
//  * X and packed W pass through a ring of four stages (three at 64 rows) of direct-to-LDS copies
//    (16-byte pieces, whole lines), one exact wait count and one LDS-only
//    barrier per round; scales and biases (at most 64 groups a row) are read
//    once into an LDS slab.
//  * After the last round the waves' tiles are summed in LDS in wave order.
// Measured at M = 6144, K = 2048, N = 128: 16.5 us (3.3 TB/s) against the GEMM's
// 25.2.  A round is 0.53 us at 32 rows, 0.8 at 64, whatever the number of
// blocks: the chain of LDS reads, casts and dequantization between two
// barriers, not HBM, is what bounds it; bf16 x, whose dequantization is longer
// and whose GEMM needs no cast, gained nothing and keeps the GEMM.
#include <type_traits>

#include "q4_common.hpp"
#include "q4_dequant.hpp"
#include "q4_epilogue.hpp"
#include "q4_launch.hpp"
#include "q4_ring.hpp"

namespace sltx {

namespace {

constexpr int NWV = 8;               // waves, one K-group each
constexpr int ST = 64 * NWV;         // threads per block
constexpr int SBN = 128;             // weight rows per block
constexpr int NJ = SBN / 32;         // MFMA tiles along N
constexpr int RK = NWV * 16;         // k per round
constexpr int WRD = RK / 8;          // packed words of a weight row per round (16)
constexpr int SLAB_G = 64;           // scale / bias groups a block holds

// W word (row, w) of a stage: the row's 16-byte piece p at position
// p ^ ((row >> 2) & 3) (q4_wide.hip's layout).
__device__ __forceinline__ int wpos(int row, int w) {
    return row * WRD + ((((w >> 2) ^ (row >> 2)) & 3) << 2) + (w & 3);
}
// Slab entry (group gi, row).
__device__ __forceinline__ int spos(int gi, int row) { return gi * SBN + (row ^ (gi & 63)); }

// Two activations as fp16, half(clamp(x, -65504, 65504)).  v_med3_f32 of a NaN
// and the two bounds is the lower one, as the reference's clamp gives it.
typedef float f32p2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t clamp_f16x2(float lo, float hi) {
    const f32p2 v = {__builtin_amdgcn_fmed3f(lo, -65504.0f, 65504.0f),
                     __builtin_amdgcn_fmed3f(hi, -65504.0f, 65504.0f)};
    return as_u32(__builtin_convertvector(v, f16x2));
}

// MT: 32-row MFMA tiles along M per block.
template <int MT>
__global__ __launch_bounds__(ST, 1) void q4_strip_kernel(GemmParams p) {
    constexpr int SBM = 32 * MT;              // activation rows per block
    constexpr int NS = MT == 1 ? 4 : 3;       // ring stages
    constexpr int XB = 4;                     // bytes of an activation
    constexpr int XCH = RK * XB / 16;         // 16-byte pieces of an X row per round (32)
    constexpr int XS = SBM * XCH;             // pieces of an X stage
    constexpr int NXC = XS / ST;              // X copies per thread per round (2 MT)
    constexpr int WPC = SBN * WRD / 4;        // 16-byte W pieces per round
    static_assert(WPC == ST && NXC * ST == XS, "whole copies");
    constexpr int CPR = NXC + 1;              // vector-memory ops per thread per round
    __shared__ u32x4 xs0[XS], xs1[XS], xs2[XS], xs3[NS > 3 ? XS : 1];
    __shared__ u32x4 ws0[WPC], ws1[WPC], ws2[WPC], ws3[NS > 3 ? WPC : 1];
    __shared__ uint32_t slab[SLAB_G * SBN];
    auto xstage = [&](auto sc) -> u32x4* {
        constexpr int S = decltype(sc)::value % NS;
        if constexpr (S == 0) return xs0;
        else if constexpr (S == 1) return xs1;
        else if constexpr (S == 2) return xs2;
        else return xs3;
    };
    auto wstage = [&](auto sc) -> u32x4* {
        constexpr int S = decltype(sc)::value % NS;
        if constexpr (S == 0) return ws0;
        else if constexpr (S == 1) return ws1;
        else if constexpr (S == 2) return ws2;
        else return ws3;
    };

    // XCD x (blocks x, x + 8, ...) takes logical blocks x G/8 .. (G = grid, a
    // multiple of 8), columns fastest.
    const int logical = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    if (logical >= p.tiles_m * p.tiles_n) return;
    const int m0 = logical / p.tiles_n * SBM, n0 = logical % p.tiles_n * SBN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = p.K, nr = K / RK;

    // ---- copy sources: a block base and 32-bit byte offsets ----
    // X copy i of thread t fills piece s = t + ST i: row s / XCH, physical piece
    // s % XCH = logical piece ^ (row % XCH); rows past M read row M - 1.  W:
    // thread t fills piece t, row t / 4; rows past N read row N - 1.  Neither is
    // stored.
    const char* const xb = reinterpret_cast<const char*>(p.a) + (size_t)m0 * K * XB;
    const char* const wb = reinterpret_cast<const char*>(p.w0) + (size_t)n0 * (K / 2);
    uint32_t xoff[NXC], woff;
#pragma unroll
    for (int i = 0; i < NXC; ++i) {
        const int s = tid + ST * i, row = s / XCH, c = (s % XCH) ^ (row % XCH);
        xoff[i] = (uint32_t)min(row, p.M - 1 - m0) * (uint32_t)(K * XB) + c * 16;
    }
    {
        const int row = tid >> 2, lp = (tid & 3) ^ ((row >> 2) & 3);
        woff = (uint32_t)min(row, p.N - 1 - n0) * (uint32_t)(K / 2) + lp * 16;
    }
    auto issue = [&](auto sc, int q) {   // CPR vector-memory ops (past the end: the last round again)
        const int qc = min(q, nr - 1);
        const char* const xq = xb + (size_t)qc * (RK * XB);
        const char* const wq = wb + (size_t)qc * (RK / 2);
        u32x4* const xd = xstage(sc) + 64 * wave;
#pragma unroll
        for (int i = 0; i < NXC; ++i)
            __builtin_amdgcn_global_load_lds((const void*)(xq + xoff[i]), (lds_ptr_t)(xd + ST * i), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const void*)(wq + woff), (lds_ptr_t)(wstage(sc) + 64 * wave), 16, 0, 0);
    };
    static_for<NS - 1>([&](auto sc) { issue(sc, decltype(sc)::value); });

    // ---- scale / bias slab: wave w fills rows 16 w .. 16 w + 15, lanes along
    // a row's groups ----
    const int ng = p.groups;   // <= SLAB_G
    {
        uint32_t sv[16], bv[16];
        const int gi = min(lane, ng - 1);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const size_t o = (size_t)min(n0 + 16 * wave + u, p.N - 1) * ng + gi;
            sv[u] = p.s0[o];
            bv[u] = p.b0[o];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (lane < ng) slab[spos(lane, 16 * wave + u)] = sv[u] | (bv[u] << 16);
    }

    const int r = lane & 31, h = lane >> 5;
    const int c = 2 * wave + h;         // this lane's 8 k of a round: X piece(s) and W word
    const int glog2 = 5 + p.gshift;
    f32x16 acc[MT][NJ];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    u32x4 a[MT], b[NJ];                 // operands of the round whose MFMAs run next
    u32x4 xn[MT][2];                    // raw operands of the round after it
    uint32_t wn[NJ], sn[NJ];
    auto reads = [&](auto sc, int q) {
        const uint32_t xl = lds_addr(xstage(sc)), wl = lds_addr(wstage(sc)), sl = lds_addr(slab);
#pragma unroll
        for (int i = 0; i < MT; ++i) {   // row 32 i + r, so row % XCH = r
            xn[i][0] = ds_read16(xl + 16 * ((32 * i + r) * XCH + ((2 * c) ^ r)));
            xn[i][1] = ds_read16(xl + 16 * ((32 * i + r) * XCH + ((2 * c + 1) ^ r)));
        }
        const int gi = (min(q, nr - 1) * RK + 8 * c) >> glog2;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            wn[j] = ds_read4(wl + 4 * wpos(32 * j + r, c));
            sn[j] = ds_read4(sl + 4 * spos(gi, 32 * j + r));
        }
    };
    auto settle = [&]() {
        static_assert(NJ == 4 && (MT == 1 || MT == 2) && XCH == 32, "operands of the wait, swizzle");
        if constexpr (MT == 1)
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(xn[0][0]), "+v"(xn[0][1]), "+v"(wn[0]), "+v"(wn[1]),
                         "+v"(wn[2]), "+v"(wn[3]), "+v"(sn[0]), "+v"(sn[1]), "+v"(sn[2]), "+v"(sn[3]));
        else
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(xn[0][0]), "+v"(xn[0][1]), "+v"(xn[MT - 1][0]),
                         "+v"(xn[MT - 1][1]), "+v"(wn[0]), "+v"(wn[1]), "+v"(wn[2]), "+v"(wn[3]),
                         "+v"(sn[0]), "+v"(sn[1]), "+v"(sn[2]), "+v"(sn[3]));
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const f32x4 x0 = __builtin_bit_cast(f32x4, xn[i][0]), x1 = __builtin_bit_cast(f32x4, xn[i][1]);
            a[i] = u32x4{clamp_f16x2(x0[0], x0[1]), clamp_f16x2(x0[2], x0[3]),
                         clamp_f16x2(x1[0], x1[1]), clamp_f16x2(x1[2], x1[3])};
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            b[j] = dequant_word_f16(wn[j], as_f16x2(__builtin_amdgcn_perm(sn[j], sn[j], 0x01000100u)),
                                    as_f16x2(__builtin_amdgcn_perm(sn[j], sn[j], 0x03020302u)));
    };
    // Every wave's copies of the next round to read have landed (NS - 2 later
    // rounds' may be in flight).
    auto ready = [&]() {
        __builtin_amdgcn_s_waitcnt(vmcnt_only((NS - 2) * CPR));
        RING_LDS_BARRIER();
    };
    // Round q: round q + 1's stage is waited for, the stage round q read is
    // refilled with round q + NS, round q + 1's operands are read, round q's
    // MFMAs run while they return.  A last round's copies and reads repeat it.
    auto round = [&](auto sc, int q) {
        constexpr int S = decltype(sc)::value % NS;
        ready();
        issue(std::integral_constant<int, S>{}, q + NS);
        reads(std::integral_constant<int, (S + 1) % NS>{}, q + 1);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = mfma32_f16(a[i], b[j], acc[i][j]);
        settle();
    };
    ready();
    reads(std::integral_constant<int, 0>{}, 0);
    settle();
    issue(std::integral_constant<int, NS - 1>{}, NS - 1);
    int q = 0;
    for (; q + NS - 1 < nr; q += NS)
        static_for<NS>([&](auto sc) { round(sc, q + decltype(sc)::value); });
    static_for<NS - 1>([&](auto sc) {
        if (q + decltype(sc)::value < nr) round(sc, q + decltype(sc)::value);
    });

    // ---- the K-groups' sums, two tiles of a row strip at a time (all eight
    // waves' partial tiles, 64 KB, in the X ring) ----
    // D[m][col] of a 32 x 32 tile is element 4 (m / 8) + m % 4 of lane
    // col + 32 ((m / 4) % 2).  Every thread sums 4 columns of one row over the
    // 8 waves, in wave order.
    constexpr int SPS = XS * 16 / 4096;   // partial tiles an X stage holds
    static_assert(NS * SPS >= 2 * NWV, "the ring holds two tiles of every wave");
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    auto buf = [&](int w, int d) -> float* {   // wave w's tile d of the pass
        const int slot = 2 * w + d, st = slot / SPS;
        u32x4* const x = st == 0 ? xs0 : st == 1 ? xs1 : st == 2 ? xs2 : xs3;
        return reinterpret_cast<float*>(x) + (slot % SPS) * 1024;
    };
    const int ml = tid >> 4, cq = tid & 15;
    const int l0 = 32 * ((ml >> 2) & 1), v = 4 * (ml >> 3) + (ml & 3);
    const int d0 = cq >> 3, c0 = 4 * (cq & 7);
#pragma unroll
    for (int t = 0; t < MT * NJ; t += 2) {
        const int i = t / NJ, j = t % NJ;
        RING_LDS_BARRIER();
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            float* const mine = buf(wave, d);
#pragma unroll
            for (int e = 0; e < 16; ++e) mine[e * 64 + lane] = acc[i][j + d][e];
        }
        RING_LDS_BARRIER();
        const int m = m0 + 32 * i + ml;
        if (m >= p.M) continue;
        float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < NWV; ++w) {
            const f32x4 g = *reinterpret_cast<const f32x4*>(buf(w, d0) + v * 64 + l0 + c0);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] += g[e];
        }
        epi_storev<4>(p, (size_t)m * p.N, n0 + 32 * (j + d0) + c0, x);
    }
}

}  // namespace

// The tile height (32-row tiles per block) for p: the lower one that covers it
// in one round of blocks (a second round repeats the whole per-block time),
// 0 where neither does.
static int strip_height(const GemmParams& p) {
    const long nb = ((long)p.N + SBN - 1) / SBN;
    for (int mt : {1, 2})
        if (((long)p.M + 32 * mt - 1) / (32 * mt) * nb <= kCUs) return mt;
    return 0;
}

// Where the kernel is the faster one (us, against the GEMM's fp32 path): at K
// = 2048 and N = 128, M = 33 / 1000 / 6144 / 12000 14.3 / 15.3 / 16.5 / 27.7
// against 17.0 / 20.3 / 25.2 / 43.4; N = 256, M = 6144 21.1 against 29.6; K =
// 128, N = 128, M = 1000 7.7 against 10.0.  Two rounds lose (K = 128, N = 512,
// M = 9000 24.4 against 13.9; K = 2048, N = 512, M = 9000 62.0 / 60.7).  A
// longer K wants more rows, since the GEMM splits K and this kernel does not:
// at K = 4096, N = 128, M = 300 / 2000 / 6144 23.0 / 23.4 / 26.9 against 18.8 /
// 23.0 / 38.4; N = 512, M = 300 / 1000 23.4 / 23.5 against 22.6 / 29.4.
int strip_rows(const GemmParams& p) {
    if (!p.a_f32 || p.w1 != nullptr || (p.epilogue != kEpiNone && p.epilogue != kEpiGeluTanh)) return 0;
    if (p.M < 1 || p.N < 1 || p.N > 4 * SBN || p.K % RK != 0 || p.groups > SLAB_G) return 0;
    if (p.K > 4096 || (p.K > 2048 && (long)p.M * p.N < 1L << 18)) return 0;
    return (reinterpret_cast<uintptr_t>(p.a) & 15) == 0 ? 32 * strip_height(p) : 0;
}

hipError_t launch_strip(GemmParams p, hipStream_t st) {
    const int mt = strip_height(p);
    p.tiles_m = (p.M + 32 * mt - 1) / (32 * mt);
    p.tiles_n = (p.N + SBN - 1) / SBN;
    const dim3 grid((p.tiles_m * p.tiles_n + 7) / 8 * 8);
    if (mt == 1)
        hipLaunchKernelGGL(q4_strip_kernel<1>, grid, dim3(ST), 0, st, p);
    else
        hipLaunchKernelGGL(q4_strip_kernel<2>, grid, dim3(ST), 0, st, p);
    return hipGetLastError();
}

}  // namespace sltx
