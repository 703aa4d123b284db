// q4_gemm_kernel.hpp -- 4-bit dequant GEMM (prefill / DiT, M > 1) on CDNA4 MFMA.
//
// Y[M,N] = A[M,K] . dequant(W)[N,K]^T, fp32 accumulate, where
// dequant(W)[n,k] = s[n,k/g]*q[n,k] + b[n,k/g].  This is the computation
// swift-ltx routes through matmulQ4Fast / matmulQ4FastF32 (Ops.swift:312-381),
// whose quantized-B GEMM kernel lives in an external package.  The SILU_MUL
// epilogue fuses linear(gate), linear(up) and siluMul
// (LlamaModel.swift:275-277); the bias + GELU-tanh epilogue covers
// DiTLinear.applyF32in + geluApproximateF32 (DiTModel.swift:102-125, :953).
//
// Block: 512 threads = 8 waves, two per SIMD.  The block tile is BM x 256 x 64
// (BM = 64*WM activation rows, 256 weight rows); wave w owns weight rows
// 32w..32w+31 and all BM activation rows, i.e. BM/32 tiles of
// v_mfma_f32_32x32x16_{f16,bf16} along M.  No weight row is dequantized
// twice, and each dequantized B fragment feeds BM/32 MFMAs.  Two waves per
// SIMD let one wave's dequantization and LDS reads issue while the other's
// MFMAs occupy the matrix core (an MFMA blocks its own wave's issue for about
// half of its 32 cycles).
//  * The B operand never passes through LDS as fp16.  In a 32x32x16 MFMA lane
//    l supplies 8 consecutive k of column l%32.  Inside each 64-wide k-tile, k
//    is permuted so that k-step s of lane half h covers 8-nibble word 4h+s of
//    the row: over a k-tile a lane reads one aligned 16-byte piece of its row,
//    and each k-step's B fragment is exactly one packed word, dequantized in
//    registers just before use (v_perm_b32 byte pairing, mantissa insertion,
//    one v_pk_fma_f16 q*s+b per pair).  The A fragments follow the same
//    permutation by reading 16-byte column 4h+s of the A tile.
//  * Packed W (256 rows x 64 B per pair of k-tiles) and the per-group
//    (scale, bias) pairs are staged through LDS with coalesced loads (four
//    lanes per 64-byte row segment), so no lane gathers 16 bytes per row.
//  * A (BM x 64 fp16/bf16 per k-tile) is copied global -> LDS directly
//    (global_load_lds_dwordx4) into a 4-stage ring, three k-tiles ahead.
//  * LDS rows are 128 bytes with an XOR swizzle of the 16-byte columns (swz):
//    the A fragment reads (16 consecutive rows, one logical column) and the
//    copies are free of bank conflicts.
//  * SILU: a wave's 32 weight rows are the 16 gate and the 16 up rows of the
//    same 16 output columns, so silu(gate) * up is formed in the lane that
//    holds both (register epilogue below).
//  * One barrier per k-tile.  Everything the next k-tile's first k-step needs
//    (its A fragments, its packed words and scale/bias) is already visible
//    before that barrier, so it is read during the last k-step of the current
//    k-tile and the MFMA stream does not drain at k-tile boundaries.
//  * Tile order is XCD-aware: the 8 XCDs receive workgroups round-robin, so
//    consecutive logical tiles (M fastest) are mapped to one XCD and the
//    M-blocks sharing a weight column block share that XCD's L2.
//  * More tiles than CUs (the lm_head and DiT up shapes): one persistent
//    block per CU walks a tile list, the copy ring running on across tiles.
//  * Outputs are stored from registers (SiLU pairs, persistent launches) or
//    staged through LDS into whole row segments (single-round launches of one
//    weight set); see the epilogue.
//  * Shapes with too few output tiles to fill 256 CUs split K; partial sums
//    go to an fp32 workspace and a second kernel adds them in split order.
#pragma once

#include <type_traits>

#include "q4_common.hpp"
#include "q4_dequant.hpp"
#include "q4_epilogue.hpp"
#include "q4_launch.hpp"

namespace sltx {

constexpr int BN = 256, BK = 64;
constexpr int NW = 8;                  // waves per block (two per SIMD)
constexpr int kThreads = 64 * NW;
constexpr int NT = BN / 32 / NW;       // 32-row weight tiles (MFMA N-tiles) per wave
constexpr int NSA = 4;     // A stages in LDS
constexpr int GPMAX = 4;   // scale/bias groups per row per 128 k (group size 32)

template <bool BF16>
__device__ __forceinline__ f32x16 mfma32(const u32x4 a, const u32x4 b, f32x16 c) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding:
// vmcnt bits [3:0] and [15:14], expcnt [6:4] = 7, lgkmcnt [11:8] = 15).
#define SLTX_WAIT_VMCNT(n) \
    __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Workgroup barrier for LDS hand-offs only.  __syncthreads() adds a
// workgroup release fence, which on gfx950 waits for every outstanding
// vector-memory op (vmcnt(0)), including the direct-to-LDS copies issued for
// k-tiles still three steps ahead.  Here each wave waits for its own LDS ops
// (lgkmcnt(0)); the copies a barrier must cover are waited for explicitly
// with SLTX_WAIT_VMCNT before it.  The memory clobber keeps the compiler from
// moving memory accesses across the barrier.
#define SLTX_LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

// Scale and bias of one (row, group), packed as fp16 bits scale | bias << 16.
struct SB {
    uint32_t v[NT];
};

// GEN = false: K % 128 == 0 and group size 32 << GS (GS = 2: K % 256 == 0);
// every load is a direct-to-LDS copy with a fixed count per k-tile and exact
// wait counts.  GEN = true: any supported shape (K % 32 == 0, group
// 32/64/128): scale/bias staged through registers, clamped tails, zero-filled
// A past K, full waits.
// KG = 2: tiles of 128 weight rows, for launches whose 256-row tiles are too
// few.  Four waves share the rows, and the two halves of the block each take
// two of a k-tile's four k-steps: every packed word is still dequantized once
// and feeds BM/32 MFMAs, and the halves' sums meet in LDS after the loop.
// Half the work between barriers makes a k-tile 0.55 us, not half of 0.95: it
// pays only where it saves K splits or fills idle CUs (figures at the plan).
// Measured and not kept: a ring reaching five k-tiles ahead (the same time: it
// does not wait for copies), and waves of 64 weight rows x half of the
// activation rows, which halve the LDS reads but dequantize every word twice
// (M = 750, N = 5120, K = 3072: 36 us against 33.7).
// A32: fp32 activations (the generic path only), each cast to fp16 as
// half(clamp(x, -65504, 65504)) -- cast_f32_to_f16, Kernels.swift:816-822,
// which DiTLinear.applyF32in runs before matmulQ4FastF32
// (DiTModel.swift:104-110) -- while it is staged: a k-tile's A is loaded into
// registers three k-tiles ahead, then cast and written to its LDS stage at
// the end of the k-tile that loaded it.
// PERSIST: the fast path over more output tiles than one round of blocks.
// Each block walks a fixed list of tiles (see the tile selection below);
// the copy ring runs on across tile boundaries -- the last three k-tiles of
// a tile issue the next tile's first A tiles and packed-W / scale-bias
// super-stages -- and the register epilogue of one tile runs while those
// copies are in flight, so neither the next tile's first memory latency nor
// its stores stall the MFMA stream for long.
// GS: the fast path's scale / bias staging.  Group 32 (GS = 0) has two scale
// dwords and two bias dwords per row and super-stage, group 64 one of each;
// group 128 has half of one, so its super-stages copy the dword of an even /
// odd pair of groups and read the half of their own.  On the generic kernel,
// which waits for every copy at the end of each k-tile, groups 32 and 128 ran
// at two thirds of group 64's rate: a 2048-8192-2048 feed-forward at M = 1537
// and group 128 took 200 us, 159 here; a Llama layer at M = 96 and group 32
// 97.4, 91.4 here.
template <int WM, bool BF16, bool SILU, bool GEN, bool SPLIT, bool A32 = false, bool PERSIST = false,
          int GS = 1, int KG = 1>
__global__ __launch_bounds__(kThreads, 1) void q4_gemm_kernel(GemmParams p) {
    static_assert(!A32 || (GEN && !BF16 && !SILU), "fp32 activations: the generic fp16 path");
    static_assert(!PERSIST || (!GEN && !SPLIT && !A32), "persistent tiles: the fast unsplit path");
    static_assert(KG == 1 || (KG == 2 && !GEN && !PERSIST && WM % 2 == 0), "k-step halves: the fast single-round path");
    constexpr int BM = 64 * WM;
    constexpr int TM = BM / 32;                // MFMA tiles along M per wave
    constexpr int A_STAGE = BM * BK / 8;       // 16-byte slots per A stage
    constexpr int NA = A_STAGE / kThreads;     // A copies per thread per k-tile
    constexpr int BNB = BN / KG, NWN = NW / KG;    // weight rows per block, waves along them
    constexpr int KSN = BK / 16 / KG;              // k-steps per wave and k-tile
    constexpr int WP_STAGE = BNB * 4;          // packed W of two k-tiles: 64 B per row
    constexpr int NWP = WP_STAGE / kThreads;   // packed-W copies per thread per super-stage
    constexpr int NPAIR = BNB * GPMAX / kThreads;   // GEN: (row, group) pairs per thread per super-stage
    constexpr int SBW = GS == 0 ? 4 : 2;           // fast path: scale/bias dwords per row per super-stage
    // and copies of them per thread (128 rows x 2 dwords: waves 4-7 repeat
    // the copies of waves 0-3, same bytes and slots)
    constexpr int NSB = (BNB * SBW + kThreads - 1) / kThreads;
    // Each stage is its own array: the compiler then knows that reads of one
    // stage do not alias a direct-to-LDS copy in flight into another, and
    // does not wait for that copy (stage indices are compile-time below).
    __shared__ u32x4 lds_a0[A_STAGE], lds_a1[A_STAGE], lds_a2[A_STAGE], lds_a3[A_STAGE];
    __shared__ u32x4 lds_wp0[WP_STAGE], lds_wp1[WP_STAGE];   // [row][piece ^ ((row >> 2) & 3)]
    // Scale/bias.  Fast path: per super-stage and row [scales, biases] dwords
    // of two groups (GS = 0: [k-tile][scales, biases]), copied direct to LDS.
    // Generic path: [row * GP + group] = scale | bias << 16, staged through
    // registers.
    __shared__ uint32_t lds_sb0[GEN ? BNB * GPMAX : BNB * SBW], lds_sb1[GEN ? BNB * GPMAX : BNB * SBW];
    static_assert(NSA == 4, "stage arrays");
    // A stage of k-tile t is t % 4, packed-W stage of super-stage ss is ss % 2.
    auto a_stage = [&](auto sc) -> u32x4* {
        constexpr int S = decltype(sc)::value & 3;
        if constexpr (S == 0) return lds_a0;
        else if constexpr (S == 1) return lds_a1;
        else if constexpr (S == 2) return lds_a2;
        else return lds_a3;
    };
    auto wp_stage = [&](auto sc) -> u32x4* {
        if constexpr ((decltype(sc)::value & 1) == 0) return lds_wp0;
        else return lds_wp1;
    };
    auto sb_stage = [&](auto sc) -> uint32_t* {
        if constexpr ((decltype(sc)::value & 1) == 0) return lds_sb0;
        else return lds_sb1;
    };

    // ---- tile selection (XCD-aware) ----
    // The 8 XCDs receive workgroups round-robin (block b on XCD b % 8).  One
    // tile per block: consecutive logical tiles (M fastest) go to one XCD.
    // PERSIST (grid a multiple of 8): XCD x owns logical tiles [x T8,
    // min((x + 1) T8, T)), T8 = ceil(T / 8), and its i-th block takes tiles
    // x T8 + i, + G / 8, + 2 G / 8, ... (G = grid): the blocks of one XCD
    // work on neighbouring tiles, which share weight columns, at any time.
    const int ntiles = p.tiles_m * p.tiles_n;
    int logical = blockIdx.x;
    int pstride = 0, pend = 0;
    if constexpr (PERSIST) {
        const int per_x = (ntiles + 7) >> 3;
        logical = (blockIdx.x & 7) * per_x + (blockIdx.x >> 3);
        pend = min(((int)(blockIdx.x & 7) + 1) * per_x, ntiles);
        pstride = gridDim.x >> 3;
        if (logical >= pend) return;
    } else {
        if ((gridDim.x & 7) == 0) {
            const int per_xcd = gridDim.x >> 3;
            logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        }
        if (logical >= ntiles * (SPLIT ? p.splits : 1)) return;
    }
    const int split = SPLIT ? logical / ntiles : 0;
    const int tile = SPLIT ? logical % ntiles : logical;
    // K range of this block: k-tiles [kb, kb + nk); Kl = its extent in k.
    const int nk_all = (p.K + BK - 1) / BK;
    const int kb = SPLIT ? split * p.split_tiles : 0;
    const int nk = SPLIT ? min(p.split_tiles, nk_all - kb) : nk_all;
    const int Kl = min(p.K - kb * BK, nk * BK);
    const int nss = (nk + 1) / 2;   // super-stages (pairs of k-tiles)
    // SILU: a tile covers 128 output columns, as 128 gate rows + 128 up rows.
    // m0 / n0: the tile the copies are reading (PERSIST: the next one from
    // its first prefetch on); em0 / en0: the tile the accumulators hold.
    int m0 = (tile % p.tiles_m) * BM;
    int n0 = (tile / p.tiles_m) * (SILU ? BNB / 2 : BNB);
    int em0 = m0, en0 = n0;
    bool has_next = PERSIST && logical + pstride < pend;

    const int tid = threadIdx.x;
    // KG = 2: wave wv owns weight rows 32 (wv % 4) .. and k-steps 2 (wv / 4) ..
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = KG == 1 ? wv : wv % NWN, kg = KG == 1 ? 0 : wv / NWN;
    const int lrow = lane & 31, h = lane >> 5;
    const int GP = 4 >> p.gshift;   // scale/bias groups per 128 k (g = 32, 64, 128)

    // Virtual W row -> matrix row (and which matrix, for SILU).  Wave wn owns
    // virtual rows 32wn..32wn+31 (one 32-row MFMA tile); with SILU its rows
    // 0-15 are the gate rows and 16-31 the up rows of the same 16 output
    // columns, n0 + 16wn .. +15, so that both halves of each output land in
    // one lane (see the epilogue).  Rows past N are clamped to the last row:
    // computed, never stored.
    auto wrow = [&](int v, const uint32_t*& W, const uint16_t*& S, const uint16_t*& B) {
        int n;
        if (SILU) {
            const int tn = (v >> 4) & 1;
            n = n0 + (v >> 5) * 16 + (v & 15);
            W = tn ? p.w1 : p.w0;
            S = tn ? p.s1 : p.s0;
            B = tn ? p.b1 : p.b0;
        } else {
            n = n0 + v;
            W = p.w0;
            S = p.s0;
            B = p.b0;
        }
        return n < p.N ? n : p.N - 1;
    };

    // ---- A: direct global -> LDS (global_load_lds_dwordx4) ----
    // Copy i of wave wn fills slots (wn + 4 i) * 64 .. +63, lane l landing in
    // slot +l.  Slot s is physical column s % 8 of row s / 8, i.e. logical
    // column (s % 8) ^ xor(row): the swizzle is applied on the global side.
    // Rows past M are clamped to M-1.
    // A source is a base that is the same for the whole wave (SGPRs: the tile
    // and the k offset) plus a byte offset per lane that no k-tile changes, so
    // a copy needs no address arithmetic in vector registers (fast path: 32
    // bits, K <= 2^22 keeps a tile's rows within them; 24 VGPRs fewer at 192
    // rows, and the DiT up, lm_head and M = 333 gate/up launches 1% faster).
    using off_t = std::conditional_t<GEN, size_t, uint32_t>;
    constexpr int AB = A32 ? 4 : 2;   // bytes of an activation
    const char* a_base;
    off_t a_off[NA];
    int a_col8[NA];
    auto set_a_src = [&]() {
        a_base = reinterpret_cast<const char*>(p.a) + ((size_t)m0 * p.K + kb * BK) * AB;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int slot = (wv + NW * i) * 64 + lane;
            const int row = slot >> 3;
            const int c16 = (slot & 7) ^ (row & 7) ^ ((row >> 3) & 1);
            a_col8[i] = c16 * 8;
            a_off[i] = ((off_t)(m0 + row < p.M ? row : p.M - 1 - m0) * (off_t)p.K + c16 * 8) * AB;
        }
    };
    set_a_src();

    // ---- packed W: direct global -> LDS, two k-tiles (64 B per row) ----
    // Four lanes cover a row's 64 bytes, so each wave-wide copy reads 16 rows
    // of 64 contiguous bytes.  Slot s is row s / 4, physical piece s % 4 =
    // logical piece ^ ((row >> 2) & 3) (conflict-free reads below).
    // SILU: copy i covers virtual rows 16 (wv + NW i) .. +15, so all of a
    // wave's copies are gate rows (even wv) or up rows (odd wv): one base.
    const char* wp_base;
    off_t wp_off[NWP];
    int wp_piece[NWP];
    auto set_wp_src = [&]() {
        wp_base = reinterpret_cast<const char*>(SILU && (wv & 1) ? p.w1 : p.w0) +
                  ((size_t)n0 * p.K + kb * BK) / 2;
#pragma unroll
        for (int i = 0; i < NWP; ++i) {
            const int slot = (wv + NW * i) * 64 + lane;
            const int row = slot >> 2;
            const int piece = (slot & 3) ^ ((row >> 2) & 3);
            const uint32_t* W;
            const uint16_t *S, *B;
            const int n = wrow(row, W, S, B) - n0;
            wp_piece[i] = piece;
            wp_off[i] = (off_t)n * (off_t)(p.K / 2) + piece * 16;
        }
    };
    set_wp_src();

    // ---- scale / bias ----
    const int g_base = (2 * kb) >> p.gshift;
    // Fast path: copy i of wave wn fills dwords (wn + NW i) * 64 + lane of the
    // stage: dword slot % SBW of row slot / SBW, scales (even) or biases
    // (odd).  GS = 1: the dword holding groups 2 ss and 2 ss + 1; GS = 0:
    // dword 2 tl (+ 1) the two groups of k-tile tl; GS = 2: the dword of
    // groups g & ~1 and g | 1, g = g_base + ss.  All are 4-byte aligned: a
    // row's groups are even in number (K % 128 == 0, GS = 2: K % 256), and so
    // is g_base for GS < 2 (splits cover whole super-stages).
    auto sb_slot0 = [&](int i) { return (wv + NW * i) * 64 % (BNB * SBW); };
    const uint32_t* sbd_src[NSB];
    auto set_sbd_src = [&]() {
#pragma unroll
        for (int i = 0; i < NSB; ++i) {
            const int slot = sb_slot0(i) + lane;
            const uint32_t* W;
            const uint16_t *S, *B;
            const int n = wrow(slot / SBW, W, S, B);
            const int g0 = GS == 2 ? 0 : g_base + (GS == 0 ? slot & 2 : 0);
            sbd_src[i] = reinterpret_cast<const uint32_t*>((slot & 1 ? B : S) + (size_t)n * p.groups + g0);
        }
    };
    set_sbd_src();
    // Generic path: pair v = tid + 256 u is (row v / GP, group v % GP).
    // Consecutive threads read consecutive groups of a row.  Values land in
    // registers and are written to LDS one k-tile later; pairs past the tile
    // (v >= 256 GP) read row 0 and land in unused LDS slots.
    const uint16_t* s_src[NPAIR];
    const uint16_t* b_src[NPAIR];
    int sb_g[NPAIR];
#pragma unroll
    for (int u = 0; u < NPAIR; ++u) {
        const int v = tid + kThreads * u;
        const int row = v / GP, g = v % GP;
        const uint32_t* W;
        const uint16_t *S, *B;
        const int n = wrow(row < BNB ? row : 0, W, S, B);
        s_src[u] = S + (size_t)n * p.groups + g_base + g;
        b_src[u] = B + (size_t)n * p.groups + g_base + g;
        sb_g[u] = g;
    }

    // load_a / zero_a_tail / fetch_w take the tile index t with its value mod
    // 4 as a compile-time constant TP; load_wp / store_sb take the super-stage
    // with its parity.
    // A32: this thread's eight fp32 values of each of its NA slots.
    f32x4 a32[A32 ? NA : 1][2];
    auto load_a = [&](auto tp, int t) {   // NA (A32: 2 NA) vector-memory ops (tiles past the end re-read the last)
        const int k0 = min(t, nk - 1) * BK;
        u32x4* stage = a_stage(tp);
        const char* base = GEN ? a_base : a_base + (size_t)k0 * AB;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            off_t off = a_off[i];
            if constexpr (GEN) off += (k0 + a_col8[i] >= Kl ? Kl - 8 - a_col8[i] : k0) * AB;
            if constexpr (A32) {
                const f32x4* src = reinterpret_cast<const f32x4*>(base + off);
                a32[i][0] = src[0];
                a32[i][1] = src[1];
            } else {
                __builtin_amdgcn_global_load_lds((const void*)(base + off),
                                                 (lds_ptr_t)(stage + (wv + NW * i) * 64), 16, 0, 0);
            }
        }
    };
    // A32: tile t's slots from the registers load_a filled, cast with the
    // clamp, into stage tp (zeros past K).
    auto store_a32 = [&](auto tp, int t) {
        if constexpr (A32) {
            const int k0 = t * BK;
            u32x4* stage = a_stage(tp);
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                u32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float lo = a32[i][e >> 1][2 * (e & 1)], hi = a32[i][e >> 1][2 * (e & 1) + 1];
                    o[e] = (uint32_t)f2h(fminf(fmaxf(lo, -65504.0f), 65504.0f)) |
                           ((uint32_t)f2h(fminf(fmaxf(hi, -65504.0f), 65504.0f)) << 16);
                }
                if (k0 + a_col8[i] >= Kl) o = u32x4{0u, 0u, 0u, 0u};
                stage[(wv + NW * i) * 64 + lane] = o;
            }
        }
    };
    auto zero_a_tail = [&](auto tp, int t) {   // GEN: after the copy of tile t landed
        const int k0 = t * BK;
        if (t >= nk || k0 + BK <= Kl) return;
        u32x4* stage = a_stage(tp);
        const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < NA; ++i)
            if (k0 + a_col8[i] >= Kl) stage[(wv + NW * i) * 64 + lane] = z;
    };
    auto load_wp = [&](auto sp, int ss) {   // NWP vector-memory ops
        const int sc = min(ss, nss - 1);
        u32x4* stage = wp_stage(sp);
        const char* base = GEN ? wp_base : wp_base + (size_t)sc * 64;   // 64 bytes per super-stage
#pragma unroll
        for (int i = 0; i < NWP; ++i) {
            off_t off = wp_off[i];
            if constexpr (GEN)
                off += sc * 128 + wp_piece[i] * 32 >= Kl ? Kl / 2 - 16 - wp_piece[i] * 16 : sc * 64;
            __builtin_amdgcn_global_load_lds((const void*)(base + off),
                                             (lds_ptr_t)(stage + (wv + NW * i) * 64), 16, 0, 0);
        }
    };
    auto load_sb_dma = [&](auto sp, int ss) {   // fast path: NSB vector-memory ops
        const int sc = min(ss, nss - 1);
        const int off = GS == 0 ? 2 * sc : GS == 1 ? sc : (g_base + sc) >> 1;   // dwords
        uint32_t* stage = sb_stage(sp);
#pragma unroll
        for (int i = 0; i < NSB; ++i)
            __builtin_amdgcn_global_load_lds((const void*)(sbd_src[i] + off),
                                             (lds_ptr_t)(stage + sb_slot0(i)), 4, 0, 0);
    };
    uint32_t s_reg[NPAIR], b_reg[NPAIR];
    auto load_sb = [&](int ss) {   // generic path: 2 NPAIR vector-memory ops
        const int sc = min(ss, nss - 1);
        const int groups_l = p.groups - g_base;
#pragma unroll
        for (int u = 0; u < NPAIR; ++u) {
            int g = sc * GP;
            if (GEN && g + sb_g[u] >= groups_l) g = groups_l - 1 - sb_g[u];
            s_reg[u] = s_src[u][g];
            b_reg[u] = b_src[u][g];
        }
    };
    auto store_sb = [&](auto sp) {
        uint32_t* stage = sb_stage(sp);
#pragma unroll
        for (int u = 0; u < NPAIR; ++u)
            stage[tid + kThreads * u] = (s_reg[u] & 0xFFFFu) | (b_reg[u] << 16);
    };

    // Packed words (16 bytes: this lane's k-steps; KG = 2: its half) and scale|bias of
    // tile t for both of the wave's 32-row MFMA tiles.
    typedef uint32_t wk_t __attribute__((ext_vector_type(KSN)));
    auto fetch_w = [&](auto tp, int t, wk_t (&wk)[NT], SB& sb) {
        constexpr int TP = decltype(tp)::value & 3;
        constexpr int TL = TP & 1, SP = (TP >> 1) & 1;   // tile within / parity of super-stage
        const u32x4* ws = wp_stage(std::integral_constant<int, SP>{});
        const int piece = TL * 2 + h;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int vr = wn * 32 * NT + j * 32 + lrow;
            wk[j] = reinterpret_cast<const wk_t*>(ws + vr * 4 + (piece ^ ((vr >> 2) & 3)))[kg];
            uint32_t v;
            if constexpr (GEN) {
                v = sb_stage(std::integral_constant<int, SP>{})[vr * GP + (piece >> p.gshift)];
            } else {
                // The half of the scale and bias dwords: GS = 1, group TL of
                // the super-stage; GS = 0, the group of this lane's 32 k of
                // k-tile TL; GS = 2, the super-stage's own group of the pair.
                const uint2* sd = reinterpret_cast<const uint2*>(sb_stage(std::integral_constant<int, SP>{}));
                const uint2 d = GS == 0 ? sd[vr * 2 + TL] : sd[vr];
                const int half = GS == 0 ? h : GS == 1 ? TL : (SP ^ g_base) & 1;
                v = __builtin_amdgcn_perm(d.y, d.x, half ? 0x07060302u : 0x05040100u);
            }
            if (GEN && t * BK + h * 32 >= Kl) v = 0;   // k past K: w = 0
            sb.v[j] = v;
        }
    };
    // B fragment of k-step ks for MFMA tile j.
    auto dequant = [&](const wk_t (&wk)[NT], const SB& sb, int ks, u32x4 (&dst)[NT]) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const uint32_t v = sb.v[j];
            if constexpr (BF16) {
                dst[j] = dequant_word_bf16(wk[j][ks], p.nib_mask, h2f((uint16_t)(v & 0xFFFFu)),
                                           h2f((uint16_t)(v >> 16)));
            } else {
                const f16x2 s2 = as_f16x2(__builtin_amdgcn_perm(v, v, 0x01000100u));
                const f16x2 b2 = as_f16x2(__builtin_amdgcn_perm(v, v, 0x03020302u));
                dst[j] = dequant_word_f16(wk[j][ks], s2, b2);
            }
        }
    };
    auto read_a = [&](const u32x4* sa, int ks, u32x4 (&dst)[TM]) {
        const int c16 = 4 * h + KSN * kg + ks;
#pragma unroll
        for (int i = 0; i < TM; ++i) dst[i] = sa[swz(i * 32 + lrow, c16)];
    };

    // TRANS: the packed-weight fragment is the MFMA's A operand, so the
    // accumulators hold D^T (weight rows along the lane's 16 values) -- the
    // layout the register epilogue stores from.  Otherwise (the LDS-staged
    // epilogue) the activation fragment is A, as measured 1.3% faster on the
    // bf16 DiT down loop (the dequantized fragment is then read as the B
    // operand).
    constexpr bool TRANS = PERSIST || SILU;
    f32x16 acc[TM][NT];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;

    // Prologue: A tiles 0..2 and packed W / scale-bias of super-stages 0 and
    // 1 in flight.  k-tile 0 needs A tiles 0 and 1 and super-stage 0 before
    // it starts; A tile 2 and super-stage 1 (issued last) may still land
    // during it (the wait at the end of k-tile 0 covers them).  Generic path:
    // scale/bias of super-stage 0 to LDS, super-stage 1's stay in registers
    // and are written at the end of k-tile 0.
    if constexpr (A32) {
        // one tile of A registers: tiles 0, 1, 2 one after another
        load_wp(I0{}, 0);
        load_wp(I1{}, 1);
        load_sb(0);
        load_a(I0{}, 0);
        SLTX_WAIT_VMCNT(0);
        store_sb(I0{});
        store_a32(I0{}, 0);
        load_sb(1);
        load_a(I1{}, 1);
        SLTX_WAIT_VMCNT(0);
        store_a32(I1{}, 1);
        load_a(I2{}, 2);
        SLTX_WAIT_VMCNT(0);
        store_a32(I2{}, 2);
    } else if constexpr (GEN) {
        load_a(I0{}, 0);
        load_a(I1{}, 1);
        load_a(I2{}, 2);
        load_wp(I0{}, 0);
        load_wp(I1{}, 1);
        load_sb(0);
        SLTX_WAIT_VMCNT(0);
        store_sb(I0{});
        load_sb(1);
        SLTX_WAIT_VMCNT(0);
        zero_a_tail(I0{}, 0);
        zero_a_tail(I1{}, 1);
        zero_a_tail(I2{}, 2);
    } else {
        load_a(I0{}, 0);
        load_a(I1{}, 1);
        load_wp(I0{}, 0);
        load_sb_dma(I0{}, 0);
        load_a(I2{}, 2);
        load_wp(I1{}, 1);
        load_sb_dma(I1{}, 1);
        SLTX_WAIT_VMCNT(NA + NWP + NSB);
    }
    SLTX_LDS_BARRIER();

    wk_t wk_c[NT], wk_n[NT];
    SB sb_c, sb_n;
    u32x4 af[2][TM], bq[2][NT];
    fetch_w(I0{}, 0, wk_c, sb_c);
    read_a(a_stage(I0{}), 0, af[0]);
    dequant(wk_c, sb_c, 0, bq[0]);

    // k-tile kt (TP = kt % 4, compile-time): MFMAs on A stage TP with B
    // dequantized from tile kt's packed words.  Issued during kt: A tile kt+3;
    // for odd kt = 2j+1 the packed W and scale/bias registers of super-stage
    // j+2 (the latter written to LDS at the end of k-tile kt+1).  The operands
    // of tile kt+1's first k-step are formed during the last k-step.  Each
    // tile is one branch-free block with a constant wait count.
    auto step = [&](auto tp, int kt) {
        constexpr int TP = decltype(tp)::value;
        constexpr bool ODD = TP & 1;
        using N1 = std::integral_constant<int, (TP + 1) & 3>;
        using N3 = std::integral_constant<int, (TP + 3) & 3>;
        int ta = kt + NSA - 1, tw = (kt + 3) >> 1;   // A tile and super-stage to copy
        if constexpr (PERSIST) {
            if (has_next) {
                // from k-tile nk - 3 on, the copies read the next tile
                if (kt == nk - (NSA - 1)) {
                    const int nt = logical + pstride;
                    m0 = (nt % p.tiles_m) * BM;
                    n0 = (nt / p.tiles_m) * (SILU ? BN / 2 : BN);
                    set_a_src();
                    set_wp_src();
                    set_sbd_src();
                }
                if (ta >= nk) ta -= nk;
                if (tw >= nss) tw -= nss;
            }
        }
        load_a(N3{}, ta);
        if constexpr (ODD) {
            // super-stage (kt+3)/2: parity ((TP+3) >> 1) & 1
            load_wp(std::integral_constant<int, ((TP + 3) >> 1) & 1>{}, tw);
            if constexpr (GEN) load_sb(tw);
            else load_sb_dma(std::integral_constant<int, ((TP + 3) >> 1) & 1>{}, tw);
        }
        const u32x4* sa = a_stage(tp);
        const u32x4* sa_n = a_stage(N1{});
        __builtin_amdgcn_sched_barrier(0);
        // Each k-step: this step's MFMAs (operands read / dequantized during
        // the previous step) with the next step's A fragment reads and B
        // dequantization interleaved.  The first MFMA goes before any new LDS
        // read: the compiler's wait for its operands then covers only reads
        // issued a full k-step earlier (it cannot count LDS reads separately
        // while direct-to-LDS copies are in flight, so every LDS wait it
        // emits waits for all of them).  The scheduling-group barriers fix
        // that order: 1 MFMA, half the step's reads, 1 MFMA, the other half,
        // then MFMAs with up to six VALU ops each, so the dequantization
        // finishes early in the step (measured 1-3% faster than one read per
        // MFMA with three VALU ops, and than all reads after the first MFMA;
        // the bf16 shapes and split down gain most).  Step 0
        // also reads tile kt+1's packed words and scale/bias (used from step 3
        // on).
#pragma unroll
        for (int ks = 0; ks < KSN; ++ks) {
            const int b = ks & 1;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = TRANS ? mfma32<BF16>(bq[b][j], af[b][i], acc[i][j])
                                      : mfma32<BF16>(af[b][i], bq[b][j], acc[i][j]);
            if (ks + 1 < KSN) {
                read_a(sa, ks + 1, af[b ^ 1]);
                dequant(wk_c, sb_c, ks + 1, bq[b ^ 1]);
            } else {
                read_a(sa_n, 0, af[b ^ 1]);
                dequant(wk_n, sb_n, 0, bq[b ^ 1]);
            }
            if (ks == 0) fetch_w(N1{}, kt + 1, wk_n, sb_n);
            constexpr int NR0 = TM + 2 * NT;   // LDS reads in step 0
            static_assert(NT * TM >= 2, "two MFMAs per step to spread the reads over");
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // MFMA
            if (ks == 0) __builtin_amdgcn_sched_group_barrier(0x100, (NR0 + 1) / 2, 0);   // DS reads
            else __builtin_amdgcn_sched_group_barrier(0x100, (TM + 1) / 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);       // VALU
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // MFMA
            if (ks == 0) __builtin_amdgcn_sched_group_barrier(0x100, NR0 / 2, 0);   // DS reads
            else __builtin_amdgcn_sched_group_barrier(0x100, TM / 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);       // VALU
#pragma unroll
            for (int q = 2; q < NT * TM; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);   // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // even kt: scale/bias of super-stage (kt+2)/2 (parity ((TP+2) >> 1) & 1)
        if constexpr (GEN && !ODD) store_sb(std::integral_constant<int, ((TP + 2) >> 1) & 1>{});
        // Before the barrier, A tile kt+2 and the packed W / scale-bias of
        // tile kt+2 must have landed (they are read during k-tile kt+1).
        // vmcnt retires in issue order.  Even kt issued only A tile kt+3;
        // odd kt issued A tile kt+3 and super-stage (kt+3)/2 after A tile
        // kt+2 (issued at kt-1, which issued nothing else).
        if constexpr (A32) {
            // tile kt+3 (loaded at the start of this k-tile) into its stage,
            // which k-tile kt-1 read before the last barrier
            SLTX_WAIT_VMCNT(0);
            store_a32(N3{}, kt + NSA - 1);
        } else if constexpr (GEN) {
            SLTX_WAIT_VMCNT(0);
            zero_a_tail(std::integral_constant<int, (TP + 2) & 3>{}, kt + 2);
        } else if constexpr (ODD) {
            SLTX_WAIT_VMCNT(NA + NWP + NSB);
        } else {
            SLTX_WAIT_VMCNT(NA);
        }
        SLTX_LDS_BARRIER();
#pragma unroll
        for (int j = 0; j < NT; ++j) wk_c[j] = wk_n[j];
        sb_c = sb_n;
    };

    // ---- KG = 2: the two K halves of each tile ----
    // Waves wv and wv + 4 hold partial sums of the same outputs.  Each gives
    // the other half of its tiles through the idle A stages (two waves a
    // stage) and keeps TM / 2 tiles, from tile kg TM / 2 on, in acc[0..].
    constexpr int TMO = TM / KG;
    auto add_k_halves = [&]() {
        static_assert(KG == 1 || 2 * TMO * 4096 <= A_STAGE * 16, "two waves' exchange fits an A stage");
        SLTX_WAIT_VMCNT(0);
        SLTX_LDS_BARRIER();
        auto buf = [&](int w) -> float* {
            u32x4* st = (w >> 1) == 0 ? lds_a0 : (w >> 1) == 1 ? lds_a1 : (w >> 1) == 2 ? lds_a2 : lds_a3;
            return reinterpret_cast<float*>(st) + (w & 1) * TMO * 1024 + lane;
        };
        float* const mine = buf(wv);
#pragma unroll
        for (int i = 0; i < TMO; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) mine[(i * 16 + v) * 64] = kg ? acc[i][0][v] : acc[TM - TMO + i][0][v];
        SLTX_LDS_BARRIER();
        const float* const other = buf(wv ^ NWN);
#pragma unroll
        for (int i = 0; i < TMO; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                acc[i][0][v] = (kg ? acc[TM - TMO + i][0][v] : acc[i][0][v]) + other[(i * 16 + v) * 64];
    };

    // ---- epilogue, from registers (TRANS) ----
    // The MFMAs compute D^T = W_tile . A_tile^T, so lane l holds, for activation row em0 + 32 i + l % 32,
    // the wave's weight rows 8 g + 4 h + r (r = 0..3, h = l / 32) in
    // acc[i][0][4 g + r]: four consecutive output columns per g.  One
    // v_permlane32_swap per value gives each lane eight consecutive columns
    // (groups g and g + 1 of lanes l and l + 32): lane l < 32 columns 0-7 of
    // the pair, lane l + 32 columns 8-15, stored as one 16-byte vector.  With
    // SILU, g = 0, 1 are gate rows and g + 2 the up rows of the same columns,
    // so silu(gate) * up is formed before the swap.  No LDS and no barrier:
    // a persistent block goes on to the next tile's k-tiles (copied during
    // the last three of this one) while the stores drain.
    static_assert(NT == 1, "one 32-row MFMA tile of W rows per wave");
    auto swap8 = [&](const float (&lo)[4], const float (&hi)[4], float (&o)[8]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, lo[r]),
                                                             __builtin_bit_cast(uint32_t, hi[r]),
                                                             false, false);
            o[r] = __builtin_bit_cast(float, (uint32_t)sw[0]);
            o[4 + r] = __builtin_bit_cast(float, (uint32_t)sw[1]);
        }
    };
    auto group = [&](const f32x16& t, int g, float (&o)[4]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = t[4 * g + r];
    };
    auto epilogue = [&]() {
        const bool vec = out_vec_ok(p);
        const int cw = en0 + (SILU ? 16 : 32) * wn + 8 * h;   // this lane's first column
#pragma unroll
        for (int i = 0; i < TMO; ++i) {
            const int m = em0 + (kg * TMO + i) * 32 + lrow;   // lanes l and l + 32 share a row
            float x[8];
            if constexpr (SPLIT) {
                // raw fp32 partial sums; the reduce kernel applies the epilogue
                const size_t nw = SILU ? 2 * (size_t)p.N : (size_t)p.N;
                float* wsr = p.ws + ((size_t)split * p.M + (m < p.M ? m : 0)) * nw;
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    float lo[4], hi[4];
                    group(acc[i][0], 2 * q, lo);
                    group(acc[i][0], 2 * q + 1, hi);
                    swap8(lo, hi, x);
                    // SILU: q = 1 is up, whose partials follow gate's
                    if (m < p.M) store_f32x8(SILU && q ? wsr + p.N : wsr, cw + (SILU ? 0 : 16 * q), p.N, x);
                }
            } else if constexpr (SILU) {
                const bool gelu = p.epilogue == kEpiGeluMul;
                float lo[4], hi[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    lo[r] = glu_f32(gelu, acc[i][0][r], acc[i][0][8 + r]);
                    hi[r] = glu_f32(gelu, acc[i][0][4 + r], acc[i][0][12 + r]);
                }
                swap8(lo, hi, x);
                if (m < p.M) store_out8(p, (size_t)m * p.N, cw, x, vec);
            } else {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    float lo[4], hi[4];
                    group(acc[i][0], 2 * q, lo);
                    group(acc[i][0], 2 * q + 1, hi);
                    swap8(lo, hi, x);
                    if (m < p.M) epi_store8(p, (size_t)m * p.N, cw + 16 * q, x, vec);
                }
            }
        }
    };

    // One launch of a single round, one weight set (no SiLU pair): each
    // 32-row accumulator tile (D, activation rows along the lane's 16 values,
    // row 8 (v / 4) + 4 h + v % 4, column l % 32) is staged through LDS (the
    // A stages, idle once the last copy into them has landed) as two fp32
    // [32][128] buffers, output columns 0-127 and 128-255, so that all 512
    // threads store whole 256-byte row segments: 16-byte pieces at 8 (t % 16)
    // of row t / 16.  Measured against the register epilogue at DiT down
    // (M = 6144, 25 MB of output at once): 2 us faster; the register stores
    // put 32 rows in each store instruction.
    auto staged_epilogue = [&]() {
        static_assert(32 * 128 * 4 <= A_STAGE * 16, "a 32 x 128 fp32 tile fits one A stage");
        SLTX_WAIT_VMCNT(0);
        SLTX_LDS_BARRIER();
        float* const eb0 = reinterpret_cast<float*>(lds_a0);
        float* const eb1 = reinterpret_cast<float*>(lds_a1);
        // KG = 2: the second buffer holds the other K half's tile (128 columns)
        float* const wdst = (wv >> 2) ? eb1 : eb0;
        const int wcol = (wn & 3) * 32 + lrow;
        const int er = tid >> 4, ec = (tid & 15) * 8;
        const bool vec = out_vec_ok(p);
#pragma unroll
        for (int i = 0; i < TMO; ++i) {
#pragma unroll
            for (int v = 0; v < 16; ++v) wdst[(8 * (v >> 2) + 4 * h + (v & 3)) * 128 + wcol] = acc[i][0][v];
            SLTX_LDS_BARRIER();
            const int m = em0 + i * 32 + er;
            // eb1's rows and columns
            const int m1 = KG == 1 ? m : m + TMO * 32, c1 = KG == 1 ? en0 + 128 + ec : en0 + ec;
            float x0[8], x1[8];
            const f32x4* r0 = reinterpret_cast<const f32x4*>(eb0 + er * 128 + ec);
            const f32x4* r1 = reinterpret_cast<const f32x4*>(eb1 + er * 128 + ec);
            const f32x4 a0 = r0[0], a1 = r0[1], b0 = r1[0], b1 = r1[1];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x0[e] = a0[e];
                x0[4 + e] = a1[e];
                x1[e] = b0[e];
                x1[4 + e] = b1[e];
            }
            if constexpr (SPLIT) {
                // raw fp32 partial sums; the reduce kernel applies the epilogue
                if (m < p.M) store_f32x8(p.ws + ((size_t)split * p.M + m) * (size_t)p.N, en0 + ec, p.N, x0);
                if (m1 < p.M) store_f32x8(p.ws + ((size_t)split * p.M + m1) * (size_t)p.N, c1, p.N, x1);
            } else {
                if (m < p.M) epi_store8(p, (size_t)m * p.N, en0 + ec, x0, vec);
                if (m1 < p.M) epi_store8(p, (size_t)m1 * p.N, c1, x1, vec);
            }
            SLTX_LDS_BARRIER();
        }
    };

    for (;;) {
        int kt = 0;
        for (; kt + 3 < nk; kt += 4) {
            step(I0{}, kt);
            step(I1{}, kt + 1);
            step(I2{}, kt + 2);
            step(I3{}, kt + 3);
        }
        if constexpr (!PERSIST) {   // PERSIST: nk % 4 == 0
            if (kt < nk) step(I0{}, kt);
            if (kt + 1 < nk) step(I1{}, kt + 1);
            if (kt + 2 < nk) step(I2{}, kt + 2);
        }
        if constexpr (KG == 2) add_k_halves();
        if constexpr (PERSIST || SILU) {
            // the block's last copies (clamped re-reads of the last k-tile)
            // land before it ends and its LDS is released; the stores need
            // no wait
            if (!has_next) SLTX_WAIT_VMCNT(0);
            epilogue();
        } else {
            static_assert(!TRANS, "the staged epilogue reads D, not D^T");
            staged_epilogue();
        }
        if (!has_next) break;
        // the next tile: its copies are in flight, its first k-step's operands
        // were formed during the last k-step
        logical += pstride;
        em0 = m0;
        en0 = n0;
        has_next = logical + pstride < pend;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][0][v] = 0.0f;
    }
}

}  // namespace sltx
