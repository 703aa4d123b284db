// q4_skinny.hip -- 4-bit dequant matmul for small M (1..32 activation rows:
// short prompts, the T5 encoder's S <= 128 layers, batched decode) on CDNA4
// MFMA, as a weight stream.
//
// Same product as q4_gemm_kernel.hpp, Y[M,N] = X[M,K] . dequant(W)[N,K]^T with fp32
// accumulation (matmulQ4Fast, Ops.swift:312-381).  At small M each weight
// byte feeds only M multiply-adds, so the kernel is bound by the weight
// stream, like the GEMV: the block tile of the large-M GEMM (128 or 192
// activation rows, LDS-staged weights) would pad M and re-stage weights for
// nothing.  Here:
//  * A block owns 16 * RT weight rows (of each weight set: gate and up for
//    the gated epilogues) and all K; its W waves split K into equal slices of
//    128 * STEPS.  In wave w, lane l covers row l % 16 of each 16-row tile
//    and, in each 128-wide k-step, the 32 k at offset 32 * (l / 16): one
//    16-byte load of packed words per step.  Two steps are loaded together
//    as 8 rows x 128 contiguous bytes per wave-wide load and swapped into
//    that layout with one DPP move per word.  Every load of a wave is issued
//    before the first MFMA, in the order of use.
//  * The block's scales and biases (one contiguous slab per array) are
//    copied to LDS with direct 16-byte global -> LDS loads, issued first.
//  * The wave's slice of X (all M rows, 16 per MFMA tile) stays in
//    registers for the whole kernel.  Every 16-byte load through the vector
//    memory path costs that path 16 cycles whatever its lanes hold, so
//    fragments loaded for all 16 rows (zeros past M) cost the CU more load
//    issue than its weights at small M.  Hence three ways (SkinnyX):
//    - M <= 8 (kXHalf), but for the shapes of skinny_plan's rule: the lanes of rows 8..15 load rows 0..7 of the next
//      fragment, so that one load fills two; a row rotation by 8 lanes (DPP)
//      gives the second.  The tile's rows 8..15 then hold other rows' data,
//      which reaches only outputs that are not stored.  Against X in LDS at
//      M = 8: Llama down 10.2 -> 9.5 us, 16384 x 4096 16.9 -> 13.2, 12000 x
//      6144 21.7 -> 17.7; and half the X registers, so that 16 waves reach K = 14336 (4096 rows at M = 2 / 8:
//      13.0 / 16.9 us against the GEMM's 32).
//    - one tile of 9..16 rows that fit, and those shapes (kXLds): the block first copies the M
//      real rows to LDS (rows padded by 16 bytes: the 16 rows of a fragment
//      read hit distinct banks), before its weight loads, and each wave reads
//      its fragments from there; rows past M read row 0.
//    - otherwise (kXRegs) all 16 rows of a tile are read through a buffer
//      resource of M * K fp16, so that rows past M read as zeros.
//  * Each word is dequantized in registers without leaving fp16: its
//    nibbles are spread to bytes (q0 q2 q4 q6 and q1 q3 q5 q7), and
//    v_cvt_scalef32_pk_f16_fp8 turns two bytes into two fp16 at a time: read
//    as fp8 e4m3, a byte b < 16 is b * 2^-9 exactly (the subnormals and the
//    first binade share one spacing), and the instruction's scale, of which
//    only the exponent counts, is 2^9.  One v_pk_fma_f16 per pair then gives
//    s * q + b with the GEMM's single rounding.  The k order inside a word
//    is 0,2,1,3,4,6,5,7; X is permuted alike when it is loaded, once per
//    wave.  Four MFMAs per 16-byte load accumulate into the tile's
//    accumulators directly.
//  * The partial tiles of the W waves are summed through LDS once, then the
//    epilogue (gated SiLU / GELU-tanh pair, bias, GELU-tanh, residual add)
//    runs on the fp32 sums.
#include "q4_common.hpp"
#include "q4_dequant.hpp"
#include "q4_launch.hpp"

namespace sltx {

namespace {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// 16-byte pieces of one array's scale / bias slab (rows x groups fp16), and
// the pieces reserved per slab in LDS (whole waves of 64).
__host__ __device__ constexpr int slab_pieces(int rows, int groups) { return rows * groups / 8; }
__host__ __device__ constexpr int slab_alloc(int rows, int groups) {
    return (slab_pieces(rows, groups) + 63) / 64 * 64;
}

__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// W waves, MT tiles of 16 activation rows, STEPS 128-wide k-steps per wave,
// PAIR: two weight sets (gate, up) and a gated epilogue, RT tiles of 16
// weight rows per block.  OCC: blocks per CU the register budget is sized for.
template <int W, int MT, int STEPS, bool PAIR, int RT, int OCC, int XM>
__global__ __launch_bounds__(64 * W, OCC) void q4_skinny_kernel(GemmParams p) {
    constexpr int NS = PAIR ? 2 : 1;
    constexpr int ROWS = 16 * RT;
    constexpr bool XL = XM == kXLds, XH = XM == kXHalf;
    static_assert(XM == kXRegs || MT == 1, "one 16-row tile");
    __shared__ f32x4 red[W][RT][NS][MT][64];
    // [2 * NS slabs][ROWS][groups] fp16, then (XL) X rows [M][K + 8] fp16
    extern __shared__ u32x4 sb_lds[];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kq = lane >> 4;
    const int n0 = blockIdx.x * ROWS;
    const int K = p.K, groups = p.groups;
    const int kw0 = wave * (128 * STEPS) + 32 * kq;   // this lane's first k

    // ---- scales and biases -> LDS (slab a: s0, b0[, s1, b1]) ----
    const int pieces = slab_pieces(ROWS, groups), alloc = slab_alloc(ROWS, groups);
    const int valid = min(ROWS, p.N - n0) * groups * 2;   // slab bytes inside the arrays
    constexpr int RA = (RT * STEPS + 7) / 8;              // rounds per slab (groups <= K/32)
#pragma unroll
    for (int a = 0; a < 2 * NS; ++a) {
        const uint16_t* arr = a == 0 ? p.s0 : a == 1 ? p.b0 : a == 2 ? p.s1 : p.b1;
        const char* src = reinterpret_cast<const char*>(arr + (size_t)n0 * groups);
#pragma unroll
        for (int r = 0; r < RA; ++r) {
            const int c0 = r * 64 * W + 64 * wave;   // wave-uniform
            if (c0 < pieces) {
                int off = (c0 + lane) * 16;
                if (off >= valid) off = 0;          // a spare copy of piece 0
                __builtin_amdgcn_global_load_lds((const void*)(src + off),
                                                 (lds_ptr_t)(sb_lds + a * alloc + c0), 16, 0, 0);
            }
        }
    }
    // ---- XL: X rows [0, M) -> LDS, 1 KB (one wave-wide copy) at a time ----
    const int xrow16 = K / 8 + 1;   // LDS row stride in 16-byte units (one of padding)
    u32x4* const xl = sb_lds + 2 * NS * alloc;
    if constexpr (XL) {
        const int per_row = K / 512;   // 1 KB chunks per row (K % 1024 == 0)
        for (int c = wave; c < p.M * per_row; c += W) {   // wave-uniform
            const int m = c / per_row, j = c - m * per_row;
            const char* src = reinterpret_cast<const char*>(p.a) + (size_t)m * K * 2 +
                              j * 1024 + lane * 16;
            __builtin_amdgcn_global_load_lds((const void*)src,
                                             (lds_ptr_t)(xl + m * xrow16 + j * 64), 16, 0, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- the wave's slice of X: fragment r of step t is x[k .. k+7] with
    // k = kw0 + 128 t + 8 r, the k of word r of the lane's packed load ----
    u32x4 xa[MT][STEPS][4];
    if constexpr (!XL) {
        const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<void*>(p.a), (short)0, p.M * K * 2, 0x00020000);
        if constexpr (XH) {
            // lanes with r16 >= 8 take row r16 - 8 of the next fragment
            const int xrow = ((r16 & 7) * K + kw0 + (r16 & 8)) * 2;
#pragma unroll
            for (int t = 0; t < STEPS; ++t)
#pragma unroll
                for (int r = 0; r < 4; r += 2)
                    xa[0][t][r] = __builtin_bit_cast(
                        u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, xrow + 256 * t + 16 * r, 0, 0));
        } else {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int xrow = ((mt * 16 + r16) * K + kw0) * 2;
#pragma unroll
                for (int t = 0; t < STEPS; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        xa[mt][t][r] = __builtin_bit_cast(
                            u32x4,
                            __builtin_amdgcn_raw_buffer_load_b128(xrs, xrow + 256 * t + 16 * r, 0, 0));
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- packed words, step by step ----
    // Steps t, t+1 of a tile and set are loaded as 2 x 8 rows x 128 bytes
    // (whole lines: load h, lane l reads row (l & 7) | 8h, piece
    // 4 * bit3(l) + l / 16 of the 128-byte run) and swapped into the MFMA
    // layout before use: a load of the layout itself is 16 rows x 64 bytes,
    // every request half a line, and streams ~15% slower.  An odd last step
    // keeps that layout.
    u32x4 wq[STEPS][RT][NS];
    const int prow = lane & 7, ppiece = 4 * ((lane >> 3) & 1) + (lane >> 4);
#pragma unroll
    for (int t = 0; t < STEPS; t += 2) {
        if (t + 1 < STEPS) {
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int row = min(n0 + 16 * i + (prow | (h << 3)), p.N - 1);
                        const uint32_t* wr = (s ? p.w1 : p.w0) + (size_t)row * (K / 8) +
                                             (wave * 128 * STEPS + 128 * t) / 8 + ppiece * 4;
                        wq[t + h][i][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wr));
                    }
        } else {
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int row = min(n0 + 16 * i + r16, p.N - 1);
                    const uint32_t* wr = (s ? p.w1 : p.w0) + (size_t)row * (K / 8) + kw0 / 8;
                    wq[t][i][s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wr + 16 * t));
                }
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // The slabs are complete once at most the X and weight loads issued after
    // them are outstanding (every wave issues all of those).  Both waits are
    // builtins: with a wait in inline assembly the compiler loses its count
    // of the loads in flight and waits for all of them at the next use.  The
    // barrier is assembly with a memory clobber, so that no LDS read moves
    // above it.
    __builtin_amdgcn_s_waitcnt(vmcnt_only((XL ? 0 : XH ? STEPS * 2 : MT * STEPS * 4) + STEPS * RT * NS));
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (XL) {   // rows past M (outputs that are not stored) read row 0
        const u32x4* xr = xl + (r16 < p.M ? r16 : 0) * xrow16 + kw0 / 8;
#pragma unroll
        for (int t = 0; t < STEPS; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) xa[0][t][r] = xr[16 * t + r];
    }

#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < STEPS; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (XH && (r & 1)) {   // rows 8.. of the fragment before (rows 8.. here unused)
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        xa[mt][t][r][c] = (uint32_t)__builtin_amdgcn_mov_dpp((int)xa[mt][t][r - 1][c],
                                                                            0x128, 0xF, 0xF, true);
                } else {
                    xa[mt][t][r] = permute_x(xa[mt][t][r]);
                }
            }

    const uint16_t* sbl = reinterpret_cast<const uint16_t*>(sb_lds);
    const int gshift = 5 + p.gshift;   // log2(group size)
    f32x4 acc[RT][NS][MT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[i][s][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < STEPS; ++t) {
        if ((t & 1) == 0 && t + 1 < STEPS) {
            // lane l of the pair's load h holds row (l & 7) | 8h, piece
            // 4 * bit3(l) + l / 16: lanes whose bit 3 is h already hold their
            // step-h data; the others take it from lane l ^ 8 of the other
            // load (a row rotation by 8 inside each 16-lane row, written
            // only to the banks of 4 lanes that need it)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int r0 = (int)wq[t][i][s][c], r1 = (int)wq[t + 1][i][s][c];
                        wq[t][i][s][c] = (uint32_t)__builtin_amdgcn_update_dpp(r0, r1, 0x128, 0xF, 0xC, false);
                        wq[t + 1][i][s][c] = (uint32_t)__builtin_amdgcn_update_dpp(r1, r0, 0x128, 0xF, 0x3, false);
                    }
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                // the lane's 32 k lie in one group (group sizes 32, 64, 128)
                const int gi = (kw0 + 128 * t) >> gshift;
                const uint16_t* srow = sbl + (size_t)(2 * s) * alloc * 8 + (16 * i + r16) * groups;
                const uint32_t sv = srow[gi], bv = srow[alloc * 8 + gi];
                const f16x2 s2 = as_f16x2(sv | (sv << 16));
                const f16x2 b2 = as_f16x2(bv | (bv << 16));
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const u32x4 b = dequant_word(wq[t][i][s][r], s2, b2);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        acc[i][s][mt] = mfma16(xa[mt][t][r], b, acc[i][s][mt]);
                }
            }
    }

#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) red[wave][i][s][mt][lane] = acc[i][s][mt];
    __syncthreads();

    // one output per thread: D[m][n] of a 16x16 tile sits in lane
    // 16 * (m / 4) + n, element m % 4
    for (int o = threadIdx.x; o < RT * MT * 256; o += 64 * W) {
        const int i = o / (MT * 256), mt = (o >> 8) % MT, ml = (o >> 4) & 15, nl = o & 15;
        const int m = mt * 16 + ml, n = n0 + 16 * i + nl;
        if (m >= p.M || n >= p.N) continue;
        const int src = 16 * (ml >> 2) + nl, e = ml & 3;
        float v[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            float a = 0.0f;
#pragma unroll
            for (int w = 0; w < W; ++w) a += red[w][i][s][mt][src][e];
            v[s] = a;
        }
        float out;
        if constexpr (PAIR) {
            out = glu_f32(p.epilogue == kEpiGeluMul, v[0], v[NS - 1]);
        } else {
            out = v[0];
            if (p.bias) out += p.bias[n];
            if (p.epilogue == kEpiGeluTanh) out = gelu_tanh_f32(out);
        }
        const size_t oi = (size_t)m * p.N + n;
        if (!PAIR && p.epilogue == kEpiResidual)
            reinterpret_cast<uint16_t*>(p.y)[oi] = residual_add_f16(p.residual[oi], out);
        else
            store_one(p, oi, out);
    }
}

// Registers of a configuration, roughly: X fragments, the packed words in
// flight, accumulators, and about 40 for the rest.
constexpr int skinny_vgprs(int mt, int steps, int ns, int rt, int xm = kXRegs) {
    return (xm == kXHalf ? 8 : 16) * mt * steps + 4 * rt * ns * steps + 4 * rt * ns * mt + 40;
}
constexpr int kSkinnyMaxVgprs = 224;   // of the 256 one block of 8 waves may use

// Dynamic LDS of a launch: the scale / bias slabs, then (kXLds) X's rows.
size_t skinny_lds(const GemmParams& p, int rt, bool pair, bool xl) {
    return (size_t)(pair ? 4 : 2) * slab_alloc(16 * rt, p.groups) * 16 +
           (xl ? (size_t)p.M * (p.K / 8 + 1) * 16 : 0);
}

// Blocks per CU a configuration is compiled for: two when a wave fits in
// 128 VGPRs.
constexpr int skinny_occ(int w, int mt, int steps, int ns, int rt, int xm) {
    return (w == 8 && skinny_vgprs(mt, steps, ns, rt, xm) <= 120) ? 2 : 1;
}

template <int W, int MT, int STEPS, bool PAIR, int RT, int XM>
hipError_t launch_cfg(const GemmParams& p, hipStream_t st) {
    constexpr int OCC = skinny_occ(W, MT, STEPS, PAIR ? 2 : 1, RT, XM);
    const dim3 grid((unsigned)((p.N + 16 * RT - 1) / (16 * RT))), block(64 * W);
    const size_t lds = skinny_lds(p, RT, PAIR, XM == kXLds);
    hipLaunchKernelGGL((q4_skinny_kernel<W, MT, STEPS, PAIR, RT, OCC, XM>), grid, block, lds, st, p);
    return hipGetLastError();
}

template <int W, int MT, int STEPS, bool PAIR, int RT>
hipError_t launch_x(const GemmParams& p, int xm, hipStream_t st) {
    if constexpr (MT == 1) {
        if (xm == kXHalf) return launch_cfg<W, MT, STEPS, PAIR, RT, kXHalf>(p, st);
    }
    if constexpr (STEPS > (W == 8 ? 6 : 5)) {
        return hipErrorInvalidValue;
    } else {
        if constexpr (MT == 1 && W == 8) {   // (16 waves: more than 8 rows of their K don't fit)
            if (xm == kXLds) return launch_cfg<W, MT, STEPS, PAIR, RT, kXLds>(p, st);
        }
        return launch_cfg<W, MT, STEPS, PAIR, RT, kXRegs>(p, st);
    }
}

template <int W, int MT, int STEPS>
hipError_t launch_steps(const GemmParams& p, const SkinnyPlan& pl, hipStream_t st) {
    const bool pair = p.w1 != nullptr;
    if (pl.RT == 2) {
        if constexpr (W == 8 && skinny_vgprs(MT, STEPS, 2, 2) <= kSkinnyMaxVgprs)
            return pair ? launch_x<W, MT, STEPS, true, 2>(p, pl.XM, st)
                        : launch_x<W, MT, STEPS, false, 2>(p, pl.XM, st);
        return hipErrorInvalidValue;
    }
    if (pair) {
        // a gated pair of 5 steps does not fit the 128 VGPRs of 16 waves
        if constexpr (W == 16 && STEPS >= 5) return hipErrorInvalidValue;
        else return launch_x<W, MT, STEPS, true, 1>(p, pl.XM, st);
    }
    return launch_x<W, MT, STEPS, false, 1>(p, pl.XM, st);
}

}  // namespace

bool skinny_plan(const GemmParams& p, bool a_bf16, SkinnyPlan* out) {
    if (a_bf16 || p.M < 1 || p.M > 32 || p.N < 1 || p.K <= 0) return false;
    if (p.gshift < 0 || p.gshift > 2) return false;
    if ((long)p.M * p.K * 2 > 0x7fffffffL) return false;   // X buffer offsets are 32-bit
    const bool pair = p.w1 != nullptr;
    if (pair && p.epilogue != kEpiSiluMul && p.epilogue != kEpiGeluMul) return false;
    if (!pair && p.epilogue != kEpiNone && p.epilogue != kEpiGeluTanh &&
        p.epilogue != kEpiResidual)
        return false;
    const int mt = p.M <= 16 ? 1 : 2;
    SkinnyPlan pl{0, mt, 0, 1, 1, kXRegs};
    // 8 waves of 1..6 steps (1..4 with 32 activation rows), else 16 waves of
    // 4..5 steps (4 for a gated pair; one set of at most 8 rows 4..7)
    if (p.K % 1024 == 0 && p.K / 1024 <= (mt == 1 ? 6 : 4)) {
        pl.W = 8;
        pl.STEPS = p.K / 1024;
    } else if (mt == 1 && p.K % 2048 == 0 && p.K / 2048 <= (pair ? 4 : p.M <= 8 ? 7 : 5)) {
        // (a gated pair of 5 steps does not fit the 128 VGPRs of 16 waves)
        pl.W = 16;
        pl.STEPS = p.K / 2048;
    } else {
        return false;
    }
    // Two row tiles per block (the X slice serves twice the weight rows), with
    // 8 waves and at least one block per CU: when the two-tile block still
    // fits two per CU, or above 8 activation rows.  Measured: the vocabulary
    // head at M = 8 takes 59.3 us with two tiles (two blocks per CU) against
    // 75.2 us with one, 16384 x 4096 13.2 against 15.0; the gate/up pair at
    // M = 16 11.2 against 12.4.  A pair of at most 8 rows keeps one tile:
    // 10.8 against 11.3 us (8192 x 3072), 6.3 against 6.9 (12000 x 1024).
    const int ns = pair ? 2 : 1;
    pl.XM = p.M <= 8 ? kXHalf : kXRegs;
    // (launch_steps instantiates two tiles where a gated pair of them fits
    // the register budget; every two-tile block that fits two per CU does)
    if (pl.W == 8 && !(pair && pl.XM == kXHalf) && (p.N + 31) / 32 >= kCUs &&
        (skinny_occ(8, mt, pl.STEPS, ns, 2, pl.XM) == 2 ||
         (p.M > 8 && skinny_vgprs(mt, pl.STEPS, 2, 2) <= kSkinnyMaxVgprs)))
        pl.RT = 2;
    pl.OCC = skinny_occ(pl.W, mt, pl.STEPS, ns, pl.RT, pl.XM);
    // X of 9..16 rows in LDS: where the rows fit beside the slabs, so that a
    // block still gets its share of the CU's LDS (all of it where the grid has
    // no second block for a CU: 3072 x 3072 at M = 16 takes 5.6 us with X in
    // LDS, 6.2 without).  Of at most 8 rows too, where blocks of three steps, or
    // of two of one set, share CUs (at one step and from four, at one block per CU
    // and for pairs of group 32, whose scales fill more of the LDS, halves are the
    // faster).  Measured, LDS against halves: 5120 x 3072 at M
    // = 5 / 6 / 8 6.27 / 6.32 / 6.77 us against 6.51 / 6.80 / 7.34, the gate/up pair at
    // M = 2 / 4 / 6 / 8 9.05 / 9.40 / 9.56 / 9.85 against 9.09 / 9.70 / 9.88 / 10.28, 5120 x
    // 2048 at M = 5 / 8 4.72 / 4.96 against 5.01 / 5.52; pairs of two steps at M = 5 / 8
    // 6.96 / 7.19 against 6.67 / 7.17, the gate/up pair of group 32 at M = 2 / 8 9.80 /
    // 10.57 against 9.28 / 10.72, 8000 x 1024 at M = 5 3.85 / 3.74, 8000 x 4096 8.18 / 8.02.
    const long blocks = (p.N + 16L * pl.RT - 1) / (16 * pl.RT);
    const bool few_in_lds = blocks > kCUs && pl.RT == 1 &&
                            (pair ? pl.STEPS == 3 && p.gshift > 0 : pl.STEPS == 3 || pl.STEPS == 2);
    if (pl.W == 8 && mt == 1 && (pl.XM == kXRegs || few_in_lds) &&
        skinny_lds(p, pl.RT, pair, true) <= (size_t)(pl.RT == 2 || blocks <= kCUs ? 128 : 64) * 1024)
        pl.XM = kXLds;
    // scales and biases are staged with 16-byte loads
    const uintptr_t sb = reinterpret_cast<uintptr_t>(p.s0) | reinterpret_cast<uintptr_t>(p.b0) |
                         (pair ? reinterpret_cast<uintptr_t>(p.s1) | reinterpret_cast<uintptr_t>(p.b1)
                               : 0);
    if ((sb & 15) != 0) return false;
    *out = pl;
    return true;
}

hipError_t launch_skinny(const GemmParams& p, const SkinnyPlan& pl, hipStream_t st) {
    if (pl.W == 8 && pl.MT == 1) {
        switch (pl.STEPS) {
            case 1: return launch_steps<8, 1, 1>(p, pl, st);
            case 2: return launch_steps<8, 1, 2>(p, pl, st);
            case 3: return launch_steps<8, 1, 3>(p, pl, st);
            case 4: return launch_steps<8, 1, 4>(p, pl, st);
            case 5: return launch_steps<8, 1, 5>(p, pl, st);
            case 6: return launch_steps<8, 1, 6>(p, pl, st);
        }
    } else if (pl.W == 8 && pl.MT == 2) {
        switch (pl.STEPS) {
            case 1: return launch_steps<8, 2, 1>(p, pl, st);
            case 2: return launch_steps<8, 2, 2>(p, pl, st);
            case 3: return launch_steps<8, 2, 3>(p, pl, st);
            case 4: return launch_steps<8, 2, 4>(p, pl, st);
        }
    } else if (pl.W == 16 && pl.MT == 1) {
        switch (pl.STEPS) {
            case 4: return launch_steps<16, 1, 4>(p, pl, st);
            case 5: return launch_steps<16, 1, 5>(p, pl, st);
            case 6: return launch_steps<16, 1, 6>(p, pl, st);
            case 7: return launch_steps<16, 1, 7>(p, pl, st);
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace sltx
