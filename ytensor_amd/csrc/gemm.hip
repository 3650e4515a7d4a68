// gemm.hip — MFMA GEMM for gfx950 (CDNA4), the device replacement of YTensor's
// blocked AVX2 sgemm / hgemm (src/kernel/avx2/sgemm.inl:268-340, 586-787;
// src/kernel/avx2/hgemm.inl:139-273).
//
// Design (MI355X-first, not a translation of the CPU Goto loop):
//  * Block tile BM x BN, k step of 128 bytes per row (64 bf16/fp16 or 32 fp32).
//    Both operands live in LDS K-contiguous, [rows][8 chunks of 16 B], so an
//    MFMA operand fragment is one ds_read_b128 per lane. A row-major B ("NN",
//    B[k][n]) stays [k][n] in LDS and its fragments are read with the gfx950
//    transposing read ds_read_b64_tr_b16, so nothing is transposed in registers.
//  * Tiles move global -> LDS by direct-to-LDS DMA (global_load_lds_dwordx4):
//    no VGPR staging. Two stages where the tile fills the LDS (256 x 256) or two
//    workgroups share a CU (128 x 128 of four waves), three at 256 x 128 and where two 128 x 64
//    share one, a 4-deep ring for 64 x 64, 64 x 32 and the one-per-CU 128 x 64 and 128 x 128 of
//    eight waves. The
//    bytes each CU can pull through its vector-memory path (~28 B/clk) are close to what
//    256 x 256 MFMA work consumes, so the 256 x 256 tile is the only one that keeps up
//    at 4096^3.
//  * LDS swizzles were chosen by measuring gfx950's LDS read rate per pattern
//    (see swz_dma / nn_blk): fragment reads are bank-conflict free.
//  * Inside a k step the A fragments stream through a 3-register ring read two
//    MFMA groups ahead, pinned by schedule barriers, so LDS latency overlaps
//    the matrix cores.
//  * MFMA operands are swapped (src0 = B rows, src1 = A rows): each lane then
//    holds 4 consecutive output columns of one row, stored as one vector.
//  * Tiles are assigned XCD-aware: the hardware places workgroup w on XCD
//    w % 8; each XCD receives a contiguous, M-grouped range of tiles so its
//    32 CUs share A and B panels in their own L2.
//  * What the DMA cannot take (rows that are not 16-byte aligned, k or n that are
//    no whole chunks, a transposed A, other strides) runs in gemm_any.hip.

#include <algorithm>

#include "common.hpp"
#include "launch.hpp"

namespace ythip {

struct GemmArgs {
    const void* A;
    const void* B;
    void* C;
    int m, n, k;
    int64_t rsa, rsb, csb, rsc;  // csa == 1 and csc == 1 on this path
    int64_t sa_b, sb_b, sc_b;
    float alpha, beta;
    int tiles_m, tiles_n;
    int c_vec_ok;   // C rows allow 4-element vector stores
    int c_line_ok;  // 16-bit C: 16-byte aligned base and rows (the ping-pong kernel's line stores)
    MaskDesc mask;  // (never on the ping-pong and GEMV kernels)
};

// Swizzles of the DMA-staged kernel, chosen by measuring gfx950's LDS read rate
// per access pattern (64 banks; ds_read_b128 and ds_read_b64_tr_b16):
//  * K-major tiles [row][8 x 16 B]: chunk c of row r at c ^ ((r >> 1) & 7). Rows
//    r and r+1 share one 256-byte bank window and take the same XOR, so a
//    fragment read (16 rows, one logical chunk) covers all 64 banks without
//    conflict; the previous row-XOR swizzle ran at ~60% of that rate.
//  * NN B tiles [k][n] in 32-byte column blocks: block b of k-row r at
//    b ^ h(r), h(r) = (r ^ ((r >> 3) << 2)) & mask, so the transposing reads of
//    k-rows r and r + 8 (served together) land in different blocks.
__device__ __forceinline__ int swz_dma(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }
__device__ __forceinline__ int nn_blk(int row, int blk, int mask) { return blk ^ ((row ^ ((row >> 3) << 2)) & mask); }

// ---------------------------------------------------------------------------
// DMA-staged variant (the fast path). Tiles go global -> LDS with
// global_load_lds (16 bytes per lane, no VGPR staging); the XOR swizzle is
// applied on the global-address side because the DMA writes 64 consecutive
// 16-byte LDS slots per wave. While the matrix cores work on one LDS stage the
// DMA fills the other; fragments for the second 32-wide k step are read from
// LDS before the first step's MFMAs, and a scheduling pattern interleaves the
// LDS reads with the MFMAs.
//   NN (B row-major [k][n], 16-bit): the B tile stays [k][n] in LDS (rows of
//   BN elements, 32-byte blocks XOR-swizzled by row) and is read with
//   ds_read_b64_tr_b16: within each 16-lane group, lane j addresses the 4
//   columns 4*(j%4).. of k-row j/4 and lane i receives column i of those 4
//   k-rows -- exactly the MFMA B operand (two reads per 16x32 fragment).
// Requirements (checked on the host): k % VEC == 0, 16-byte aligned rows, and
// for NN: n % 8 == 0. Rows past M / N are clamped (their outputs are never
// stored).
// ---------------------------------------------------------------------------

// What the DMA reads in place of k past the end.
static __device__ const u32x4 dma_zero[1] = {{0u, 0u, 0u, 0u}};

// SOFF: every operand spans less than 2^31 bytes (checked on the host): the DMA
// then goes from a wave-uniform base, moved by scalar adds per k step, plus a
// per-lane 32-bit byte offset fixed for the whole k loop (dma16_soff), and the
// LDS destination is the wave's base plus constants -- no VALU address work
// between the MFMAs of consecutive k steps.
// FORM (templates, since the forms' code would cost the others its length):
//   PLAIN; MASKED: a masked product;
//   SWIGLU (NT): B = [gate rows | up rows], a.n columns of C each: a wave's fragments
//   alternate between 16 gate rows and the same 16 up rows, so a lane holds both
//   factors of its activations and the [m][2 n] product is never written.
// RAGGED: k need not be whole steps. Without it the k loop is the compiler's for a plain
// count of steps; with it, a few more scalar instructions per step show where a chain of steps is
// all there is (64 x 64 x 8192 NT 27.6 us, 28.6 with it; 512 x 1024 x 3072 NT 11.9 / 12.3).
enum { PLAIN = 0, MASKED = 1, SWIGLU = 2 };
template <class T, class TO, int BM, int BN, int WM, int WN, bool NN, int STAGES, bool SOFF, int FORM, bool RAGGED = true>
__global__ __launch_bounds__(64 * WM * WN) void gemm_mfma_dma_kernel(GemmArgs a) {
    using raw = typename T::raw;
    constexpr int THREADS = 64 * WM * WN;
    constexpr int VEC = 16 / sizeof(raw);
    constexpr int BK = 8 * VEC;
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int A_PT = BM * 8 / THREADS, B_PT = BN * 8 / THREADS;
    static_assert(A_PT * THREADS == BM * 8 && B_PT * THREADS == BN * 8, "tile/thread mismatch");
    static_assert(!NN || sizeof(raw) == 2, "the transposing LDS read is 16-bit");
    constexpr int STA = BM * 8, STB = BN * 8;             // 16-byte slots per stage
    constexpr int NBLK = BN / 16;                          // NN: 32-byte blocks per k-row
    constexpr int BLK_MASK = (NBLK < 8 ? NBLK : 8) - 1;
    constexpr int MF_PER_CHUNK = sizeof(raw) == 2 ? 1 : 4;

    constexpr int PER = A_PT + B_PT;  // DMA instructions per thread per stage
    static_assert(STAGES >= 2 && STAGES <= 4 && (STAGES - 2) * PER < 64, "pipeline depth");

    __shared__ u32x4 sbuf[STAGES * (STA + STB)];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int lrow = lane & 15, lgrp = lane >> 4;

    int tm, tn;
    tile_coords(blockIdx.x, a.tiles_m, a.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int bz = blockIdx.y;
    const raw* __restrict__ Ap = static_cast<const raw*>(a.A) + bz * a.sa_b;
    const raw* __restrict__ Bp = static_cast<const raw*>(a.B) + bz * a.sb_b;
    // A ragged k makes the FIRST step short, [0, first): its missing chunks come
    // from 16 bytes of zeros (dma_zero), and the loop has whole steps only.
    const int KT_all = RAGGED ? (a.k + BK - 1) / BK : a.k / BK;
    const int first = RAGGED ? a.k - (KT_all - 1) * BK : BK;
    // a tile that the mask hides whole: its sums are not used
    const int KT = FORM == MASKED && hidden_tile(a.mask, min(m0 + BM, a.m) - 1, n0) ? 1 : KT_all;

    // the B row behind row r of an NT tile
    auto b_row = [&](int r) -> int64_t {
        if constexpr (FORM == SWIGLU) {
            const int f = (r % WTN) / 16;
            const int col = n0 / 2 + r / WTN * (WTN / 2) + f / 2 * 16 + r % 16;
            return (f & 1 ? a.n : 0) + min(col, a.n - 1);
        } else {
            return min(n0 + r, a.n - 1);
        }
    };

    // Step 0 of a ragged k, and every step of operands too large for SOFF.
    auto issue_a = [&](int kt, u32x4* sA) {
        const int k0 = kt == 0 ? 0 : kt * BK - (BK - first);
#pragma unroll (SOFF ? 1 : A_PT)
        for (int i = 0; i < A_PT; ++i) {
            const int slot = i * THREADS + wave * 64 + lane;
            const int r = slot >> 3;
            const int c = swz_dma(r, slot & 7);  // the swizzle is an involution on the chunk index
            const int row = min(m0 + r, a.m - 1);
            const raw* g = Ap + (int64_t)row * a.rsa + k0 + c * VEC;
            if (kt == 0 && c * VEC >= first) g = reinterpret_cast<const raw*>(dma_zero);
            dma16_async(g, &sA[i * THREADS + wave * 64]);
        }
    };
    auto issue_b = [&](int kt, u32x4* sB) {
        const int k0 = kt == 0 ? 0 : kt * BK - (BK - first);
#pragma unroll (SOFF ? 1 : B_PT)
        for (int i = 0; i < B_PT; ++i) {
            const int slot = i * THREADS + wave * 64 + lane;
            const raw* g;
            if constexpr (!NN) {
                const int r = slot >> 3;
                const int c = swz_dma(r, slot & 7);
                g = Bp + b_row(r) * a.csb + k0 + c * VEC;
                if (kt == 0 && c * VEC >= first) g = reinterpret_cast<const raw*>(dma_zero);
            } else {
                const int r = slot / (2 * NBLK), ps = slot % (2 * NBLK);
                const int lb = nn_blk(r, ps >> 1, BLK_MASK);
                g = Bp + (int64_t)(k0 + r) * a.rsb + min(n0 + lb * 16 + (ps & 1) * 8, a.n - 8);
                if (kt == 0 && r >= first) g = reinterpret_cast<const raw*>(dma_zero);
            }
            dma16_async(g, &sB[i * THREADS + wave * 64]);
        }
    };
    // SOFF: per-lane byte offsets of the stage-0 loads (the k loop moves the base)
    uint32_t offA[SOFF ? A_PT : 1], offB[SOFF ? B_PT : 1];
    uint32_t ldsA0 = 0, ldsB0 = 0;
    if constexpr (SOFF) {
#pragma unroll
        for (int i = 0; i < A_PT; ++i) {
            const int slot = i * THREADS + wave * 64 + lane;
            const int r = slot >> 3;
            const int c = swz_dma(r, slot & 7);
            const int row = min(m0 + r, a.m - 1);
            offA[i] = (uint32_t)(((int64_t)row * a.rsa + c * VEC) * (int64_t)sizeof(raw));
        }
#pragma unroll
        for (int i = 0; i < B_PT; ++i) {
            const int slot = i * THREADS + wave * 64 + lane;
            int64_t e;
            if constexpr (!NN) {
                const int r = slot >> 3;
                const int c = swz_dma(r, slot & 7);
                e = b_row(r) * a.csb + c * VEC;
            } else {
                const int r = slot / (2 * NBLK), ps = slot % (2 * NBLK);
                const int lb = nn_blk(r, ps >> 1, BLK_MASK);
                e = (int64_t)r * a.rsb + min(n0 + lb * 16 + (ps & 1) * 8, a.n - 8);
            }
            offB[i] = (uint32_t)(e * (int64_t)sizeof(raw));
        }
        ldsA0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)&sbuf[wave * 64]);
        ldsB0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)&sbuf[STAGES * STA + wave * 64]);
    }
    // DMA of k step kt into stage st
    auto issue_st = [&](int kt, int st) {
        if (SOFF && (kt > 0 || first == BK)) {
            const int64_t k0 = (int64_t)kt * BK - (BK - first);
            const char* bA = reinterpret_cast<const char*>(Ap) + k0 * (int64_t)sizeof(raw);
            const char* bB = reinterpret_cast<const char*>(Bp) + k0 * (NN ? a.rsb : (int64_t)1) * (int64_t)sizeof(raw);
#pragma unroll
            for (int i = 0; i < A_PT; ++i) dma16_soff(bA, offA[i], ldsA0 + (uint32_t)(st * STA + i * THREADS) * 16u);
#pragma unroll
            for (int i = 0; i < B_PT; ++i) dma16_soff(bB, offB[i], ldsB0 + (uint32_t)(st * STB + i * THREADS) * 16u);
        } else {
            issue_a(kt, sbuf + st * STA);
            issue_b(kt, sbuf + STAGES * STA + st * STB);
        }
    };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Fragment reads. A fragment (16 rows x one 16-byte chunk) is one ds_read_b128;
    // a B fragment is one ds_read_b128 (NT) or two transposing reads (NN).
    auto ldA = [&](const u32x4* sA, int ks, int i) -> u32x4 {
        const int r = wm * WTM + i * 16 + lrow;
        return sA[r * 8 + swz_dma(r, ks * 4 + lgrp)];
    };
    auto ldB = [&](const u32x4* sB, int ks, int j) -> u32x4 {
        if constexpr (!NN) {
            const int r = wn * WTN + j * 16 + lrow;
            return sB[r * 8 + swz_dma(r, ks * 4 + lgrp)];
        } else {
            const int nb = (wn * WTN + j * 16) >> 4;
            u32x4 v;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = ks * 32 + 8 * lgrp + 4 * h + (lrow >> 2);
                const int byte = r * (BN * 2) + (nn_blk(r, nb, BLK_MASK) << 5) + 8 * (lrow & 3);
                const u32x2 w = lds_read_tr16(sB, byte);
                v[2 * h] = w[0];
                v[2 * h + 1] = w[1];
            }
            return v;
        }
    };
    // One k step = 2 x 32 k = 2*FM A fragments (t = ks*FM + i). A fragments stream
    // through a ring of 3 registers, read two steps ahead; the B fragments of the
    // second half are read right after the first step. The schedule barriers pin
    // the order (reads for t+2, then the FN MFMAs of t), so every wait before an
    // MFMA is a partial lgkmcnt and the reads overlap the matrix work.
    constexpr int BR = NN ? 2 : 1;
    constexpr int NTS = 2 * FM;
    static_assert(FM >= 2, "the A ring needs at least 4 fragments per k step");
    auto compute = [&](const u32x4* sA, const u32x4* sB) {
        u32x4 fb[2][FN], fa[3];
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[0][j] = ldB(sB, 0, j);
        fa[0] = ldA(sA, 0, 0);
        fa[1] = ldA(sA, 1 / FM, 1 % FM);
        __builtin_amdgcn_sched_group_barrier(0x100, FN * BR + 2, 0);
        static_for<0, NTS>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            constexpr int ks = t / FM, i = t % FM;
            constexpr int nrd = (t + 2 < NTS ? 1 : 0) + (t == 1 ? FN * BR : 0);
            if constexpr (t + 2 < NTS) fa[(t + 2) % 3] = ldA(sA, (t + 2) / FM, (t + 2) % FM);
            if constexpr (t == 1) {
#pragma unroll
                for (int j = 0; j < FN; ++j) fb[1][j] = ldB(sB, 1, j);
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = mfma_chunk(T{}, fb[ks][j], fa[t % 3], acc[i][j]);
            if constexpr (nrd > 0) __builtin_amdgcn_sched_group_barrier(0x100, nrd, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, FN * MF_PER_CHUNK, 0);
        });
    };

    u32x4* sA = sbuf;
    u32x4* sB = sbuf + STAGES * STA;
    if constexpr (STAGES == 2) {
        // Double buffer: DMA of step kt+1 overlaps the MFMAs of step kt.
        issue_st(0, 0);
        wait_vmcnt<0>();
        __syncthreads();
        for (int kt = 0; kt < KT; ++kt) {
            const int cur = kt & 1;
            if (kt + 1 < KT) issue_st(kt + 1, cur ^ 1);
            compute(sA + cur * STA, sB + cur * STB);
            wait_vmcnt<0>();  // this wave's DMA for the next step has landed
            __syncthreads();
        }
    } else {
    // STAGES-deep ring: STAGES-1 k steps are in flight while one is computed.
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st)
        if (st < KT) issue_st(st, st);
    for (int kt = 0; kt < KT; ++kt) {
        // Stage kt has landed for this wave once at most `ahead` later stages are outstanding.
        const int ahead = min(STAGES - 2, KT - 1 - kt);
        if (STAGES > 2 && ahead >= 2) wait_vmcnt<(STAGES > 2 ? 2 : 0) * PER>();
        else if (STAGES > 2 && ahead == 1) wait_vmcnt<PER>();
        else wait_vmcnt<0>();
        __syncthreads();  // every wave's share of stage kt is in LDS; stage kt-1 is consumed
        const int nxt = kt + STAGES - 1;
        if (nxt < KT) issue_st(nxt, nxt % STAGES);
        compute(sA + (kt % STAGES) * STA, sB + (kt % STAGES) * STB);
    }
    }

    using oraw = typename TO::raw;
    oraw* Cp = static_cast<oraw*>(a.C) + bz * a.sc_b;
    if constexpr (FORM == SWIGLU) {
        static_assert(FN % 2 == 0 && !NN && sizeof(oraw) == 2, "gate and up fragments in pairs");
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int m = m0 + wm * WTM + i * 16 + lrow;
            if (m >= a.m) continue;
#pragma unroll
            for (int j = 0; j < FN; j += 2) {
                const int n = n0 / 2 + wn * (WTN / 2) + j * 8 + lgrp * 4;
                uint32_t v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t gu = pack2<TO>(acc[i][j][r], acc[i][j + 1][r]);  // both rounded first
                    const float y = swish_mul(lo_as_f32(TO{}, gu), hi_as_f32(TO{}, gu));
                    // silu_mul's conversion, element by element (fp16 subnormals)
                    v[r] = std::is_same_v<TO, F16> ? f32_to_f16_bits(y) : f32_to_bf16_bits(y);
                }
                if (n < a.n)  // a.n % 4 == 0
                    *reinterpret_cast<u32x2*>(Cp + (int64_t)m * a.rsc + n) = u32x2{v[0] | v[1] << 16, v[2] | v[3] << 16};
            }
        }
        return;
    }
    float alpha = a.alpha;
    const bool filled = FORM == MASKED && a.mask.fill && a.beta == 0.0f;
    if (FORM == MASKED && filled) {  // every entry is written: the value where hidden, then the stores of a plain product
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int m = min(m0 + wm * WTM + i * 16 + lrow, a.m - 1);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const uint32_t vis = visible4(a.mask, m, n0 + wn * WTN + j * 16 + lgrp * 4, a.n);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = (vis >> r) & 1 ? alpha * acc[i][j][r] : a.mask.value;
            }
        }
        alpha = 1.0f;
    }
    if constexpr (sizeof(oraw) == 2 && BN >= 64) {
        if (a.beta == 0.0f && (FORM != MASKED || filled) && a.c_line_ok && m0 + BM <= a.m && n0 + BN <= a.n) {
            // A whole 16-bit tile leaves through LDS in rows of BN elements (chunk c of
            // row r at c ^ (r % CPR)): each thread stores 16-byte chunks of whole tile
            // rows, 128-byte lines and up, instead of the fragments' 8-byte pieces of
            // 16 rows (1040 x 12288 x 512: 24.6 -> 20.4 us; 512 x 6144 x 1024: 11.2 ->
            // 10.0 us). Tiles 32 wide keep the fragment stores: half lines gain nothing
            // there and the extra barriers cost.
            constexpr int CPR = BN / 8;  // 16-byte chunks per tile row
            static_assert(BM * BN * 2 <= STAGES * (STA + STB) * 16, "the C tile fits in the stages");
            char* t = reinterpret_cast<char*>(sbuf);
            __syncthreads();  // every wave is done reading the stages
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int r = wm * WTM + i * 16 + lrow;
                    const int cb = (wn * WTN + j * 16 + lgrp * 4) * 2;
                    *reinterpret_cast<u32x2*>(t + r * (2 * BN) + ((((cb >> 4) ^ (r & (CPR - 1))) << 4) | (cb & 15))) =
                        u32x2{pack2<TO>(alpha * acc[i][j][0], alpha * acc[i][j][1]),
                              pack2<TO>(alpha * acc[i][j][2], alpha * acc[i][j][3])};
                }
            __syncthreads();
#pragma unroll
            for (int id = tid; id < BM * CPR; id += THREADS) {
                const int r = id / CPR, c = id % CPR;
                *reinterpret_cast<u32x4*>(Cp + (int64_t)(m0 + r) * a.rsc + n0 + c * 8) =
                    *reinterpret_cast<const u32x4*>(t + r * (2 * BN) + ((c ^ (r & (CPR - 1))) << 4));
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = m0 + wm * WTM + i * 16 + lrow;
        if (m >= a.m) continue;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + wn * WTN + j * 16 + lgrp * 4;
            if (n >= a.n) continue;
            oraw* crow = Cp + (int64_t)m * a.rsc;
            if (FORM == MASKED && !filled) {
                masked_store4<TO>(a.mask, crow, 1, m, n, a.n, acc[i][j] * alpha, a.beta);
                continue;
            }
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = alpha * acc[i][j][r];
            if (a.beta != 0.0f) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < a.n) v[r] += a.beta * load_as_f32<TO>(crow, n + r);
            }
            if (a.c_vec_ok && n + 3 < a.n) {
                if constexpr (sizeof(oraw) == 2) {
                    *reinterpret_cast<u32x2*>(crow + n) = u32x2{pack2<TO>(v[0], v[1]), pack2<TO>(v[2], v[3])};
                } else {
                    *reinterpret_cast<f32x4*>(crow + n) = f32x4{v[0], v[1], v[2], v[3]};
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < a.n) store_from_f32<TO>(crow, n + r, v[r]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Ping-pong variant of the 256 x 256 DMA kernel for whole 256-row tiles.
// Waves 0-3 (group A) own tile rows 0-127, waves 4-7 (group B) rows 128-255;
// the hardware places waves w and w+4 on one SIMD. Per 64-wide k step kt, after
// one workgroup barrier,
//   group A: stages step kt+1 (DMA), reads every fragment of step kt from LDS
//            into registers (X), then runs the step's 64 MFMAs from registers at
//            raised issue priority (Y);
//   group B: runs Y(kt-1) on the fragments it read before the barrier, then
//            X(kt), and drains its LDS reads;
// so on each SIMD one wave's MFMA cluster runs while the other wave loads.
// Group A waits for its DMA of step kt+1 before the next barrier; group B's
// reads of a stage end before the barrier after which group A refills it.
// Same LDS layouts, swizzles, fragments and MFMA order as
// gemm_mfma_dma_kernel (bit-identical C).
// Requirements (host): m % 256 == 0, k % 64 == 0, every operand spans < 2^31
// bytes, and NN: n % 16 == 0 / NT: n % 256 == 0. Each DMA is a scalar base
// plus a 32-bit lane offset fixed for the kernel: A's (and NT B's) chunk
// swizzle repeats every 32 rows of a stage and NN B's block swizzle depends on
// the 8-k-row group only through its parity. A partial last column of NN
// tiles re-reads B's last 16 columns and stores only columns below N. A 16-bit
// C with beta == 0 and 16-byte aligned rows leaves through LDS as whole lines.
template <class T, class TO, bool NN>
__global__ __launch_bounds__(512, 1) void gemm_pingpong_kernel(GemmArgs a) {
    using raw = typename T::raw;
    static_assert(sizeof(raw) == 2, "16-bit operands");
    constexpr int BM = 256, BN = 256, BK = 64, GT = 256;
    constexpr int WTM = 128, WTN = 64, FM = 8, FN = 4;
    constexpr int STA = BM * 8, STB = BN * 8;        // 16-byte slots per stage
    constexpr int A_PT = STA / GT, B_PT = STB / GT;  // DMA per group-A thread per step
    constexpr int NBLK = BN / 16, BLK_MASK = 7;
    __shared__ u32x4 sbuf[2 * (STA + STB)];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool grpB = wave >= 4;
    const int wm = wave >> 2, wn = wave & 3;
    const int lrow = lane & 15, lgrp = lane >> 4;
    int tm, tn;
    tile_coords(blockIdx.x, a.tiles_m, a.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int bz = blockIdx.y;
    const raw* __restrict__ Ap = static_cast<const raw*>(a.A) + bz * a.sa_b;
    const raw* __restrict__ Bp = static_cast<const raw*>(a.B) + bz * a.sb_b;
    const int KT = a.k / BK;
    u32x4* sA = sbuf;
    u32x4* sB = sbuf + 2 * STA;

    // DMA slot i*256 + t of a stage (t < 256: group A)
    const int t = tid & (GT - 1);
    uint32_t offA, offB0, offB1;
    {
        const int r0 = t >> 3;
        const int c = swz_dma(r0, t & 7);
        offA = (uint32_t)(((int64_t)(m0 + r0) * a.rsa + c * 8) * 2);
        if constexpr (NN) {
            // columns past N (a partial last tile column) re-read the last 16 (never stored)
            const int kr = t / (2 * NBLK), ps = t % (2 * NBLK);
            const int lb0 = nn_blk(kr, ps >> 1, BLK_MASK), lb1 = nn_blk(kr + 8, ps >> 1, BLK_MASK);
            offB0 = (uint32_t)(((int64_t)kr * a.rsb + min(n0 + lb0 * 16, a.n - 16) + (ps & 1) * 8) * 2);
            offB1 = (uint32_t)(((int64_t)kr * a.rsb + min(n0 + lb1 * 16, a.n - 16) + (ps & 1) * 8) * 2);
        } else {
            offB0 = offB1 = (uint32_t)(((int64_t)(n0 + r0) * a.csb + c * 8) * 2);
        }
    }
    const uint32_t ldsA = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)&sA[(wave & 3) * 64]);
    const uint32_t ldsB = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)&sB[(wave & 3) * 64]);
    // the DMA of step kt: A's slice, then B's
    auto issueA = [&](int kt) {
        const int st = kt & 1;
        const char* bA = reinterpret_cast<const char*>(Ap) + (int64_t)kt * BK * 2;
#pragma unroll
        for (int i = 0; i < A_PT; ++i)
            dma16_soff(bA + (int64_t)i * 32 * a.rsa * 2, offA, ldsA + (uint32_t)(st * STA + i * GT) * 16u);
    };
    auto issueB = [&](int kt) {
        const int st = kt & 1;
        const char* bB = reinterpret_cast<const char*>(Bp) + (int64_t)kt * BK * (NN ? a.rsb : (int64_t)1) * 2;
#pragma unroll
        for (int i = 0; i < B_PT; ++i) {
            const int64_t step = NN ? (int64_t)i * 8 * a.rsb * 2 : (int64_t)i * 32 * a.csb * 2;
            dma16_soff(bB + step, (i & 1) ? offB1 : offB0, ldsB + (uint32_t)(st * STB + i * GT) * 16u);
        }
    };
    // half hf of A's or B's slice of step kt
    auto issueAh = [&](int kt, int hf) {
        const int st = kt & 1;
        const char* bA = reinterpret_cast<const char*>(Ap) + (int64_t)kt * BK * 2;
#pragma unroll
        for (int i = hf * (A_PT / 2); i < (hf + 1) * (A_PT / 2); ++i)
            dma16_soff(bA + (int64_t)i * 32 * a.rsa * 2, offA, ldsA + (uint32_t)(st * STA + i * GT) * 16u);
    };
    auto issueBh = [&](int kt, int hf) {
        const int st = kt & 1;
        const char* bB = reinterpret_cast<const char*>(Bp) + (int64_t)kt * BK * (NN ? a.rsb : (int64_t)1) * 2;
#pragma unroll
        for (int i = hf * (B_PT / 2); i < (hf + 1) * (B_PT / 2); ++i) {
            const int64_t step = NN ? (int64_t)i * 8 * a.rsb * 2 : (int64_t)i * 32 * a.csb * 2;
            dma16_soff(bB + step, (i & 1) ? offB1 : offB0, ldsB + (uint32_t)(st * STB + i * GT) * 16u);
        }
    };
    auto ldA = [&](const u32x4* s, int ks, int i) -> u32x4 {
        const int r = wm * WTM + i * 16 + lrow;
        return s[r * 8 + swz_dma(r, ks * 4 + lgrp)];
    };
    auto ldB = [&](const u32x4* s, int ks, int j) -> u32x4 {
        if constexpr (!NN) {
            const int r = wn * WTN + j * 16 + lrow;
            return s[r * 8 + swz_dma(r, ks * 4 + lgrp)];
        } else {
            const int nb = (wn * WTN + j * 16) >> 4;
            u32x4 v;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = ks * 32 + 8 * lgrp + 4 * h + (lrow >> 2);
                const int byte = r * (BN * 2) + (nn_blk(r, nb, BLK_MASK) << 5) + 8 * (lrow & 3);
                const u32x2 w = lds_read_tr16(s, byte);
                v[2 * h] = w[0];
                v[2 * h + 1] = w[1];
            }
            return v;
        }
    };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 fa[2][FM], fb[2][FN];
    // the fragments of step kt's 32-wide k chunk ks
    auto Xk = [&](int kt, int ks) {
        const u32x4* cA = sA + (kt & 1) * STA;
        const u32x4* cB = sB + (kt & 1) * STB;
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[ks][j] = ldB(cB, ks, j);
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[ks][i] = ldA(cA, ks, i);
    };
    auto X = [&](int kt) {
        Xk(kt, 0);
        Xk(kt, 1);
    };
    auto XB = [&](int kt, int ks) {
        const u32x4* cB = sB + (kt & 1) * STB;
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[ks][j] = ldB(cB, ks, j);
    };
    auto XA = [&](int kt, int ks) {
        const u32x4* cA = sA + (kt & 1) * STA;
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[ks][i] = ldA(cA, ks, i);
    };
    // the MFMA order of gemm_mfma_dma_kernel: per output fragment, k chunk 0 then 1
    auto Y = [&]() {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = mfma_chunk(T{}, fb[ks][j], fa[ks][i], acc[i][j]);
        __builtin_amdgcn_s_setprio(0);
    };
    constexpr int LGKM0 = 0xc07f;  // s_waitcnt lgkmcnt(0), vmcnt and expcnt not waited
    if (!grpB) {
        issueA(0);
        issueB(0);
        for (int kt = 0; kt < KT; ++kt) {
            wait_vmcnt<0>();               // this wave's share of step kt has landed
            __builtin_amdgcn_s_barrier();  // step kt in LDS; group B done with stage (kt+1)&1
            // step kt+1's DMA interleaved with step kt's fragment reads, the same
            // bits. NT: A's slice, the first k chunk, B's slice, the second (4096^3
            // NT 96.7 -> 94.6 us, the LM head 563 -> 559 us). NN, in quarters: half
            // of A's slice before each of the first chunk's B and A fragment reads,
            // then half of B's before the second chunk's (4096^3 NN 98.7 -> 98.0 ->
            // 97.0 us over the two steps)
            const bool nx = kt + 1 < KT;
            if constexpr (NN) {
                if (nx) issueAh(kt + 1, 0);
                XB(kt, 0);
                if (nx) issueAh(kt + 1, 1);
                XA(kt, 0);
                if (nx) issueBh(kt + 1, 0);
                XB(kt, 1);
                if (nx) issueBh(kt + 1, 1);
                XA(kt, 1);
            } else {
                if (nx) issueA(kt + 1);
                Xk(kt, 0);
                if (nx) issueB(kt + 1);
                Xk(kt, 1);
            }
            Y();
        }
    } else {
        for (int kt = 0; kt < KT; ++kt) {
            __builtin_amdgcn_s_barrier();
            if (kt > 0) Y();  // step kt-1, read before the barrier
            X(kt);
            __builtin_amdgcn_s_waitcnt(LGKM0);  // the stage's reads end before group A refills it
        }
        Y();
    }

    using oraw = typename TO::raw;
    oraw* Cp = static_cast<oraw*>(a.C) + bz * a.sc_b;
    if constexpr (sizeof(oraw) == 2) {
        if (a.beta == 0.0f && a.c_line_ok) {
            // Whole 128-byte lines of C. A fragment store writes 32 bytes into each
            // of 16 rows, a quarter of a line per row, and the launch then spends
            // microseconds per tile in the store path (the LM head's 18 rounds of
            // tiles lose ~10% to it). Instead each wave rounds its 128 x 64 tile into
            // 16 KiB of a free operand stage (row r at r * 128 bytes, 16-byte chunk c
            // at c ^ (r & 7)) and stores 8 whole rows per instruction. Group A's waves
            // take the stage no wave reads in the last k step and go at once; group
            // B's take the other one after a barrier that group A meets once its
            // stores are out.
            const int sl = ((KT - 1) & 1) ^ (grpB ? 0 : 1);
            const bool bhalf = (wave & 3) >= 2;  // waves 0, 1, 4, 5 use A's stage, 2, 3, 6, 7 B's
            char* wl = reinterpret_cast<char*>(bhalf ? sB + sl * STB : sA + sl * STA) + (wave & 1) * (WTM * WTN * 2);
            if (grpB) __builtin_amdgcn_s_barrier();
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int r = i * 16 + lrow;
                    const int cb = j * 32 + lgrp * 8;  // byte of the lane's 4 columns in the row
                    *reinterpret_cast<u32x2*>(wl + r * 128 + ((((cb >> 4) ^ (r & 7)) << 4) | (cb & 15))) =
                        u32x2{pack2<TO>(a.alpha * acc[i][j][0], a.alpha * acc[i][j][1]),
                              pack2<TO>(a.alpha * acc[i][j][2], a.alpha * acc[i][j][3])};
                }
            // the wave reads back only its own writes: LDS keeps a wave's accesses in order
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_s_waitcnt(LGKM0);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int q = 0; q < WTM / 8; ++q) {
                const int r = q * 8 + (lane >> 3), c = lane & 7;
                const u32x4 v = *reinterpret_cast<const u32x4*>(wl + r * 128 + ((c ^ (r & 7)) << 4));
                const int n = n0 + wn * WTN + c * 8;  // n % 16 == 0: the 8 columns are all in or all out
                if (n < a.n) *reinterpret_cast<u32x4*>(Cp + (int64_t)(m0 + wm * WTM + r) * a.rsc + n) = v;
            }
            if (!grpB) __builtin_amdgcn_s_barrier();
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = m0 + wm * WTM + i * 16 + lrow;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + wn * WTN + j * 16 + lgrp * 4;
            if (n >= a.n) continue;  // n % 16 == 0: the lane's 4 columns are all in or all out
            oraw* crow = Cp + (int64_t)m * a.rsc;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = a.alpha * acc[i][j][r];
            if (a.beta != 0.0f) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] += a.beta * load_as_f32<TO>(crow, n + r);
            }
            if (a.c_vec_ok) {
                if constexpr (sizeof(oraw) == 2) {
                    *reinterpret_cast<u32x2*>(crow + n) = u32x2{pack2<TO>(v[0], v[1]), pack2<TO>(v[2], v[3])};
                } else {
                    *reinterpret_cast<f32x4*>(crow + n) = f32x4{v[0], v[1], v[2], v[3]};
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) store_from_f32<TO>(crow, n + r, v[r]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Skinny GEMM, M <= 16 (the decode GEMVs: x [1..16, K] . W^T). HBM-bound on
// the weight stream, so the design goal is bytes in flight, not MFMA reuse.
//   NT (W^T, the `linear` layout): gemv_kernel in gemv.hip.
//   NN (B [K][N] row-major): M == 1 in gemv_nn_kernel (16-byte chunks of 8
//   k-rows per load), few fp32 rows in gemm_skinny_nn_kernel, else the tile kernels.
// ---------------------------------------------------------------------------
constexpr int SKINNY_M = 16;
constexpr int SKINNY_WAVES = 8;

// A few fp32 rows (m <= 16) with row-major B: lane = one output column, coalesced row
// loads, 8 waves split k, fp32 sums reduced through LDS. Bound by the weight stream
// at 2 to 4 rows, by the row loads of A above.
__global__ __launch_bounds__(64 * SKINNY_WAVES) void gemm_skinny_nn_kernel(GemmArgs a) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = blockIdx.x * 64 + lane;
    const int bz = blockIdx.y;
    const float* __restrict__ Ap = static_cast<const float*>(a.A) + bz * a.sa_b;
    const float* __restrict__ Bp = static_cast<const float*>(a.B) + bz * a.sb_b;
    const int per_wave = (a.k + SKINNY_WAVES - 1) / SKINNY_WAVES;
    const int k_begin = wave * per_wave, k_end = min(a.k, k_begin + per_wave);
    float acc[SKINNY_M];
#pragma unroll
    for (int i = 0; i < SKINNY_M; ++i) acc[i] = 0.f;
    const bool col = n < a.n;
    const float* bp = Bp + (col ? n : 0);
    constexpr int UNR = 8;
    int k = k_begin;
    for (; k + UNR <= k_end; k += UNR) {
        float b[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) b[u] = col ? bp[(int64_t)(k + u) * a.rsb] : 0.f;
#pragma unroll
        for (int i = 0; i < SKINNY_M; ++i) {
            if (i < a.m) {
#pragma unroll
                for (int u = 0; u < UNR; ++u) acc[i] = fmaf(Ap[(int64_t)i * a.rsa + k + u], b[u], acc[i]);
            }
        }
    }
    for (; k < k_end; ++k) {
        const float b = col ? bp[(int64_t)k * a.rsb] : 0.f;
#pragma unroll
        for (int i = 0; i < SKINNY_M; ++i)
            if (i < a.m) acc[i] = fmaf(Ap[(int64_t)i * a.rsa + k], b, acc[i]);
    }
    __shared__ float red[SKINNY_WAVES][SKINNY_M][64];
#pragma unroll
    for (int i = 0; i < SKINNY_M; ++i) red[wave][i][lane] = acc[i];
    __syncthreads();
    if (wave != 0 || !col) return;
    for (int i = 0; i < a.m; ++i) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < SKINNY_WAVES; ++w) t += red[w][i][lane];
        float* crow = static_cast<float*>(a.C) + bz * a.sc_b + (int64_t)i * a.rsc;
        float v = a.alpha * t;
        if (a.beta != 0.0f) v += a.beta * crow[n];
        crow[n] = v;
    }
}

// M == 1 with row-major B [K][N] (the configs' weight layout): a workgroup owns
// CPR * VEC consecutive columns (CPR 16-byte chunks of a k-row); its 16 waves
// split K, and within a wave lane (r, c) = (lane / CPR, lane % CPR) reads chunk c
// of k-rows r, r + 64/CPR, ... (all of a wave's loads issued before the first
// use). CPR is chosen so the grid covers the CUs: narrower column tiles read
// shorter row pieces but keep more CUs streaming. Per lane VEC fp32 partials in
// k order, a butterfly over the row lanes, then a fixed-order sum of the 16
// waves' partials in LDS.
template <class T, class TO, int CPR>
__global__ __launch_bounds__(1024) void gemv_nn_kernel(GemmArgs a) {
    using raw = typename T::raw;
    constexpr int VEC = 16 / sizeof(raw), WAVES = 16, UNR = 8, RPI = 64 / CPR;  // k-rows per load
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane % CPR, r = lane / CPR;
    // column tiles t..t+T/8-1 on one XCD (workgroups are dealt to the 8 XCDs
    // round-robin): tiles narrower than a 128-byte line share its fetch in one L2
    int tile = blockIdx.x;
    if ((gridDim.x & 7) == 0) tile = (tile & 7) * (gridDim.x >> 3) + (tile >> 3);
    const int n0 = tile * CPR * VEC;
    const int bz = blockIdx.y;
    const raw* __restrict__ Ap = static_cast<const raw*>(a.A) + bz * a.sa_b;
    const raw* __restrict__ Bp = static_cast<const raw*>(a.B) + bz * a.sb_b + n0 + c * VEC;
    const bool col = n0 + c * VEC < a.n;  // the host guarantees n % VEC == 0
    const int kper = ((a.k + WAVES - 1) / WAVES + RPI - 1) / RPI * RPI;
    const int kb = wave * kper, ke = min(a.k, kb + kper);
    float acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
    for (int k0 = kb; k0 < ke; k0 += RPI * UNR) {
        u32x4 w[UNR];
        float x[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int kk = k0 + RPI * u + r;
            const bool ok = col && kk < ke;
            w[u] = ok ? __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(Bp + (int64_t)kk * a.rsb))
                      : u32x4{0u, 0u, 0u, 0u};
            x[u] = kk < ke ? load_as_f32<T>(Ap, kk) : 0.f;
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            if constexpr (sizeof(raw) == 2) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t we = w[u][e];
                    acc[2 * e] = fmaf(x[u], lo_as_f32(T{}, we), acc[2 * e]);
                    acc[2 * e + 1] = fmaf(x[u], hi_as_f32(T{}, we), acc[2 * e + 1]);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = fmaf(x[u], __uint_as_float(w[u][e]), acc[e]);
            }
        }
    }
#pragma unroll
    for (int off = CPR; off < 64; off <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
    __shared__ float red[WAVES][CPR * VEC];
    if (r == 0) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) red[wave][c * VEC + e] = acc[e];
    }
    __syncthreads();
    if (tid >= CPR * VEC) return;
    const int n = n0 + tid;
    if (n >= a.n) return;
    float t = 0.f;
#pragma unroll
    for (int w2 = 0; w2 < WAVES; ++w2) t += red[w2][tid];
    using oraw = typename TO::raw;
    oraw* crow = static_cast<oraw*>(a.C) + bz * a.sc_b;
    float v = a.alpha * t;
    if (a.beta != 0.0f) v += a.beta * load_as_f32<TO>(crow, n);
    store_from_f32<TO>(crow, n, v);
}

// fp32 GEMM on v_mfma_f32_16x16x4_f32 with DMA-staged tiles (configs[0], the
// reference's sgemm_rowmajor, src/kernel/avx2/sgemm.inl:268-340, and its
// transposed-B forms). Block tile BM x BN, k step BK = 32 (one 128-byte row of
// fp32), an LDS ring of STAGES steps filled by global_load_lds (two in flight
// ahead of the one being computed with 4 stages). Operands are swapped
// (src0 = B^T fragment, src1 = A fragment) so lane l holds C[m = l % 16][n =
// 4 g + 0..3], g = l / 16: one 16-byte store per output fragment.
//   A tile [BM rows][8 chunks of 16 B]: chunk c of row r at c ^ (r & 7); the
//     fragment of a 16-wide k block kb is one ds_read_b128 (chunk 4 kb + g) per
//     lane feeding 4 MFMAs.
//   B, NT (B = W^T, W [n][k] rows): the same layout as A.
//   B, NN (row-major [k][n]): [BK rows][BN / 4 chunks], chunk c of k-row r at
//     c ^ (((r >> 2) & 3) << 2); MFMA step j of lane group g reads k-row
//     16 kb + 4 g + j, one ds_read_b32 of n = 16 fn + l % 16: the four groups'
//     rows land in four bank ranges.
// Rows of A / B past m / n re-read the last row (never stored); k % 4 == 0.
template <int BM, int BN, int WM, int WN, bool NN, int STAGES, bool MASK>
__global__ __launch_bounds__(64 * WM * WN) void gemm_f32_kernel(GemmArgs a) {
    constexpr int THREADS = 64 * WM * WN;
    constexpr int BK = 32;
    static_assert(STAGES >= 3, "the ring keeps two k steps in flight");
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int STA = BM * 8;                        // 16-byte chunks of an A stage
    constexpr int STB = NN ? BK * (BN / 4) : BN * 8;   // ... of a B stage
    constexpr int A_PT = STA / THREADS, B_PT = STB / THREADS;
    static_assert(A_PT * THREADS == STA && B_PT * THREADS == STB, "tile / thread mismatch");
    static_assert(!NN || BN >= 64, "the NN swizzle needs 16 chunks per k-row");
    constexpr int PER = A_PT + B_PT;
    __shared__ u32x4 sA[STAGES * STA];
    __shared__ u32x4 sB[STAGES * STB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;
    int tm, tn;
    tile_coords(blockIdx.x, a.tiles_m, a.tiles_n, tm, tn);
    const int bz = blockIdx.y;
    const int m0 = tm * BM, n0 = tn * BN;
    const float* Ap = static_cast<const float*>(a.A) + bz * a.sa_b;
    const float* Bp = static_cast<const float*>(a.B) + bz * a.sb_b;

    // DMA element offsets within a k step (the base moves by BK along k)
    int aoff[A_PT], boff[B_PT];  // source chunk of each DMA slot
    int64_t arow[A_PT];
#pragma unroll
    for (int i = 0; i < A_PT; ++i) {
        const int slot = i * THREADS + tid;
        const int row = slot / 8, c = slot % 8;
        aoff[i] = c ^ (row & 7);
        arow[i] = (int64_t)min(m0 + row, a.m - 1) * a.rsa;
    }
    int64_t bbase[B_PT];
#pragma unroll
    for (int i = 0; i < B_PT; ++i) {
        const int slot = i * THREADS + tid;
        if constexpr (NN) {
            constexpr int BCH = BN / 4;
            const int row = slot / BCH, c = slot % BCH;   // k-row, n chunk
            const int src = c ^ (((row >> 2) & 3) << 2);
            const int nn = min(n0 + 4 * src, a.n - 4);    // n % 4 == 0 on this path
            bbase[i] = (int64_t)row * a.rsb + nn;
            boff[i] = 0;
        } else {
            const int row = slot / 8, c = slot % 8;       // n-row, k chunk
            bbase[i] = (int64_t)min(n0 + row, a.n - 1) * a.csb;
            boff[i] = (c ^ (row & 7)) * 4;
        }
    }
    // A ragged k makes the first step short, as in gemm_mfma_dma_kernel. (A form without it gains 1% NT,
    // 0.5% NN and loses 4% at 2048 x 768 x 4672 NT.)
    const int nks_all = (a.k + BK - 1) / BK;
    const int first = a.k - (nks_all - 1) * BK;
    const int nks = MASK && hidden_tile(a.mask, min(m0 + BM, a.m) - 1, n0) ? 1 : nks_all;
    auto issue = [&](int ks) {
        const int k0 = ks == 0 ? 0 : ks * BK - (BK - first);
        u32x4* dA = sA + (ks % STAGES) * STA;
        u32x4* dB = sB + (ks % STAGES) * STB;
#pragma unroll
        for (int i = 0; i < A_PT; ++i) {
            const float* p = Ap + arow[i] + k0 + aoff[i] * 4;
            if (ks == 0 && aoff[i] * 4 >= first) p = reinterpret_cast<const float*>(dma_zero);
            dma16_async(p, &dA[i * THREADS + wave * 64]);
        }
#pragma unroll
        for (int i = 0; i < B_PT; ++i) {
            const float* p = Bp + bbase[i] + (NN ? (int64_t)k0 * a.rsb : (int64_t)k0 + boff[i]);
            const int bk = NN ? (i * THREADS + tid) / (BN / 4) : boff[i];  // the chunk's (first) k in the step
            if (ks == 0 && bk >= first) p = reinterpret_cast<const float*>(dma_zero);
            dma16_async(p, &dB[i * THREADS + wave * 64]);
        }
    };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = f32x4{0.f, 0.f, 0.f, 0.f};

    constexpr int AHEAD = STAGES - 1;  // steps issued before the first one is computed
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
        if (i < nks) issue(i);
    for (int ks = 0; ks < nks; ++ks) {
        // this thread's DMA of step ks has landed (the later steps' may still fly)
        const int later = min(nks - 1 - ks, AHEAD - 1);
        if (later >= 2) wait_vmcnt<2 * PER>();
        else if (later == 1) wait_vmcnt<PER>();
        else wait_vmcnt<0>();
        __syncthreads();
        if (ks + AHEAD < nks) issue(ks + AHEAD);
        const u32x4* cA = sA + (ks % STAGES) * STA;
        const u32x4* cB = sB + (ks % STAGES) * STB;
        const float* cBf = reinterpret_cast<const float*>(cB);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            f32x4 af[FM];
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) {
                const int row = wm * WTM + fm * 16 + r16;
                af[fm] = __builtin_bit_cast(f32x4, cA[row * 8 + ((4 * kb + g) ^ (row & 7))]);
            }
            if constexpr (!NN) {
                f32x4 bf[FN];
#pragma unroll
                for (int fn = 0; fn < FN; ++fn) {
                    const int row = wn * WTN + fn * 16 + r16;
                    bf[fn] = __builtin_bit_cast(f32x4, cB[row * 8 + ((4 * kb + g) ^ (row & 7))]);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                        for (int fn = 0; fn < FN; ++fn)
                            acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[fn][j], af[fm][j], acc[fm][fn], 0, 0, 0);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int krow = 16 * kb + 4 * g + j;  // (krow >> 2) & 3 == g
                    float bf[FN];
#pragma unroll
                    for (int fn = 0; fn < FN; ++fn) {
                        const int nl = wn * WTN + fn * 16 + r16;  // n within the tile
                        const int ch = (nl >> 2) ^ (g << 2);
                        bf[fn] = cBf[krow * BN + ch * 4 + (nl & 3)];
                    }
#pragma unroll
                    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                        for (int fn = 0; fn < FN; ++fn)
                            acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[fn], af[fm][j], acc[fm][fn], 0, 0, 0);
                }
            }
        }
    }
    // epilogue: lane holds C[m0 + wm WTM + 16 fm + l % 16][n0 + wn WTN + 16 fn + 4 g + i]
    float* Cp = static_cast<float*>(a.C) + bz * a.sc_b;
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
        const int m = m0 + wm * WTM + fm * 16 + r16;
        if (m >= a.m) continue;
        float* crow = Cp + (int64_t)m * a.rsc;
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
            const int n = n0 + wn * WTN + fn * 16 + 4 * g;
            f32x4 v = acc[fm][fn] * a.alpha;
            if constexpr (MASK) {
                if (n < a.n) masked_store4<F32>(a.mask, crow, 1, m, n, a.n, v, a.beta);
                continue;
            }
            if (a.c_vec_ok && n + 3 < a.n) {
                if (a.beta != 0.0f) v += a.beta * *reinterpret_cast<const f32x4*>(crow + n);
                *reinterpret_cast<f32x4*>(crow + n) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < a.n) crow[n + i] = a.beta != 0.0f ? v[i] + a.beta * crow[n + i] : v[i];
            }
        }
    }
}

// C = beta * C (k == 0 or alpha == 0), sgemm.inl:594-604.
template <class TO>
__global__ __launch_bounds__(256) void gemm_scale_kernel(void* C, int m, int n, int64_t rsc, int64_t csc,
                                                         int64_t sc_b, float beta) {
    const int j = blockIdx.x * 16 + (threadIdx.x & 15);
    const int i = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (i >= m || j >= n) return;
    const int64_t co = blockIdx.z * sc_b + i * rsc + j * csc;
    const float v = (beta == 0.0f) ? 0.0f : beta * load_as_f32<TO>(C, co);
    store_from_f32<TO>(C, co, v);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
namespace {

template <class T, class TO, int BM, int BN, int WM, int WN, int STAGES, bool SOFF = true, int FORM = PLAIN>
hipError_t launch_dma_tile(const GemmArgs& a0, bool nn, int batch, hipStream_t s) {
    GemmArgs a = a0;
    a.tiles_m = (a.m + BM - 1) / BM;
    a.tiles_n = (a.n + BN - 1) / BN;
    dim3 grid(a.tiles_m * a.tiles_n, batch);
    dim3 block(64 * WM * WN);
    auto launch = [&](auto ragged) {
        constexpr bool R = decltype(ragged)::value;
        if (nn) gemm_mfma_dma_kernel<T, TO, BM, BN, WM, WN, true, STAGES, SOFF, FORM, R><<<grid, block, 0, s>>>(a);
        else gemm_mfma_dma_kernel<T, TO, BM, BN, WM, WN, false, STAGES, SOFF, FORM, R><<<grid, block, 0, s>>>(a);
    };
    constexpr int BK = 128 / sizeof(typename T::raw);
    if constexpr (FORM == PLAIN) {
        if (a.k % BK == 0) launch(std::false_type{});
        else launch(std::true_type{});
    } else {
        launch(std::true_type{});
    }
    return hipGetLastError();
}

// 16-bit operands that span 2^31 bytes or more
bool dma_far(int m, int n, int k, int64_t rsa, int64_t rsb, int64_t csb, bool nn) {
    const int64_t span_a = ((int64_t)(m - 1) * rsa + k) * 2;
    const int64_t span_b = (nn ? (int64_t)(k - 1) * rsb + n : (int64_t)(n - 1) * csb + k) * 2;
    return span_a >= (int64_t(1) << 31) || span_b >= (int64_t(1) << 31);
}
bool dma_far(const GemmArgs& a, bool nn) { return dma_far(a.m, a.n, a.k, a.rsa, a.rsb, a.csb, nn); }

template <class T, class TO>
hipError_t launch_dma(const GemmArgs& a, bool nn, int batch, hipStream_t s) {
    auto tiles = [&](int bm, int bn) {
        return (int64_t)((a.m + bm - 1) / bm) * ((a.n + bn - 1) / bn) * batch;
    };
    // bytes spanned by one batch entry's A and B: below 2^31 the DMA goes from a
    // scalar base plus 32-bit lane offsets
    const bool far = dma_far(a, nn);
    auto cost = [&](int bm, int bn) { return (tiles(bm, bn) + 255) / 256 * (bm + bn); };
    if (a.mask.kind != YTHIP_MASK_NONE) {  // (the caller sends far operands elsewhere)
        if (cost(128, 128) < cost(64, 64)) return launch_dma_tile<T, TO, 128, 128, 2, 4, 4, true, MASKED>(a, nn, batch, s);
        return launch_dma_tile<T, TO, 64, 64, 2, 2, 4, true, MASKED>(a, nn, batch, s);
    }
    if (far) {
        if (tiles(256, 256) >= 192) return launch_dma_tile<T, TO, 256, 256, 2, 4, 2, false>(a, nn, batch, s);
        if (tiles(128, 128) >= 256) return launch_dma_tile<T, TO, 128, 128, 2, 2, 2, false>(a, nn, batch, s);
        return launch_dma_tile<T, TO, 64, 64, 2, 2, 4, false>(a, nn, batch, s);
    }
    if (tiles(256, 256) >= 192) {
        // whole 256-row tiles: the ping-pong schedule (same bits). NT with a partial
        // last column of tiles: the whole tiles on the ping-pong kernel, the last
        // N % 256 columns as a product of their own (disjoint columns of C; B rows
        // and C columns offset).
        if (a.m % 256 == 0 && a.k % 64 == 0) {
            if (!nn && a.n % 256 != 0 && a.n > 256) {
                using oraw = typename TO::raw;
                GemmArgs g = a;
                g.n = a.n / 256 * 256;
                g.tiles_m = a.m / 256;
                g.tiles_n = g.n / 256;
                gemm_pingpong_kernel<T, TO, false><<<dim3(g.tiles_m * g.tiles_n, batch), 512, 0, s>>>(g);
                const hipError_t e = hipGetLastError();
                if (e != hipSuccess) return e;
                GemmArgs r = a;
                r.n = a.n - g.n;
                r.B = static_cast<const typename T::raw*>(a.B) + (int64_t)g.n * a.csb;
                r.C = static_cast<oraw*>(a.C) + g.n;
                return launch_dma<T, TO>(r, nn, batch, s);
            }
            if (nn ? a.n % 16 == 0 : a.n % 256 == 0) {
                GemmArgs g = a;
                g.tiles_m = a.m / 256;
                g.tiles_n = (a.n + 255) / 256;
                const dim3 grid(g.tiles_m * g.tiles_n, batch);
                if (nn) gemm_pingpong_kernel<T, TO, true><<<grid, 512, 0, s>>>(g);
                else gemm_pingpong_kernel<T, TO, false><<<grid, 512, 0, s>>>(g);
                return hipGetLastError();
            }
        }
        return launch_dma_tile<T, TO, 256, 256, 2, 4, 2>(a, nn, batch, s);
    }
    // Every tile's k loop runs at about the same bytes a clock into its CU's LDS
    // (20 to 27, one workgroup or several), so the time is what the busiest CU
    // stages: passes over the 256 CUs times BM + BN rows a k step. The smallest wins,
    // the smaller tile when even (its ramp is shorter). Measured on bf16, the rule's
    // tile against the one of a rule by tile counts that stood here: 2048^3 NN 24.0 /
    // 31.3 us, 2400^3 40.5 / 62.9, 1536^3 16.2 / 19.1, 2048 x 1024 x 3072 NT 23.4 / 24.6
    // (weights from HBM 25.1 / 29.5); as graph nodes 512 x 6144 x 1024 NT 10.9 / 10.1 (12.8 / 15.1),
    // 512 x 4096 x 1024 NT 8.3 / 8.0 (9.7 / 11.0). A ring deeper than 4 steps loses at
    // every size (512 x 1024 x 3072: 13.6, 8 deep 14.8, 12 deep 17.6 us).
    const int64_t c0 = cost(64, 32), c1 = cost(64, 64), c2 = cost(128, 64), c3 = cost(128, 128);
    // The 256-wide tiles of a small matrix in a batch share little of the XCDs' L2s, and lose
    // more by it than the smaller ones do: 256 x 128 / 128 x 128 NT at 32 tiles a matrix (8 x 1024 x 1024 x
    // 1024) 26.3 / 20.5 us, at 60 (4 x 1280 x 1536 x 640) 15.4 / 14.4, at 72 (3 x 1500 x 1500 x 1504)
    // 26.6 / 28.4, at 100 (2 x 2560 x 1280 x 1280) 20.8 / 22.2.
    const int64_t c4 = batch == 1 || tiles(256, 128) >= 72 * (int64_t)batch ? cost(256, 128) : INT64_MAX;
    const int64_t best = std::min(std::min(std::min(c0, c1), std::min(c2, c3)), c4);
    if (c0 == best) return launch_dma_tile<T, TO, 64, 32, 2, 1, 4>(a, nn, batch, s);
    if (c1 == best) return launch_dma_tile<T, TO, 64, 64, 2, 2, 4>(a, nn, batch, s);
    if (c2 == best) {
        // one per CU: eight waves and a deep ring, as four waves with two steps in flight leave
        // the CU waiting. Two resident 64 x 64 tiles / one 128 x 64 of four waves / of eight, NT, weights
        // from HBM: 200 x 6144 x 1024 10.1 / 10.2 / 8.8 us, 448 x 4096 x 1024 11.0 / 10.2 / 9.0; weights that
        // stay cached: 7.2 / 8.8 / 7.9 and 7.6 / 9.1 / 8.2
        if (tiles(128, 64) <= 256) return launch_dma_tile<T, TO, 128, 64, 4, 2, 4>(a, nn, batch, s);
        return launch_dma_tile<T, TO, 128, 64, 2, 2, 3>(a, nn, batch, s);
    }
    if (c3 == best) {
        // one per CU: eight waves and a deep ring; several: two resident per CU
        // (3072^3: 75.9 us, 80.2 with the deep ring)
        if (tiles(128, 128) <= 256) return launch_dma_tile<T, TO, 128, 128, 2, 4, 4>(a, nn, batch, s);
        return launch_dma_tile<T, TO, 128, 128, 2, 2, 2>(a, nn, batch, s);
    }
    return launch_dma_tile<T, TO, 256, 128, 2, 4, 3>(a, nn, batch, s);
}

template <class TO>
hipError_t launch_scale(void* C, int m, int n, int64_t rsc, int64_t csc, int64_t sc_b, float beta, int batch,
                        hipStream_t s) {
    dim3 grid((n + 15) / 16, (m + 15) / 16, batch);
    gemm_scale_kernel<TO><<<grid, 256, 0, s>>>(C, m, n, rsc, csc, sc_b, beta);
    return hipGetLastError();
}

// Few fp32 rows against a row-major B: the tile kernel walks the whole k in one chain of
// 32-wide steps whatever the rows, 18.5 ns per k and pass over the CUs; the skinny kernel
// cuts k over 8 waves and pays per row, more once A no longer stays in the caches that the
// workgroups of an XCD share. Fitted to 770 products (k 256 to 8192, n 36 to 40000, 2 to 16
// rows, batches of 8 and 64). Skinny / tiles, us, k = 8192: n = 64, 2 rows 82 / 153, 8 rows 135 / 153;
// n = 8192, 4 rows 150 / 155, 8 rows 223 / 155; n = 40000, 8 rows 283 / 436.
bool skinny_nn_pays(int m, int n, int k, int batch) {
    const int64_t tiles = (int64_t)((n + 63) / 64) * batch, passes = (tiles + 255) / 256;
    double row = 1.15;  // ns per k and row
    if (tiles * k > 65536 && (int64_t)m * k > 3072) {
        row = batch == 1 && passes > 1 && k <= 2048 ? 1.8 : 2.2;
        if (batch > 1) row *= std::min(1.6, std::max(1.0, tiles / 330.0));
    }
    return 8.0 + 7.0 * (passes - 1) + row * m <= (passes < 4 ? 18.5 : 20.5) * passes;
}

bool aligned(const void* p, int bytes) { return (reinterpret_cast<uintptr_t>(p) % bytes) == 0; }

// The operand forms that the aligned kernels take: A's rows in 16-byte chunks, B as [n][k]
// rows (nt), as [k][n] rows in pieces of 4 (nn) or in 16-byte chunks (nn16).
struct Forms {
    bool a, nt, nn, nn16;
};
Forms forms_of(int es, int n, int k, const void* A, int64_t sa_b, int64_t rsa, int64_t csa, const void* B, int64_t sb_b,
               int64_t rsb, int64_t csb) {
    const int vec = 16 / es;
    Forms f;
    f.a = csa == 1 && rsa % vec == 0 && sa_b % vec == 0 && aligned(A, 16) && k % vec == 0;
    f.nt = rsb == 1 && csb % vec == 0 && sb_b % vec == 0 && aligned(B, 16);
    f.nn = !f.nt && csb == 1 && rsb % 4 == 0 && sb_b % 4 == 0 && n % 4 == 0 && aligned(B, 4 * es);
    f.nn16 = f.nn && rsb % vec == 0 && sb_b % vec == 0 && n % vec == 0 && aligned(B, 16);
    return f;
}

template <class T, class TO>
int gemm_typed(int batch, int m, int n, int k, const void* A, int64_t sa_b, int64_t rsa, int64_t csa,
               const void* B, int64_t sb_b, int64_t rsb, int64_t csb, void* C, int64_t sc_b, int64_t rsc,
               int64_t csc, float alpha, float beta, const MaskDesc& mask, hipStream_t s) {
    using raw = typename T::raw;
    using oraw = typename TO::raw;
    constexpr int VEC = 16 / sizeof(raw);
    const bool plain = mask.kind == YTHIP_MASK_NONE;
    if (k == 0 || alpha == 0.0f) return status_of(launch_scale<TO>(C, m, n, rsc, csc, sc_b, beta, batch, s));

    const Forms fo = forms_of(sizeof(raw), n, k, A, sa_b, rsa, csa, B, sb_b, rsb, csb);
    const bool nt = fo.nt, nn = fo.nn;
    if (fo.a && (nt || nn) && csc == 1) {
        GemmArgs g{};
        g.A = A; g.B = B; g.C = C;
        g.m = m; g.n = n; g.k = k;
        g.rsa = rsa; g.rsb = rsb; g.csb = csb; g.rsc = rsc;
        g.sa_b = sa_b; g.sb_b = sb_b; g.sc_b = sc_b;
        g.alpha = alpha; g.beta = beta;
        g.c_vec_ok = (rsc % 4 == 0) && (sc_b % 4 == 0) && aligned(C, 4 * sizeof(oraw));
        g.c_line_ok = sizeof(oraw) == 2 && (rsc % 8 == 0) && (sc_b % 8 == 0) && aligned(C, 16);
        g.mask = mask;
        if (m <= SKINNY_M && plain) {
            if (nt) {
                GemvArgs v{};
                v.A = A; v.lda = rsa; v.W = B; v.ldw = csb; v.C = C; v.ldc = rsc;
                v.sa_b = sa_b; v.sw_b = sb_b; v.sc_b = sc_b;
                v.m = m; v.n = n; v.k = k; v.alpha = alpha; v.beta = beta;
                return gemv_dispatch(0, T::code, TO::code, v, batch, s);
            }
            if (m == 1 && fo.nn16) {
                auto tiles = [&](int cpr) { return (int64_t)((n + cpr * VEC - 1) / (cpr * VEC)) * batch; };
                // >= 192 workgroups: (1, 3072, 1024) 8.0 us with 96 workgroups of 32
                // columns, 7.1 us with 192 of 16 (XCD-remapped, lines shared in L2)
                if (tiles(8) >= 192)
                    gemv_nn_kernel<T, TO, 8><<<dim3((n + 8 * VEC - 1) / (8 * VEC), batch), 1024, 0, s>>>(g);
                else if (tiles(4) >= 192)
                    gemv_nn_kernel<T, TO, 4><<<dim3((n + 4 * VEC - 1) / (4 * VEC), batch), 1024, 0, s>>>(g);
                else
                    gemv_nn_kernel<T, TO, 2><<<dim3((n + 2 * VEC - 1) / (2 * VEC), batch), 1024, 0, s>>>(g);
                return status_of(hipGetLastError());
            }
            // 2..16 rows of a row-major fp32 B: see skinny_nn_pays
            if constexpr (std::is_same_v<T, F32>)
                if (nn && skinny_nn_pays(m, n, k, batch)) {
                    gemm_skinny_nn_kernel<<<dim3((n + 63) / 64, batch), 64 * SKINNY_WAVES, 0, s>>>(g);
                    return status_of(hipGetLastError());
                }
            // 2..16 rows of a row-major, 16-bit B: the MFMA DMA path (one partial
            // 64-row tile per column tile) streams B at full width
            if constexpr (sizeof(raw) == 2)
                if (fo.nn16) return status_of(launch_dma<T, TO>(g, true, batch, s));
        }
        if constexpr (std::is_same_v<T, F32> && std::is_same_v<TO, F32>) {
            // fp32 on the DMA-staged fp32 MFMA kernel: 16-byte aligned rows of A and
            // of B (NT) or B's k-rows (NN). 1000^3: 37.8 us on the register-staged
            // kernel that took k % 32 != 0 before, 24.6 us here
            const bool f_nn = fo.nn16;
            if (nt || f_nn) {
                auto ntiles = [&](int bm, int bn) { return (int64_t)((m + bm - 1) / bm) * ((n + bn - 1) / bn) * batch; };
                const bool big = ntiles(128, 128) >= 512;
                GemmArgs f = g;
                f.tiles_m = (m + (big ? 127 : 63)) / (big ? 128 : 64);
                f.tiles_n = (n + (big ? 127 : 63)) / (big ? 128 : 64);
                const dim3 grid(f.tiles_m * f.tiles_n, batch);
                // 1024^3 (256 tiles of 64 x 64): 8 waves of 32 x 16 and a 4-step ring,
                // 99 TFLOP/s NN; 4 waves or 3 steps 86-98, 32 x 64 or 64 x 128 tiles <= 92
                auto launch = [&](auto masked) {
                    constexpr bool M = decltype(masked)::value;
                    if (big) {
                        if (f_nn) gemm_f32_kernel<128, 128, 2, 4, true, 3, M><<<grid, 512, 0, s>>>(f);
                        else gemm_f32_kernel<128, 128, 2, 4, false, 3, M><<<grid, 512, 0, s>>>(f);
                    } else {
                        if (f_nn) gemm_f32_kernel<64, 64, 2, 4, true, 4, M><<<grid, 512, 0, s>>>(f);
                        else gemm_f32_kernel<64, 64, 2, 4, false, 4, M><<<grid, 512, 0, s>>>(f);
                    }
                };
                if (plain) launch(std::false_type{});
                else launch(std::true_type{});
                return status_of(hipGetLastError());
            }
        }
        // DMA-staged fast path: 16-byte aligned rows everywhere, k in whole chunks
        // (k % 64 != 0, 4096 x 4096 x 4072 NN: 228 -> 119 us, 1000^3 17.3 -> 7.8 us
        // against the register-staged kernel that took those before).
        if constexpr (sizeof(raw) == 2)
            if ((nt || fo.nn16) && (plain || !dma_far(g, nn))) return status_of(launch_dma<T, TO>(g, nn, batch, s));
    }
    return gemm_any_dispatch(T::code, TO::code, batch, m, n, k, A, sa_b, rsa, csa, B, sb_b, rsb, csb, C, sc_b, rsc, csc,
                             alpha, beta, mask, s);
}

// C = alpha * sum of the S parts' fp32 products + beta * C, four columns a thread; all
// parts' loads are in flight at once.
template <class TO, int S>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ parts, int64_t mn, int n4,
                                                            void* C, int64_t rsc, float alpha, float beta) {
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id * 4 >= mn) return;
    f32x4 p[S];
#pragma unroll
    for (int s = 0; s < S; ++s) p[s] = *reinterpret_cast<const f32x4*>(parts + s * mn + id * 4);
    f32x4 v = p[0];
#pragma unroll
    for (int s = 1; s < S; ++s) v += p[s];
    const int64_t at = id / n4 * rsc + id % n4 * 4;
    v *= alpha;
    if (beta != 0.0f)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += beta * load_as_f32<TO>(C, at + r);
    auto* c = static_cast<typename TO::raw*>(C) + at;
    if constexpr (sizeof(*c) == 2) *reinterpret_cast<u32x2_any*>(c) = u32x2{pack2<TO>(v[0], v[1]), pack2<TO>(v[2], v[3])};
    else *reinterpret_cast<f32x4_any*>(c) = v;
}

template <class T>
int swiglu_typed(const GemmArgs& a, hipStream_t s) {
    auto cost = [&](int bm, int bn) {
        return ((int64_t)((a.m + bm - 1) / bm) * ((2 * a.n + bn - 1) / bn) + 255) / 256 * (bm + bn);
    };
    auto launch = [&](auto bm, auto bn, auto wm, auto wn, auto stages) {
        GemmArgs g = a;
        g.tiles_m = (a.m + bm.value - 1) / bm.value;
        g.tiles_n = (2 * a.n + bn.value - 1) / bn.value;
        gemm_mfma_dma_kernel<T, T, bm.value, bn.value, wm.value, wn.value, false, stages.value, true, SWIGLU>
            <<<dim3(g.tiles_m * g.tiles_n), 64 * wm.value * wn.value, 0, s>>>(g);
        return status_of(hipGetLastError());
    };
    using std::integral_constant;
#define YT_I(x) integral_constant<int, x> {}
    // the tile rule of launch_dma
    const int64_t c0 = cost(64, 32), c1 = cost(64, 64), c2 = cost(128, 64), c3 = cost(128, 128);
    const int64_t best = std::min(std::min(c0, c1), std::min(c2, c3));
    if (c0 == best) return launch(YT_I(64), YT_I(32), YT_I(2), YT_I(1), YT_I(4));
    if (c1 == best) return launch(YT_I(64), YT_I(64), YT_I(2), YT_I(2), YT_I(4));
    if (c2 == best) return launch(YT_I(128), YT_I(64), YT_I(2), YT_I(2), YT_I(3));
    return launch(YT_I(128), YT_I(128), YT_I(2), YT_I(4), YT_I(4));
#undef YT_I
}

}  // namespace

int gemm_masked_dispatch(int dtype_in, int dtype_out, int batch, int m, int n, int k, const void* A, int64_t sa_b,
                         int64_t rsa, int64_t csa, const void* B, int64_t sb_b, int64_t rsb, int64_t csb, void* C,
                         int64_t sc_b, int64_t rsc, int64_t csc, float alpha, float beta, const MaskDesc& mask,
                         hipStream_t s) {
#define YTHIP_GEMM(TI, TOUT)                                                                                        \
    return gemm_typed<TI, TOUT>(batch, m, n, k, A, sa_b, rsa, csa, B, sb_b, rsb, csb, C, sc_b, rsc, csc, alpha, beta, \
                                mask, s)
    if (dtype_in == YTHIP_F32 && dtype_out == YTHIP_F32) YTHIP_GEMM(F32, F32);
    if (dtype_in == YTHIP_BF16 && dtype_out == YTHIP_BF16) YTHIP_GEMM(BF16, BF16);
    if (dtype_in == YTHIP_BF16 && dtype_out == YTHIP_F32) YTHIP_GEMM(BF16, F32);
    if (dtype_in == YTHIP_F16 && dtype_out == YTHIP_F16) YTHIP_GEMM(F16, F16);
    if (dtype_in == YTHIP_F16 && dtype_out == YTHIP_F32) YTHIP_GEMM(F16, F32);
#undef YTHIP_GEMM
    return fail(YTHIP_EUNSUPPORTED, "ythip_gemm: unsupported dtype_in/dtype_out combination %d/%d", dtype_in,
                dtype_out);
}

// Whether a masked product is faster with the mask in its store than as an fp32 product in
// a workspace and a blend. What the store costs: it exists on 64- and 128-wide tiles only.
//  * m <= 16 rows that the plain product gives to a GEMV kernel: the tile kernel walks k in one
//    chain. 1 x 1024 x 8192 NT, store / workspace: bf16 30 / 16 us, fp32 154 / 16; at k = 1024
//    bf16 10 / 15, fp32 22 / 16. Many columns fill the chip with tiles: bf16 16 x 8192 x 8192 NT 30 / 40.
//  * 16-bit products of 192 and more 256 x 256 tiles: the plain one is the ping-pong kernel (1.54 us
//    a 64-wide step and pass over the CUs, 128 x 128 tiles 0.656), against the blend's own
//    bytes and blocks. bf16 4096^3 NN byte mask kept 152 / 137 us, filled 145 / 137; 8192^3 causal 1031 /
//    898, bytes 1133 / 924; 4096 x 4096 x 1024 bytes 54 / 101. The constants are fitted to 940 products
//    (k 256 to 8192, five mask shapes, kept and filled): none is slower than the workspace form.
//    A diagonal's hidden tiles only help where the busiest XCD, which holds the last eighth of the
//    rows (tile_coords), has some.
//  * operands of 2^31 bytes and more have no masked DMA form; register-staged 64 x 64 tiles
//    re-read both operands per tile (131200 x 256 x 8192 bytes 1092 / 818 us, one row or column
//    of tiles 466 / 637).
//  * aligned operands and a strided C: only the register-staged kernel stores it.
bool gemm_masked_store_pays(int dtype_in, int batch, int m, int n, int k, const void* A, int64_t sa_b, int64_t rsa,
                            int64_t csa, const void* B, int64_t sb_b, int64_t rsb, int64_t csb, int64_t csc,
                            const MaskDesc& mask) {
    if (mask.kind == YTHIP_MASK_NONE) return true;
    const bool f32 = dtype_in == YTHIP_F32;
    const Forms f = forms_of(f32 ? 4 : 2, n, k, A, sa_b, rsa, csa, B, sb_b, rsb, csb);
    if (!f.a || !(f.nt || f.nn16 || (f32 && f.nn))) return true;
    if (m <= SKINNY_M && (f.nt || (m == 1 && f.nn16) || (f32 && skinny_nn_pays(m, n, k, batch))))
        return f32 ? k <= 512 : k <= 2048 || (n > 4096 && !(m == 1 && f.nt));
    if (csc != 1) return false;
    if (f32) return true;
    double share = 1.0;  // visible, of the last eighth of the rows
    if (mask.kind == YTHIP_MASK_CAUSAL || mask.kind == YTHIP_MASK_DIAG) {
        share = 0.0;
        for (int t = 0; t < 16; ++t) {
            const int64_t row = m - 1 - (int64_t)(m / 8) * t / 16;
            share += std::max<int64_t>(0, std::min<int64_t>(n, row + mask.off + 1)) / (16.0 * n);
        }
    }
    if (dma_far(m, n, k, rsa, rsb, csb, f.nn16)) return m <= 64 || n <= 64 || share < 0.7;
    auto tiles = [&](int b) { return (int64_t)((m + b - 1) / b) * ((n + b - 1) / b) * batch; };
    if (tiles(256) < 192) return true;
    const double steps = (k + 63) / 64, cells = (double)batch * m * n;
    const double blocks = (double)batch * m * std::min(8, (n + 255) / 256);
    const double bytes = mask.kind == YTHIP_MASK_BOOL && mask.fill ? 0.6e-6 * cells : 0.0;
    const double blend = 1.83e-6 * cells + 0.848e-3 * blocks + bytes;
    const double store = mask.fill ? 3.3 : mask.kind == YTHIP_MASK_BOOL ? 8.24 : 3.7;  // kept bytes: entry by entry
    return (tiles(128) + 255) / 256 * (0.656 * share * steps + store) <=
           (tiles(256) + 255) / 256 * 1.54 * steps + blend;
}

int gemm_dispatch(int dtype_in, int dtype_out, int batch, int m, int n, int k, const void* A, int64_t sa_b,
                  int64_t rsa, int64_t csa, const void* B, int64_t sb_b, int64_t rsb, int64_t csb, void* C,
                  int64_t sc_b, int64_t rsc, int64_t csc, float alpha, float beta, hipStream_t s) {
    return gemm_masked_dispatch(dtype_in, dtype_out, batch, m, n, k, A, sa_b, rsa, csa, B, sb_b, rsb, csb, C, sc_b, rsc,
                                csc, alpha, beta, MaskDesc{YTHIP_MASK_NONE, nullptr, 0, 0, 0, 0.f}, s);
}

// How many parts k is cut into for a product too small for the chip (1: none). Such a
// grid has at most one 64 x 32 tile per CU and each walks the whole k, one step of about
// 280 ns after the other, whatever the number of rows (64 or 512 x 1024 x 3072: 11.8 and
// 12.6 us). The parts run side by side as a batch of fp32 products, on larger tiles
// where there are rows for them, and a second launch sums them.
int gemm_splits(int m, int n, int k) {
    const int64_t tiles = (int64_t)((m + 63) / 64) * ((n + 31) / 32);
    if (m < 2 || n % 4 != 0 || tiles > 256) return 1;
    for (int s = 8; s > 1; s >>= 1)
        if (k % (64 * s) == 0 && k / s >= 384 && tiles * s <= 1024) return s;
    return 1;
}

// The same where the sum is a launch of its own and not part of one that runs anyway:
// only a long k over half the CUs or fewer pays for it. bf16, one launch / parts and
// sum: 128 x 1024 x 3072 11.8 / 8.9 us, 64 x 1024 x 3072 11.8 / 7.2, 24 x 1024 x 2048 9.2 / 6.1,
// 256 x 512 x 4096 14.9 / 9.9; not taken: 300 x 1024 x 3072 12.1 / 12.2, 512 x 1024 x 2048
// 9.3 / 12.8, 64 x 4096 x 1024 5.9 / 7.3.
int gemm_splits_alone(int m, int n, int k) {
    const int64_t tiles = (int64_t)((m + 63) / 64) * ((n + 31) / 32);
    return m > 16 && k >= 2048 && tiles <= 128 ? gemm_splits(m, n, k) : 1;
}

}  // namespace ythip

using namespace ythip;

extern "C" {

__attribute__((visibility("default"))) int ythip_gemm_splits(int dtype, int m, int n, int k) {
    if ((dtype != YTHIP_BF16 && dtype != YTHIP_F16) || m <= 0 || n <= 0 || k <= 0) return 1;
    return gemm_splits(m, n, k);
}

__attribute__((visibility("default"))) size_t ythip_gemm_workspace_size(int dtype, int m, int n, int k) {
    if ((dtype != YTHIP_BF16 && dtype != YTHIP_F16) || m <= 0 || n <= 0 || k <= 0) return 0;
    const int s = gemm_splits_alone(m, n, k);
    return s > 1 ? (size_t)s * m * n * sizeof(float) : 0;
}

__attribute__((visibility("default"))) int ythip_gemm_ws(int dtype_in, int dtype_out, int m, int n, int k, const void* A,
                                                         int64_t rsa, int64_t csa, const void* B, int64_t rsb, int64_t csb,
                                                         void* C, int64_t rsc, int64_t csc, float alpha, float beta,
                                                         void* workspace, size_t ws_bytes, void* stream) {
    const size_t need = ythip_gemm_workspace_size(dtype_in, m, n, k);
    // rows that the DMA kernels take, and a C that the sum can write
    const bool ok = need > 0 && alpha != 0.0f && A && B && C && workspace && csa == 1 && rsb == 1 && csc == 1 &&
                    rsa % 8 == 0 && csb % 8 == 0 && aligned(A, 16) && aligned(B, 16) && aligned(workspace, 16) &&
                    ws_bytes >= need &&
                    (dtype_out == dtype_in || dtype_out == YTHIP_F32);
    if (!ok)
        return ythip_gemm(dtype_in, dtype_out, 1, m, n, k, A, 0, rsa, csa, B, 0, rsb, csb, C, 0, rsc, csc, alpha, beta,
                          stream);
    const int s = gemm_splits(m, n, k);
    hipStream_t st = static_cast<hipStream_t>(stream);
    float* parts = static_cast<float*>(workspace);
    if (const int e = gemm_dispatch(dtype_in, YTHIP_F32, s, m, n, k / s, A, k / s, rsa, 1, B, k / s, 1, csb, parts,
                                    (int64_t)m * n, n, 1, 1.0f, 0.0f, st))
        return e;
    const int64_t mn = (int64_t)m * n;
    const dim3 grid((unsigned)((mn / 4 + 255) / 256));
    auto sum = [&](auto to) {
        using TO = decltype(to);
        if (s == 8) splitk_reduce_kernel<TO, 8><<<grid, 256, 0, st>>>(parts, mn, n / 4, C, rsc, alpha, beta);
        else if (s == 4) splitk_reduce_kernel<TO, 4><<<grid, 256, 0, st>>>(parts, mn, n / 4, C, rsc, alpha, beta);
        else splitk_reduce_kernel<TO, 2><<<grid, 256, 0, st>>>(parts, mn, n / 4, C, rsc, alpha, beta);
        return status_of(hipGetLastError());
    };
    if (dtype_out == YTHIP_F32) return sum(F32{});
    return dtype_out == YTHIP_BF16 ? sum(BF16{}) : sum(F16{});
}

__attribute__((visibility("default"))) int ythip_gemm_swiglu(int dtype, int m, int inter, int k, const void* A, int64_t lda,
                                                             const void* W, int64_t ldw, void* C, int64_t ldc,
                                                             void* stream) {
    const char* who = "ythip_gemm_swiglu";
    if (m < 0 || inter < 0 || k < 0) return fail(YTHIP_EINVAL, "%s: negative size", who);
    if (dtype != YTHIP_BF16 && dtype != YTHIP_F16) return fail(YTHIP_EUNSUPPORTED, "%s: 16-bit types only", who);
    if (m == 0 || inter == 0) return 0;
    if (!A || !W || !C) return fail(YTHIP_EINVAL, "%s: NULL pointer", who);
    if (k == 0 || k % 8 || inter % 4 || lda % 8 || ldw % 8 || ldc % 4 || lda < k || ldw < k || ldc < inter ||
        !aligned(A, 16) || !aligned(W, 16) || !aligned(C, 8) || (int64_t)m * lda * 2 >= (int64_t(1) << 31) ||
        (int64_t)2 * inter * ldw * 2 >= (int64_t(1) << 31))
        return fail(YTHIP_EUNSUPPORTED, "%s: 16-byte aligned rows below 2^31 bytes, k %% 8 == 0, inter %% 4 == 0", who);
    GemmArgs g{};
    g.A = A; g.B = W; g.C = C;
    g.m = m; g.n = inter; g.k = k;
    g.rsa = lda; g.rsb = 1; g.csb = ldw; g.rsc = ldc;
    g.alpha = 1.0f;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dtype == YTHIP_BF16 ? swiglu_typed<BF16>(g, s) : swiglu_typed<F16>(g, s);
}

}  // extern "C"
