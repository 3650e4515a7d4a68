// gemm_any.hip — the matrix product for every layout that the DMA-staged kernels
// of gemm.hip cannot take: sizes that are multiples of nothing, rows at any
// element alignment, a transposed A, strided views, a column-major C
// (YTensor::matmul over arbitrary strides, src/ytensor_math.inl:284-316,
// 954-1051; sgemm.inl:586-787 packs its panels from any stride the same way).
//
// Bound by the operand stream into LDS (about 28 bytes a clock and CU from L2)
// in 16 bits, by the matrix cores in fp32. global_load_lds needs 16-byte aligned
// sources and whole k steps, so the tiles go through registers here:
//  * both operands land in LDS as [row][8 chunks of 16 bytes] of one 128-byte k
//    step, so the compute loop is the same for every layout;
//  * an operand whose k runs contiguously (KC) is read in 16-byte pieces, one
//    whose rows run contiguously (RC: a row-major B, a transposed A) in pieces of
//    4 rows x one k, transposed in registers. gfx950 takes such loads at any
//    element address, so neither alignment nor an odd stride costs extra
//    instructions. Anything else (ST) gathers element by element;
//  * no load is predicated: a row past the end re-reads a row inside (its results
//    are never stored), a piece that would run past the end is read from the last
//    place where it fits and shifted. A ragged k makes the FIRST step short (zeros
//    in both operands), so that the loop has whole steps only. Every load stays
//    inside the operand;
//  * the next PF k steps are in flight in registers while one is computed from
//    LDS (two stages): these grids often have one workgroup per CU, so nothing
//    else hides the load latency.
// (1021 x 779) . (779 x 1003): bf16 303 -> 10.8 us, fp32 362 -> 22 us (one output
// per thread before); 1024^3 bf16 with a transposed A 493 -> 12 us.

#include <utility>

#include "common.hpp"
#include "launch.hpp"

namespace ythip {

struct AnyArgs {
    const void* A;
    const void* B;
    void* C;
    int m, n, k;
    int64_t rsa, csa, rsb, csb, rsc, csc;
    int64_t sa_b, sb_b, sc_b;
    float alpha, beta;
    int tiles_m, tiles_n;
    MaskDesc mask;
    int mask_t;  // C is the transpose of the masked matrix
};

enum { KC = 0, RC = 1, ST = 2 };

__device__ __forceinline__ int any_swz(int row, int chunk) { return chunk ^ ((row ^ (row >> 3)) & 7); }

// v moved down by `bytes` (0..15), zeros in the freed top bytes; no branch, so
// that nothing makes the compiler wait for a load early
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int bytes) {
    uint64_t lo = (uint64_t)v[1] << 32 | v[0], hi = (uint64_t)v[3] << 32 | v[2];
    const bool far = bytes >= 8;
    lo = far ? hi : lo;
    hi = far ? 0 : hi;
    const int bits = (bytes & 7) * 8;
    lo = (lo >> bits) | ((hi << 1) << (63 - bits));
    hi >>= bits;
    return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}
__device__ __forceinline__ u32x2 shift_down(u32x2 v, int bytes) {
    const uint64_t x = ((uint64_t)v[1] << 32 | v[0]) >> (bytes * 8);
    return u32x2{(uint32_t)x, (uint32_t)(x >> 32)};
}
// the first `bytes` of v, zeros after them (bytes <= 0: all zero)
__device__ __forceinline__ u32x4 keep_low(u32x4 v, int bytes) {
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int left = min(max(bytes - 4 * q, 0), 4);
        o[q] = v[q] & (uint32_t)((uint64_t(1) << (8 * left)) - 1);
    }
    return o;
}

// One operand's tile: ROWS rows (m of A, n of B) by one 128-byte k step, held in
// registers between its loads and its LDS writes. A piece is 16 bytes of one row
// (KC, ST) or 4 rows of KP consecutive k (RC; KP spreads the tile over all threads).
template <class T, int ROWS, int THREADS, int MODE>
struct Stager {
    using raw = typename T::raw;
    static constexpr int ES = sizeof(raw), VEC = 16 / ES, BK = 8 * VEC;
    static constexpr int SHARE = ROWS * BK / THREADS / 4;
    static constexpr int KP = SHARE < 1 ? 1 : (SHARE > VEC ? VEC : SHARE);
    static constexpr int ITEMS = MODE == RC ? ROWS / 4 * (BK / KP) : ROWS * 8;
    static constexpr int PT = ITEMS / THREADS;
    static_assert(PT * THREADS == ITEMS, "tile / thread mismatch");
    using rc_t = typename std::conditional<ES == 2, u32x2, u32x4>::type;
    using rc_any = typename std::conditional<ES == 2, u32x2_any, u32x4_any>::type;

    struct Regs {
        u32x4 kc[MODE == RC ? 1 : PT];
        rc_t rc[MODE == RC ? PT : 1][MODE == RC ? KP : 1];
    };

    const raw* base[PT];             // where each piece starts at k = 0
    int shift[MODE == RC ? PT : 1];  // bytes, for the last group of rows

    __device__ __forceinline__ static int piece_k(int id) { return MODE == RC ? id / (ROWS / 4) * KP : (id & 7) * VEC; }

    __device__ __forceinline__ void init(const raw* p, int row0, int rows, int64_t rs, int64_t ks, int tid) {
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int id = tid + i * THREADS;
            if constexpr (MODE == RC) {
                const int row = row0 + id % (ROWS / 4) * 4, at = min(row, rows - 4);
                shift[i] = min(row - at, 3) * ES;
                base[i] = p + at + (int64_t)piece_k(id) * ks;
            } else {
                base[i] = p + (int64_t)min(row0 + (id >> 3), rows - 1) * rs + (int64_t)piece_k(id) * ks;
            }
        }
    }

    // The first step holds k in [0, first), the ones after it are whole: a ragged
    // k costs nothing in the loop. What lies past `first` is masked in put_first;
    // what lies past k is not read.
    __device__ __forceinline__ void get_first(Regs& r, int k, int64_t ks, int tid) const {
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int kk = piece_k(tid + i * THREADS);
            if constexpr (MODE == RC) {
#pragma unroll
                for (int e = 0; e < KP; ++e)
                    r.rc[i][e] = *reinterpret_cast<const rc_any*>(base[i] + (int64_t)(min(kk + e, k - 1) - kk) * ks);
            } else if constexpr (MODE == KC) {
                r.kc[i] = *reinterpret_cast<const u32x4_any*>(base[i] + (min(kk, k - VEC) - kk));
            } else {
                raw e[VEC];
#pragma unroll
                for (int j = 0; j < VEC; ++j) e[j] = base[i][(int64_t)(min(kk + j, k - 1) - kk) * ks];
                r.kc[i] = __builtin_bit_cast(u32x4, e);
            }
        }
    }

    __device__ __forceinline__ void get(Regs& r, int k0, int64_t ks) const {
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const raw* p = base[i] + (int64_t)k0 * ks;
            if constexpr (MODE == RC) {
#pragma unroll
                for (int e = 0; e < KP; ++e) r.rc[i][e] = *reinterpret_cast<const rc_any*>(p + (int64_t)e * ks);
            } else if constexpr (MODE == KC) {
                r.kc[i] = *reinterpret_cast<const u32x4_any*>(p);
            } else {
                raw e[VEC];
#pragma unroll
                for (int j = 0; j < VEC; ++j) e[j] = p[(int64_t)j * ks];
                r.kc[i] = __builtin_bit_cast(u32x4, e);
            }
        }
    }

    // ragged (uniform): this tile holds the operand's last group of rows and it is not whole
    template <bool FIRST>
    __device__ __forceinline__ void put(Regs r, u32x4* s, int tid, int first, int k, bool ragged) const {
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int id = tid + i * THREADS, kk = piece_k(id);
            if constexpr (MODE == RC) {
                if (ragged) {
#pragma unroll
                    for (int e = 0; e < KP; ++e) r.rc[i][e] = shift_down(r.rc[i][e], shift[i]);
                }
                if constexpr (FIRST) {
#pragma unroll
                    for (int e = 0; e < KP; ++e)
                        if (kk + e >= first) r.rc[i][e] = rc_t{};
                }
                const int g = id % (ROWS / 4), at = kk * ES;
                char* b = reinterpret_cast<char*>(s);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int row = g * 4 + j;
                    char* d = b + row * 128 + any_swz(row, at >> 4) * 16 + (at & 15);
                    if constexpr (ES == 2) {
                        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
                        uint32_t o[KP / 2];
#pragma unroll
                        for (int q = 0; q < KP / 2; ++q)
                            o[q] = __builtin_amdgcn_perm(r.rc[i][2 * q + 1][j >> 1], r.rc[i][2 * q][j >> 1], sel);
                        if constexpr (KP == 8) *reinterpret_cast<u32x4*>(d) = u32x4{o[0], o[1], o[2], o[3]};
                        else if constexpr (KP == 4) *reinterpret_cast<u32x2*>(d) = u32x2{o[0], o[1]};
                        else *reinterpret_cast<uint32_t*>(d) = o[0];
                    } else {
                        if constexpr (KP == 4)
                            *reinterpret_cast<u32x4*>(d) =
                                u32x4{r.rc[i][0][j], r.rc[i][1][j], r.rc[i][2][j], r.rc[i][3][j]};
                        else if constexpr (KP == 2)
                            *reinterpret_cast<u32x2*>(d) = u32x2{r.rc[i][0][j], r.rc[i][1][j]};
                        else
                            *reinterpret_cast<uint32_t*>(d) = r.rc[i][0][j];
                    }
                }
            } else {
                u32x4 v = r.kc[i];
                if constexpr (FIRST) {
                    if constexpr (MODE == KC) v = shift_down(v, min(kk - min(kk, k - VEC), VEC - 1) * ES);
                    v = keep_low(v, (first - kk) * ES);
                }
                s[(id >> 3) * 8 + any_swz(id >> 3, id & 7)] = v;
            }
        }
    }
};

template <class T, class TO, int BM, int BN, int WM, int WN, int AM, int BMODE, bool MASKED>
__global__ __launch_bounds__(64 * WM * WN) void gemm_any_kernel(AnyArgs a) {
    using raw = typename T::raw;
    constexpr int THREADS = 64 * WM * WN;
    constexpr int WTM = BM / WM, WTN = BN / WN, FM = WTM / 16, FN = WTN / 16;
    constexpr int STAGE = (BM + BN) * 8;  // 16-byte chunks
    constexpr int PF = (AM == ST || BM > 64) ? 1 : 2;
    using SA = Stager<T, BM, THREADS, AM>;
    using SB = Stager<T, BN, THREADS, BMODE>;
    constexpr int BK = SA::BK;
    __shared__ u32x4 lds[2 * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int r16 = lane & 15, g = lane >> 4;
    int tm, tn;
    tile_coords(blockIdx.x, a.tiles_m, a.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN, bz = blockIdx.y;

    SA sa;
    SB sb;
    sa.init(static_cast<const raw*>(a.A) + bz * a.sa_b, m0, a.m, a.rsa, a.csa, tid);
    sb.init(static_cast<const raw*>(a.B) + bz * a.sb_b, n0, a.n, a.csb, a.rsb, tid);
    typename SA::Regs ra[PF];
    typename SB::Regs rb[PF];
    const bool raga = a.m < m0 + BM && (a.m & 3) != 0, ragb = a.n < n0 + BN && (a.n & 3) != 0;

    // (a tile that the mask hides whole: one step, its sums are not used)
    const bool hidden = MASKED && !a.mask_t && hidden_tile(a.mask, min(m0 + BM, a.m) - 1, n0);
    const int all = (a.k + BK - 1) / BK;
    const int first = a.k - (all - 1) * BK;  // k in the first step
    const int steps = hidden ? 1 : all;
    // Past the last step the last one is read again: a load under a condition would
    // make every later wait a wait for all loads.
    auto load = [&](int p, int kt) {
        const int k0 = first + (min(kt, steps - 1) - 1) * BK;
        sa.get(ra[p], k0, a.csa);
        sb.get(rb[p], k0, a.rsb);
    };
    auto store = [&](int p, int kt) {
        u32x4* s = lds + (kt & 1) * STAGE;
        sa.template put<false>(ra[p], s, tid, first, a.k, raga);
        sb.template put<false>(rb[p], s + BM * 8, tid, first, a.k, ragb);
    };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](int kt) {
        const u32x4* cA = lds + (kt & 1) * STAGE;
        const u32x4* cB = cA + BM * 8;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const int r = wm * WTM + i * 16 + r16;
                fa[i] = cA[r * 8 + any_swz(r, h * 4 + g)];
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int r = wn * WTN + j * 16 + r16;
                fb[j] = cB[r * 8 + any_swz(r, h * 4 + g)];
            }
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = mfma_chunk(T{}, fb[j], fa[i], acc[i][j]);
        }
    };

    sa.get_first(ra[0], a.k, a.csa, tid);
    sb.get_first(rb[0], a.k, a.rsb, tid);
    if (PF == 2 && steps > 1) load(PF - 1, 1);
    sa.template put<true>(ra[0], lds, tid, first, a.k, raga);
    sb.template put<true>(rb[0], lds + BM * 8, tid, first, a.k, ragb);
    // Step kt computes from LDS stage kt % 2; its successor's pieces, in register
    // set (kt + 1) % PF, go to the other stage (last read in step kt - 1, before
    // the barrier), and that set then takes the loads of step kt + 1 + PF.
    if (steps > 1) {
        load(0, PF);
        __syncthreads();
        auto step = [&](int set, int kt) {
            compute(kt);
            store(set, kt + 1);
            load(set, kt + 1 + PF);
            __syncthreads();
        };
        int kt = 0;
        if constexpr (PF == 1) {
            do step(0, kt);
            while (++kt < steps - 1);
        } else {
            // pairs of steps, and the odd one out afterwards: with an exit between the
            // two the compiler would take either set for the newest and wait for both
            for (; kt + 2 < steps; kt += 2) {
                step(1, kt);
                step(0, kt + 1);
            }
            if (kt < steps - 1) step(1, kt);
        }
    } else {
        __syncthreads();
    }
    compute(steps - 1);

    // lane: C[m = r16][n = 4 g .. 4 g + 3] of each 16 x 16 tile
    using oraw = typename TO::raw;
    oraw* Cp = static_cast<oraw*>(a.C) + bz * a.sc_b;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = m0 + wm * WTM + i * 16 + r16;
        if (m >= a.m) continue;
        oraw* crow = Cp + (int64_t)m * a.rsc;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + wn * WTN + j * 16 + g * 4;
            if (n >= a.n) continue;
            f32x4 v = acc[i][j];
            if constexpr (MASKED) {
                if (!a.mask_t) {
                    masked_store4<TO>(a.mask, crow, a.csc, m, n, a.n, v * a.alpha, a.beta);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (n + r >= a.n) continue;
                        const int64_t at = (n + r) * a.csc;
                        float x = v[r] * a.alpha;
                        if (a.beta != 0.0f) x += a.beta * load_as_f32<TO>(crow, at);
                        if (visible(a.mask, n + r, m)) store_from_f32<TO>(crow, at, x);
                        else if (a.mask.fill) store_from_f32<TO>(crow, at, a.mask.value);
                    }
                }
                continue;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] *= a.alpha;
                if (a.beta != 0.0f && n + r < a.n) v[r] += a.beta * load_as_f32<TO>(crow, (n + r) * a.csc);
            }
            if (a.csc == 1 && n + 3 < a.n) {
                if constexpr (sizeof(oraw) == 2)
                    *reinterpret_cast<u32x2_any*>(crow + n) = u32x2{pack2<TO>(v[0], v[1]), pack2<TO>(v[2], v[3])};
                else
                    *reinterpret_cast<f32x4_any*>(crow + n) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < a.n) store_from_f32<TO>(crow, (n + r) * a.csc, v[r]);
            }
        }
    }
}

namespace {

template <class T, class TO, int AM, int BMODE>
hipError_t launch_any_mode(AnyArgs a, int batch, hipStream_t s) {
    // passes over the 256 CUs that a grid of b x b tiles takes
    auto rounds = [&](int b) { return ((int64_t)((a.m + b - 1) / b) * ((a.n + b - 1) / b) * batch + 255) / 256; };
    auto grid = [&](int b) {
        a.tiles_m = (a.m + b - 1) / b;
        a.tiles_n = (a.n + b - 1) / b;
        return dim3(a.tiles_m * a.tiles_n, batch);
    };
    constexpr int WN = sizeof(typename T::raw) == 4 ? 4 : 2;  // fp32: two waves a SIMD
    if constexpr (AM != ST) {
        // The tile that leaves the busiest CU less to do: bytes staged per k step
        // (the edge) in 16 bits, matrix work (the area) in fp32. 2400 x 2401 x 2402:
        // bf16 97 us on 64 x 64 tiles, 67 us on 128 x 128; fp32 251 us on 64 x 64.
        const bool wide = sizeof(typename T::raw) == 2 ? rounds(128) * 128 < rounds(64) * 64
                                                       : rounds(128) * 128 * 128 <= rounds(64) * 64 * 64;
        if (wide && a.mask.kind == YTHIP_MASK_NONE) {
            const dim3 gr = grid(128);
            gemm_any_kernel<T, TO, 128, 128, 2, WN, AM, BMODE, false><<<gr, 128 * WN, 0, s>>>(a);
            return hipGetLastError();
        }
    }
    const dim3 gr = grid(64);
    if (a.mask.kind == YTHIP_MASK_NONE) gemm_any_kernel<T, TO, 64, 64, 2, WN, AM, BMODE, false><<<gr, 128 * WN, 0, s>>>(a);
    else gemm_any_kernel<T, TO, 64, 64, 2, WN, AM, BMODE, true><<<gr, 128 * WN, 0, s>>>(a);
    return hipGetLastError();
}

template <class T, class TO>
hipError_t launch_any(const AnyArgs& a, int batch, hipStream_t s) {
    // a piece has to fit: VEC elements of k (KC), 4 rows (RC)
    constexpr int VEC = 16 / sizeof(typename T::raw);
    auto mode = [&](int rows, int64_t rs, int64_t ks) {
        if (ks == 1 && a.k >= VEC) return (int)KC;
        if (rs == 1 && rows >= 4) return (int)RC;
        return (int)ST;
    };
    const int am = mode(a.m, a.rsa, a.csa), bm = mode(a.n, a.csb, a.rsb);
    if (am == ST || bm == ST) return launch_any_mode<T, TO, ST, ST>(a, batch, s);
    if (am == KC) {
        if (bm == KC) return launch_any_mode<T, TO, KC, KC>(a, batch, s);
        return launch_any_mode<T, TO, KC, RC>(a, batch, s);
    }
    if (bm == KC) return launch_any_mode<T, TO, RC, KC>(a, batch, s);
    return launch_any_mode<T, TO, RC, RC>(a, batch, s);
}

}  // namespace

int gemm_any_dispatch(int dtype_in, int dtype_out, int batch, int m, int n, int k, const void* A, int64_t sa_b,
                      int64_t rsa, int64_t csa, const void* B, int64_t sb_b, int64_t rsb, int64_t csb, void* C,
                      int64_t sc_b, int64_t rsc, int64_t csc, float alpha, float beta, const MaskDesc& mask, hipStream_t s) {
    AnyArgs a{A, B, C, m, n, k, rsa, csa, rsb, csb, rsc, csc, sa_b, sb_b, sc_b, alpha, beta, 0, 0, mask, 0};
    if (csc != 1 && rsc == 1) {  // a column-major C: C^T = B^T . A^T, so that its stores run along memory
        a.mask_t = 1;
        std::swap(a.A, a.B);
        std::swap(a.m, a.n);
        std::swap(a.rsa, a.csb);
        std::swap(a.csa, a.rsb);
        std::swap(a.sa_b, a.sb_b);
        std::swap(a.rsc, a.csc);
    }
    if (dtype_in == YTHIP_F32) return status_of(launch_any<F32, F32>(a, batch, s));
    if (dtype_in == YTHIP_BF16)
        return status_of(dtype_out == YTHIP_F32 ? launch_any<BF16, F32>(a, batch, s) : launch_any<BF16, BF16>(a, batch, s));
    return status_of(dtype_out == YTHIP_F32 ? launch_any<F16, F32>(a, batch, s) : launch_any<F16, F16>(a, batch, s));
}

}  // namespace ythip
