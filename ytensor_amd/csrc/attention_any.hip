// attention_any.hip — attention for the layouts the MFMA kernels of attention.hip
// cannot take: any element strides (the ymodel2 example's transposed ring cache
// [b, 2, hd, L], example/ymodel2-s-2/ymodel2.cpp:47-144, 188-262), any alignment,
// head dims other than 64 and 128 (up to 256, d != dv included), every type, mask
// and bias; flash semantics (src/kernel/avx2/flash_attention.inl:202-443: rows
// that see no key are zero).
//
// Bound by latency and by the fp32 matrix cores: all arithmetic is fp32 on
// v_mfma_f32_16x16x4_f32, whatever the input type. No LDS staging: a wave owns 16
// queries and reads its K and V fragments straight from L1 / L2 in the layout the
// MFMA wants, so any stride is only another address --
//   S^T = K . Q^T: lane (r, g) holds K[key r][d = 16 b + 4 g + j] and ends with
//     S[query r][keys 4 g .. 4 g + 3]: 16 bytes along d when d runs contiguously,
//     else 4 loads (contiguous over the 16 lanes r when keys do);
//   O^T += V^T . P^T: lane (r, g) holds V[key 4 g + j][d = 16 t + r]: 16 bytes
//     along the keys when they run contiguously, else 4 loads over d.
// The W waves of a workgroup (eight, four at the largest head dims, or one: see
// launch_any) share the same 16 queries and each take a run of the visible key
// blocks, with an online softmax of their own; they are merged through LDS at the end.
// That keeps every SIMD busy at a few hundred queries and evens out causal rows. 8
// heads x 256 queries x 1024 keys, d = 64, transposed cache, byte mask, fp32: 323 us
// one wave per query before, 26 us here (8.5 us of it the 64 MB that the 128
// workgroups read from L2, 7.5 us matrix work on the 128 CUs they cover); 16 heads x
// 1024 x 80 bf16 causal 2311 -> 127 us.

#include <algorithm>

#include "attention_args.hpp"

namespace ythip {

// What a lane reads where no mask word is (no mask, or fewer keys than four): K may
// be smaller than the word.
static __device__ const uint32_t no_mask_word = 0x01010101u;

// Four elements as they were loaded: consecutive ones in one load (PIECE), or one
// by one at a stride. Converted only where they are used, so that a load in flight
// is not waited for.
template <class T, bool PIECE>
struct Four {
    using raw = typename T::raw;
    using piece = typename std::conditional<sizeof(raw) == 4, f32x4, u32x2>::type;
    using piece_any = typename std::conditional<sizeof(raw) == 4, f32x4_any, u32x2_any>::type;
    typename std::conditional<PIECE, piece, raw[4]>::type v;

    __device__ __forceinline__ void load(const void* p, int64_t i) {
        v = *reinterpret_cast<const piece_any*>(static_cast<const raw*>(p) + i);
    }
    __device__ __forceinline__ f32x4 get() const {
        if constexpr (!PIECE) {
            return f32x4{load_as_f32<T>(v, 0), load_as_f32<T>(v, 1), load_as_f32<T>(v, 2), load_as_f32<T>(v, 3)};
        } else if constexpr (sizeof(raw) == 4) {
            return v;
        } else {
            return f32x4{lo_as_f32(T{}, v[0]), hi_as_f32(T{}, v[0]), lo_as_f32(T{}, v[1]), hi_as_f32(T{}, v[1])};
        }
    }
};

// x[i + by], zero past the fourth (by <= 4)
__device__ __forceinline__ f32x4 moved(f32x4 x, int by) {
    f32x4 y = by & 1 ? f32x4{x[1], x[2], x[3], 0.f} : x;
    y = by & 2 ? f32x4{y[2], y[3], 0.f, 0.f} : y;
    return by >= 4 ? f32x4{0.f, 0.f, 0.f, 0.f} : y;
}

// NB: 16-wide d blocks (d and dv <= 16 NB; FULL: both equal); KD: K is read in
// pieces along d; VK: V is read in pieces along the keys; NKT: 16-key tiles per
// block. The code is straight and runs once or twice per wave, so its length is
// time (instruction fetch): the forms are templates and not branches.
template <class T, int NB, bool FULL, bool KD, bool VK, int W, int NKT>
__global__ __launch_bounds__(64 * W) void attn_any_kernel(AttnArgs a) {
    constexpr int BKV = 16 * NKT;
    constexpr float BIG = 3.402823466e38f;  // the largest finite float
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int nbh = a.B * a.Hq;
    const int nqb = (a.Sq + 15) / 16;
    // heads fastest: the workgroups that share K / V run together; last query
    // blocks first, they see the most keys under a causal mask
    const int bh = blockIdx.x % nbh, qb = nqb - 1 - blockIdx.x / nbh;
    const int b = bh / a.Hq, h = bh % a.Hq, kvh = h / (a.Hq / a.Hkv);
    const int64_t ko = b * a.ks0 + kvh * a.ks1, vo = b * a.vs0 + kvh * a.vs1;
    const int q0 = qb * 16, qrow = q0 + r, qr = min(qrow, a.Sq - 1);

    static_assert(FULL || !VK, "V in pieces: whole d blocks only");
    f32x4 qf[NB];
    {
        const int64_t qo = b * a.qs0 + h * a.qs1 + (int64_t)qr * a.qs2;
        if (FULL && a.qs3 == 1) {
            Four<T, true> q[NB];
#pragma unroll
            for (int bb = 0; bb < NB; ++bb) q[bb].load(a.Q, qo + 16 * bb + 4 * g);
#pragma unroll
            for (int bb = 0; bb < NB; ++bb) qf[bb] = q[bb].get() * a.scale_log2;
        } else {
#pragma unroll
            for (int bb = 0; bb < NB; ++bb)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int d = 16 * bb + 4 * g + j;
                    const float v = load_as_f32<T>(a.Q, qo + min(d, a.D - 1) * a.qs3);
                    qf[bb][j] = d < a.D ? v * a.scale_log2 : 0.f;
                }
        }
    }

    int kv_end = a.Skv;
    if (a.causal) kv_end = min(a.Skv, min(q0 + 15, a.Sq - 1) + a.diag_off + 1);
    const int nblk = kv_end > 0 ? (kv_end + BKV - 1) / BKV : 0;
    // This wave's blocks: a run of n, begun at a place that differs from workgroup
    // to workgroup. In a transposed cache the rows of a block lie a power of two
    // apart, in one L2 channel; waves that walk together would all wait for it.
    const int per = (nblk + W - 1) / W, b0 = wave * per, n = min(max(nblk - b0, 0), per);
    const int turn = n > 0 ? (int)(blockIdx.x % (unsigned)n) : 0;
    // the mask word of four keys is read where it fits; without a mask, or with
    // fewer keys than four, a constant stands in for it
    const bool words = a.mask != nullptr && a.Skv >= 4;
    // (in the global address space by name: the choice of two origins would be read by flat
    // loads, which wait for every load in flight -- bf16, d = 128, 2048 keys 76 us, 84 flat)
    using global_word = const __attribute__((address_space(1))) u32_any*;
    using global_byte = const __attribute__((address_space(1))) uint8_t*;
    const global_byte mrow = words ? (global_byte)(a.mask + (int64_t)qr * a.mask_ld) : (global_byte)&no_mask_word;

    // One block's operands. The next block's K is loaded as soon as the scores have
    // used this one's, its V after the output product: each load has the other
    // half of a block's work to arrive in, without a second set of registers.
    // Offsets are a lane part plus a part the whole wave shares.
    uint32_t mw[NKT];
    Four<T, KD> kr[NKT][NB];
    Four<T, VK> vr[NKT][NB];
    auto first_key = [&](int i) {
        const int j = min(i, n - 1) + turn;
        return (b0 + (j < n ? j : j - n)) * BKV;
    };
    auto load_k = [&](int i) {
        const int k0 = first_key(i);
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
            mw[kt] = *(global_word)(mrow + (words ? min(k0 + 16 * kt + 4 * g, a.Skv - 4) : 0));
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
            const int64_t row = ko + (int64_t)min(k0 + 16 * kt + r, a.Skv - 1) * a.ks2;
            const int64_t lane_d = row + 4 * g * a.ks3;
#pragma unroll
            for (int bb = 0; bb < NB; ++bb) {
                const int d = 16 * bb + 4 * g;
                if constexpr (KD) {
                    kr[kt][bb].load(a.K, row + (FULL ? d : min(d, a.D - 4)));  // D % 4 == 0
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        kr[kt][bb].v[j] = static_cast<const typename T::raw*>(
                            a.K)[FULL ? lane_d + (16 * bb + j) * a.ks3 : row + min(d + j, a.D - 1) * a.ks3];
                }
            }
        }
    };
    auto load_v = [&](int i) {
        const int k0 = first_key(i);
        const int64_t lane_d = vo + (int64_t)min(r, a.Dv - 1) * a.vs3;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
            const int key = k0 + 16 * kt + 4 * g;
            int64_t at[VK ? 1 : 4];
            if constexpr (VK) {
                at[0] = lane_d + min(key, a.Skv - 4);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) at[j] = lane_d + (int64_t)min(key + j, a.Skv - 1) * a.vs2;
            }
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                const int64_t col = FULL ? 16 * t * a.vs3 : (int64_t)(min(16 * t + r, a.Dv - 1) - min(r, a.Dv - 1)) * a.vs3;
                if constexpr (VK) {
                    vr[kt][t].load(a.V, at[0] + col);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) vr[kt][t].v[j] = static_cast<const typename T::raw*>(a.V)[at[j] + col];
                }
            }
        }
    };

    float m = -INFINITY, lsum = 0.f;
    f32x4 o[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};

    if (n > 0) {
        load_k(0);
        load_v(0);
    }
    for (int i = 0; i < n; ++i) {
        const int k0 = first_key(i);
        const bool whole = k0 + BKV <= a.Skv;
        uint32_t vis = 0;  // bit 4 kt + e: key k0 + 16 kt + 4 g + e is visible to qrow
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
            const int key0 = k0 + 16 * kt + 4 * g;
            uint32_t w = mw[kt];
            if (!words) {
                w = 0x01010101u;
                if (a.mask != nullptr) {
                    w = 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        w |= (uint32_t)a.mask[(int64_t)qr * a.mask_ld + min(key0 + e, a.Skv - 1)] << (8 * e);
                }
            } else if (!whole) {
                const int by = min(key0 - min(key0, a.Skv - 4), 4) * 8;
                w = by < 32 ? w >> by : 0u;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                bool v = key0 + e < a.Skv && ((w >> (8 * e)) & 0xffu) != 0u;
                if (a.causal) v = v && key0 + e <= qrow + a.diag_off;
                vis |= (uint32_t)v << (4 * kt + e);
            }
        }
        if (__ballot(vis != 0) == 0) {  // no row sees a key of the block
            load_k(i + 1);
            load_v(i + 1);
            continue;
        }

        f32x4 s[NKT];
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int bb = 0; bb < NB; ++bb) {
            f32x4 kf[NKT];
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt) {
                kf[kt] = kr[kt][bb].get();
                if constexpr (!FULL) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) kf[kt][j] = 16 * bb + 4 * g + j < a.D ? kf[kt][j] : 0.f;
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int kt = 0; kt < NKT; ++kt)
                    s[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kt][j], qf[bb][j], s[kt], 0, 0, 0);
        }
        load_k(i + 1);
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (a.bias != nullptr) {
                    const int key = min(k0 + 16 * kt + 4 * g + e, a.Skv - 1);
                    s[kt][e] += a.bias[(int64_t)qr * a.brs + (int64_t)key * a.bcs] * LOG2E;
                }
                s[kt][e] = (vis >> (4 * kt + e)) & 1 ? s[kt][e] : -INFINITY;
                mx = __builtin_elementwise_maximum(mx, s[kt][e]);
            }
        mx = max_across_rows(mx);
        const float m_new = __builtin_elementwise_maximum(m, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = exp2f(m - m_use);
        float psum = 0.f;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[kt][e] = exp2f(s[kt][e] - m_use);
                psum += s[kt][e];
            }
        lsum = fmaf(lsum, alpha, psum);
        m = m_new;
        // A key that a row does not see must not reach it, whatever its V row holds (a
        // cache row not yet written, say), and 0 . V would carry an infinity or NaN
        // over. Such values are rare: they leave the product, and every row that
        // gives them weight gets them back.
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            f32x4 vf[NKT];
            bool odd = false;
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt) {
                vf[kt] = vr[kt][t].get();
                const int key0 = k0 + 16 * kt + 4 * g;
                if (!whole) {
                    if constexpr (VK) {
                        vf[kt] = moved(vf[kt], min(key0 - min(key0, a.Skv - 4), 4));
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j) vf[kt][j] = key0 + j < a.Skv ? vf[kt][j] : 0.f;
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) odd = odd || !(fabsf(vf[kt][j]) <= BIG);
            }
            o[t] = alpha == 0.f ? f32x4{0.f, 0.f, 0.f, 0.f} : o[t] * alpha;
            if (__ballot(odd) != 0) {
                f32x4 up = {0.f, 0.f, 0.f, 0.f}, down = {0.f, 0.f, 0.f, 0.f};  // weight of +inf or NaN, of -inf or NaN
#pragma unroll
                for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float v = vf[kt][j];
                        const bool fin = fabsf(v) <= BIG;
                        up = __builtin_amdgcn_mfma_f32_16x16x4f32(fin || v < 0.f ? 0.f : 1.f, s[kt][j], up, 0, 0, 0);
                        down = __builtin_amdgcn_mfma_f32_16x16x4f32(fin || v > 0.f ? 0.f : 1.f, s[kt][j], down, 0, 0, 0);
                        vf[kt][j] = fin ? v : 0.f;
                    }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[t][e] += up[e] > 0.f ? INFINITY : 0.f;
                    o[t][e] += down[e] > 0.f ? -INFINITY : 0.f;
                }
            }
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[kt][j], s[kt][j], o[t], 0, 0, 0);
        }
        load_v(i + 1);
    }

    // the row's denominator over its four lanes
    lsum += __shfl_xor(lsum, 16, 64);
    lsum += __shfl_xor(lsum, 32, 64);
    // Merge of the waves, 16 d at a time: O = sum_w 2^(m_w - m) O_w / sum_w 2^(m_w - m) l_w
    __shared__ float sm[W][16], sl[W][16];
    __shared__ f32x4 so[W][NB][64];
    if (g == 0) {
        sm[wave][r] = m;
        sl[wave][r] = lsum;
    }
#pragma unroll
    for (int t = 0; t < NB; ++t) so[wave][t][lane] = o[t];
    __syncthreads();
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) top = __builtin_elementwise_maximum(top, sm[w][r]);
    const float base = top == -INFINITY ? 0.f : top;
    float wt[W], L = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        wt[w] = exp2f(sm[w][r] - base);
        L = fmaf(sl[w][r], wt[w], L);
    }
    if (qrow >= a.Sq) return;
    // a row that sees no key, or whose scores hold a NaN or +inf (L is NaN), is zero
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    const int64_t oo = b * a.os0 + h * a.os1 + (int64_t)qrow * a.os2;
    for (int t = wave; t < NB; t += W) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < W; ++w) acc += wt[w] == 0.f ? f32x4{0.f, 0.f, 0.f, 0.f} : so[w][t][lane] * wt[w];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 16 * t + 4 * g + i;
            if (d < a.Dv) store_from_f32<T>(a.O, oo + d * a.os3, L > 0.f ? acc[i] * inv : 0.f);
        }
    }
}

namespace {

template <class T, int NB, int W>
hipError_t launch_full(const AttnArgs& a, const dim3 grid, hipStream_t s) {
    constexpr int NKT = NB <= 4 ? 2 : 1;  // what the registers hold at two waves a SIMD
    const bool kd = a.ks3 == 1, vk = a.vs2 == 1 && a.Skv >= 4;
    if (kd && vk) attn_any_kernel<T, NB, true, true, true, W, NKT><<<grid, 64 * W, 0, s>>>(a);
    else if (kd) attn_any_kernel<T, NB, true, true, false, W, NKT><<<grid, 64 * W, 0, s>>>(a);
    else if (vk) attn_any_kernel<T, NB, true, false, true, W, NKT><<<grid, 64 * W, 0, s>>>(a);
    else attn_any_kernel<T, NB, true, false, false, W, NKT><<<grid, 64 * W, 0, s>>>(a);
    return hipGetLastError();
}

template <class T, int NB, int W>
hipError_t launch_part(const AttnArgs& a, const dim3 grid, hipStream_t s) {
    constexpr int NKT = NB <= 8 ? 2 : 1;
    if (a.ks3 == 1 && a.D % 4 == 0) attn_any_kernel<T, NB, false, true, false, W, NKT><<<grid, 64 * W, 0, s>>>(a);
    else attn_any_kernel<T, NB, false, false, false, W, NKT><<<grid, 64 * W, 0, s>>>(a);
    return hipGetLastError();
}

template <class T>
hipError_t launch_any(const AttnArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)((int64_t)((a.Sq + 15) / 16) * a.B * a.Hq));
    const int d = std::max(a.D, a.Dv);
    // One wave a workgroup where the queries fill the chip by themselves, or the keys are one or
    // two blocks: of eight most would idle, and all pay the merge. Many keys stay with eight,
    // which read a block's K and V from L2 together, and under a mask, where rows see different
    // numbers of keys, the eight even them out: there the line lies lower. Eight waves / one, us:
    // 2048 workgroups, fp32, no mask: d 8, 16 keys 57 / 23; d 80, 16 keys 106 / 27; d 128, 128
    // keys 89 / 44; bf16 d 64, 512 keys 125 / 85; bf16 d 128 transposed, 1024 keys 353 / 362,
    // 2048 keys 643 / 712. Causal, fp32, d 80, 128 keys: one wave takes 0.47 of eight's time,
    // 512 keys 1.11.
    const bool masked = a.causal || a.mask != nullptr;
    const unsigned wgs = grid.x;
    const int top = wgs < 1024 ? 32 : !masked || wgs >= 8192 ? 512 : wgs >= 2048 ? 128 : 64;
    const bool one = a.Skv <= top;
    if (a.D == 64 && a.Dv == 64) return one ? launch_full<T, 4, 1>(a, grid, s) : launch_full<T, 4, 8>(a, grid, s);
    if (a.D == 128 && a.Dv == 128) return one ? launch_full<T, 8, 1>(a, grid, s) : launch_full<T, 8, 8>(a, grid, s);
    if (d <= 64) return one ? launch_part<T, 4, 1>(a, grid, s) : launch_part<T, 4, 8>(a, grid, s);
    if (d <= 128) return one ? launch_part<T, 8, 1>(a, grid, s) : launch_part<T, 8, 8>(a, grid, s);
    return one ? launch_part<T, 16, 1>(a, grid, s) : launch_part<T, 16, 4>(a, grid, s);  // 64 KB of O tiles in LDS
}

}  // namespace

hipError_t attn_any(int dtype, const AttnArgs& a, hipStream_t s) {
    switch (dtype) {
        case YTHIP_F32: return launch_any<F32>(a, s);
        case YTHIP_F16: return launch_any<F16>(a, s);
        default: return launch_any<BF16>(a, s);
    }
}

}  // namespace ythip
