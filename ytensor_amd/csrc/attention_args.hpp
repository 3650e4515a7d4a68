// attention_args.hpp — the arguments that the prefill attention kernels share.
#pragma once

#include "common.hpp"

namespace ythip {

constexpr float LOG2E = 1.4426950408889634f;

struct AttnArgs {
    const void* Q;
    const void* K;
    const void* V;
    void* O;
    int64_t qs0, qs1, qs2, ks0, ks1, ks2, vs0, vs1, vs2, os0, os1, os2;
    int64_t qs3, ks3, vs3, os3;  // element strides along d (1 on the MFMA path)
    int B, Hq, Hkv, Sq, Skv, D, Dv;
    int diag_off;  // causal / diagonal masks: key j visible to query i iff j <= i + diag_off
    float scale_log2;  // scale * log2(e)
    const uint8_t* mask;
    int64_t mask_ld;
    int causal;
    const float* bias;
    int64_t brs, bcs;
    int nqb;
    int balance;  // causal: the grid is resident at once, two workgroups per CU (see attn_fwd_mfma)
    uint8_t* tcls;        // byte mask's tile classes (mask_tile_class_kernel), or null
    int nkbt;             // 64-key blocks of the mask rows: ceil(Skv / 64)
    int o_line;           // O: unit d stride, 16-byte aligned base, rows and heads
    int mask_words;       // byte mask, no bias, 4-byte aligned base and rows (attn_fwd_f32)
    float scale;          // MODE 4: the scale itself
    int any_mask;         // MODE 4: a mask was given, so rows that see no key are zero
};

// Any layout, type, mask and bias, d and dv up to 256 (attention_any.hip).
hipError_t attn_any(int dtype, const AttnArgs& a, hipStream_t s);

}  // namespace ythip
