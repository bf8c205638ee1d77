// Shared by the attention kernels (attention.hip, attention_decode.hip).
#pragma once

#include <stdint.h>

#include "nvr_device.h"
#include "nvr_internal.h"

namespace nvr {

// The q/k norm + RoPE + KV-slot write that the decode-batch entry point runs
// inside the attention launch; unused otherwise.
struct QkvRopeArgs {
    const uint16_t* qkv;   // [rows, qh + 2 kvh, 128]
    const uint16_t* qw;    // q norm weight [128]
    const uint16_t* kw;    // k norm weight [128]
    const int* slots;      // [rows]
    const float* rope;     // [max_positions, 128]: cos | sin
    int max_positions;
    float eps;
};

// One 16-lane group per head in the layout of qkv_rope's d128 kernel: lane m
// holds elements 8m .. 8m + 7 of the head (xw) and of its norm weight (wv). Returns the normalised and rotated elements.
__device__ __forceinline__ uint4 qkv_rotate(const float* rope, int max_positions, float eps, const uint4& xw,
                                            const uint4& wv, int pos, int m) {
    constexpr int D = 128;
    float cs[8], sn[8], wf[8];
    if (pos >= 0 && pos < max_positions) {
        const float4* t = reinterpret_cast<const float4*>(rope + int64_t(pos) * D + 8 * (m & 7));
        const float4 c0 = t[0], c1 = t[1], s0 = t[D / 8], s1 = t[D / 8 + 1];
        cs[0] = c0.x; cs[1] = c0.y; cs[2] = c0.z; cs[3] = c0.w;
        cs[4] = c1.x; cs[5] = c1.y; cs[6] = c1.z; cs[7] = c1.w;
        sn[0] = s0.x; sn[1] = s0.y; sn[2] = s0.z; sn[3] = s0.w;
        sn[4] = s1.x; sn[5] = s1.y; sn[6] = s1.z; sn[7] = s1.w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) { cs[i] = 1.0f; sn[i] = 0.0f; }
    }
    if (m < 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i) sn[i] = -sn[i];
    }
    unpack8(wv, wf);
    return norm_rotate_d128(xw, wf, cs, sn, eps);
}

// 32-lane shuffle-down fold of the reference's warp_sum, valid in lanes 0 and
// 32 of the wave (the reference's warps are the two 32-lane halves).
__device__ __forceinline__ float half_wave_sum(float v) {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) v += xor_lane(v, o);
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v = fmaxf(v, xor_lane(v, o));
    return v;
}

// The reference's final fold of its 8 warp sums (zeros in lanes 8..31).
__device__ __forceinline__ float fold8(const float* w) {
    return ((w[0] + w[4]) + (w[2] + w[6])) + ((w[1] + w[5]) + (w[3] + w[7]));
}

// nvr_expf for x <= 0 or NaN, with its bits: the same polynomial, and 2^k
// applied as 2^(k + 64) (exact, k >= -159) times 2^-64 (the one rounding), so
// neither branch nor select remains but the one below -110.
__device__ __forceinline__ float exp_nonpositive(float x) {
    const float kf = __builtin_rintf(x * 0x1.715476p+0f);
    float r = __builtin_fmaf(kf, -0x1.62e400p-1f, x);
    r = __builtin_fmaf(kf, -0x1.7f7d1cp-20f, r);
    float p = 0x1.a01a02p-13f;
    p = __builtin_fmaf(p, r, 0x1.6c16c2p-10f);
    p = __builtin_fmaf(p, r, 0x1.111112p-7f);
    p = __builtin_fmaf(p, r, 0x1.555556p-5f);
    p = __builtin_fmaf(p, r, 0x1.555556p-3f);
    p = __builtin_fmaf(p, r, 0.5f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_fmaf(p, r, 1.0f);
    const int k = int(fmaxf(kf, -160.0f));
    const float y = (p * pow2i(k + 64)) * 0x1.0p-64f;
    return x < -110.0f ? 0.0f : y;
}

// attention_decode.hip: decode batches at head dim 128, one block per CU.
// Needs 16-byte aligned q (or qkv, norm weights and RoPE table) and caches,
// blocks * bs below 2^31 and attention_decode_fits.
bool attention_decode_fits(int bs, int kvh, int max_context);
template <int HPB, bool FUSED>
void launch_attention_decode(nv_context* c, const uint16_t* q, uint16_t* k, uint16_t* v, const int* p, const int* s,
                             const int* t, uint16_t* o, int rows, int qh, int kvh, int bs, int blocks, int stride,
                             int batch, int max_context, const QkvRopeArgs& fa);

}  // namespace nvr
