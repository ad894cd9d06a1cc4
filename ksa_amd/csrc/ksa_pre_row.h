// One q / k head row in front of the attention - RMSNorm, norm weight, rotary embedding - for the decode kernel that
// does this step itself, and the lane exchanges it shares with the pre-attention kernel.  A row of D 16-bit elements
// is held by LPR = D / 8 consecutive lanes, eight elements each; arithmetic and rounding points are those of
// ksa_pre.hip, whose loop has the same statements in place (as calls of these functions they are scheduled
// otherwise there: 177 against 162 us at 32k tokens of 32 + 8 heads).
#pragma once
#include "ksa_cvt.h"

// value of the lane `n` places further inside the same row of 16 lanes (cyclic)
template <int N>
__device__ __forceinline__ uint32_t pre_row_ror(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + N, 0xf, 0xf, false);
}

// sum over the LPR lanes that hold one head row; every lane of the row gets the total
template <int LPR>
__device__ __forceinline__ float pre_row_sum(float ss) {
    if constexpr (LPR == 16) {  // rotations inside a DPP row (16 lanes)
        ss += __builtin_bit_cast(float, pre_row_ror<8>(__builtin_bit_cast(uint32_t, ss)));
        ss += __builtin_bit_cast(float, pre_row_ror<4>(__builtin_bit_cast(uint32_t, ss)));
        ss += __builtin_bit_cast(float, pre_row_ror<2>(__builtin_bit_cast(uint32_t, ss)));
        ss += __builtin_bit_cast(float, pre_row_ror<1>(__builtin_bit_cast(uint32_t, ss)));
    } else {
#pragma unroll
        for (int m = 1; m < LPR; m <<= 1) ss += __shfl_xor(ss, m);
    }
    return ss;
}

// 1 / RMS of a row from this lane's eight elements
template <typename T, int LPR>
__device__ __forceinline__ float ksa_row_inv_rms(const u32x4 raw, float eps) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = KsaCvt<T>::dot2(raw[i], raw[i], ss);
    ss = pre_row_sum<LPR>(ss);
    return rsqrtf(ss * (1.0f / (8 * LPR)) + eps);
}

// z = round(w * round(x * inv)), kept packed for the exchange; wl / wh: this lane's slice of the weight,
// each packed word split into (low, 0) and (0, high)
template <typename T>
__device__ __forceinline__ u32x4 ksa_row_scale(const u32x4 raw, float inv, const uint32_t (&wl)[4], const uint32_t (&wh)[4]) {
    using C = KsaCvt<T>;
    u32x4 zp;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t y = C::down2(C::lo(raw[i]) * inv, C::hi(raw[i]) * inv);
        float z0, z1;
        C::dot2z_x2(y, wl[i], y, wh[i], z0, z1);
        zp[i] = C::down2(z0, z1);
    }
    return zp;
}

// out = round(round(z cos) + round(rot(z) sin)), cosines and sines split like the weights, the sines with the
// rotate_half sign; the two rounded terms of an element are packed together and added by a dot product with (1, 1)
template <typename T, int LPR>
__device__ __forceinline__ u32x4 ksa_row_rope(const u32x4 zp, const uint32_t (&cl)[4], const uint32_t (&ch)[4],
                                              const uint32_t (&sl)[4], const uint32_t (&sh)[4]) {
    using C = KsaCvt<T>;
    u32x4 outp;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t pp;  // the partner half of the row
        if constexpr (LPR == 16) pp = pre_row_ror<8>(zp[i]);
        else pp = (uint32_t)__shfl_xor((int)zp[i], LPR / 2);
        float c0, s0, c1, s1, o0, o1;
        C::dot2z_x4(zp[i], cl[i], pp, sl[i], zp[i], ch[i], pp, sh[i], c0, s0, c1, s1);
        const uint32_t e0 = C::down2(c0, s0), e1 = C::down2(c1, s1);
        C::dot2z_x2(e0, C::kOnes, e1, C::kOnes, o0, o1);
        outp[i] = C::down2(o0, o1);
    }
    return outp;
}
