// Block fixed point as the mat-vec kernels hold activations (gemv.hip, gemv_quad.hip, gemv_wide.hip, each built once per precision with
// FHIP_GEMV_PLANES = 2 or 3): a run of 16 or 32 columns is one f32 scale and NP signed byte planes. The kernels promise each other's bits,
// so the quantiser and what turns a run's plane sums back into f32 stand here, once. Anonymous: the two precisions are different functions.
#pragma once
#include <stdint.h>

#ifndef FHIP_GEMV_PLANES
#define FHIP_GEMV_PLANES 2
#endif

namespace {

constexpr int NP = FHIP_GEMV_PLANES;   // byte planes per activation run
static_assert(NP == 2 || NP == 3, "two or three activation planes");
// Largest quantised magnitude: every digit at 127; the run's largest activation maps onto it. With two planes the rounding
// of the reciprocal and of the product moves that by at most 0.02, never to the next integer; with three (8.4e6 * 2^-22 = 2)
// the quantiser clamps.
constexpr float QMAX = NP == 2 ? 32639.0f : 8355711.0f;
constexpr float TINY_RUN = 7.888609052210118e-31f;   // 2^-100: below this QMAX / amax leaves the f32 range's comfortable part
constexpr float HUGE_RUN = 7.922816251426434e28f;    // 2^96

__device__ __forceinline__ int dot4(uint32_t a, uint32_t b, int c) { return __builtin_amdgcn_sdot4((int)a, (int)b, c, false); }

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true); }
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E;   // quad_perm [1,0,3,2], [2,3,0,1]

// exact integer plane sums -> f32 (one rounding, at most 2^-24 relative)
__device__ __forceinline__ float planes_f32(const int (&a)[NP]) {
    if constexpr (NP == 2) return (float)((a[0] << 8) + a[1]);
    else return fmaf((float)a[0], 65536.0f, (float)((a[1] << 8) + a[NP - 1]));
}

// Eight consecutive activations of one run -> NP plane dword pairs, the run's scale and the run's quantised sum.
// The 2 (RUN 16) or 4 (RUN 32) lanes of a run sit in one quad and agree on amax, the scale and the sum afterwards.
template <int RUN>
__device__ __forceinline__ void quantize8(const float (&v)[8], uint32_t (&pl)[NP][2], float& scale_out, float& sum_out) {
    float amax = fmaxf(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))),
                       fmaxf(fmaxf(fabsf(v[4]), fabsf(v[5])), fmaxf(fabsf(v[6]), fabsf(v[7]))));
    float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));   // NaN / inf detector (fmaxf drops NaNs)
    amax = fmaxf(amax, dpp_f<DPP_XOR1>(amax));
    sum += dpp_f<DPP_XOR1>(sum);
    if (RUN == 32) {
        amax = fmaxf(amax, dpp_f<DPP_XOR2>(amax));
        sum += dpp_f<DPP_XOR2>(sum);
    }
    // not representable in block fixed point: non-finite members (their sum is not finite either), a run so large that a
    // format's offset term (up to 128 times the run's sum) could leave the f32 range where the element-wise products do not,
    // or a run so small that QMAX / amax would overflow
    const bool special = !(fabsf(sum) <= 3.4028234663852886e38f) || amax > HUGE_RUN || (amax < TINY_RUN && amax > 0.f);
    const float inv = amax > 0.f ? QMAX * __builtin_amdgcn_rcpf(amax) : 0.f;
    uint32_t t[8];
    if constexpr (NP == 2) {
        // round to nearest by adding 1.5 * 2^23; the 128 makes the low byte an offset-binary digit
#pragma unroll
        for (int i = 0; i < 8; i++) t[i] = __float_as_uint(fmaf(v[i], inv, 12582912.0f + 128.0f));
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            // (clamped before the rounding: the bounds are whole numbers, and it is one instruction)
            const int q = __float2int_rn(__builtin_amdgcn_fmed3f(v[i] * inv, -QMAX, QMAX));
            t[i] = (uint32_t)(q + 0x8080);
        }
    }
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        const uint32_t t0 = t[4 * hh], t1 = t[4 * hh + 1], t2 = t[4 * hh + 2], t3 = t[4 * hh + 3];
        const uint32_t p01 = __builtin_amdgcn_perm(t1, t0, 0x05010400u), p23 = __builtin_amdgcn_perm(t3, t2, 0x05010400u);
        pl[NP - 1][hh] = __builtin_amdgcn_perm(p23, p01, 0x05040100u) ^ 0x80808080u;   // bytes 0, back to signed digits
        if constexpr (NP == 2) {
            pl[0][hh] = __builtin_amdgcn_perm(p23, p01, 0x07060302u);                  // bytes 1: the signed top digit
        } else {
            pl[1][hh] = __builtin_amdgcn_perm(p23, p01, 0x07060302u) ^ 0x80808080u;
            const uint32_t u01 = __builtin_amdgcn_perm(t1, t0, 0x00000602u), u23 = __builtin_amdgcn_perm(t3, t2, 0x00000602u);
            pl[0][hh] = __builtin_amdgcn_perm(u23, u01, 0x05040100u);                  // bytes 2
        }
    }
    int qs[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) qs[p] = dot4(pl[p][1], 0x01010101u, dot4(pl[p][0], 0x01010101u, 0));
    int qsum = qs[0];
#pragma unroll
    for (int p = 1; p < NP; p++) qsum = (qsum << 8) + qs[p];
    qsum += dpp_i<DPP_XOR1>(qsum);
    if (RUN == 32) qsum += dpp_i<DPP_XOR2>(qsum);
    const float scale = amax * (1.0f / QMAX);
    scale_out = special ? __uint_as_float(0x7FC00000u) : scale;
    sum_out = scale * (float)qsum;
}

}  // namespace
