// mq_wave.h -- wave64 reductions and the fp32 arithmetic shared by the runner kernels (gfx950):
// where two kernels have to round alike, every fused multiply-add is written out.
#pragma once
#include <hip/hip_runtime.h>

namespace mq {

// DPP path: xor 1, xor 2 (quad_perm), i <-> 7-i, i <-> 15-i inside each 16-lane row, then
// the four row results via readlane (the result is wave-uniform).
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float lane_f(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ float wave_sum_f(float v) {
    v += dpp_f<0xB1>(v);
    v += dpp_f<0x4E>(v);
    v += dpp_f<0x141>(v);
    v += dpp_f<0x140>(v);
    return (lane_f(v, 0) + lane_f(v, 16)) + (lane_f(v, 32) + lane_f(v, 48));
}
__device__ __forceinline__ float wave_max_f(float v) {
    v = fmaxf(v, dpp_f<0xB1>(v));
    v = fmaxf(v, dpp_f<0x4E>(v));
    v = fmaxf(v, dpp_f<0x141>(v));
    v = fmaxf(v, dpp_f<0x140>(v));
    return fmaxf(fmaxf(lane_f(v, 0), lane_f(v, 16)), fmaxf(lane_f(v, 32), lane_f(v, 48)));
}

// Mean and reciprocal deviation of a row of n values, lane l holding values l, l + 64, ... (V of them)
template <int V>
__device__ __forceinline__ void ln_stats(const float (&v)[V], int n, int lane, float eps, float &mean, float &rstd) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < V; i++)
        if (lane + 64 * i < n) s += v[i];
    mean = wave_sum_f(s) / (float)n;
    float s2 = 0.f;
#pragma unroll
    for (int i = 0; i < V; i++)
        if (lane + 64 * i < n) {
            const float d = v[i] - mean;
            s2 = __builtin_fmaf(d, d, s2);
        }
    rstd = 1.0f / sqrtf(wave_sum_f(s2) / (float)n + eps);
}
__device__ __forceinline__ float ln_value(float v, float mean, float rstd, float w, float b) {
    return __builtin_fmaf((v - mean) * rstd, w, b);
}

// The encoder's fp32 attention (k_attention and its few-row form): keys a block of its online
// softmax, and s + a . b of four dims of a score
constexpr int ATT_KB = 16;
__device__ __forceinline__ float score4(float s, const float4 a, const float4 b) {
    return s + __builtin_fmaf(a.w, b.w, __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.x, b.x, a.y * b.y)));
}

}  // namespace mq
