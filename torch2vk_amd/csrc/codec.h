// Pieces the audio codec's kernels share.
#pragma once

#include "common.h"

namespace t2h {

// sin(y)^2 to fp32 accuracy for |y| <= SIN_SQUARED_MAX (1.2e-7 absolute and 2.8e-7 relative against 64 bits; the
// library's sinf squared: 1.3e-7 absolute).  y is reduced to r = y - k pi / 2, k = rint(2 y / pi), by Cody and Waite's
// method in double, pi / 2 in two parts (fp64 runs at the unpacked fp32 rate here, so the two multiply-adds cost
// no more than three in fp32 and hold for large arguments); sin(r) on [-pi / 4, pi / 4] is its Taylor series to
// r^11 (the next term is below 7e-12), and an odd k turns the square into cos(r)^2 = 1 - sin(r)^2.  About 20
// instructions and no branch, so several run side by side in an epilogue.
constexpr float SIN_SQUARED_MAX = 1073741824.0f;  // 2^30: k stays an int
__device__ __forceinline__ float sin_squared(float y) {
    const double k = rint((double)y * 0.63661977236758134308);
    double rd = fma(k, -1.57079632679489655800, (double)y);  // pi / 2 rounded to 53 bits
    rd = fma(k, -6.12323399573676603587e-17, rd);             // what is left of it
    const float r = (float)rd;
    const float q = r * r;
    float p = fmaf(q, -2.5052108385441719e-8f, 2.7557319223985893e-6f);  // -1 / 11!, 1 / 9!, ...
    p = fmaf(q, p, -1.9841269841269841e-4f);
    p = fmaf(q, p, 8.3333333333333333e-3f);
    p = fmaf(q, p, -1.6666666666666667e-1f);
    const float s = fmaf(q * r, p, r);
    const float s2 = s * s;
    return ((int)k & 1) != 0 ? 1.0f - s2 : s2;
}

// The codec's activation: x + sin(alpha x)^2 / (alpha + eps)
// (src/models/quantized_omnivoice/dispatch/audio_decode.py:151-161).
__device__ __forceinline__ float snake_f32(float v, float alpha, float eps) {
    const float y = alpha * v, inv = 1.0f / (alpha + eps);
    if (fabsf(y) <= SIN_SQUARED_MAX) return v + inv * sin_squared(y);
    const float s = sinf(y);  // large arguments, infinities and NaN
    return v + inv * (s * s);
}

// t2h_conv_transpose1d_q8_0, and with `snaked` also bf16(snake(y, alpha)) of every output, [B, L_out, Co].
int conv_transpose1d_q8_0_launch(const float* x, const int64_t* x_strides, const void* w, const float* bias,
                                 float* out, uint32_t batch, uint32_t ci, uint32_t li, uint32_t co, uint32_t kh,
                                 uint32_t stride, uint32_t pad, uint32_t lo, uint16_t* snaked, const float* alpha,
                                 float eps, void* stream);

}  // namespace t2h
