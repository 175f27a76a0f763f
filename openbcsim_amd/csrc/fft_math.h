// Arithmetic of the convolution kernels: complex products, small DFTs, and the
// normal variates of the noise path.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bcsim_hip {

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
#pragma clang fp contract(fast)
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
// multiply by -i (forward) or +i (inverse)
template <bool INV>
__device__ __forceinline__ float2 rot90(float2 a) {
    return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

// 4-point DFT (forward: exp(-2 pi i nk / 4); inverse: conjugate kernel).
template <bool INV>
__device__ __forceinline__ void dft4(float2 u0, float2 u1, float2 u2, float2 u3, float2& y0, float2& y1,
                                     float2& y2, float2& y3) {
    const float2 a0 = cadd(u0, u2);
    const float2 a1 = csub(u0, u2);
    const float2 a2 = cadd(u1, u3);
    const float2 a3 = rot90<INV>(csub(u1, u3));
    y0 = cadd(a0, a2);
    y2 = csub(a0, a2);
    y1 = cadd(a1, a3);
    y3 = csub(a1, a3);
}

// 8-point DFT as two 4-point DFTs of the even and odd inputs joined by the
// eighth roots of unity: X[k] = E[k] + w^k O[k], X[k+4] = E[k] - w^k O[k].
template <bool INV>
__device__ __forceinline__ void dft8(const float2* x, float2* y) {
    constexpr float h = 0.70710678118654752f;  // 1/sqrt(2)
    float2 e[4], o[4];
    dft4<INV>(x[0], x[2], x[4], x[6], e[0], e[1], e[2], e[3]);
    dft4<INV>(x[1], x[3], x[5], x[7], o[0], o[1], o[2], o[3]);
    // w = exp(-i pi/4) forward, exp(+i pi/4) inverse
    const float2 o1 = INV ? make_float2(h * (o[1].x - o[1].y), h * (o[1].x + o[1].y))
                          : make_float2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
    const float2 o2 = rot90<INV>(o[2]);
    const float2 o3 = INV ? make_float2(-h * (o[3].x + o[3].y), h * (o[3].x - o[3].y))
                          : make_float2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y));
    y[0] = cadd(e[0], o[0]);
    y[4] = csub(e[0], o[0]);
    y[1] = cadd(e[1], o1);
    y[5] = csub(e[1], o1);
    y[2] = cadd(e[2], o2);
    y[6] = csub(e[2], o2);
    y[3] = cadd(e[3], o3);
    y[7] = csub(e[3], o3);
}

// Counter-based normal variates for the noise path: a 32-bit integer hash
// (Wang's mix, then a multiply-xorshift round) feeds a Box-Muller transform.
__device__ __forceinline__ uint32_t mix32(uint32_t x) {
    x = (x ^ 61u) ^ (x >> 16);
    x *= 9u;
    x = x ^ (x >> 4);
    x *= 0x27d4eb2du;
    x = x ^ (x >> 15);
    x *= 0x85ebca6bu;
    x ^= x >> 13;
    return x;
}

__device__ __forceinline__ float2 normal_pair(uint32_t seed, uint32_t counter, uint32_t line, uint32_t n) {
    const uint32_t h0 = mix32(seed ^ mix32(counter ^ mix32(line * 0x9e3779b9u ^ mix32(n))));
    const uint32_t h1 = mix32(h0 ^ 0x68bc21ebu);
    const float u1 = ((h0 >> 8) + 1u) * (1.0f / 16777217.0f);  // (0, 1]
    const float u2 = (h1 >> 8) * (1.0f / 16777216.0f);         // [0, 1)
    const float rad = sqrtf(-2.0f * logf(u1));
    float s, co;
    sincospif(2.0f * u2, &s, &co);
    return make_float2(rad * co, rad * s);
}

}  // namespace bcsim_hip
