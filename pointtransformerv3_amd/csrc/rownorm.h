// A row of C channels over C/8 neighbouring lanes of a wave, 8 channels a lane: loads, stores and LayerNorm statistics, in
// the one order of additions that every kernel on such rows shares (norm.hip, lintile.hip).
#pragma once
#include "common.h"

namespace {

template <typename T> struct Vec8 { T v[8]; };

template <typename T>
__device__ __forceinline__ void load8(const T* p, float (&f)[8]) {
    const Vec8<T> r = *(const Vec8<T>*)p;
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = (float)r.v[i];
}
template <typename T>
__device__ __forceinline__ void store8(T* p, const float (&f)[8]) {
    Vec8<T> r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r.v[i] = (T)f[i];
    *(Vec8<T>*)p = r;
}

template <typename T> __device__ __forceinline__ float round_to(float v) { return (float)(T)v; }

// statistics of 8 values per lane over the LPR lanes of a row
template <int LPR>
__device__ __forceinline__ void row_stats(const float (&v)[8], float eps, float& mean, float& rstd) {
    constexpr int C = 8 * LPR;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += v[i];
#pragma unroll
    for (int o = 1; o < LPR; o <<= 1) s += __shfl_xor(s, o, PTV3_WAVE);
    mean = s * (1.f / C);
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) q += (v[i] - mean) * (v[i] - mean);
#pragma unroll
    for (int o = 1; o < LPR; o <<= 1) q += __shfl_xor(q, o, PTV3_WAVE);
    rstd = rsqrtf(q * (1.f / C) + eps);
}

}  // namespace
