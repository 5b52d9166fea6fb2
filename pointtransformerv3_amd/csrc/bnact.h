// Inference-mode BatchNorm1d and exact GELU as the epilogue of a reduction (the stem's pair sum, the pooling's segments), to the
// bits of ptv3_bn_act over its stored rows. A pass by itself, it is bound by its launch and trip to memory below 100k rows and
// by memory above: five launches fewer took a float16 forward of 16 clouds of 2k points from 1922 to 1906 us, a bfloat16 one of a
// lidar sweep of 86k from 3324 to 3306, a room of 100k from 3335 to 3324; 400k voxels: 9750, within the runs' spread.
#pragma once
#include "common.h"

struct BnGelu {
    const void *mean, *var;      // running statistics, float where stats_f32, else of the rows' type
    const void *gamma, *beta;    // of the rows' type, or null
    float eps;
    int stats_f32;
};

namespace {

__device__ __forceinline__ float gelu_exact(float x) {
    // 0.5 x (1 + erf(x / sqrt 2)); erf by Abramowitz-Stegun 7.1.26, |error| < 1.5e-7
    const float z = fabsf(x) * 0.70710678118654752f;
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, z, 1.0f));
    float p = fmaf(1.061405429f, t, -1.453152027f);
    p = fmaf(p, t, 1.421413741f);
    p = fmaf(p, t, -0.284496736f);
    p = fmaf(p, t, 0.254829592f);
    const float e = __builtin_amdgcn_exp2f(-z * z * 1.4426950408889634f);
    const float erf_abs = fmaf(-p * t, e, 1.0f);
    const float half_x = 0.5f * x;
    return fmaf(copysignf(erf_abs, x), half_x, half_x);
}

// V neighbouring channels' parameters, asked for together and ahead of the sums they meet: a kernel of few rows is a chain of
// trips to memory, and at its end these were one more (85 against 59 us at 309k x 64 that way).
template <typename T, int V> struct BnChannels {
    typedef T tv __attribute__((ext_vector_type(V)));
    typedef float fv __attribute__((ext_vector_type(V)));
    fv mean, var, gamma, beta;
    __device__ __forceinline__ void load(const BnGelu& bn, int ch) {
        if (bn.stats_f32) {
            mean = *(const fv*)((const float*)bn.mean + ch);
            var = *(const fv*)((const float*)bn.var + ch);
        } else {
            const tv m = *(const tv*)((const T*)bn.mean + ch), v = *(const tv*)((const T*)bn.var + ch);
#pragma unroll
            for (int k = 0; k < V; ++k) {
                mean[k] = (float)m[k];
                var[k] = (float)v[k];
            }
        }
#pragma unroll
        for (int k = 0; k < V; ++k) {
            gamma[k] = 1.f;
            beta[k] = 0.f;
        }
        if (bn.gamma) {
            const tv g = *(const tv*)((const T*)bn.gamma + ch);
#pragma unroll
            for (int k = 0; k < V; ++k) gamma[k] = (float)g[k];
        }
        if (bn.beta) {
            const tv b = *(const tv*)((const T*)bn.beta + ch);
#pragma unroll
            for (int k = 0; k < V; ++k) beta[k] = (float)b[k];
        }
    }
    // x as the reduction would have stored it. Rounded here: from a half the compiler forms v_fma_mixlo_f16, which rounds the last
    // sum once, as it does in ptv3_bn_act; left to the caller's packing it would be rounded to float in between.
    __device__ __forceinline__ float apply(float x, int k, float eps) const {
        return (float)(T)gelu_exact((float)(T)(((float)(T)x - mean[k]) * rsqrtf(var[k] + eps) * gamma[k] + beta[k]));
    }
};

// A channel's mean and biased variance from the sums of bn_stats_kernel, which are around the first row's value
struct BnMoments {
    float mean, var;
};
__device__ __forceinline__ BnMoments bn_moments(float pivot, float s1, float s2, int64_t n) {
    const float m1 = s1 / (float)n;
    return BnMoments{pivot + m1, fmaxf(s2 / (float)n - m1 * m1, 0.f)};
}
// running averages follow (unbiased variance, as torch does)
__device__ __forceinline__ void bn_running(BnMoments m, int64_t n, float momentum, float* mean, float* var) {
    *mean = (1.f - momentum) * *mean + momentum * m.mean;
    const float unbiased = n > 1 ? m.var * ((float)n / (float)(n - 1)) : m.var;
    *var = (1.f - momentum) * *var + momentum * unbiased;
}

}  // namespace

// ptv3_segment_reduce, BatchNorm, GELU. rows: (m, c) scratch, for shapes whose reduction has no such epilogue.
int ptv3_segment_reduce_bn_gelu(const void* src, int dtype, int64_t n, int c, const int64_t* indices, const int64_t* idx_ptr,
                                int64_t m, int op, const BnGelu& bn, void* rows, void* out, hipStream_t stream);
// ptv3_subm_conv_pairs_fwd without a bias, BatchNorm, GELU; y as there
int ptv3_conv_pairs_bn_gelu(const void* feat, int dtype, int64_t n, int cin, int taps, int64_t n_pairs, const int32_t* tap_ptr,
                            const int32_t* row_ptr, const int32_t* pair_in, const int32_t* pair_slot, const void* weight, int cout,
                            const BnGelu& bn, void* y, void* out, hipStream_t stream);
