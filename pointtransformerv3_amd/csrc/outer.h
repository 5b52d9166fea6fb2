// The second half of a weight gradient: adding up the slabs its work-groups left (backward.hip). A caller that queues
// many weight gradients defers these sums and has several done by one launch.
#pragma once
#include "common.h"

struct SlabJob {
    const float* slabs;
    int64_t stride, total;      // floats per slab, of which the first `total` are summed
    int splits;                 // 0: nothing to sum, the result is in place
    float* out;                 // values [0, first)
    int64_t first;
    float* out2;                // values [first, total)
    const int32_t* tap_ptr;     // ranges over pair lists: a tap's values have only the slabs its list reaches
    int taps, k_total;
    int64_t rows_per_split;
};
constexpr int SLAB_JOBS = 16;

// as ptv3_linear_wgrad / ptv3_subm_conv_wgrad / ptv3_subm_conv_wgrad_pairs (half precision, channels in 8s), the sum over
// the slabs left to ptv3_slab_sums; `workspace` must stay until then. The Linear layers of up to 8 jobs, all of as many
// rows, share a launch (two where some have a side below 128 channels); slabs[i] is job i's sum.
struct LinearGrad {
    const void *x, *dy;         // (n, k), (n, nout)
    int64_t n;
    int k, nout;
    float *dweight, *dbias;
};
size_t ptv3_linear_wgrads_bytes(const LinearGrad* jobs, int count);
int ptv3_linear_wgrads_slabs(const LinearGrad* jobs, int count, int dtype, void* workspace, size_t workspace_bytes, SlabJob* slabs,
                             hipStream_t stream);
int ptv3_subm_conv_wgrad_slabs(const void* feat, const void* dout, int dtype, int64_t n, int cin, int cout, const int32_t* nbr,
                               const int32_t* tap_ptr, const int32_t* pair_in, int taps, float* dweight, float* dbias,
                               void* workspace, size_t workspace_bytes, SlabJob* job, hipStream_t stream);
int ptv3_slab_sums(const SlabJob* jobs, int count, hipStream_t stream);
// BatchNorm in training, the sums that its kernels add onto zeroed by the caller, who has many layers: the sums of
// ptv3_batch_norm_stats (2c); then statistics (3c, as there), running averages (both or none) and, of half rows, BatchNorm with
// GELU in one; and ptv3_batch_norm_bwd
int ptv3_batch_norm_sums(const void* x, int dtype, int64_t n, int c, float* sums, hipStream_t stream);
int ptv3_batch_norm_gelu_train(const void* x, int dtype, int64_t n, int c, const float* sums, const void* gamma, const void* beta,
                               float eps, float momentum, float* running_mean, float* running_var, float* stats, void* out,
                               hipStream_t stream);
int ptv3_batch_norm_bwd_onto(const void* x, int x_dtype, const void* dout, int dout_dtype, const float* stats, const void* gamma,
                             const void* beta, int param_dtype, int64_t n, int c, int gelu, int batch_stats, void* dx, int dx_dtype,
                             float* dgamma_dbeta, hipStream_t stream);
// a + b * scale_in -> out32 (float) and, times scale_out, out16 (half): both optional, so are a and the row scales
int ptv3_two_sums(const void* a, int a_dtype, const void* b, int b_dtype, const void* scale_in, const void* scale_out,
                  int scale_dtype, int64_t n, int c, void* out32, void* out16, int out16_dtype, hipStream_t stream);
