// fp32 products on the matrix cores (v_mfma_f32_32x32x2f32: full fp32 operands and accumulation): Linear layers of the
// float model and the pair form of the float submanifold convolution.
//
// A work-group of four waves owns TM rows x TN outputs. 16 inputs of its rows and of its weight rows at a time go
// global -> registers -> LDS (two buffers, one barrier per step); a lane reads four consecutive inputs of its row or
// weight row as one 16-byte LDS word and feeds them to four MFMAs (the inputs of a step are taken in the order
// {j, 4 + j}, the same on both sides). The matrix pipe bounds it: a 32 x 32 x 2 product holds the pipe for 64 cycles and
// needs one register per operand, so LDS and L2 are nearly idle and a plain two-buffer pipeline is enough; the fp32
// rate of the pipe (157 TFLOP/s) is twice what unpacked VALU FMAs could reach.
//
// Measured (MI355X, float model on one room of 100k voxels): the 23 convolutions of a forward take 3.7 ms with their
// segment sums, where one thread per (voxel, output) walking the stored neighbour map took 506 ms; its dense layers
// 5.2 ms, where 64 x 64 tiles of VALU FMAs took 10 ms. Forward 530 -> 11.6 ms. A large product runs at 60 % of the
// 153 TFLOP/s a library reaches on this part.
#include "rowtile.h"

namespace {

constexpr int F32_KC = 16;              // inputs per step
constexpr int F32_STRIDE = F32_KC + 4;  // floats per LDS row: 5 16-byte words, rows start in distinct bank groups
constexpr int F32_THREADS = 256;

struct F32Args {
    const void* x;          // (rows, k) float or half
    const float* w;         // row c of output c: w + c * w_row + tap * w_tap
    int64_t w_row, w_tap;
    const float* bias;      // (nout,) or null
    const float* resid;     // (n, nout) or null
    void* out;              // (n, nout) float or half; PAIRS: the pair rows
    int64_t n;
    int k, nout, gelu, row_tiles, col_tiles;
    // PAIRS
    const int32_t *tap_ptr, *pair_in, *pair_slot;
    int taps;
};

template <typename XT, bool VEC> struct Load4;
template <> struct Load4<float, true> {
    static __device__ __forceinline__ f32x4 at(const float* p, int left) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (left >= 4) v = *(const f32x4*)p;
        return v;
    }
};
template <> struct Load4<float, false> {
    static __device__ __forceinline__ f32x4 at(const float* p, int left) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < left) v[j] = p[j];
        return v;
    }
};
template <> struct Load4<_Float16, true> {
    static __device__ __forceinline__ f32x4 at(const _Float16* p, int left) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (left >= 4) {
            const u32x2 r = *(const u32x2*)p;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                v[2 * j] = H16<_Float16>::lo(r[j]);
                v[2 * j + 1] = H16<_Float16>::hi(r[j]);
            }
        }
        return v;
    }
};

template <int TM, int TN, int WM, int WN, typename XT, typename OT, bool VEC, bool PAIRS>
__global__ __launch_bounds__(F32_THREADS, 2) void gemm_f32_kernel(F32Args g) {
    static_assert(WM * WN == 4 && TM % (32 * WM) == 0 && TN % (32 * WN) == 0, "four waves share the tile");
    constexpr int MT = TM / (32 * WM), NT = TN / (32 * WN);
    constexpr int XP = (TM * 4 + F32_THREADS - 1) / F32_THREADS, WP = (TN * 4 + F32_THREADS - 1) / F32_THREADS;
    __shared__ float lds[2][(TM + TN) * F32_STRIDE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, hf = lane >> 5;
    const int wm = wave / WN, wn = wave % WN;

    const int item = xcd_chunked_id((int)blockIdx.x, g.row_tiles * g.col_tiles);
    const int rt = item / g.col_tiles, col0 = (item % g.col_tiles) * TN;

    int64_t start = (int64_t)rt * TM;
    int count, tap = 0;
    if (PAIRS) {
        // lane l looks at taps l and l + 64: a wave prefix sum over the taps' tile counts finds this tile's tap
        int carry = 0;
        bool found = false;
        count = 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int t = lane + 64 * q;
            const int first = t < g.taps ? g.tap_ptr[t] : 0;
            const int cnt = t < g.taps ? g.tap_ptr[t + 1] - first : 0;
            const int tiles = (cnt + TM - 1) / TM;
            int incl = tiles;
#pragma unroll
            for (int off = 1; off < PTV3_WAVE; off <<= 1) {
                const int v = __shfl_up(incl, off, PTV3_WAVE);
                if (lane >= off) incl += v;
            }
            incl += carry;
            const uint64_t hit = __ballot(rt < incl && rt >= incl - tiles);
            if (hit && !found) {
                found = true;
                const int l = __ffsll((unsigned long long)hit) - 1;
                const int rel = rt - (__shfl(incl, l, PTV3_WAVE) - __shfl(tiles, l, PTV3_WAVE));
                tap = 64 * q + l;
                start = __shfl(first, l, PTV3_WAVE) + rel * TM;
                count = min(TM, __shfl(cnt, l, PTV3_WAVE) - rel * TM);
            }
            carry = __shfl(incl, PTV3_WAVE - 1, PTV3_WAVE);
        }
        if (!found) return;   // the grid is an upper bound on the number of tiles; the whole work-group agrees
    } else {
        count = (int)(g.n - start < TM ? g.n - start : TM);
    }

    // staging: piece e of a tile is 16 bytes of row e / 4; rows and outputs past the end repeat the last one
    const XT* xrow[XP];
    const float* wrow[WP];
    const int pc = (tid & 3) * 4;
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        int r = (tid + i * F32_THREADS) >> 2;
        r = min(r, count - 1);
        const int64_t src = PAIRS ? (int64_t)g.pair_in[start + r] : start + r;
        xrow[i] = (const XT*)g.x + src * g.k + pc;
    }
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const int c = min(col0 + ((tid + i * F32_THREADS) >> 2), g.nout - 1);
        wrow[i] = g.w + (int64_t)c * g.w_row + (int64_t)tap * g.w_tap + pc;
    }
    f32x4 xr[XP], wr[WP];
    auto fetch = [&](int k0) {
        const int left = g.k - k0 - pc;
#pragma unroll
        for (int i = 0; i < XP; ++i) xr[i] = Load4<XT, VEC>::at(xrow[i] + k0, left);
#pragma unroll
        for (int i = 0; i < WP; ++i) wr[i] = Load4<float, VEC>::at(wrow[i] + k0, left);
    };
    auto park = [&](int buf) {
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const int e = tid + i * F32_THREADS;
            if (TM * 4 % F32_THREADS == 0 || e < TM * 4) *(f32x4*)(&lds[buf][(e >> 2) * F32_STRIDE + pc]) = xr[i];
        }
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            const int e = tid + i * F32_THREADS;
            if (TN * 4 % F32_THREADS == 0 || e < TN * 4) *(f32x4*)(&lds[buf][(TM + (e >> 2)) * F32_STRIDE + pc]) = wr[i];
        }
    };

    f32x16 acc[MT][NT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

    const int steps = (g.k + F32_KC - 1) / F32_KC;
    fetch(0);
    park(0);
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
        if (s + 1 < steps) fetch((s + 1) * F32_KC);
        const float* xs = &lds[s & 1][(wm * MT * 32 + col) * F32_STRIDE + hf * 4];
        const float* ws = &lds[s & 1][(TM + wn * NT * 32 + col) * F32_STRIDE + hf * 4];
#pragma unroll
        for (int c = 0; c < F32_KC / 8; ++c) {
            f32x4 xa[MT], wb[NT];
#pragma unroll
            for (int a = 0; a < MT; ++a) xa[a] = *(const f32x4*)(xs + a * 32 * F32_STRIDE + c * 8);
#pragma unroll
            for (int b = 0; b < NT; ++b) wb[b] = *(const f32x4*)(ws + b * 32 * F32_STRIDE + c * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int a = 0; a < MT; ++a)
#pragma unroll
                    for (int b = 0; b < NT; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[a][j], wb[b][j], acc[a][b], 0, 0, 0);
        }
        if (s + 1 < steps) park((s + 1) & 1);
        __syncthreads();
    }

    // acc[a][b][v]: row 8*(v/4) + 4*hf + v%4 of its 32, output `col`: a store instruction writes two 128-byte runs
#pragma unroll
    for (int b = 0; b < NT; ++b) {
        const int c = col0 + (wn * NT + b) * 32 + col;
        if (c >= g.nout) continue;
        const float bias = g.bias ? g.bias[c] : 0.f;
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = (wm * MT + a) * 32 + 8 * (v / 4) + 4 * hf + (v & 3);
                if (r >= count) continue;
                const int64_t at = (PAIRS ? (int64_t)g.pair_slot[start + r] : start + r) * g.nout + c;
                float y = acc[a][b][v] + bias;
                if (!PAIRS) {
                    if (g.gelu) y = 0.5f * y * (1.f + erff(y * 0.70710678118654752f));
                    if (g.resid) y += g.resid[at];
                }
                ((OT*)g.out)[at] = (OT)y;
            }
    }
}

// Tile of a launch: rounds of work-groups over the 256 CUs times the products of a tile, smaller tiles a little dearer
// for the operands they re-read.
template <typename XT, typename OT, bool VEC, bool PAIRS>
int launch_f32(F32Args& g, int64_t rows, hipStream_t stream) {
    const int extra = PAIRS ? g.taps : 0;   // every tap may end with a partial tile
    auto cost = [&](int tm, int tn, double weight) {
        const int64_t tiles = (rows / tm + (PAIRS ? extra : (rows % tm != 0))) * ptv3_ceil_div(g.nout, tn);
        return (double)ptv3_ceil_div(tiles, 256) * tm * tn * weight;
    };
#define PTV3_TILE(TM, TN, WM, WN)                                                                              \
    do {                                                                                                      \
        const int64_t rt = rows / TM + (PAIRS ? extra : (rows % TM != 0));                                    \
        g.col_tiles = (int)ptv3_ceil_div(g.nout, TN);                                                         \
        if (rt * g.col_tiles >= (1ll << 31)) return PTV3_EINVAL;                                              \
        g.row_tiles = (int)rt;                                                                                \
        hipLaunchKernelGGL((gemm_f32_kernel<TM, TN, WM, WN, XT, OT, VEC, PAIRS>),                             \
                           dim3((unsigned)(rt * g.col_tiles)), dim3(F32_THREADS), 0, stream, g);              \
        PTV3_RETURN_LAUNCH();                                                                                 \
    } while (0)
    if (g.nout <= 32) PTV3_TILE(128, 32, 4, 1);
    const double c11 = cost(128, 128, 1.0), c10 = cost(128, 64, 1.05), c00 = cost(64, 64, 1.12);
    if (g.nout > 64 && c11 <= c10 && c11 <= c00) PTV3_TILE(128, 128, 2, 2);
    if (c10 <= c00) PTV3_TILE(128, 64, 2, 2);
    PTV3_TILE(64, 64, 2, 2);
#undef PTV3_TILE
}

// y (pairs, cout) in output-major slot order -> out[i] = bias + sum of voxel i's slots, V channels per thread
template <int V>
__global__ __launch_bounds__(256) void pair_segment_sum_f32_kernel(const float* __restrict__ y,
                                                                   const int32_t* __restrict__ row_ptr, int64_t n,
                                                                   int cout, const float* __restrict__ bias,
                                                                   float* __restrict__ out) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const int groups = cout / V;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * groups) return;
    const int64_t i = e / groups;
    const int c = (int)(e - i * groups) * V;
    vec acc;
#pragma unroll
    for (int k = 0; k < V; ++k) acc[k] = bias ? bias[c + k] : 0.f;
    const int s0 = row_ptr[i], s1 = row_ptr[i + 1];
    const float* src = y + (int64_t)s0 * cout + c;
    for (int s = s0; s < s1; s += 4, src += 4 * (int64_t)cout) {
        vec r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (s + j < s1) r[j] = *(const vec*)(src + (int64_t)j * cout);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (s + j < s1) acc += r[j];
    }
    *(vec*)(out + i * cout + c) = acc;
}

bool aligned16(const void* a, const void* b) { return (((uintptr_t)a | (uintptr_t)b) & 15) == 0; }

}  // namespace

int ptv3_subm_conv_pairs_f32(const float* feat, int64_t n, int cin, int taps, int64_t n_pairs, const int32_t* tap_ptr,
                             const int32_t* row_ptr, const int32_t* pair_in, const int32_t* pair_slot,
                             const float* weight, const float* bias, int cout, float* y, float* out,
                             hipStream_t stream) {
    if (taps > 128) return PTV3_ESHAPE;
    if (n_pairs > 0) {
        F32Args g = {};
        g.x = feat; g.w = weight; g.w_row = (int64_t)taps * cin; g.w_tap = cin; g.out = y;
        g.n = n_pairs; g.k = cin; g.nout = cout;
        g.tap_ptr = tap_ptr; g.pair_in = pair_in; g.pair_slot = pair_slot; g.taps = taps;
        const int rc = cin % 4 == 0 && aligned16(feat, weight) ? launch_f32<float, float, true, true>(g, n_pairs, stream)
                                    : launch_f32<float, float, false, true>(g, n_pairs, stream);
        if (rc != PTV3_OK) return rc;
    }
    if (cout % 4 == 0)
        hipLaunchKernelGGL(pair_segment_sum_f32_kernel<4>, dim3((unsigned)ptv3_ceil_div(n * (cout / 4), 256)), dim3(256),
                           0, stream, y, row_ptr, n, cout, bias, out);
    else
        hipLaunchKernelGGL(pair_segment_sum_f32_kernel<1>, dim3((unsigned)ptv3_ceil_div(n * cout, 256)), dim3(256), 0,
                           stream, y, row_ptr, n, cout, bias, out);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_linear_f32_fwd(const void* x, int x_dtype, const float* w, const float* bias, const float* resid,
                                   int64_t n, int k, int nout, int gelu, void* out, int out_dtype, void* stream_) {
    if (n < 0 || k < 1 || nout < 1) return PTV3_EINVAL;
    if ((x_dtype != PTV3_F32 && x_dtype != PTV3_F16) || (out_dtype != PTV3_F32 && out_dtype != PTV3_F16)) return PTV3_EINVAL;
    const bool vec = k % 4 == 0 && aligned16(x, w);
    if (x_dtype == PTV3_F16 && out_dtype == PTV3_F16) return PTV3_ESHAPE;
    if ((x_dtype == PTV3_F16 || out_dtype == PTV3_F16) && !vec && n > 0) return PTV3_ESHAPE;
    if (n == 0) return PTV3_OK;
    if (!x || !w || !out) return PTV3_EINVAL;
    hipStream_t stream = (hipStream_t)stream_;
    F32Args g = {};
    g.x = x; g.w = w; g.w_row = k; g.bias = bias; g.resid = resid; g.out = out;
    g.n = n; g.k = k; g.nout = nout; g.gelu = gelu; g.taps = 0;
    if (x_dtype == PTV3_F16) return launch_f32<_Float16, float, true, false>(g, n, stream);
    if (out_dtype == PTV3_F16) return launch_f32<float, _Float16, true, false>(g, n, stream);
    return vec ? launch_f32<float, float, true, false>(g, n, stream)
               : launch_f32<float, float, false, false>(g, n, stream);
}
