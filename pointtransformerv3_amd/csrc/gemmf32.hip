// fp32 products on the matrix cores: Linear layers of the float model and the pair form of the float submanifold
// convolution.
//
// A float is taken as the sum of three bf16, each the rest of the one before rounded: 8 + 8 + 8 bits, all that a float has,
// with a float's range (G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019). Of the nine products of two such floats the six largest are taken, six
// v_mfma_f32_32x32x16_bf16 in 192 cycles where eight v_mfma_f32_32x32x2_f32 take 512; what is left out is 2^-24 of a
// product at most, 2^-27 of it on average. The first pieces' products have a sum of their own, the smaller ones another, put
// together at the end: sixteen products a rounding instead of two, so sums are closer to 64 bits than the float
// instruction's, whatever the operands.
// Error (2-norm, unit normal operands), float instruction -> pieces: K = 6 4.7e-8 -> 2.8e-8, 32 1.03e-7 -> 0.39e-7,
// 64 1.44e-7 -> 0.50e-7, 256 2.87e-7 -> 0.89e-7, 2048 8.1e-7 -> 2.7e-7; rows of one value of order 1 under a weight of 1e-8
// and the rest the other way round, K = 256, 2.87e-7 -> 0.89e-7. (Two halves a float, 22 bits under a fixed scale, three
// products, take 0.75 of the time but lose such rows: 2.3e-4.)
//
// A work-group of four waves owns TM rows x TN outputs. KC inputs of its rows and of its weight rows at a time go
// global -> registers -> pieces in LDS, two buffers and one barrier per step; the loads of two steps are on the way, none of
// them under a condition (a condition made the compiler wait for all of them), and the splitting of the next step is
// scheduled between the products of this one. Bound by the matrix cores and the splitting (VALU), by the latency of a step
// where a launch has few tiles, by memory at 32 and 64 inputs.
// Measured (MI355X; us, float instruction -> pieces): 100k x 64 -> 192 40 -> 35, 36k x 128 -> 384 51 -> 35, 11.6k x 256 -> 1024
// 70 -> 42, 2.1k x 2048 -> 512 93 -> 73, 300 x 512 -> 512 18 -> 13; rows of 1e-6, 100k x 64 -> 64 17.5 -> 16.1; a float forward
// of one room of 100k voxels 10.9 -> 8.5 ms.
#include "bnact.h"
#include "rowtile.h"

namespace {

constexpr int F32_THREADS = 256;
constexpr uint32_t F32_TINY = (127u - 102u) * (1u << 24) - 1u;   // 2^-102 as `least` sees it

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

// Four values of a row of k from place `at` on; places past the row's end read its last ones again, and are made zero
// before they are parked (cut).
template <typename XT, bool VEC> struct Load4;
template <> struct Load4<float, true> {
    typedef f32x4 raw;
    static __device__ __forceinline__ raw at(const float* p, int at, int k) { return *(const f32x4*)(p + min(at, k - 4)); }
    static __device__ __forceinline__ f32x4 value(raw v) { return v; }
    static __device__ __forceinline__ raw cut(raw v, int left) { return left > 0 ? v : (f32x4){0.f, 0.f, 0.f, 0.f}; }
};
template <> struct Load4<float, false> {
    typedef f32x4 raw;
    static __device__ __forceinline__ raw at(const float* p, int at, int k) {
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = p[min(at + j, k - 1)];
        return v;
    }
    static __device__ __forceinline__ f32x4 value(raw v) { return v; }
    static __device__ __forceinline__ raw cut(raw v, int left) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = j < left ? v[j] : 0.f;
        return v;
    }
};
template <> struct Load4<_Float16, true> {
    typedef u32x2 raw;
    static __device__ __forceinline__ raw at(const _Float16* p, int at, int k) { return *(const u32x2*)(p + min(at, k - 4)); }
    static __device__ __forceinline__ f32x4 value(raw v) {
        return (f32x4){H16<_Float16>::lo(v[0]), H16<_Float16>::hi(v[0]), H16<_Float16>::lo(v[1]), H16<_Float16>::hi(v[1])};
    }
    static __device__ __forceinline__ raw cut(raw v, int left) { return left > 0 ? v : (u32x2){0u, 0u}; }
};

// four consecutive values of a row as PIECES pieces, each KC of them behind the one before
template <int PIECES, int KC> __device__ __forceinline__ void park_pieces(unsigned char* at, f32x4 v) {
#pragma unroll
    for (int q = 0; q < PIECES; ++q) {
        u32x2 p;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            p[j] = H16<__bf16>::pack2(v[2 * j], v[2 * j + 1]);
            v[2 * j] -= __builtin_bit_cast(float, p[j] << 16);
            v[2 * j + 1] -= __builtin_bit_cast(float, p[j] & 0xffff0000u);
        }
        *(u32x2*)(at + q * KC * 2) = p;
    }
}
// the least of m and the sizes of v, in the order of their bits; zero is none
__device__ __forceinline__ uint32_t least(uint32_t m, f32x4 v) {
#pragma unroll
    for (int j = 0; j < 4; j += 2)
        m = min(m, min(__builtin_bit_cast(uint32_t, v[j]) * 2u - 1u, __builtin_bit_cast(uint32_t, v[j + 1]) * 2u - 1u));
    return m;
}

template <int TM, int TN, int WM, int WN, int KC, typename XT, typename OT, bool VEC, bool PAIRS>
__global__ __launch_bounds__(F32_THREADS, 2) void gemm_f32_kernel(F32Args g) {
    static_assert(WM * WN == 4 && TM % (32 * WM) == 0 && TN % (32 * WN) == 0, "four waves share the tile");
    constexpr int MT = TM / (32 * WM), NT = TN / (32 * WN);
    constexpr int RL = KC / 4;                  // lanes that hold a row's values of a step, four each
    constexpr int XP = (TM * RL + F32_THREADS - 1) / F32_THREADS, WP = (TN * RL + F32_THREADS - 1) / F32_THREADS;
    constexpr int ROW = 3 * KC * 2 + 16;        // bytes of an LDS row of pieces: rows start in distinct bank groups
    constexpr int STRIDE = KC + 4;              // floats of an LDS row of whole values
    constexpr int XQ = sizeof(XT) == 2 ? 2 : 3;   // pieces of a row's value: 11 bits of a half are in two
    __shared__ __align__(16) unsigned char lds[2][(TM + TN) * ROW];
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
    const int pc = (tid % RL) * 4;
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        int r = (tid + i * F32_THREADS) / RL;
        r = min(r, count - 1);
        const int64_t src = PAIRS ? (int64_t)g.pair_in[start + r] : start + r;
        xrow[i] = (const XT*)g.x + src * g.k;
    }
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const int c = min(col0 + ((tid + i * F32_THREADS) / RL), g.nout - 1);
        wrow[i] = g.w + (int64_t)c * g.w_row + (int64_t)tap * g.w_tap;
    }
    uint32_t tiny = ~0u;   // the least value that is not zero among this thread's pieces
    struct Stage {   // two steps are on the way
        typename Load4<XT, VEC>::raw x[XP];
        f32x4 w[WP];
    } st0, st1;
    auto fetch = [&](Stage& t, int k0) {
#pragma unroll
        for (int i = 0; i < XP; ++i) t.x[i] = Load4<XT, VEC>::at(xrow[i], k0 + pc, g.k);
#pragma unroll
        for (int i = 0; i < WP; ++i) t.w[i] = Load4<float, VEC>::at(wrow[i], k0 + pc, g.k);
    };
    auto trim = [&](Stage& t, int s) {   // the last step of a row that is no whole number of steps
        const int left = g.k - s * KC - pc;
        if (left >= KC - pc) return;
#pragma unroll
        for (int i = 0; i < XP; ++i) t.x[i] = Load4<XT, VEC>::cut(t.x[i], left);
#pragma unroll
        for (int i = 0; i < WP; ++i) t.w[i] = Load4<float, VEC>::cut(t.w[i], left);
    };
    auto park = [&](const Stage& t, int s) {
        unsigned char* to = lds[s & 1] + pc * 2;
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const int e = tid + i * F32_THREADS;
            const f32x4 v = Load4<XT, VEC>::value(t.x[i]);
            if (XQ == 3) tiny = least(tiny, v);
            if (TM * RL % F32_THREADS == 0 || e < TM * RL) park_pieces<XQ, KC>(to + (e / RL) * ROW, v);
        }
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            const int e = tid + i * F32_THREADS;
            tiny = least(tiny, t.w[i]);
            if (TN * RL % F32_THREADS == 0 || e < TN * RL) park_pieces<3, KC>(to + (TM + (e / RL)) * ROW, t.w[i]);
        }
    };

    f32x16 acc[MT][NT], low[MT][NT];   // sums of the first pieces' products, and of the five smaller ones
    const int steps = (g.k + KC - 1) / KC;
    auto clear = [&](f32x16 (&t)[MT][NT]) {
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
            for (int b = 0; b < NT; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) t[a][b][v] = 0.f;
    };

    // step s from buffer s & 1; `t` holds step s + 1 and takes step s + 3
    auto step = [&](int s, Stage& t) {
        trim(t, s + 1);
        const unsigned char* xs = lds[s & 1] + (wm * MT * 32 + col) * ROW + hf * 16;
        const unsigned char* ws = lds[s & 1] + (TM + wn * NT * 32 + col) * ROW + hf * 16;
#pragma unroll
        for (int c = 0; c < KC / 16; ++c) {
            bf16x8 xa[MT][3], wb[NT][3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int off = c * 32 + q * KC * 2;
#pragma unroll
                for (int a = 0; a < MT; ++a)
                    if (q < XQ) xa[a][q] = __builtin_bit_cast(bf16x8, *(const u32x4*)(xs + a * 32 * ROW + off));
#pragma unroll
                for (int b = 0; b < NT; ++b) wb[b][q] = __builtin_bit_cast(bf16x8, *(const u32x4*)(ws + b * 32 * ROW + off));
            }
#pragma unroll
            for (int i = 0; i < 6; ++i)   // the third piece of a row comes last: a half has none, and the same sums
#pragma unroll
                for (int a = 0; a < MT; ++a)
#pragma unroll
                    for (int b = 0; b < NT; ++b) {
                        constexpr int QX[6] = {0, 0, 1, 1, 0, 2}, QW[6] = {0, 1, 0, 1, 2, 0};
                        if (QX[i] >= XQ) continue;
                        f32x16& sum = i == 0 ? acc[a][b] : low[a][b];
                        sum = H16<__bf16>::mfma(xa[a][QX[i]], wb[b][QW[i]], sum);
                    }
        }
        park(t, s + 1);
        fetch(t, (s + 3) * KC);
#pragma unroll
        for (int i = 0; i < KC / 16 * MT * NT * (XQ == 2 ? 5 : 6); ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one product, then the splitting of the next step's values
            __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
        }
        __syncthreads();
    };
    clear(acc);
    clear(low);
    fetch(st0, 0);
    fetch(st1, KC);
    trim(st0, 0);
    park(st0, 0);
    fetch(st0, 2 * KC);
    __syncthreads();
    for (int s = 0; s < steps; s += 2) {
        step(s, st1);
        if (s + 1 < steps) step(s + 1, st0);
    }

    // Where the pieces do not hold every bit - a sum that is not finite (infinities, NaN, values that round past the largest
    // bf16), a value below 2^-102 whose last piece would be subnormal - the work-group takes its tile again on whole floats.
    float odd = 0.f;
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[a][b][v] += low[a][b][v];
                odd = fmaf(acc[a][b][v], 0.f, odd);
            }
    if (__syncthreads_or(odd != 0.f || tiny < F32_TINY)) {
        float* whole = (float*)lds;
        clear(acc);
        for (int s = 0; s < steps; ++s) {
            fetch(st0, s * KC);
            trim(st0, s);
#pragma unroll
            for (int i = 0; i < XP; ++i) {
                const int e = tid + i * F32_THREADS;
                if (TM * RL % F32_THREADS == 0 || e < TM * RL)
                    *(f32x4*)(whole + (e / RL) * STRIDE + pc) = Load4<XT, VEC>::value(st0.x[i]);
            }
#pragma unroll
            for (int i = 0; i < WP; ++i) {
                const int e = tid + i * F32_THREADS;
                if (TN * RL % F32_THREADS == 0 || e < TN * RL) *(f32x4*)(whole + (TM + (e / RL)) * STRIDE + pc) = st0.w[i];
            }
            __syncthreads();
            const float* xs = whole + (wm * MT * 32 + col) * STRIDE + hf;
            const float* ws = whole + (TM + wn * NT * 32 + col) * STRIDE + hf;
#pragma unroll 2
            for (int c = 0; c < KC; c += 2)
#pragma unroll
                for (int a = 0; a < MT; ++a)
#pragma unroll
                    for (int b = 0; b < NT; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[a * 32 * STRIDE + c],
                                                                         ws[b * 32 * STRIDE + c], acc[a][b], 0, 0, 0);
            __syncthreads();
        }
    }

    // acc[a][b][v]: row 8*(v/4) + 4*hf + v%4 of its 32, output `col`: a store instruction writes two 128-byte runs
#pragma unroll
    for (int a = 0; a < MT; ++a) {
        const int r0 = (wm * MT + a) * 32 + 4 * hf;
        int64_t at[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int r = min(r0 + 8 * (v / 4) + (v & 3), count - 1);
            at[v] = (PAIRS ? (int64_t)g.pair_slot[start + r] : start + r) * g.nout;
        }
#pragma unroll
        for (int b = 0; b < NT; ++b) {
            const int c = col0 + (wn * NT + b) * 32 + col;
            if (c >= g.nout) continue;
            const float bias = g.bias ? g.bias[c] : 0.f;
            f32x16 y = acc[a][b];
#pragma unroll
            for (int v = 0; v < 16; ++v) y[v] += bias;
            if (!PAIRS && g.gelu) {
#pragma unroll
                for (int v = 0; v < 16; ++v) y[v] = gelu_f32(y[v]);
            }
            if (!PAIRS && g.resid) {
                f32x16 r;
#pragma unroll
                for (int v = 0; v < 16; ++v) r[v] = g.resid[at[v] + c];
#pragma unroll
                for (int v = 0; v < 16; ++v) y[v] += r[v];
            }
            if (count == TM) {
#pragma unroll
                for (int v = 0; v < 16; ++v) ((OT*)g.out)[at[v] + c] = (OT)y[v];
            } else {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (r0 + 8 * (v / 4) + (v & 3) < count) ((OT*)g.out)[at[v] + c] = (OT)y[v];
            }
        }
    }
}

// Tile of a launch: rounds of work-groups over the CUs times the products of a tile, smaller tiles a little dearer
// for the operands they re-read.
template <typename XT, typename OT, bool VEC, bool PAIRS>
int launch_f32(F32Args& g, int64_t rows, hipStream_t stream) {
    const int extra = PAIRS ? g.taps : 0;   // every tap may end with a partial tile
    const int64_t cus = ptv3_cus();
    auto cost = [&](int tm, int tn, double weight) {
        const int64_t tiles = (rows / tm + (PAIRS ? extra : (rows % tm != 0))) * ptv3_ceil_div(g.nout, tn);
        return (double)ptv3_ceil_div(tiles, cus) * tm * tn * weight;
    };
#define PTV3_TILE(TM, TN, WM, WN, KC)                                                                          \
    do {                                                                                                      \
        const int64_t rt = rows / TM + (PAIRS ? extra : (rows % TM != 0));                                    \
        g.col_tiles = (int)ptv3_ceil_div(g.nout, TN);                                                         \
        if (rt * g.col_tiles >= (1ll << 31)) return PTV3_EINVAL;                                              \
        g.row_tiles = (int)rt;                                                                                \
        hipLaunchKernelGGL((gemm_f32_kernel<TM, TN, WM, WN, KC, XT, OT, VEC, PAIRS>),                             \
                           dim3((unsigned)(rt * g.col_tiles)), dim3(F32_THREADS), 0, stream, g);              \
        PTV3_RETURN_LAUNCH();                                                                                 \
    } while (0)
    if (g.nout <= 32) PTV3_TILE(128, 32, 4, 1, 16);
    const double c11 = cost(128, 128, 1.0), c10 = cost(128, 64, 1.05), c00 = cost(64, 64, 1.12);
    if (g.nout > 64 && c11 <= c10 && c11 <= c00) PTV3_TILE(128, 128, 2, 2, 16);
    if (c10 <= c00) PTV3_TILE(128, 64, 2, 2, 16);
    // steps of 32 inputs halve the barriers of a long row (300 x 512 -> 512 15.3 -> 12.6 us, 11.6k x 1024 -> 256 54 -> 48); a short
    // one is sooner through its first step with 16 (100k x 64 -> 64 15.4 against 16.9)
    if (g.k >= 256) PTV3_TILE(64, 64, 2, 2, 32);
    PTV3_TILE(64, 64, 2, 2, 16);
#undef PTV3_TILE
}

// y (pairs, cout) in output-major slot order -> out[i] = bias + sum of voxel i's slots, V channels per thread. ONCE: see
// pair_segment_sum_kernel (a room of 100k in float 8787 -> 8648 us)
template <int V, bool BN, bool ONCE>
__global__ __launch_bounds__(256) void pair_segment_sum_f32_kernel(const float* __restrict__ y,
                                                                   const int32_t* __restrict__ row_ptr, int64_t n,
                                                                   int cout, PieceDiv groups, const float* __restrict__ bias,
                                                                   float* __restrict__ out, BnGelu bn) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = ptv3_row_of(e, groups);
    if (i >= n) return;
    const int c = (int)(e - i * groups.count) * V;
    vec acc;
#pragma unroll
    for (int k = 0; k < V; ++k) acc[k] = bias ? bias[c + k] : 0.f;
    BnChannels<float, V> norm;
    if constexpr (BN) norm.load(bn, c);
    const int s0 = row_ptr[i], s1 = row_ptr[i + 1];
    const float* src = y + (int64_t)s0 * cout + c;
    for (int s = s0; s < s1; s += 4, src += 4 * (int64_t)cout) {
        vec r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (s + j < s1) r[j] = ptv3_read<ONCE>((const vec*)(src + (int64_t)j * cout));
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (s + j < s1) acc += r[j];
    }
    if constexpr (BN)
#pragma unroll
        for (int k = 0; k < V; ++k) acc[k] = norm.apply(acc[k], k, bn.eps);
    *(vec*)(out + i * cout + c) = acc;
}

bool aligned16(const void* a, const void* b) { return (((uintptr_t)a | (uintptr_t)b) & 15) == 0; }

}  // namespace

int ptv3_subm_conv_pairs_f32(const float* feat, int64_t n, int cin, int taps, int64_t n_pairs, const int32_t* tap_ptr,
                             const int32_t* row_ptr, const int32_t* pair_in, const int32_t* pair_slot,
                             const float* weight, const float* bias, int cout, float* y, float* out,
                             hipStream_t stream, const BnGelu* bn) {
    if (taps > 128 || (bn && cout % 4 != 0)) return PTV3_ESHAPE;
    if (n_pairs > 0) {
        F32Args g = {};
        g.x = feat; g.w = weight; g.w_row = (int64_t)taps * cin; g.w_tap = cin; g.out = y;
        g.n = n_pairs; g.k = cin; g.nout = cout;
        g.tap_ptr = tap_ptr; g.pair_in = pair_in; g.pair_slot = pair_slot; g.taps = taps;
        const int rc = cin % 4 == 0 && aligned16(feat, weight) ? launch_f32<float, float, true, true>(g, n_pairs, stream)
                                    : launch_f32<float, float, false, true>(g, n_pairs, stream);
        if (rc != PTV3_OK) return rc;
    }
    if (cout % 4 == 0) {
        const bool once = n_pairs * cout * 4 > ptv3_l2_bytes();
        auto kern = bn ? (once ? pair_segment_sum_f32_kernel<4, true, true> : pair_segment_sum_f32_kernel<4, true, false>)
                       : (once ? pair_segment_sum_f32_kernel<4, false, true> : pair_segment_sum_f32_kernel<4, false, false>);
        hipLaunchKernelGGL(kern, dim3((unsigned)ptv3_ceil_div(n * (cout / 4), 256)), dim3(256), 0, stream, y, row_ptr, n, cout,
                           ptv3_piece_div(cout / 4), bias, out, bn ? *bn : BnGelu{});
    } else {
        hipLaunchKernelGGL((pair_segment_sum_f32_kernel<1, false, false>), dim3((unsigned)ptv3_ceil_div(n * cout, 256)), dim3(256), 0,
                           stream, y, row_ptr, n, cout, ptv3_piece_div(cout), bias, out, BnGelu{});
    }
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
