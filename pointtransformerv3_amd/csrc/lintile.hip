// Linear layers as tiles of the output: out = epilogue(x W^T + b), half precision, any K and N that are multiples of 32.
//
// The row kernels (linear.hip, linearw.hip, mlpwide.hip) give a work-group whole rows and let it stream or hold all weights:
// right for the 10^4 .. 10^6 rows of a large level, but the lowest levels of a scene, and every level of a small one, have
// tens to some thousand rows. Then a handful of work-groups each pull megabytes of weights through one CU's 64 bytes per
// cycle (45 us for the 512-channel MLP of 86 rows on one work-group), and what every launch pays once -- staging, a first
// pass through a long instruction stream -- is most of its time. Two forms:
//   few_kernel          32 x 32 outputs; the four waves take a quarter of the contraction each straight from global memory
//                       into MFMA operands, all loads of up to four steps in flight, and meet in LDS. Bound by one trip to
//                       memory: 2.6 - 4 us a launch up to 512 inputs.
//   linear_tile_kernel  64 x 64 or 128 x 128 outputs, both operands through LDS. Few tiles: bound by the latency of a step
//                       of 64 inputs (0.25 us); many: by the L2 -> CU operand stream (64 FLOP per byte: 540 - 700 TFLOP/s).
// Measured, 1500 rows: 256 -> 1024 12.0 -> 5.2 us, 1024 -> 256 13.2 -> 6.7, 512 -> 512 12.5 -> 4.8, 2048 -> 512 22.4 -> 10.9,
// 256 -> 1024 with the GELU's input kept 21.2 -> 6.0.
#include "lintile.h"
#include "rownorm.h"
#include "rowtile.h"

namespace {

template <typename T> __device__ __forceinline__ f32x4 few_mfma(typename H16<T>::v8 a, typename H16<T>::v8 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 few_mfma<_Float16>(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x4 few_mfma<__bf16>(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Work-group -> tile. Work-groups go to the 8 XCDs round-robin: with few row tiles a column tile's go to one XCD, one after
// the other, and its weights enter one L2; with many a row tile's do, and its rows enter one L2.
enum { TILES_PLAIN = 0, TILES_BY_COLUMN = 1, TILES_BY_ROW = 2 };
__device__ __forceinline__ bool tile_of(const LinArgs& a, int& rt, int& ct) {
    const int id = blockIdx.x, slot = id >> 3, xcd = id & 7;
    if (a.order == TILES_BY_COLUMN) {
        ct = slot / a.row_tiles * 8 + xcd;
        rt = slot % a.row_tiles;
    } else if (a.order == TILES_BY_ROW) {
        rt = slot / a.col_tiles * 8 + xcd;
        ct = slot % a.col_tiles;
    } else {
        rt = id % a.row_tiles;
        ct = id / a.row_tiles;
    }
    return rt < a.row_tiles && ct < a.col_tiles;
}
unsigned tile_grid(LinArgs& a, int rows, int cols) {
    a.row_tiles = (int)ptv3_ceil_div(a.n, rows);
    a.col_tiles = a.nout / cols;
    a.order = a.row_tiles >= 64 ? TILES_BY_ROW : a.col_tiles % 8 == 0 ? TILES_BY_COLUMN : TILES_PLAIN;
    return (unsigned)((a.order == TILES_BY_ROW ? (a.row_tiles + 7) / 8 * 8 : a.row_tiles) * a.col_tiles);
}

// What follows the sum of the products, on eight neighbouring channels c .. c + 7 of rows that `rows` walks; roundings where
// separate layers would have stored. One copy per kind: a launch of a few microseconds pays for every instruction it fetches.
// PRE: the bias and, of a layer that reads one, the second matrix's piece of the one row were asked for by the caller.
template <typename T> struct LinPre { typename H16<T>::v8 bias, other; };
template <typename T, int ACT, bool PRE, typename F>
__device__ __forceinline__ void lin_epilogue(const LinArgs& a, int c, const LinPre<T>& pre, F&& rows) {
    typedef typename H16<T>::v8 v8;
    v8 bias, gamma, beta;
    float mu[8], sc[8];
    if (PRE) bias = pre.bias;
    else if (a.bias) bias = *(const v8*)((const T*)a.bias + c);
    if (ACT >= ACT_BN) {
        if (a.gamma) gamma = *(const v8*)((const T*)a.gamma + c);
        if (a.beta) beta = *(const v8*)((const T*)a.beta + c);
        // one test for all of them: behind a test each, every value was a trip to memory of its own
        float va[8];
        if (a.stats_f32) {
            load8((const float*)a.mean + c, mu);
            load8((const float*)a.var + c, va);
        } else {
            load8((const T*)a.mean + c, mu);
            load8((const T*)a.var + c, va);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) sc[u] = rsqrtf(va[u] + a.bn_eps) * (a.gamma ? (float)gamma[u] : 1.f);
    }
    rows([&](float (&y)[8], int64_t at) {
        v8 keep, other;
        if (PRE) other = pre.other;
        else if (ACT == ACT_GELU_GRAD) other = ptv3_read<true>((const v8*)((const T*)a.aux + at));
        else if (ACT == ACT_NONE && a.resid) other = *(const v8*)((const T*)a.resid + at);
        if (a.bias)
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] += (float)bias[u];
        if (ACT == ACT_NONE && a.resid)
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] += (float)other[u];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (ACT >= ACT_BN) y[u] = (H16<T>::round(y[u]) - mu[u]) * sc[u] + (a.beta ? (float)beta[u] : 0.f);
            if (ACT == ACT_GELU_KEEP) keep[u] = (T)y[u];
            if (ACT == ACT_GELU || ACT == ACT_BN_GELU || ACT == ACT_GELU_KEEP) y[u] = gelu_erf(H16<T>::round(y[u]));
            if (ACT == ACT_GELU_GRAD) y[u] = H16<T>::round(y[u]) * gelu_erf_grad((float)other[u]);
        }
        u32x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = H16<T>::pack2(y[2 * q], y[2 * q + 1]);
        *(u32x4*)((T*)a.out + at) = o;
        if (ACT == ACT_GELU_KEEP) ptv3_write<true>((v8*)((T*)a.aux + at), keep);
    });
}
template <typename T, bool PRE, typename F>
__device__ __forceinline__ void lin_epilogue(const LinArgs& a, int c, const LinPre<T>& pre, F&& rows) {
    switch (a.act) {
        case ACT_NONE: return lin_epilogue<T, ACT_NONE, PRE>(a, c, pre, rows);
        case ACT_GELU: return lin_epilogue<T, ACT_GELU, PRE>(a, c, pre, rows);
        case ACT_GELU_KEEP: return lin_epilogue<T, ACT_GELU_KEEP, PRE>(a, c, pre, rows);
        case ACT_GELU_GRAD: return lin_epilogue<T, ACT_GELU_GRAD, PRE>(a, c, pre, rows);
        case ACT_BN: return lin_epilogue<T, ACT_BN, PRE>(a, c, pre, rows);
        default: return lin_epilogue<T, ACT_BN_GELU, PRE>(a, c, pre, rows);
    }
}

constexpr int FEW_THREADS = 256, FEW_WAVES = 4;
constexpr int64_t FEW_TILES = 208;

// The 32 normalised rows of a work-group, rounded where a launch of its own would have stored them (the same operations as
// layer_norm_kernel's, in the same order), into LDS rows of K + 8. Every column tile makes its rows again: a few KB out of
// L2 against a dependent launch.
template <typename T, int MODE, int K>
__device__ __forceinline__ void front_rows(const LinArgs& a, const LinFront& f, int64_t r0, bool first, T* xs) {
    constexpr int LPR = K / 8, RPP = FEW_THREADS / LPR;   // lanes per row, rows per pass
    const int sub = threadIdx.x % LPR;
    float g[8], b[8], g2[8], b2[8];
    load8((const T*)f.g + sub * 8, g);
    load8((const T*)f.b + sub * 8, b);
    if (MODE == LinFront::NORM_SUM_NORM) {
        load8((const T*)f.g2 + sub * 8, g2);
        load8((const T*)f.b2 + sub * 8, b2);
    }
    constexpr int P = 32 / RPP;
    u32x4 xq[P], oq[P];   // every pass's rows are on the way before the first is waited for
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int64_t r = r0 + p * RPP + threadIdx.x / LPR, at = r < a.n ? r : a.n - 1;   // rows past the end are not stored
        xq[p] = *(const u32x4*)((const T*)a.x + at * K + sub * 8);
        if (MODE == LinFront::NORM_SUM_NORM) oq[p] = *(const u32x4*)((const T*)f.res + at * K + sub * 8);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int r = p * RPP + threadIdx.x / LPR;
        float v[8], mean, rstd;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = H16<T>::lo(xq[p][i]);
            v[2 * i + 1] = H16<T>::hi(xq[p][i]);
        }
        row_stats<LPR>(v, f.eps, mean, rstd);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (v[i] - mean) * rstd * g[i] + b[i];
        if (MODE == LinFront::NORM_SUM_NORM) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[2 * i] = H16<T>::round(H16<T>::round(v[2 * i]) + H16<T>::lo(oq[p][i]));
                v[2 * i + 1] = H16<T>::round(H16<T>::round(v[2 * i + 1]) + H16<T>::hi(oq[p][i]));
            }
            if (first && r0 + r < a.n) store8((T*)f.sum + (r0 + r) * K + sub * 8, v);
            row_stats<LPR>(v, f.eps, mean, rstd);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = (v[i] - mean) * rstd * g2[i] + b2[i];
        }
        u32x4 o4;
#pragma unroll
        for (int q = 0; q < 4; ++q) o4[q] = H16<T>::pack2(v[2 * q], v[2 * q + 1]);
        *(u32x4*)(xs + r * (K + 8) + sub * 8) = o4;
    }
}

// MODE: 0, rows from memory, K of the layer in LinArgs; otherwise what LinFront says, K = KF.
template <typename T, int MB, int NB, int D, int MODE, int KF>
__global__ __launch_bounds__(FEW_THREADS) void few_kernel(LinArgs a, LinFront f) {
    typedef typename H16<T>::v8 v8;
    constexpr int ROWS = MB * 16, COLS = NB * 16, CS = COLS + 4;
    __shared__ float red[FEW_WAVES][ROWS * CS];
    __shared__ __align__(16) T xs[MODE ? ROWS * (KF + 8) : 1];
    int rt, ct;
    if (!tile_of(a, rt, ct)) return;
    const int tid = threadIdx.x, wave = tid / PTV3_WAVE, lane = tid % PTV3_WAVE, lr = lane & 15, lg = lane >> 4;
    const int64_t r0 = (int64_t)rt * ROWS;
    const int c0 = ct * COLS, K = MODE ? KF : a.k, steps = K / 32;
    const T* xr[MB];
    const T* wr[NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int64_t r = r0 + mb * 16 + lr;
        xr[mb] = MODE ? xs + (mb * 16 + lr) * (KF + 8) + lg * 8
                      : (const T*)a.x + (r < a.n ? r : a.n - 1) * K + lg * 8;   // rows past the end are multiplied and not stored
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) wr[nb] = (const T*)a.w + (int64_t)(c0 + nb * 16 + lr) * K + lg * 8;
    f32x4 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = (f32x4){0.f, 0.f, 0.f, 0.f};

    v8 xf[2][D][MB], wf[2][D][NB];   // two sets of D steps: one is multiplied, one on its way
    auto load = [&](v8 (&xv)[D][MB], v8 (&wv)[D][NB], int base, bool rows, bool weights) {   // the wave's steps base, base + 4, ...; the last one again past the end
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const int st = base + i * FEW_WAVES, at = (st < steps ? st : steps - 1) * 32;
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                if (rows) xv[i][mb] = *(const v8*)(xr[mb] + at);
            if (!weights) continue;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) wv[i][nb] = *(const v8*)(wr[nb] + at);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](v8 (&xv)[D][MB], v8 (&wv)[D][NB], int base) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const bool on = base + i * FEW_WAVES < steps;   // zeros past the end, not a branch: the loads stay where they are
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) xv[i][mb] = on ? xv[i][mb] : (v8)0;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) wv[i][nb] = on ? wv[i][nb] : (v8)0;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = few_mfma<T>(wv[i][nb], xv[i][mb], acc[nb][mb]);
        }
    };
    load(xf[0], wf[0], wave, MODE == 0, true);
    // what the epilogue reads is on its way as well: behind the sums it was one more trip to memory
    constexpr int PIECES = COLS / 8;
    static_assert(ROWS * PIECES <= FEW_THREADS, "a thread stores one piece");
    LinPre<T> pre = {};
    const int er = tid / PIECES, ec = c0 + tid % PIECES * 8;
    const bool stores = er < ROWS && r0 + er < a.n;
    const int64_t eat = (r0 + er) * a.nout + ec;
    if (a.bias) pre.bias = *(const v8*)((const T*)a.bias + ec);
    const void* second = a.act == ACT_GELU_GRAD ? a.aux : a.act == ACT_NONE ? a.resid : nullptr;
    if (second && stores) pre.other = *(const v8*)((const T*)second + eat);
    if (MODE) {   // the weights are on their way meanwhile
        front_rows<T, MODE ? MODE : 1, MODE ? KF : 64>(a, f, r0, ct == 0, xs);
        __syncthreads();
        load(xf[0], wf[0], wave, true, false);
    }
    constexpr int ROUND = D * FEW_WAVES;
    for (int base = wave;; base += 2 * ROUND) {
        const bool more = base - wave + ROUND < steps;
        if (more) load(xf[1], wf[1], base + ROUND, true, true);
        multiply(xf[0], wf[0], base);
        if (!more) break;
        const bool again = base - wave + 2 * ROUND < steps;
        if (again) load(xf[0], wf[0], base + 2 * ROUND, true, true);
        multiply(xf[1], wf[1], base + ROUND);
        if (!again) break;
    }
    // acc[nb][mb][e]: output channel nb * 16 + 4 lg + e of row mb * 16 + lr, over this wave's steps
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) *(f32x4*)&red[wave][(mb * 16 + lr) * CS + nb * 16 + 4 * lg] = acc[nb][mb];
    __syncthreads();
    lin_epilogue<T, true>(a, ec, pre, [&](auto&& store) {
        if (!stores) return;
        float y[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f32x4 s = *(const f32x4*)&red[0][er * CS + (ec - c0) + h * 4];
#pragma unroll
            for (int w = 1; w < FEW_WAVES; ++w) s += *(const f32x4*)&red[w][er * CS + (ec - c0) + h * 4];
#pragma unroll
            for (int u = 0; u < 4; ++u) y[h * 4 + u] = s[u];
        }
        store(y, eat);
    });
}

// ---- tiles through LDS ------------------------------------------------------------------------------------------------

constexpr int TL_THREADS = 256, TL_KC = 64, TL_STRIDE = TL_KC + 8;

// A tile of MT * 64 rows x NT * 64 output channels per work-group, a quadrant per wave; both operands staged 64 inputs at a
// time, DEPTH steps ahead in registers, two LDS buffers and one barrier per step.
template <typename T, int MT, int NT, int DEPTH>
__global__ __launch_bounds__(TL_THREADS, 2) void linear_tile_kernel(LinArgs a) {
    typedef typename H16<T>::v8 v8;
    constexpr int XBUF = MT * 64 * TL_STRIDE, WBUF = NT * 64 * TL_STRIDE, OS = NT * 32 + 4;
    constexpr int RPS = TL_THREADS / (TL_KC / 8), XP = MT * 64 / RPS, WP = NT * 64 / RPS;   // rows per pass, pieces per thread
    extern __shared__ __align__(16) unsigned char tl_smem[];
    T* lds = (T*)tl_smem;                              // [2][rows | weights], then a quadrant of sums per wave
    static_assert(4 * 32 * OS * 4 <= 2 * (XBUF + WBUF) * 2, "a wave's 32 rows of sums fit where the operands were");
    int rt, ct;
    if (!tile_of(a, rt, ct)) return;
    const int tid = threadIdx.x, wave = tid / PTV3_WAVE, lane = tid % PTV3_WAVE, col = lane & 31, hf = lane >> 5;
    const int64_t m0 = (int64_t)rt * (MT * 64);
    const int n0 = ct * (NT * 64), K = a.k;
    const int wr = (wave >> 1) * (MT * 32), wc = (wave & 1) * (NT * 32);
    const int srow = tid / (TL_KC / 8), spc = tid % (TL_KC / 8);
    const T* xp[XP];
    const T* wp[WP];
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        const int64_t r = m0 + srow + RPS * i;
        xp[i] = (const T*)a.x + (r < a.n ? r : a.n - 1) * K + spc * 8;   // rows past the end repeat the last one
    }
#pragma unroll
    for (int i = 0; i < WP; ++i) wp[i] = (const T*)a.w + (int64_t)(n0 + srow + RPS * i) * K + spc * 8;
    const int steps = K / TL_KC;                       // a multiple of DEPTH
    u32x4 xr[DEPTH][XP], wr4[DEPTH][WP];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
#pragma unroll
        for (int i = 0; i < XP; ++i) xr[d][i] = *(const u32x4*)(xp[i] + d * TL_KC);
#pragma unroll
        for (int i = 0; i < WP; ++i) wr4[d][i] = *(const u32x4*)(wp[i] + d * TL_KC);
    }
    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][b][v] = 0.f;
    // nothing in flight when the loop is entered: the wait-count bookkeeping of a loop is the union of its entry
    // and its back edge, and with loads pending at entry it settles for draining everything once per trip
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
#pragma unroll
        for (int i = 0; i < XP; ++i) asm volatile("" ::"v"(xr[d][i]));
#pragma unroll
        for (int i = 0; i < WP; ++i) asm volatile("" ::"v"(wr4[d][i]));
    }
    for (int s0 = 0; s0 < steps; s0 += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            T* xb = lds + ((DEPTH % 2 ? s0 + d : d) & 1) * (XBUF + WBUF);   // the buffer of two steps ago: read before the last barrier
            T* wb = xb + XBUF;
#pragma unroll
            for (int i = 0; i < XP; ++i) *(u32x4*)(xb + (srow + RPS * i) * TL_STRIDE + spc * 8) = xr[d][i];
#pragma unroll
            for (int i = 0; i < WP; ++i) *(u32x4*)(wb + (srow + RPS * i) * TL_STRIDE + spc * 8) = wr4[d][i];
            const int sn = s0 + d + DEPTH < steps ? s0 + d + DEPTH : steps - 1;   // past the end: a valid address, never used
#pragma unroll
            for (int i = 0; i < XP; ++i) xr[d][i] = *(const u32x4*)(xp[i] + sn * TL_KC);
#pragma unroll
            for (int i = 0; i < WP; ++i) wr4[d][i] = *(const u32x4*)(wp[i] + sn * TL_KC);
            __syncthreads();
#pragma unroll
            for (int ks = 0; ks < TL_KC / 16; ++ks) {
                u32x4 xf[MT], wf[NT];
#pragma unroll
                for (int i = 0; i < MT; ++i) xf[i] = *(const u32x4*)(xb + (wr + i * 32 + col) * TL_STRIDE + ks * 16 + hf * 8);
#pragma unroll
                for (int b = 0; b < NT; ++b) wf[b] = *(const u32x4*)(wb + (wc + b * 32 + col) * TL_STRIDE + ks * 16 + hf * 8);
#pragma unroll
                for (int b = 0; b < NT; ++b)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
                        acc[i][b] = H16<T>::mfma(__builtin_bit_cast(v8, wf[b]), __builtin_bit_cast(v8, xf[i]), acc[i][b]);
            }
        }
    }
    __syncthreads();   // every wave is through with the operand tiles: their room takes the sums
    // acc[i][b][v]: output channel n0 + wc + b*32 + 8*(v/4) + 4*hf + v%4 of row m0 + wr + i*32 + col
    float* stage = (float*)lds + wave * (32 * OS);
    constexpr int PIECES = NT * 4, RPI = PTV3_WAVE / PIECES;   // 16-byte pieces per row, rows per pass of the wave
    const int orow = lane / PIECES, opc = lane % PIECES;
    lin_epilogue<T, false>(a, n0 + wc + opc * 8, LinPre<T>{}, [&](auto&& store) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
#pragma unroll
            for (int b = 0; b < NT; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *(f32x4*)(stage + col * OS + b * 32 + 8 * q + 4 * hf) =
                        (f32x4){acc[i][b][4 * q], acc[i][b][4 * q + 1], acc[i][b][4 * q + 2], acc[i][b][4 * q + 3]};
            asm volatile("" ::: "memory");
#pragma unroll 2
            for (int it = 0; it < 32 / RPI; ++it) {
                const int r = it * RPI + orow;
                const int64_t row = m0 + wr + i * 32 + r;
                float y[8];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const f32x4 s = *(const f32x4*)(stage + r * OS + opc * 8 + h * 4);
#pragma unroll
                    for (int u = 0; u < 4; ++u) y[h * 4 + u] = s[u];
                }
                if (row < a.n) store(y, row * a.nout + n0 + wc + opc * 8);
            }
            asm volatile("" ::: "memory");
        }
    });
}

template <typename T, int MT, int NT, int DEPTH>
int tile_launch(LinArgs& a, hipStream_t stream) {
    const size_t lds = 2 * (size_t)(MT + NT) * 64 * TL_STRIDE * sizeof(T);
    auto kern = linear_tile_kernel<T, MT, NT, DEPTH>;
    static LdsGrant grant;
    if (const int rc = ptv3_allow_lds((const void*)kern, lds, grant)) return rc;
    const unsigned grid = tile_grid(a, MT * 64, NT * 64);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(TL_THREADS), lds, stream, a);
    PTV3_RETURN_LAUNCH();
}

template <typename T, int D>
int few_launch(LinArgs& a, hipStream_t stream) {
    const unsigned grid = tile_grid(a, 32, 32);
    hipLaunchKernelGGL((few_kernel<T, 2, 2, D, 0, 0>), dim3(grid), dim3(FEW_THREADS), 0, stream, a, LinFront{});
    PTV3_RETURN_LAUNCH();
}

template <typename T, int MODE>
int front_launch(LinArgs& a, const LinFront& f, hipStream_t stream) {
    const unsigned grid = tile_grid(a, 32, 32);
    if (a.k == 64) hipLaunchKernelGGL((few_kernel<T, 2, 2, 1, MODE, 64>), dim3(grid), dim3(FEW_THREADS), 0, stream, a, f);
    else if (a.k == 256) hipLaunchKernelGGL((few_kernel<T, 2, 2, 2, MODE, 256>), dim3(grid), dim3(FEW_THREADS), 0, stream, a, f);
    else return PTV3_ESHAPE;
    PTV3_RETURN_LAUNCH();
}

// Which tile. 32 x 32 while they do not outnumber the CUs (700 rows, 256 -> 256: 3.1 us against 3.7 with 64 x 64, 256 -> 768:
// 5.0 against 4.0) and where 64 does not divide the layer; 128 x 128 once there is three quarters of a work-group per CU
// (3000 rows, 2048 -> 512: 22.7 against 19.2 us; 12000 rows: 37 against 44), later for short contractions whose epilogue reads
// or writes a second matrix (9000 rows, 256 -> 1024: 22 against 18 us; 20000: 32 against 34).
template <typename T>
int lin_tiled_t(LinArgs& a, hipStream_t stream) {
    const int64_t t32 = ptv3_ceil_div(a.n, 32) * (a.nout / 32), t128 = ptv3_ceil_div(a.n, 128) * (a.nout / 128);
    if (a.k % 64 != 0 || a.nout % 64 != 0 || t32 <= FEW_TILES) {
        if (a.k <= 128) return few_launch<T, 1>(a, stream);
        if (a.k <= 256) return few_launch<T, 2>(a, stream);
        return few_launch<T, 4>(a, stream);
    }
    const bool second = (a.act == ACT_GELU_KEEP || a.act == ACT_GELU_GRAD) && a.k <= 256;
    if (a.k % 128 == 0 && a.nout % 128 == 0 && t128 >= (second ? 1024 : 188)) return tile_launch<T, 2, 2, 2>(a, stream);
    if (a.k % 256 == 0) return tile_launch<T, 1, 1, 4>(a, stream);
    return a.k % 128 == 0 ? tile_launch<T, 1, 1, 2>(a, stream) : tile_launch<T, 1, 1, 1>(a, stream);
}

}  // namespace

bool lin_tiled_takes(int k, int nout) { return k >= 32 && k % 32 == 0 && nout >= 32 && nout % 32 == 0; }

// Against the kernels that keep weights on the CU and walk rows (linear.hip; 256 inputs: linearw.hip), by the size of the
// output: those cost 3.5 - 14 us however few the rows and win once every CU has many rows to walk. Where the two meet, in
// outputs: 32 inputs 0.8M, 64: 7M, 128: 6M, 256: 3M (4096 rows of 768); with the second matrix of the GELU's training
// forms 2.5M, -, 19M, 16M. With 512 inputs and more the tiles are the faster form at every size measured (37,000 rows:
// 512 -> 512 31 against 44 us, 512 -> 2048 106 against 127).
bool lin_tiled_pays(int64_t n, int k, int nout, int act) {
    if (!lin_tiled_takes(k, nout)) return false;
    const int64_t size = n * nout;
    if (act == ACT_GELU_KEEP || act == ACT_GELU_GRAD)
        return k >= 512 || size <= (k <= 32 ? 2500000 : k <= 64 ? 20000000 : k <= 128 ? 19000000 : 16000000);
    if (k >= 512 || (k == 256 && act >= ACT_BN)) return true;
    return size <= (k <= 32 ? 800000 : k <= 96 ? (k == 96 ? 1200000 : 7000000) : k <= 192 ? 6000000 : k <= 256 ? 3100000 : 5000000);
}

int lin_tiled(LinArgs& a, int dtype, hipStream_t stream) {
    if (!lin_tiled_takes(a.k, a.nout)) return PTV3_ESHAPE;
    if (ptv3_ceil_div(a.n, 32) * (a.nout / 32) >= (1ll << 30)) return PTV3_EINVAL;
    if (dtype == PTV3_F16) return lin_tiled_t<_Float16>(a, stream);
    if (dtype == PTV3_BF16) return lin_tiled_t<__bf16>(a, stream);
    return PTV3_ESHAPE;
}

// Whether the norm goes into the layer behind it. The launch it replaces costs 3 us and every column tile's own norm 2: with
// 256 inputs while a CU has one tile (block tail of 250 rows 17.0 -> 15.7 us, of 350 no change; then the layer alone takes
// few_kernel as well, and the sums are the same bits), with 64 up to a thousand tiles (1500 rows 13.8 -> 12.1, 4000 14.2 ->
// 14.0; beyond FEW_TILES the layer alone takes linear_tile_kernel, which adds the inputs in one chain where few_kernel adds two
// halves: the same float sums in another order, rounded at the same places). With 512 the norm of 32 rows takes as long as the launch (300 rows 23.2 -> 26.1).
bool lin_front_pays(int64_t n, int k, int nout) {
    const int64_t tiles = ptv3_ceil_div(n, 32) * (nout / 32);
    return k == 64 ? tiles <= 1024 : k == 256 && tiles <= FEW_TILES;
}

int lin_front(LinArgs& a, const LinFront& f, int dtype, hipStream_t stream) {
    if (dtype != PTV3_F16 && dtype != PTV3_BF16) return PTV3_ESHAPE;
    if (a.nout % 32 != 0 || a.n >= (1ll << 31)) return PTV3_ESHAPE;
#define PTV3_FRONT(T)                                                               \
    do {                                                                            \
        if (f.mode == LinFront::NORM) return front_launch<T, LinFront::NORM>(a, f, stream); \
        return front_launch<T, LinFront::NORM_SUM_NORM>(a, f, stream);              \
    } while (0)
    if (dtype == PTV3_F16) PTV3_FRONT(_Float16);
    PTV3_FRONT(__bf16);
#undef PTV3_FRONT
}

// The second half of a block layer by layer: sum = shortcut + attn Wproj^T + b, then sum + fc2(GELU(fc1(LN(sum)))).
// Against the fused kernels, which give a work-group whole rows: at 512 channels one streams 4 MB of weights through a CU
// (53 us whatever the rows, against 21 - 49 us here up to 3000; 62 against 71 at 6000), at 256 (18 us against 15 - 18 up to
// 600 rows) and 64 channels (15.7 us against 11 - 12 up to 3000) a work-group's chain of layers is the longer one.
extern "C" int ptv3_block_tail_few_pays(int64_t n, int channels) {
    return channels == 512 ? n <= 4096 : channels == 256 ? n <= 600 : channels == 64 ? n <= 4096 : 0;
}

extern "C" size_t ptv3_block_tail_few_bytes(int64_t n, int channels) { return n < 0 ? 0 : (size_t)n * channels * 12; }

extern "C" int ptv3_block_tail_few(const void* attn, const void* shortcut, const void* w_proj, const void* b_proj,
                                   const void* ln2_gamma, const void* ln2_beta, float ln2_eps, const void* w1, const void* b1,
                                   const void* w2, const void* b2, int dtype, int64_t n, int channels, void* workspace,
                                   size_t workspace_bytes, void* out, void* stream) {
    if (n < 0 || channels < 64 || channels % 64 != 0) return PTV3_EINVAL;
    if (dtype != PTV3_F16 && dtype != PTV3_BF16) return PTV3_ESHAPE;
    if (n == 0) return PTV3_OK;
    if (!attn || !shortcut || !w_proj || !w1 || !w2 || !workspace || !out) return PTV3_EINVAL;
    if (workspace_bytes < ptv3_block_tail_few_bytes(n, channels)) return PTV3_EWORKSPACE;
    const size_t rows = (size_t)n * channels * 2;
    void *sum = workspace, *normed = (char*)sum + rows, *hidden = (char*)normed + rows;
    hipStream_t s = (hipStream_t)stream;
    auto layer = [&](const void* x, const void* w, const void* b, int k, int nout, int act, const void* resid, void* y) {
        LinArgs a = {};
        a.x = x, a.w = w, a.bias = b, a.n = n, a.k = k, a.nout = nout, a.act = act, a.resid = resid, a.out = y;
        return lin_tiled(a, dtype, s);
    };
    int rc = layer(attn, w_proj, b_proj, channels, channels, ACT_NONE, shortcut, sum);
    if (rc == PTV3_OK && ln2_gamma && ln2_beta && lin_front_pays(n, channels, 4 * channels)) {
        LinArgs a = {};
        LinFront f = {};
        a.x = sum, a.w = w1, a.bias = b1, a.n = n, a.k = channels, a.nout = 4 * channels, a.act = ACT_GELU, a.out = hidden;
        f.mode = LinFront::NORM, f.g = ln2_gamma, f.b = ln2_beta, f.eps = ln2_eps;
        rc = lin_front(a, f, dtype, s);
        if (rc == PTV3_OK) rc = layer(hidden, w2, b2, 4 * channels, channels, ACT_NONE, sum, out);
        return rc;
    }
    if (rc == PTV3_OK)
        rc = ptv3_layer_norm(sum, nullptr, ln2_gamma, ln2_beta, nullptr, nullptr, nullptr, dtype, n, channels, ln2_eps, 0, normed,
                             nullptr, stream);
    if (rc == PTV3_OK) rc = layer(normed, w1, b1, channels, 4 * channels, ACT_GELU, nullptr, hidden);
    if (rc == PTV3_OK) rc = layer(hidden, w2, b2, 4 * channels, channels, ACT_NONE, sum, out);
    return rc;
}

extern "C" int ptv3_linear_gemm_fwd(const void* x, const void* w, const void* bias, const void* resid, int dtype,
                                    int64_t n, int k, int nout, void* out, void* stream) {
    if (n < 0 || k < 1 || nout < 1) return PTV3_EINVAL;
    if (dtype != PTV3_F16 && dtype != PTV3_BF16) return PTV3_ESHAPE;
    if (k % 128 != 0 || nout % 128 != 0) return PTV3_ESHAPE;
    if (n == 0) return PTV3_OK;
    if (!x || !w || !out) return PTV3_EINVAL;
    LinArgs a = {};
    a.x = x, a.w = w, a.bias = bias, a.n = n, a.k = k, a.nout = nout, a.act = ACT_NONE, a.resid = resid, a.out = out;
    return lin_tiled(a, dtype, (hipStream_t)stream);
}
