// Submanifold 3x3x3 convolution, tile form: no pair matrix in memory.
//
// Replaces spconv.SubMConv3d.forward at the xCPE call sites of the reference (model.py:546-552:
// in_channels == out_channels, 3x3x3, bias) where the pair form's round trip of one product row
// per (input, output) pair through HBM is what bounds it.
//
// A work-group owns 32 to 128 consecutive output voxels and keeps their sums as fp32 in MFMA accumulators: a wave holds 32
// output channels of all of them (64 channels: of half of them). From the tile's pair list (plan_tiles_kernel) it makes a
// table of the row that every output reads at every tap, and walks the taps that occur in the tile: the rows of a tap go
// from memory to LDS without passing through registers (buffer_load ... lds, 16 bytes a lane, 16-byte pieces swizzled by
// the row), a row per output, while the tap before is multiplied. An output without the tap has an offset past the
// end of the buffer, for which the load's own range check writes zeros: nothing is read for it, nothing is branched on.
// Groups of 32 outputs without the tap are not multiplied. Sums are fp32 in tap order whatever the tile: the same bits on
// every run and for every tile size, closer to the exact sums than the pair form (which rounds every product row).
//
// The weights come in fragment order (ptv3_subm_conv_pack_weight): the 16 bytes lane l needs for
// (tap, 32-channel slice, 16-channel step) are stored at consecutive addresses over the lanes, so a
// wave fetches a fragment as one contiguous KB straight into registers, one tap ahead.
//
// What bounds it: large levels the matrix cores - 70 % of the (tap, 32 outputs) of a level occur where 36 % of the pairs
// do, and what is multiplied runs at 750 TFLOP/s of the 1090 a large product reaches; small ones a tile's chain of taps,
// 20 us for 32 outputs to 38 for 128. Measured (fp16, MI355X), against gathering through registers into the row of the output
// with two chunks in flight, launches back to back: 128 channels, 149k voxels of 9.8 pairs 167 -> 117 us, 371k 339 -> 257, 36k
// 54 -> 39; 64 channels, 20k voxels of 5.3 pairs 18.9 (sparse tiles) -> 14.6. In a traced forward 146k take 122 us. Tried: 64-channel slices with three in flight (125 us at 149k), waves of
// 64 x 64 (137), 256 channels (93k voxels 274 - 300 us against 344 in pair form, 37k 131 - 153 against 122: half of the products
// are of absent neighbours, and those of the pair form are not).
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include "common.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));   // a caller's vector may start at any of its elements
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));

template <typename T> struct TileOps;
template <> struct TileOps<_Float16> {
    typedef f16x8 v8;
    typedef f16x4 v4;
    static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float a, float b) {
        f32x2 f = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
    }
};
template <> struct TileOps<__bf16> {
    typedef bf16x8 v8;
    typedef bf16x4 v4;
    static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float a, float b) {
        f32x2 f = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
    }
};

constexpr int CT_THREADS = 256;
constexpr int CT_TAPS = 27;
constexpr int CT_IN_MASK = (1 << 24) - 1;

// weight (c, taps, c) -> fragment order: piece ((t * c/32 + slice) * c/16 + step) * 64 + lane holds
// input channels 16 step + 8 (lane / 32) .. + 8 of output channel 32 slice + lane % 32 at tap t
template <typename T>
__global__ __launch_bounds__(CT_THREADS) void pack_weight_kernel(const T* __restrict__ w, int c, int taps,
                                                                 T* __restrict__ packed) {
    const int64_t total = (int64_t)taps * c * c / 8;
    const int64_t idx = (int64_t)blockIdx.x * CT_THREADS + threadIdx.x;
    if (idx >= total) return;
    const int lane = (int)(idx % 64);
    int64_t r = idx / 64;
    const int steps = c / 16, slices = c / 32;
    const int s = (int)(r % steps);
    r /= steps;
    const int sl = (int)(r % slices);
    const int t = (int)(r / slices);
    const int co = 32 * sl + lane % 32, k = 16 * s + 8 * (lane / 32);
    *(u32x4*)(packed + idx * 8) = *(const u32x4*)(w + ((int64_t)co * taps + t) * c + k);
}

// the same for several weights in one launch: job j owns blocks first_block[j] .. first_block[j + 1]
__global__ __launch_bounds__(CT_THREADS) void pack_weight_batch_kernel(const ptv3_pack_job* __restrict__ jobs, int n_jobs) {
    const int j = ptv3_job_of_block(jobs, n_jobs);
    const ptv3_pack_job job = jobs[j];
    const int c = job.channels, taps = job.taps;
    if (c < 32 || c % 32 != 0 || taps < 1) return;   // a row no *_blocks() helper would have sized: touch nothing
    const int64_t total = (int64_t)taps * c * c / 8;
    const int64_t idx = ((int64_t)blockIdx.x - job.first_block) * CT_THREADS + threadIdx.x;
    if (idx < 0 || idx >= total) return;
    const int lane = (int)(idx % 64);
    int64_t r = idx / 64;
    const int steps = c / 16, slices = c / 32;
    const int st = (int)(r % steps);
    r /= steps;
    const int sl = (int)(r % slices);
    const int t = (int)(r / slices);
    const int co = 32 * sl + lane % 32, k = 16 * st + 8 * (lane / 32);
    const uint16_t* w = (const uint16_t*)job.weight;   // both half types are 16-bit patterns here
    *(u32x4*)((uint16_t*)job.packed + idx * 8) = *(const u32x4*)(w + ((int64_t)co * taps + t) * c + k);
}

// output-major pair words from the tap-major lists: slot_pair[pair_slot[q]] = tap(q) << 24 | pair_in[q]
__global__ __launch_bounds__(CT_THREADS) void plan_slots_kernel(const int32_t* __restrict__ tap_ptr, int taps,
                                                                const int32_t* __restrict__ pair_in,
                                                                const int32_t* __restrict__ pair_slot, int64_t n_pairs,
                                                                int32_t* __restrict__ slot_pair) {
    __shared__ int32_t tp[129];
    for (int i = threadIdx.x; i <= taps; i += CT_THREADS) tp[i] = tap_ptr[i];
    __syncthreads();
    const int64_t q = (int64_t)blockIdx.x * CT_THREADS + threadIdx.x;
    if (q >= n_pairs) return;
    int lo = 0, hi = taps;   // largest t with tp[t] <= q: the (non-empty) tap that holds q
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (tp[mid] <= (int32_t)q) lo = mid; else hi = mid;
    }
    slot_pair[pair_slot[q]] = (int32_t)((uint32_t)lo << 24 | (uint32_t)pair_in[q]);
}

constexpr int CT_TV = 128;          // output voxels per tile of the lists (at 128 channels tiles of 96 as well)
constexpr int CT_TILE_WORDS = 32;   // int32 per tile in tile_tap: 28 tap starts (relative), the tile's first pair

// Per tile of blockDim.x (96 or 128) consecutive voxels: its pairs sorted by tap, inside a tap by output voxel.
// tile_tap[tile][t] = first pair of tap t relative to the tile's first pair (t = 27: the tile's pair
// count), [28] = the tile's first pair; tile_pair[.] = voxel inside the tile << 24 | input row, in that
// order; vox_taps[i] = bit t set when voxel i has a neighbour at tap t.
__global__ __launch_bounds__(CT_TV) void plan_tiles_kernel(const int32_t* __restrict__ row_ptr,
                                                           const int32_t* __restrict__ slot_pair, int64_t n,
                                                           int32_t* __restrict__ tile_tap, uint32_t* __restrict__ tile_pair,
                                                           uint32_t* __restrict__ vox_taps) {
    __shared__ int32_t wave_cnt[2][32], tstart[32];
    const int tid = threadIdx.x, lane = tid % PTV3_WAVE, wave = tid / PTV3_WAVE;
    const int64_t v0 = (int64_t)blockIdx.x * blockDim.x;
    const bool live = v0 + tid < n;
    int s_lo = 0, s_hi = 0;
    if (live) {
        s_lo = row_ptr[v0 + tid];
        s_hi = row_ptr[v0 + tid + 1];
    }
    const int32_t base = row_ptr[v0];
    uint32_t mine = 0;
    for (int s = s_lo; s < s_hi; ++s) mine |= 1u << (((uint32_t)slot_pair[s] >> 24) & 31);
    if (live) vox_taps[v0 + tid] = mine;
    for (int t = 0; t < CT_TAPS; ++t) {
        const uint64_t bal = __ballot((mine >> t) & 1u);
        if (lane == 0) wave_cnt[wave][t] = __popcll(bal);
    }
    __syncthreads();
    if (wave == 0) {
        const int c = lane < CT_TAPS ? wave_cnt[0][lane] + wave_cnt[1][lane] : 0;
        int x = c;
#pragma unroll
        for (int off = 1; off < 32; off <<= 1) {
            const int y = __shfl_up(x, off, PTV3_WAVE);
            if (lane >= off) x += y;
        }
        if (lane < 32) {
            tstart[lane] = x - c;
            int32_t word = x - c;           // lanes 27.. hold the total
            if (lane == 28) word = base;
            tile_tap[(int64_t)blockIdx.x * CT_TILE_WORDS + lane] = word;
        }
    }
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
    int s = s_lo;   // a voxel's slots follow tap order
    for (int t = 0; t < CT_TAPS; ++t) {
        const bool has = (mine >> t) & 1u;
        const uint64_t bal = __ballot(has);
        if (has) {
            const int pos = tstart[t] + (wave == 1 ? wave_cnt[0][t] : 0) + __popcll(bal & below);
            tile_pair[base + pos] = (uint32_t)tid << 24 | ((uint32_t)slot_pair[s] & CT_IN_MASK);
            ++s;
        }
    }
}

constexpr int CG_THREADS = 256;
constexpr uint32_t CG_ABSENT = 0xFFFFFF00u;   // offset of a row that is not there: past fewer than 2^24 rows of 256 bytes

// G groups of 32 outputs; `sub` work-groups share a tile of the lists; DMA = 0: feat does not start at a multiple of 16 bytes
template <typename T, int C, int G, int DMA>
__global__ __launch_bounds__(CG_THREADS, 2) void conv_gather_kernel(
    const T* __restrict__ feat, int64_t n, const T* __restrict__ packed_w, const T* __restrict__ bias,
    const int32_t* __restrict__ tile_tap, const uint32_t* __restrict__ tile_pair, int sub, T* __restrict__ out) {
    typedef typename TileOps<T>::v8 v8;
    typedef typename TileOps<T>::v4 v4;
    constexpr int WC = C / 32, WR = 4 / WC, NG = G / WR, KS = C / 16;   // waves across channels and outputs, groups of a wave
    constexpr int R = 32 * G, LPR = C / 8, ROWS = PTV3_WAVE / LPR;      // lanes of a row, rows of a load
    constexpr int PER = R / ROWS / 4;                                   // loads of a wave per tap
    static_assert(WC * WR == 4 && NG * WR == G && PER * ROWS * 4 == R, "four waves share channels, outputs and loads");
    // apart, so that the compiler sees that reading one does not wait for the loads into the other
    __shared__ __align__(16) T rows_a[R * C];
    __shared__ __align__(16) T rows_b[R * C];
    __shared__ uint32_t src[CT_TAPS * R];         // byte offset of the row an output reads at a tap
    __shared__ int32_t starts[CT_TAPS + 1];
    __shared__ uint32_t groups[CT_TAPS];          // groups in which a tap occurs
    __shared__ int32_t taps[CT_TAPS + 3];         // tap | groups << 8 of the taps that occur, then tap 0 with no group
    __shared__ int32_t n_taps;

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / PTV3_WAVE), lane = tid % PTV3_WAVE;
    const int col = lane & 31, hf = lane >> 5;
    const int wc = wave % WC, wr = wave / WC;
    // work-group ids go round the XCDs: every XCD works through one contiguous eighth of the tiles, so that tiles
    // which gather the same neighbour rows meet in one L2
    const int id = xcd_chunked_id(blockIdx.x, gridDim.x);
    const int tile = id / sub, first = id % sub * R;   // this work-group's outputs inside the tile of the lists
    const int64_t v0 = (int64_t)tile * (sub * R) + first;
    const int nv = (int)min((int64_t)R, n - v0);
    if (nv <= 0) return;

    const int32_t* tt = tile_tap + (int64_t)tile * CT_TILE_WORDS;
    const int total = tt[CT_TAPS];
    const uint32_t* tp = tile_pair + tt[28];
    if (tid <= CT_TAPS) starts[tid] = tt[tid];
    if (tid < CT_TAPS) groups[tid] = 0u;
    for (int e = tid; e < CT_TAPS * R; e += CG_THREADS) src[e] = CG_ABSENT;
    u32x2 b4[4] = {};
    if (bias)
#pragma unroll
        for (int q = 0; q < 4; ++q) b4[q] = *(const u32x2_a2*)(bias + wc * 32 + 8 * q + 4 * hf);
    __syncthreads();
    for (int e = tid; e < total; e += CG_THREADS) {
        const uint32_t word = tp[e];
        const int o = (int)(word >> 24) - first;
        if (o < 0 || o >= R) continue;
        int t = 0, hi = CT_TAPS;   // the tap of pair e: the largest t with starts[t] <= e
        while (hi - t > 1) {
            const int mid = (t + hi) >> 1;
            if (starts[mid] <= e) t = mid; else hi = mid;
        }
        src[t * R + o] = (word & CT_IN_MASK) * (uint32_t)(C * sizeof(T));
        atomicOr(&groups[t], 1u << (o >> 5));
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t here = lane < CT_TAPS ? groups[lane] : 0u;
        const uint64_t any = __ballot(here != 0u);
        const int count = __popcll(any);
        if (here) taps[__popcll(any & ((1ull << lane) - 1ull))] = lane | (int)(here << 8);
        if (lane >= count && lane < CT_TAPS + 3) taps[lane] = 0;
        if (lane == 0) n_taps = count;
    }
    __syncthreads();
    const int count = __builtin_amdgcn_readfirstlane(n_taps);

    f32x16 acc[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4 b = __builtin_bit_cast(v4, b4[q]);
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[g][4 * q + k] = (float)b[k];
        }

    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)feat, 0, (int)(uint32_t)(n * (int64_t)(C * sizeof(T))), 0x00020000);
    u32x4 w_a[KS], w_b[KS];
    const T* wbase = packed_w + ((int64_t)wc * KS * PTV3_WAVE + lane) * 8;
    auto weights = [&](int t, u32x4 (&w)[KS]) {
        const T* p = wbase + (int64_t)t * (WC * KS * PTV3_WAVE * 8);
#pragma unroll
        for (int i = 0; i < KS; ++i) w[i] = *(const u32x4*)(p + i * PTV3_WAVE * 8);
    };
    const uint32_t* my_src = src + wave * (PER * ROWS) + lane / LPR;
    auto gather = [&](int t, T* buf) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int at = (wave * PER + j) * ROWS;   // 1 KB of LDS, lane after lane: the swizzle is in what a lane reads
            const uint32_t row = my_src[t * R + j * ROWS], off = row + (uint32_t)(((lane % LPR) ^ ((at + lane / LPR) & 7)) * 16);
            if constexpr (DMA) {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(buf + at * C), 16, (int)off,
                                                         0, 0, 0);
            } else {
                u32x4 piece = {};
                if (row != CG_ABSENT) piece = *(const u32x4_a2*)((const char*)feat + off);
                *(u32x4*)(buf + at * C + lane * 8) = piece;
            }
        }
    };
    auto multiply = [&](int here, const T* buf, const u32x4 (&w)[KS]) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (!(here >> (wr * NG + g) & 1)) continue;
            const T* row = buf + ((wr * NG + g) * 32 + col) * C;
            u32x4 x[KS];
#pragma unroll
            for (int i = 0; i < KS; ++i) x[i] = *(const u32x4*)(row + ((2 * i + hf) ^ (col & 7)) * 8);
#pragma unroll
            for (int i = 0; i < KS; ++i)
                acc[g] = TileOps<T>::mfma(__builtin_bit_cast(v8, w[i]), __builtin_bit_cast(v8, x[i]), acc[g]);
        }
    };
    int now = __builtin_amdgcn_readfirstlane(taps[0]), next = __builtin_amdgcn_readfirstlane(taps[1]);
    gather(now & 31, rows_a);
    weights(now & 31, w_a);
    // The barrier: everyone's rows of this tap are in LDS, and everyone is through with the buffer of the tap before, which
    // takes the next one's. Past the last tap, tap 0 is gathered and not multiplied.
    auto step = [&](int i, T* mine, T* ahead, const u32x4 (&w)[KS], u32x4 (&w_ahead)[KS]) {
        const int after = taps[i + 2];
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        gather(next & 31, ahead);
        weights(next & 31, w_ahead);
        multiply(now >> 8, mine, w);
        now = next;
        next = __builtin_amdgcn_readfirstlane(after);
    };
    for (int i = 0; i < count; i += 2) {
        step(i, rows_a, rows_b, w_a, w_b);
        if (i + 1 < count) step(i + 1, rows_b, rows_a, w_b, w_a);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // ---- sums -> halfs in LDS by output row -> out, 16 bytes per lane
    // acc[g][v]: output channel 32 wc + 8 (v / 4) + 4 hf + v % 4 of output (wr NG + g) 32 + col
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = (wr * NG + g) * 32 + col;
            *(u32x2*)(rows_a + r * C + ((wc * 4 + q) ^ (r & 7)) * 8 + 4 * hf) =
                (u32x2){TileOps<T>::pack2(acc[g][4 * q], acc[g][4 * q + 1]), TileOps<T>::pack2(acc[g][4 * q + 2], acc[g][4 * q + 3])};
        }
    __syncthreads();
    for (int e = tid; e < nv * LPR; e += CG_THREADS) {
        const int r = e / LPR, pc = e % LPR;
        *(u32x4*)(out + (v0 + r) * C + pc * 8) = *(const u32x4*)(rows_a + r * C + (pc ^ (r & 7)) * 8);
    }
}

// The time of a launch at 128 channels whose fullest CU gets k work-groups of `groups` x 32 outputs and holds `at_once` of them,
// in tenths of a us: once + each k + round ceil(k / at_once). Fitted to 2.5k - 220k voxels of 8 - 10 pairs: 38 us for one
// work-group of 128 outputs a CU, 51 for two, 77 for three (measured 38, 53, 77); 32 outputs 20 us, 64 26, 96 31. A level of
// more or fewer pairs is slower or faster whatever the groups: at 5, 16 and 24 pairs a voxel from 3k to 400k voxels the row
// that comes out cheapest was the fastest of the four each time, at 9 pairs but once (3 %). A constant below zero is the
// fit's: the least a row comes to is 180. Larger levels take 128 outputs, the least per output.
struct GatherCost { int groups, once, each, round, at_once; };
constexpr GatherCost GATHER_COST[4] = {{1, 100, 80, 0, 1}, {2, -10, 70, 200, 3}, {3, 20, 90, 195, 2}, {4, 126, 129, 130, 2}};
int64_t gather_cost(int64_t n, const GatherCost& c) {
    const int64_t k = ptv3_ceil_div(ptv3_ceil_div(n, 32 * c.groups), (int64_t)ptv3_cus());
    return c.once + c.each * k + c.round * ptv3_ceil_div(k, (int64_t)c.at_once);
}

// groups per work-group on lists of tile_voxels outputs: the cheapest that divides the tile; 64 channels: two up to two work-groups
// a CU (30k voxels: 15.7 us against 17.5 with four), four on larger levels (40k: 19.9 against 22.5, 150k: 47 against 53)
int gather_groups(int64_t n, int c, int tile_voxels) {
    if (c == 64) return n <= 2 * ptv3_cus() * 64 ? 2 : 4;
    const GatherCost* best = nullptr;
    for (const GatherCost& g : GATHER_COST)
        if (tile_voxels % (32 * g.groups) == 0 && (!best || gather_cost(n, g) < gather_cost(n, *best))) best = &g;
    return best->groups;
}

template <typename T, int C, int G>
int launch_gather(const void* feat, int64_t n, int tile_voxels, const void* packed_w, const void* bias, const int32_t* tile_tap,
                  const uint32_t* tile_pair, void* out, hipStream_t stream) {
    const int sub = tile_voxels / (32 * G);
    const bool dma = (uintptr_t)feat % 16 == 0;
    hipLaunchKernelGGL((dma ? conv_gather_kernel<T, C, G, 1> : conv_gather_kernel<T, C, G, 0>),
                       dim3((unsigned)(ptv3_ceil_div(n, tile_voxels) * sub)), dim3(CG_THREADS), 0, stream, (const T*)feat, n,
                       (const T*)packed_w, (const T*)bias, tile_tap, tile_pair, sub, (T*)out);
    PTV3_RETURN_LAUNCH();
}

template <typename T>
int dispatch_tiles(const void* feat, int64_t n, int c, int tile_voxels, const void* packed_w, const void* bias,
                   const int32_t* tile_tap, const uint32_t* tile_pair, void* out, hipStream_t stream) {
    const int g = gather_groups(n, c, tile_voxels);
#define PTV3_GATHER(C, G) \
    if (c == C && g == G) return launch_gather<T, C, G>(feat, n, tile_voxels, packed_w, bias, tile_tap, tile_pair, out, stream)
    PTV3_GATHER(64, 2);
    PTV3_GATHER(64, 4);
    PTV3_GATHER(128, 1);
    PTV3_GATHER(128, 2);
    PTV3_GATHER(128, 3);
    PTV3_GATHER(128, 4);
#undef PTV3_GATHER
    return PTV3_ESHAPE;
}

}  // namespace

extern "C" int ptv3_conv_plan_slots(const int32_t* tap_ptr, int taps, const int32_t* pair_in, const int32_t* pair_slot,
                                    int64_t n_pairs, int32_t* slot_pair, void* stream_) {
    if (taps < 1 || taps > 128 || n_pairs < 0) return PTV3_EINVAL;
    if (n_pairs == 0) return PTV3_OK;
    if (!tap_ptr || !pair_in || !pair_slot || !slot_pair) return PTV3_EINVAL;
    hipLaunchKernelGGL(plan_slots_kernel, dim3((unsigned)ptv3_ceil_div(n_pairs, CT_THREADS)), dim3(CT_THREADS), 0,
                       (hipStream_t)stream_, tap_ptr, taps, pair_in, pair_slot, n_pairs, slot_pair);
    PTV3_RETURN_LAUNCH();
}

// 128, or at 128 channels 96 where three groups of 32 a work-group are the cheapest: 146k voxels are six work-groups of 96 on the
// fullest CU (114 us), nine of 64 (119) or five of 128 (118); 60k are two of 128 (53), four of 64 (67) or three of 96 (72)
extern "C" int ptv3_conv_tile_voxels(int64_t n, int channels) {
    if (channels != 128) return 128;
    const int64_t three = gather_cost(n, GATHER_COST[2]);
    for (const GatherCost& g : GATHER_COST)
        if (g.groups != 3 && gather_cost(n, g) <= three) return 128;
    return 96;
}

extern "C" int64_t ptv3_conv_plan_tile_count(int64_t n) { return n < 0 ? 0 : ptv3_ceil_div(n, CT_TV); }

extern "C" int64_t ptv3_conv_plan_tile_count_sized(int64_t n, int tile_voxels) {
    return (n < 0 || (tile_voxels != 96 && tile_voxels != 128)) ? 0 : ptv3_ceil_div(n, tile_voxels);
}

extern "C" int ptv3_conv_plan_tiles_sized(const int32_t* row_ptr, const int32_t* slot_pair, int64_t n, int taps,
                                          int tile_voxels, int32_t* tile_tap, int32_t* tile_pair, int32_t* vox_taps,
                                          void* stream_) {
    if (n < 0 || n >= (1ll << 24)) return PTV3_EINVAL;
    if (taps != CT_TAPS || (tile_voxels != 96 && tile_voxels != 128)) return PTV3_ESHAPE;
    if (n == 0) return PTV3_OK;
    if (!row_ptr || !slot_pair || !tile_tap || !tile_pair || !vox_taps) return PTV3_EINVAL;
    hipLaunchKernelGGL(plan_tiles_kernel, dim3((unsigned)ptv3_ceil_div(n, tile_voxels)), dim3(tile_voxels), 0,
                       (hipStream_t)stream_, row_ptr, slot_pair, n, tile_tap, (uint32_t*)tile_pair, (uint32_t*)vox_taps);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_conv_plan_tiles(const int32_t* row_ptr, const int32_t* slot_pair, int64_t n, int taps,
                                    int32_t* tile_tap, int32_t* tile_pair, int32_t* vox_taps, void* stream_) {
    return ptv3_conv_plan_tiles_sized(row_ptr, slot_pair, n, taps, CT_TV, tile_tap, tile_pair, vox_taps, stream_);
}

extern "C" int ptv3_subm_conv_pack_weight(const void* weight, int dtype, int channels, int taps, void* packed,
                                          void* stream_) {
    if (channels < 32 || channels % 32 != 0 || taps < 1) return PTV3_ESHAPE;
    if (dtype != PTV3_F16 && dtype != PTV3_BF16) return PTV3_ESHAPE;
    if (!weight || !packed) return PTV3_EINVAL;
    const int64_t total = (int64_t)taps * channels * channels / 8;
    const dim3 grid((unsigned)ptv3_ceil_div(total, CT_THREADS));
    // both half types are 16-bit patterns here: one instantiation moves either
    hipLaunchKernelGGL(pack_weight_kernel<_Float16>, grid, dim3(CT_THREADS), 0, (hipStream_t)stream_,
                       (const _Float16*)weight, channels, taps, (_Float16*)packed);
    PTV3_RETURN_LAUNCH();
}

extern "C" int64_t ptv3_subm_conv_pack_weight_blocks(int channels, int taps) {
    if (channels < 32 || channels % 32 != 0 || taps < 1) return 0;
    return ptv3_ceil_div((int64_t)taps * channels * channels / 8, CT_THREADS);
}

extern "C" int ptv3_subm_conv_pack_weight_batch(const ptv3_pack_job* jobs, int n_jobs, int64_t n_blocks, void* stream_) {
    if (n_jobs < 0 || n_blocks < 0 || n_blocks > 0x7fffffffLL) return PTV3_EINVAL;
    if (n_jobs == 0 || n_blocks == 0) return PTV3_OK;
    if (!jobs) return PTV3_EINVAL;
    hipLaunchKernelGGL(pack_weight_batch_kernel, dim3((unsigned)n_blocks), dim3(CT_THREADS), 0, (hipStream_t)stream_, jobs,
                       n_jobs);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_subm_conv_tiles_fwd(const void* feat, int dtype, int64_t n, int channels, int taps,
                                        const void* packed_weight, const void* bias, const int32_t* tile_tap,
                                        const int32_t* tile_pair, const int32_t* vox_taps, void* out, void* stream_) {
    return ptv3_subm_conv_tiles_fwd_sized(feat, dtype, n, channels, taps, CT_TV, packed_weight, bias, tile_tap, tile_pair,
                                          vox_taps, out, stream_);
}

extern "C" int ptv3_subm_conv_tiles_fwd_sized(const void* feat, int dtype, int64_t n, int channels, int taps,
                                              int tile_voxels, const void* packed_weight, const void* bias,
                                              const int32_t* tile_tap, const int32_t* tile_pair, const int32_t* vox_taps,
                                              void* out, void* stream_) {
    if (n < 0 || n >= (1ll << 24)) return PTV3_EINVAL;
    if (taps != CT_TAPS) return PTV3_ESHAPE;
    if (dtype != PTV3_F16 && dtype != PTV3_BF16) return PTV3_ESHAPE;
    if (channels != 64 && channels != 128) return PTV3_ESHAPE;
    if (tile_voxels != 128 && !(tile_voxels == 96 && channels == 128)) return PTV3_ESHAPE;
    if (n == 0) return PTV3_OK;
    if (!feat || !packed_weight || !tile_tap || !tile_pair || !vox_taps || !out) return PTV3_EINVAL;
    hipStream_t stream = (hipStream_t)stream_;
    const uint32_t* tp = (const uint32_t*)tile_pair;
    if (dtype == PTV3_F16)
        return dispatch_tiles<_Float16>(feat, n, channels, tile_voxels, packed_weight, bias, tile_tap, tp, out, stream);
    return dispatch_tiles<__bf16>(feat, n, channels, tile_voxels, packed_weight, bias, tile_tap, tp, out, stream);
}
