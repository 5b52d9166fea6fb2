// Batched LSD radix argsort of (k, n) int64 curve codes, with the inverse permutation, and the curve codes
// themselves when the caller starts from coordinates (ptv3_serialize).
//
// Replaces serialization/default.py:8-24 and torch.argsort + scatter_ at model.py:119-126 and :667-674 of the
// reference. Only the significant low bits are sorted (3*depth + batch bits, e.g. 29 instead of 64) in digits of 8 bits,
// or of 9 where that saves a pass; all k rows share every launch (blockIdx.y = row). 1.2 M points in 8 scenes, 4 orders,
// 33 bits: 325 us before these tiles, groups and digits, 195 now; 100k points, 28 bits: 77 and 44; 2,000: 50 and 10.
//   small rows   : up to SMALL_KEYS keys a row is one work-group's: codes, every pass in LDS, order and inverse, in one
//                  launch. (The general path queues a launch per pass and two in front; at 2,000 points each of them
//                  is 5 us of latency.)
//   totals       : one pass over the codes (or over the coordinates, writing the codes) counts, for EVERY pass at
//                  once, how many keys of a row have each digit value (LDS histograms, one global atomic per
//                  work-group, digit and pass; a wave whose digits are all equal, as the scene bits are, adds once).
//   scatter      : one launch per pass. A work-group ranks its tile of keys (stable, by wave-level digit matching),
//                  publishes the tile's digit counts, and adds up the counts in front of it: those of the tiles of
//                  its own group of GROUP tiles, then the sums of the groups in front, GROUP at a time, up to one that
//                  is already inclusive. (All tiles of a launch run at about the same time, so a walk over single
//                  tiles, sixteen at a time, cost a row of 146 tiles nine dependent trips to memory.) A word has its
//                  status in the upper half, the count in the lower, and is written and read with device-scope atomics, so
//                  that the pair is seen whole and seen across the XCDs' L2s. Work-groups are dispatched in launch
//                  order, so everything a tile waits for is already running or done; the wait is bounded all the
//                  same: a tile that has waited for seconds counts the keys in front of it itself.
//                  The tile is put in digit order in LDS first, so that the global writes of one digit are
//                  contiguous runs. Between passes a point travels as (key, 32-bit index); the key is cut to 32
//                  bits where what later passes look at fits (the first pass drops its own digit).
//   inverse      : long rows take a pass of their own over `order`, an XCD a contiguous eighth of the positions: the
//                  scenes of a batch are contiguous there, so one L2 sees the scattered 8-byte stores of one scene
//                  and can put whole lines together (from the last scatter they go out as partial lines).
// Status values grow with the pass number (2 pass + 1: counts, 2 pass + 2: inclusive sums), so the words are
// cleared once per sort, not once per pass. int64 order / inverse appear only at the end.
#include "common.h"
#include "encode_core.h"

namespace {

constexpr int SORT_THREADS = 512;
constexpr int SORT_WAVES = SORT_THREADS / PTV3_WAVE;
constexpr int MAX_RADIX = 512;
constexpr int MAX_PASSES = 8;
constexpr int GROUP = 8;              // tiles per group, and words read at a time
constexpr int SPIN_LIMIT = 1 << 20;   // look-back polls before a tile stops waiting (seconds; never reached)
constexpr int SMALL_THREADS = 1024;
// rows of one work-group: at 4,096 keys 15 us against 20 by the general path, at 8,192 (eight keys a thread) 28 against 23
constexpr int SMALL_KEYS = 4096;
constexpr int MIN_TILE = 2048;        // keys of the smallest scatter tile
// Keys per thread of a scatter tile. Short rows want many work-groups (100k x 4 keys: 44 us with 4, 46 with 8, 52 with
// 12), long ones few tiles to look back over (400k x 4: 89, 81, 89; 1.2 M x 4 at 30 bits: 234, 188, 165).
constexpr int64_t FEW_KEYS = 600000, MANY_KEYS = 2400000;
// from here on `inverse` outgrows an XCD's 4 MB of L2 by so much that it gets a pass of its own: 1.2 M keys a row 236
// against 247 us, 400k 92 against 86
constexpr int64_t INVERSE_APART = 1 << 20;

struct OrderIds { int id[8]; };

struct Points {   // where the codes come from: coordinates, or null and `code` is read
    const int32_t* grid;
    const int64_t* batch;
    int depth;
    OrderIds ids;
};

__device__ __forceinline__ uint64_t point_code(const Points& p, int row, int64_t i) {
    const uint32_t mask = (1u << p.depth) - 1u;   // depth <= 16
    const uint64_t hi = p.batch ? ((uint64_t)p.batch[i] << (3 * p.depth)) : 0ull;
    return hi | ptv3::curve_code(p.ids.id[row], (uint32_t)p.grid[3 * i] & mask, (uint32_t)p.grid[3 * i + 1] & mask,
                                 (uint32_t)p.grid[3 * i + 2] & mask, p.depth);
}

__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t* __restrict__ words, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) words[i] = 0u;
}

// totals[pass][row][digit] += keys of the block with that digit in that pass, all passes from one read
template <int BITS, bool ENCODE>
__global__ __launch_bounds__(SORT_THREADS) void digit_totals_kernel(Points pts, int64_t* __restrict__ code, int64_t n, int items,
                                                                    int passes, int k, uint32_t* __restrict__ totals) {
    constexpr int R = 1 << BITS;
    __shared__ uint32_t hist[MAX_PASSES * R];
    const int row = blockIdx.y, tid = threadIdx.x, lane = tid % PTV3_WAVE;
    for (int e = tid; e < passes * R; e += SORT_THREADS) hist[e] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * items * SORT_THREADS;
    int64_t* row_code = code + (int64_t)row * n;
    for (int j = 0; j < items; ++j) {
        const int64_t i = base + (int64_t)j * SORT_THREADS + tid;
        if (i >= n) break;   // the lanes of a wave that are left stay together
        uint64_t key;
        if (ENCODE) {
            key = point_code(pts, row, i);
            row_code[i] = (int64_t)key;
        } else {
            key = (uint64_t)row_code[i];
        }
        const uint64_t active = __ballot(1);
        for (int p = 0; p < passes; ++p) {
            const uint32_t digit = (uint32_t)(key >> (BITS * p)) & (R - 1);
            const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)digit);
            if (__ballot(digit != first) == 0) {
                if (lane == 0) atomicAdd(&hist[p * R + first], (uint32_t)__popcll(active));   // lane 0 is the lowest i
            } else {
                atomicAdd(&hist[p * R + digit], 1u);
            }
        }
    }
    __syncthreads();
    for (int e = tid; e < passes * R; e += SORT_THREADS) {
        const uint32_t c = hist[e];
        if (c) atomicAdd(&totals[((int64_t)(e / R) * k + row) * R + e % R], c);
    }
}

// A tile's count of one digit: 16 bits of status above 16 bits of count (a tile has fewer keys); a group's: 32 above 32.
using TileWord = uint32_t;
using GroupWord = uint64_t;
template <typename W> constexpr int HALF = sizeof(W) * 4;
template <typename W>
__device__ __forceinline__ W look_load(const W* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename W>
__device__ __forceinline__ void look_store(W* p, uint32_t status, uint32_t count) {
    __hip_atomic_store(p, (W)(((W)status << HALF<W>) | count), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Rank of this lane's key among the keys of its digit that the wave has counted in `hist` so far, and this item's
// lanes in front of it; adds the item to `hist`. What bounds a pass is this VALU work (a middle pass of 4.8 M keys ran
// 154 instructions per key and lane, 19 of its 54 us on all SIMDs): four instructions per digit bit, and instead of an
// atomic's result handed round by the leading lane a plain read in front of its add (the LDS operations of one wave
// execute in order).
template <int BITS, bool ALL>
__device__ __forceinline__ uint32_t wave_rank(uint32_t* hist, uint32_t digit, bool valid) {
    const uint64_t all = ALL ? ~0ull : __ballot(valid);
    uint32_t lo = (uint32_t)all, hi = (uint32_t)(all >> 32);   // lanes with this lane's digit
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
        const uint32_t m = (uint32_t)((int32_t)(digit << (31 - b)) >> 31);   // all ones where the bit is set
        const uint64_t bal = __ballot(m != 0u);
        lo &= ~((uint32_t)bal ^ m);
        hi &= ~((uint32_t)(bal >> 32) ^ m);
    }
    const uint32_t in_front = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
    const uint32_t before = __hip_atomic_load(hist + digit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    __builtin_amdgcn_wave_barrier();
    if ((ALL || valid) && in_front == 0u) atomicAdd(hist + digit, (uint32_t)(__popc(lo) + __popc(hi)));
    __builtin_amdgcn_wave_barrier();
    return before + in_front;
}

__device__ __forceinline__ uint32_t wave_inclusive(uint32_t x, int lane) {
#pragma unroll
    for (int off = 1; off < PTV3_WAVE; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, PTV3_WAVE);
        if (lane >= off) x += y;
    }
    return x;
}

// Sum of the counts of one digit in `count` (at most GROUP) words `step` apart, all read in one round trip, from
// `p` downwards; stops at the first inclusive one when `stop` is given. recount(j): the count that word j stands for, from
// the keys, where `limit` polls have not brought it (every word where limit is negative).
template <typename W, typename Recount>
__device__ __forceinline__ uint32_t look_sum(const W* p, int64_t step, int count, uint32_t s_counts, int limit, bool* stop, Recount recount) {
    constexpr W MASK = ((W)1 << HALF<W>) - 1;
    W w[GROUP];
#pragma unroll
    for (int j = 0; j < GROUP; ++j) w[j] = j < count ? look_load(p - j * step) : (W)0;
    uint32_t sum = 0;
    bool closed = false;
#pragma unroll
    for (int j = 0; j < GROUP; ++j) {
        if (closed || j >= count) continue;
        for (int spin = 0; limit < 0 || (uint32_t)(w[j] >> HALF<W>) < s_counts; ++spin) {
            if (spin >= limit) {
                w[j] = (W)s_counts << HALF<W> | recount(j);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            w[j] = look_load(p - j * step);
        }
        sum += (uint32_t)(w[j] & MASK);
        if (stop) closed = (uint32_t)(w[j] >> HALF<W>) > s_counts;
    }
    if (stop) *stop = closed;
    return sum;
}

template <typename K> struct __align__(2 * sizeof(K)) Keyed { K key; int32_t idx; };   // as a point travels between passes

// The tile's part of a pass. ALL: the tile is full. KL: keys in registers and LDS, KO: keys written (see scatter_kernel).
template <typename KL, typename KO, bool FIRST, bool LAST, int BITS, int ITEMS, bool ALL>
__device__ __forceinline__ void scatter_tile(
    const void* __restrict__ in, int count, int tbase, int shift, int drop, int pass, uint32_t row_total, TileWord* my_word,
    GroupWord* my_group, int tile, int spin_limit, Keyed<KO>* __restrict__ out, int64_t* __restrict__ order,
    int64_t* __restrict__ inverse, KO* __restrict__ sorted, uint32_t (*whist)[1 << BITS], uint32_t* gdelta, uint32_t* wsum,
    uint32_t* rsum, Keyed<KL>* stage) {
    constexpr int R = 1 << BITS;
    const int tid = threadIdx.x, wave = tid / PTV3_WAVE, lane = tid % PTV3_WAVE;
    const int mine = wave * (PTV3_WAVE * ITEMS) + lane;   // first key of this lane in the tile
    Keyed<KL> item[ITEMS];
    uint32_t rank[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int i = mine + j * PTV3_WAVE;
        item[j] = Keyed<KL>{};
        if (ALL || i < count) {
            if (FIRST) item[j] = Keyed<KL>{(KL)((const int64_t*)in)[i], tbase + i};
            else item[j] = ((const Keyed<KL>*)in)[i];
        }
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        rank[j] = wave_rank<BITS, ALL>(whist[wave], (uint32_t)(item[j].key >> shift) & (R - 1), mine + j * PTV3_WAVE < count);
    __syncthreads();
    // thread = digit (whole waves): publish the tile's count; scans over the digits of the tile's and the row's counts
    const uint32_t s_counts = 2u * (uint32_t)pass + 1u, s_sums = s_counts + 1u;
    uint32_t c[SORT_WAVES], total = 0, x = 0, rx = 0;
    if (tid < R) {
#pragma unroll
        for (int w = 0; w < SORT_WAVES; ++w) { c[w] = whist[w][tid]; total += c[w]; }
        look_store(my_word, s_counts, total);
        x = wave_inclusive(total, lane);
        rx = wave_inclusive(row_total, lane);
        if (lane == PTV3_WAVE - 1) { wsum[wave] = x; rsum[wave] = rx; }
    }
    __syncthreads();
    if (tid < R) {
        const int group = tile / GROUP, place = tile % GROUP;
        // keys of this digit in `tiles` tiles from `from` on, all of them in front of this one and therefore full; the
        // pass reads one buffer and writes another, so they stand whatever the other tiles are doing
        auto keys_in = [&](int from, int tiles) {
            constexpr int TILE = SORT_THREADS * ITEMS;
            uint32_t found = 0;
            for (int64_t i = (int64_t)from * TILE - tbase; i < (int64_t)(from + tiles) * TILE - tbase; ++i) {
                const KL key = FIRST ? (KL)((const int64_t*)in)[i] : ((const Keyed<KL>*)in)[i].key;
                found += ((uint32_t)(key >> shift) & (R - 1)) == (uint32_t)tid;
            }
            return found;
        };
        uint32_t own = 0, before = 0;
        if (place > 0)
            own = look_sum(my_word - R, R, place, s_counts, spin_limit, nullptr, [&](int j) { return keys_in(tile - 1 - j, 1); });
        if (place == GROUP - 1) look_store(my_group, group == 0 ? s_sums : s_counts, own + total);
        bool closed = false;
        for (int g = group - 1; g >= 0 && !closed; g -= GROUP)
            before += look_sum(my_group - (int64_t)(group - g) * R, R, g + 1 < GROUP ? g + 1 : GROUP, s_counts, spin_limit, &closed,
                               [&](int j) { return keys_in((g - j) * GROUP, GROUP); });
        if (place == GROUP - 1 && group > 0) look_store(my_group, s_sums, before + own + total);
        uint32_t start = x - total, rstart = rx - row_total;
        for (int w = 0; w < wave; ++w) { start += wsum[w]; rstart += rsum[w]; }
        gdelta[tid] = rstart + before + own - start;
#pragma unroll
        for (int w = 0; w < SORT_WAVES; ++w) { whist[w][tid] = start; start += c[w]; }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        if (ALL || mine + j * PTV3_WAVE < count) stage[whist[wave][(uint32_t)(item[j].key >> shift) & (R - 1)] + rank[j]] = item[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int lp = j * SORT_THREADS + tid;
        if (ALL || lp < count) {
            const Keyed<KL> v = stage[lp];
            const uint32_t pos = gdelta[(uint32_t)(v.key >> shift) & (R - 1)] + (uint32_t)lp;
            if (LAST) {
                order[pos] = v.idx;
                if (inverse) inverse[(uint32_t)v.idx] = pos;
                if (sorted) sorted[pos] = (KO)v.key;
            } else {
                out[pos] = Keyed<KO>{(KO)(v.key >> drop), v.idx};
            }
        }
    }
}

// `drop`: bits that the first pass cuts off its keys (its own digit) so that they fit KO; KL then still holds them.
// totals: this pass's digit totals of every row [k][R]; look: the tiles' published counts [k][tiles][R], glook: the
// groups' [k][groups][R].
template <typename KL, typename KO, bool FIRST, bool LAST, int BITS, int ITEMS>
__global__ __launch_bounds__(SORT_THREADS) void scatter_kernel(
    const void* __restrict__ in, int64_t n, int shift, int drop, int pass, const uint32_t* __restrict__ totals, TileWord* look,
    GroupWord* glook, int tiles, int groups, int spin_limit, Keyed<KO>* __restrict__ out, int64_t* __restrict__ order,
    int64_t* __restrict__ inverse, KO* __restrict__ sorted) {
    constexpr int R = 1 << BITS, TILE = SORT_THREADS * ITEMS;
    __shared__ uint32_t whist[SORT_WAVES][R];   // per wave and digit: count, then start inside the sorted tile
    __shared__ uint32_t gdelta[R];              // global start of the digit's run minus its start inside the tile
    __shared__ uint32_t wsum[SORT_WAVES], rsum[SORT_WAVES];
    extern __shared__ __align__(16) unsigned char sort_smem[];   // the tile in digit order
    const int row = blockIdx.y, tile = blockIdx.x, tid = threadIdx.x;
    for (int e = tid; e < SORT_WAVES * R; e += SORT_THREADS) (&whist[0][0])[e] = 0;
    const uint32_t row_total = tid < R ? totals[row * R + tid] : 0u;   // keys of digit `tid` in the whole row
    __syncthreads();
    const int64_t rbase = (int64_t)row * n, tbase = (int64_t)tile * TILE;
    const void* src = FIRST ? (const void*)((const int64_t*)in + rbase + tbase) : (const void*)((const Keyed<KL>*)in + rbase + tbase);
    TileWord* my_word = look + ((int64_t)row * tiles + tile) * R + tid;
    GroupWord* my_group = glook + ((int64_t)row * groups + tile / GROUP) * R + tid;
    out += rbase;
    order += rbase;
    if (inverse) inverse += rbase;
    if (sorted) sorted += rbase;
    Keyed<KL>* stage = (Keyed<KL>*)sort_smem;
    if (n - tbase >= TILE)
        scatter_tile<KL, KO, FIRST, LAST, BITS, ITEMS, true>(src, TILE, (int)tbase, shift, drop, pass, row_total, my_word, my_group, tile,
                                                             spin_limit, out, order, inverse, sorted, whist, gdelta, wsum, rsum, stage);
    else
        scatter_tile<KL, KO, FIRST, LAST, BITS, ITEMS, false>(src, (int)(n - tbase), (int)tbase, shift, drop, pass, row_total, my_word,
                                                              my_group, tile, spin_limit, out, order, inverse, sorted, whist, gdelta,
                                                              wsum, rsum, stage);
}

constexpr int INV_ITEMS = 8;
__global__ __launch_bounds__(256) void inverse_kernel(const int64_t* __restrict__ order, int64_t n, int blocks, int64_t* __restrict__ inverse) {
    const int64_t rbase = (int64_t)blockIdx.y * n;
    const int64_t base = (int64_t)xcd_chunked_id(blockIdx.x, blocks) * (256 * INV_ITEMS) + threadIdx.x;
    int64_t v[INV_ITEMS];
#pragma unroll
    for (int j = 0; j < INV_ITEMS; ++j) v[j] = base + j * 256 < n ? order[rbase + base + j * 256] : 0;
#pragma unroll
    for (int j = 0; j < INV_ITEMS; ++j)
        if (base + j * 256 < n) inverse[rbase + v[j]] = base + j * 256;
}

// A row of up to SMALL_THREADS * ITEMS keys, sorted by one work-group; `pts.grid`: the codes are made here.
template <typename K, int BITS, int ITEMS>
__global__ __launch_bounds__(SMALL_THREADS) void small_sort_kernel(Points pts, int64_t* __restrict__ code, int n, int passes,
                                                                   int64_t* __restrict__ order, int64_t* __restrict__ inverse,
                                                                   K* __restrict__ sorted) {
    constexpr int R = 1 << BITS, WAVES = SMALL_THREADS / PTV3_WAVE, TILE = SMALL_THREADS * ITEMS;
    extern __shared__ __align__(16) unsigned char small_smem[];
    K* skey = (K*)small_smem;
    uint16_t* sidx = (uint16_t*)(skey + TILE);
    uint32_t(*whist)[R] = (uint32_t(*)[R])(sidx + TILE);
    __shared__ uint32_t wsum[WAVES];
    const int row = blockIdx.x, tid = threadIdx.x, wave = tid / PTV3_WAVE, lane = tid % PTV3_WAVE;
    const int wbase = wave * (PTV3_WAVE * ITEMS) + lane;
    const int64_t rbase = (int64_t)row * n;
    K key[ITEMS];
    uint16_t idx[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int i = wbase + j * PTV3_WAVE;
        key[j] = 0;
        idx[j] = (uint16_t)i;
        if (i < n) {
            if (pts.grid) {
                const uint64_t v = point_code(pts, row, i);
                code[rbase + i] = (int64_t)v;
                key[j] = (K)v;
            } else {
                key[j] = (K)code[rbase + i];
            }
        }
    }
    for (int p = 0; p < passes; ++p) {
        const int shift = BITS * p;
        uint32_t rank[ITEMS];
        for (int e = tid; e < WAVES * R; e += SMALL_THREADS) (&whist[0][0])[e] = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            rank[j] = wave_rank<BITS, false>(whist[wave], (uint32_t)(key[j] >> shift) & (R - 1), wbase + j * PTV3_WAVE < n);
        }
        __syncthreads();
        uint32_t c[WAVES], total = 0, x = 0;
        if (tid < R) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) { c[w] = whist[w][tid]; total += c[w]; }
            x = wave_inclusive(total, lane);
            if (lane == PTV3_WAVE - 1) wsum[wave] = x;
        }
        __syncthreads();
        if (tid < R) {
            uint32_t start = x - total;
            for (int w = 0; w < wave; ++w) start += wsum[w];
#pragma unroll
            for (int w = 0; w < WAVES; ++w) { whist[w][tid] = start; start += c[w]; }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            if (wbase + j * PTV3_WAVE < n) {
                const uint32_t lp = whist[wave][(uint32_t)(key[j] >> shift) & (R - 1)] + rank[j];
                skey[lp] = key[j];
                sidx[lp] = idx[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int i = wbase + j * PTV3_WAVE;
            if (i < n) { key[j] = skey[i]; idx[j] = sidx[i]; }
        }
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int i = wbase + j * PTV3_WAVE;
        if (i < n) {
            order[rbase + i] = idx[j];
            inverse[rbase + idx[j]] = i;
            if (sorted) sorted[rbase + i] = key[j];
        }
    }
}

struct SortWs {
    void* items[2];     // (k, n) of Keyed<uint64_t> (or Keyed<uint32_t>: the same room is reserved either way)
    uint32_t* totals;   // [MAX_PASSES][k][R]
    TileWord* look;     // [k][tiles][R]
    GroupWord* glook;   // [k][groups][R]
    size_t zero_words;  // 32-bit words from `totals` on that are cleared before a sort
    size_t bytes;
};

SortWs carve(void* base, int64_t n, int k, int tile, int radix) {
    SortWs w;
    const int64_t tiles = ptv3_ceil_div(n > 0 ? n : 1, tile), groups = ptv3_ceil_div(tiles, GROUP);
    size_t off = 0;
    char* p = (char*)base;
    for (int i = 0; i < 2; ++i) {
        w.items[i] = (void*)(p + off);
        off += ptv3_align256((size_t)k * n * sizeof(Keyed<uint64_t>));
    }
    const size_t zero_from = off;
    w.totals = (uint32_t*)(p + off);
    off += ptv3_align256((size_t)MAX_PASSES * k * radix * sizeof(uint32_t));
    w.look = (TileWord*)(p + off);
    off += ptv3_align256((size_t)k * tiles * radix * sizeof(TileWord));
    w.glook = (GroupWord*)(p + off);
    off += ptv3_align256((size_t)k * groups * radix * sizeof(GroupWord));
    w.zero_words = (off - zero_from) / sizeof(uint32_t);
    w.bytes = off;
    return w;
}

struct Job {
    Points pts;
    int64_t* code;
    int64_t n;
    int k, key_bits, passes;
    int64_t *order, *inverse;
    void* sorted;
    void* workspace;
    hipStream_t stream;
    int spin_limit = SPIN_LIMIT;
};

template <typename K, int BITS, int ITEMS>
int run_small(const Job& j) {
    const size_t lds = (sizeof(K) + 2) * SMALL_THREADS * ITEMS + (SMALL_THREADS / PTV3_WAVE) * (sizeof(uint32_t) << BITS);
    auto kern = small_sort_kernel<K, BITS, ITEMS>;
    static LdsGrant grant;
    if (const int rc = ptv3_allow_lds((const void*)kern, lds, grant)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)j.k), dim3(SMALL_THREADS), lds, j.stream, j.pts, j.code, (int)j.n, j.passes, j.order,
                       j.inverse, (K*)j.sorted);
    return PTV3_OK;
}

template <typename KL, typename KO, bool FIRST, bool LAST, int BITS, int ITEMS>
int run_pass(const Job& j, const SortWs& w, int p, int drop, int64_t* inverse) {
    const int tile = SORT_THREADS * ITEMS;
    const int tiles = (int)ptv3_ceil_div(j.n, tile), groups = (int)ptv3_ceil_div(tiles, GROUP);
    const size_t lds = sizeof(Keyed<KL>) * tile;
    auto kern = scatter_kernel<KL, KO, FIRST, LAST, BITS, ITEMS>;
    static LdsGrant grant;
    if (const int rc = ptv3_allow_lds((const void*)kern, lds, grant)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)j.k), dim3(SORT_THREADS), lds, j.stream,
                       FIRST ? (const void*)j.code : w.items[(p & 1) ^ 1], j.n, BITS * p - (FIRST ? 0 : drop), FIRST ? drop : 0, p,
                       w.totals + ((size_t)p * j.k << BITS), w.look, w.glook, tiles, groups,
                       j.spin_limit, (Keyed<KO>*)w.items[p & 1], j.order, inverse, (KO*)j.sorted);
    return PTV3_OK;
}

// KO: type of the keys between passes
template <typename KO, int BITS, int ITEMS>
int run_passes(const Job& j, int drop) {
    const SortWs w = carve(j.workspace, j.n, j.k, SORT_THREADS * ITEMS, 1 << BITS);
    hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)ptv3_ceil_div((int64_t)w.zero_words, 256)), dim3(256), 0, j.stream,
                       w.totals, (int64_t)w.zero_words);
    // keys per work-group: a thousand work-groups or more while each still shares its table between enough keys
    int64_t items = ptv3_ceil_div(j.n * j.k, (int64_t)SORT_THREADS * 1024);
    items = items < 4 ? 4 : items > 32 ? 32 : items;
    const dim3 grid((unsigned)ptv3_ceil_div(j.n, items * SORT_THREADS), (unsigned)j.k);
    if (j.pts.grid)
        hipLaunchKernelGGL((digit_totals_kernel<BITS, true>), grid, dim3(SORT_THREADS), 0, j.stream, j.pts, j.code, j.n, (int)items,
                           j.passes, j.k, w.totals);
    else
        hipLaunchKernelGGL((digit_totals_kernel<BITS, false>), grid, dim3(SORT_THREADS), 0, j.stream, j.pts, j.code, j.n, (int)items,
                           j.passes, j.k, w.totals);
    const bool apart = j.n >= INVERSE_APART;
    int64_t* inverse = apart ? nullptr : j.inverse;
    for (int p = 0; p < j.passes; ++p) {
        const bool first = p == 0, last = p == j.passes - 1;
        int rc;
        if (first && last) rc = run_pass<KO, KO, true, true, BITS, ITEMS>(j, w, p, 0, inverse);
        else if (first && drop) rc = run_pass<uint64_t, KO, true, false, BITS, ITEMS>(j, w, p, drop, inverse);
        else if (first) rc = run_pass<KO, KO, true, false, BITS, ITEMS>(j, w, p, 0, inverse);
        else if (last) rc = run_pass<KO, KO, false, true, BITS, ITEMS>(j, w, p, drop, inverse);
        else rc = run_pass<KO, KO, false, false, BITS, ITEMS>(j, w, p, drop, inverse);
        if (rc != PTV3_OK) return rc;
    }
    if (apart) {
        const int blocks = (int)ptv3_ceil_div(j.n, 256 * INV_ITEMS);
        hipLaunchKernelGGL(inverse_kernel, dim3((unsigned)blocks, (unsigned)j.k), dim3(256), 0, j.stream, j.order, j.n, blocks, j.inverse);
    }
    return PTV3_OK;
}

template <int BITS>
int run_bits(const Job& j) {
    if (j.n <= SMALL_KEYS) {
        if (j.n <= 2 * SMALL_THREADS) return j.key_bits <= 32 ? run_small<uint32_t, BITS, 2>(j) : run_small<uint64_t, BITS, 2>(j);
        return j.key_bits <= 32 ? run_small<uint32_t, BITS, 4>(j) : run_small<uint64_t, BITS, 4>(j);
    }
    const int drop = j.key_bits > 32 && j.key_bits - BITS <= 32 && !j.sorted ? BITS : 0;
    const bool narrow = j.key_bits <= 32 || drop;
    if (j.n * j.k < FEW_KEYS)
        return narrow ? run_passes<uint32_t, BITS, 4>(j, drop) : run_passes<uint64_t, BITS, 4>(j, 0);
    // (64-bit keys: 16 bytes a point in LDS, a tile of 12 keys a thread would leave one work-group per CU)
    if (j.n * j.k < MANY_KEYS || !narrow)
        return narrow ? run_passes<uint32_t, BITS, 8>(j, drop) : run_passes<uint64_t, BITS, 8>(j, 0);
    return run_passes<uint32_t, BITS, 12>(j, drop);
}

int run(Job& j, size_t workspace_bytes) {
    if (j.n > SMALL_KEYS && (!j.workspace || workspace_bytes < ptv3_argsort_workspace_bytes(j.n, j.k))) return PTV3_EWORKSPACE;
    const int p8 = (j.key_bits + 7) / 8, p9 = (j.key_bits + 8) / 9;
    j.passes = p9 < p8 ? p9 : p8;
    const int rc = p9 < p8 ? run_bits<9>(j) : run_bits<8>(j);
    if (rc != PTV3_OK) return rc;
    PTV3_RETURN_LAUNCH();
}

}  // namespace

extern "C" size_t ptv3_argsort_workspace_bytes(int64_t n, int k) {
    if (n < 0 || k < 1) return 0;
    return carve(nullptr, n, k, MIN_TILE, MAX_RADIX).bytes;
}

// sorted_keys: where the sorted keys of every row go (uint32_t when key_bits <= 32, else uint64_t), or null
int ptv3_argsort_keys(const int64_t* code, int64_t n, int k, int key_bits, int64_t* order, int64_t* inverse,
                      void* sorted_keys, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (n < 0 || k < 1 || k > 65535 || n >= (1ll << 31)) return PTV3_EINVAL;
    if (key_bits < 1 || key_bits > 63) return PTV3_EDEPTH;
    if (n == 0) return PTV3_OK;
    if (!code || !order || !inverse || !workspace) return PTV3_EINVAL;
    // the bits above key_bits are equal across a row (the contract), so cutting the keys to 32 bits keeps the order
    Job j = {Points{}, const_cast<int64_t*>(code), n, k, key_bits, 0, order, inverse, sorted_keys, workspace, stream};
    return run(j, workspace_bytes);
}

extern "C" int ptv3_argsort(const int64_t* code, int64_t n, int k, int key_bits, int64_t* order,
                            int64_t* inverse, void* workspace, size_t workspace_bytes,
                            void* stream_) {
    return ptv3_argsort_keys(code, n, k, key_bits, order, inverse, nullptr, workspace, workspace_bytes,
                             (hipStream_t)stream_);
}

extern "C" int ptv3_argsort_impatient(const int64_t* code, int64_t n, int k, int key_bits, int spin_limit, int64_t* order,
                                      int64_t* inverse, void* workspace, size_t workspace_bytes, void* stream_) {
    if (n < 0 || k < 1 || k > 65535 || n >= (1ll << 31) || spin_limit > SPIN_LIMIT) return PTV3_EINVAL;
    if (key_bits < 1 || key_bits > 63) return PTV3_EDEPTH;
    if (n == 0) return PTV3_OK;
    if (!code || !order || !inverse || !workspace) return PTV3_EINVAL;
    Job j = {Points{}, const_cast<int64_t*>(code), n, k, key_bits, 0, order, inverse, nullptr, workspace, (hipStream_t)stream_, spin_limit};
    return run(j, workspace_bytes);
}

// The curve codes of every order and their argsort; sorted_keys as in ptv3_argsort_keys.
int ptv3_serialize_keys(const int32_t* grid_coord, const int64_t* batch, int64_t n, int depth, const int32_t* order_ids_host, int k,
                        int key_bits, int64_t* code, int64_t* order, int64_t* inverse, void* sorted_keys, void* workspace,
                        size_t workspace_bytes, hipStream_t stream) {
    if (n < 0 || n >= (1ll << 31) || k < 1 || k > 8 || !order_ids_host) return PTV3_EINVAL;
    if (depth < 1 || depth > 16 || key_bits < 1 || key_bits > 63) return PTV3_EDEPTH;
    Job j = {Points{grid_coord, batch, depth, OrderIds{}}, code, n, k, key_bits, 0, order, inverse, sorted_keys, workspace, stream};
    for (int r = 0; r < k; ++r) {
        if (order_ids_host[r] < 0 || order_ids_host[r] > 3) return PTV3_EINVAL;
        j.pts.ids.id[r] = order_ids_host[r];
    }
    if (n == 0) return PTV3_OK;
    if (!grid_coord || !code || !order || !inverse || !workspace) return PTV3_EINVAL;
    return run(j, workspace_bytes);
}

extern "C" int ptv3_serialize(const int32_t* grid_coord, const int64_t* batch, int64_t n, int depth, const int32_t* order_ids_host,
                              int k, int key_bits, int64_t* code, int64_t* order, int64_t* inverse, void* workspace,
                              size_t workspace_bytes, void* stream_) {
    return ptv3_serialize_keys(grid_coord, batch, n, depth, order_ids_host, k, key_bits, code, order, inverse, nullptr, workspace,
                               workspace_bytes, (hipStream_t)stream_);
}
