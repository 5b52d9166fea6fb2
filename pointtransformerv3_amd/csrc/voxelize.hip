// Voxelisation in front of the model: coordinates -> grid coordinates, one point kept per voxel.
//
// What Pointcept's data pipeline does on the host before PointTransformerV3.forward sees a batch
// (the model's own fallback, model.py:88-96, only derives grid_coord): per scene,
// grid_coord = floor((coord - min over the scene) / grid_size), and of the points that fall into one
// voxel the first in input order is kept. Here on the device, in input order, deterministic:
//   scene_min        per-scene minimum of every axis;
//   split_count, split_scan, split   points to 64 .. 4096 parts by a hash of their voxel, as (voxel key, point) pairs;
//   part             one work-group per part: table of its voxels in LDS, first point of every voxel to its members;
//   count/scan/assign   kept flags -> positions, the kept points' grid coordinates and indices, scene ends;
//   inverse          voxel of every input point.
// Bound by memory (about 130 bytes move per point). One table of all voxels in device memory cost two atomics per point
// on lines that eight L2 caches hand to each other (170 us for 1.56M points in 3 scenes); a part's table never leaves the
// CU (part 30 us, split 22, split_count and split_scan 13). Every point is read four times instead, in order, from the
// last-level cache. All kernels of that size: 409 -> 149 us, with the rows of three arrays gathered behind them (41 -> 26).
#include "voxelhash.h"

namespace {

constexpr int VX_THREADS = 512;
constexpr int VX_WAVES = VX_THREADS / PTV3_WAVE;
constexpr int VX_ITEMS = 8;
constexpr int VX_TILE = VX_THREADS * VX_ITEMS;   // points per work-group of the streaming kernels
constexpr uint64_t VX_EMPTY = ~0ull;
// A part holds 1024 .. 2048 points on average where n allows: its table fills LDS to at most half, and 64 parts at
// least keep the launch wide for the smallest inputs. Beyond 4096 parts a tile's runs would be single points; parts
// of more voxels than a table holds (from 12M points on, or by accident of the hash) take their table in memory.
constexpr int VX_MIN_PART_BITS = 6, VX_MAX_PART_BITS = 12, VX_PART = 2048;
constexpr int VX_SLOTS = 4096, VX_FILL = 3072;

struct VoxWs {
    uint64_t* keys;       // [n] voxel keys, part by part
    int32_t* point;       // [n] the points they belong to
    uint64_t* table;      // [2n] tables of parts that do not fit LDS: part p's at twice its first pair
    int32_t* table_first; // [2n]
    int32_t* rep;         // [n] the point kept of the voxel of every point
    int32_t* pos;         // [n] position among the kept points, of points that are kept
    uint32_t* tile_parts; // [tiles][parts] points per tile and part, then their places within the part
    uint32_t* part_size;  // [parts]
    uint32_t* tile_kept;  // [tiles]
    uint32_t* scene_min;  // [nb][3] order-preserving encoding of the float minimum
    int32_t* status;      // [1] non-zero: a grid coordinate does not fit 16 bits
    int64_t tiles;
    int part_bits;
    size_t bytes;
};

VoxWs vx_carve(void* base, int64_t n, int nb) {
    VoxWs w;
    char* p = (char*)base;
    size_t off = 0;
    const size_t m = (size_t)(n > 0 ? n : 1);
    w.tiles = ptv3_ceil_div((int64_t)m, VX_TILE);
    w.part_bits = VX_MIN_PART_BITS;
    while (w.part_bits < VX_MAX_PART_BITS && ((int64_t)VX_PART << w.part_bits) < n) ++w.part_bits;
    const size_t parts = (size_t)1 << w.part_bits;
    auto take = [&](size_t bytes) {
        void* at = p + off;
        off += ptv3_align256(bytes);
        return at;
    };
    w.keys = (uint64_t*)take(m * 8);
    w.point = (int32_t*)take(m * 4);
    w.table = (uint64_t*)take(2 * m * 8);
    w.table_first = (int32_t*)take(2 * m * 4);
    w.rep = (int32_t*)take(m * 4);
    w.pos = (int32_t*)take(m * 4);
    w.tile_parts = (uint32_t*)take((size_t)w.tiles * parts * 4);
    w.part_size = (uint32_t*)take(parts * 4);
    w.tile_kept = (uint32_t*)take((size_t)w.tiles * 4);
    w.scene_min = (uint32_t*)take((size_t)(nb > 0 ? nb : 1) * 3 * 4);
    w.status = (int32_t*)take(4);
    w.bytes = off;
    return w;
}

// floats order like these unsigned integers
__device__ __forceinline__ uint32_t f2ord(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// scene of point i: the first of the scenes lo .. hi whose end is > i (hi where none is)
__device__ __forceinline__ int scene_in(const int64_t* __restrict__ offset, int lo, int hi, int64_t i) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (offset[mid] <= i) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// The points of one tile and the scenes they lie in: nearly always one, found once per tile.
struct VoxTile {
    int64_t base;
    int count, lo, hi;
};
__device__ __forceinline__ VoxTile vx_tile(const int64_t* __restrict__ offset, int nb, int64_t n) {
    VoxTile t;
    t.base = (int64_t)blockIdx.x * VX_TILE;
    t.count = (int)min((int64_t)VX_TILE, n - t.base);
    t.lo = scene_in(offset, 0, nb - 1, t.base);
    t.hi = scene_in(offset, t.lo, nb - 1, t.base + t.count - 1);
    return t;
}

__global__ __launch_bounds__(256) void vx_init_kernel(VoxWs w, int nb, int64_t* __restrict__ offset_out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < 3 * (int64_t)nb) w.scene_min[i] = 0xffffffffu;
    if (i < nb) offset_out[i] = 0;
    if (i == 0) w.status[0] = 0;
}

// Three atomics per tile of one scene: all 24 loads of a thread are in flight together (a wave that walked 1024 points
// with a scene search per step took 71 us for 1.56M points).
__global__ __launch_bounds__(VX_THREADS) void vx_scene_min_kernel(const float* __restrict__ coord, int64_t n,
                                                                  const int64_t* __restrict__ offset, int nb, VoxWs w) {
    __shared__ uint32_t red[VX_WAVES][3];
    const VoxTile t = vx_tile(offset, nb, n);
    const int lane = threadIdx.x % PTV3_WAVE, wave = threadIdx.x / PTV3_WAVE;
    float c[VX_ITEMS][3];
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int64_t i = t.base + min(k * VX_THREADS + (int)threadIdx.x, t.count - 1);   // a point twice does not matter
#pragma unroll
        for (int a = 0; a < 3; ++a) c[k][a] = coord[3 * i + a];
    }
    if (t.lo == t.hi) {
        uint32_t m[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu};
#pragma unroll
        for (int k = 0; k < VX_ITEMS; ++k)
#pragma unroll
            for (int a = 0; a < 3; ++a) m[a] = min(m[a], f2ord(c[k][a]));
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) m[a] = min(m[a], (uint32_t)__shfl_xor((int)m[a], off, PTV3_WAVE));
            if (lane == 0) red[wave][a] = m[a];
        }
        __syncthreads();
        if (threadIdx.x < 3) {
            uint32_t r = red[0][threadIdx.x];
#pragma unroll
            for (int k = 1; k < VX_WAVES; ++k) r = min(r, red[k][threadIdx.x]);
            atomicMin(&w.scene_min[3 * t.lo + threadIdx.x], r);
        }
        return;
    }
    // several scenes: per wave and step where it lies in one of them, per point elsewhere
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int64_t i = t.base + min(k * VX_THREADS + (int)threadIdx.x, t.count - 1);
        const int s = scene_in(offset, t.lo, t.hi, i), s0 = __shfl(s, 0, PTV3_WAVE);
        const bool uniform = __ballot(s != s0) == 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            uint32_t v = f2ord(c[k][a]);
            if (uniform) {
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, off, PTV3_WAVE));
            }
            if (!uniform || lane == 0) atomicMin(&w.scene_min[3 * s + a], v);
        }
    }
}

__device__ __forceinline__ void vx_grid(const float* __restrict__ coord, int64_t i, int s, const VoxWs& w, float grid_size,
                                        int32_t (&g)[3]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) g[a] = (int32_t)floorf((coord[3 * i + a] - ord2f(w.scene_min[3 * s + a])) / grid_size);
}

// part of a voxel: the top bits of the hash; its place in the part's table: the low half
__device__ __forceinline__ uint32_t vx_part(uint64_t hash, int part_bits) { return (uint32_t)(hash >> (64 - part_bits)); }

__device__ __forceinline__ uint64_t vx_key(const float* __restrict__ coord, int64_t i, const int64_t* __restrict__ offset,
                                           const VoxTile& t, const VoxWs& w, float grid_size, bool* fits) {
    const int s = scene_in(offset, t.lo, t.hi, i);
    int32_t g[3];
    vx_grid(coord, i, s, w, grid_size, g);
    *fits = ((g[0] | g[1] | g[2]) >> 16) == 0;   // (negative cannot happen: the minimum is subtracted)
    return vh_block_key(s, g[0], g[1], g[2]);
}

__global__ __launch_bounds__(VX_THREADS) void vx_split_count_kernel(const float* __restrict__ coord, int64_t n,
                                                                    const int64_t* __restrict__ offset, int nb,
                                                                    float grid_size, VoxWs w) {
    extern __shared__ uint32_t cnt[];   // [parts]
    const int parts = 1 << w.part_bits;
    const VoxTile t = vx_tile(offset, nb, n);
    for (int b = threadIdx.x; b < parts; b += VX_THREADS) cnt[b] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int at = k * VX_THREADS + (int)threadIdx.x;
        if (at < t.count) {
            bool fits;
            const uint64_t key = vx_key(coord, t.base + at, offset, t, w, grid_size, &fits);
            if (!fits) w.status[0] = 1;
            atomicAdd(&cnt[vx_part(vh_mix(key), w.part_bits)], 1u);
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < parts; b += VX_THREADS) w.tile_parts[(int64_t)blockIdx.x * parts + b] = cnt[b];
}

// Down the tiles: SEGS threads of a part that take a share of the tiles each, eight tiles in one trip to memory. Bound by that
// trip and by the chain of adding up the shares. Up to 128 tiles (524k points) 16 shares of 64 parts a work-group do it in one
// trip: more shares make the chain longer and the runs that a wave reads shorter. Beyond, 64 shares of 16 parts do. 16 | 64
// shares, us: 10k points 2.1 | 3.3, 50k 3.2 | 3.4, 150k 3.4 | 4.7, 400k 3.7 | 5.2, 530k 5.1 | 4.8, 1.5M 6.5 | 5.4, 3M 11.0 | 9.8.
constexpr int VX_SCAN_THREADS = 1024, VX_SCAN_AT_ONCE = 8;
template <int SEGS>
__global__ __launch_bounds__(VX_SCAN_THREADS) void vx_split_scan_kernel(VoxWs w) {
    constexpr int PARTS = VX_SCAN_THREADS / SEGS;
    static_assert(PARTS <= 1 << VX_MIN_PART_BITS, "whole work-groups");
    __shared__ uint32_t sum[SEGS][PARTS];
    const int parts = 1 << w.part_bits, mine = threadIdx.x % PARTS, seg = threadIdx.x / PARTS;
    const int64_t per = (w.tiles + SEGS - 1) / SEGS, t0 = min(w.tiles, seg * per), t1 = min(w.tiles, t0 + per);
    uint32_t* __restrict__ col = w.tile_parts + blockIdx.x * PARTS + mine;
    uint32_t v[VX_SCAN_AT_ONCE], total = 0;
    for (int64_t t = t0; t < t1; t += VX_SCAN_AT_ONCE) {
#pragma unroll
        for (int k = 0; k < VX_SCAN_AT_ONCE; ++k) v[k] = t + k < t1 ? col[(t + k) * parts] : 0u;
#pragma unroll
        for (int k = 0; k < VX_SCAN_AT_ONCE; ++k) total += v[k];
    }
    sum[seg][mine] = total;
    __syncthreads();
    uint32_t run = 0, all = 0;
#pragma unroll
    for (int s = 0; s < SEGS; ++s) {
        const uint32_t c = sum[s][mine];
        if (s < seg) run += c;
        all += c;
    }
    if (seg == 0) w.part_size[blockIdx.x * PARTS + mine] = all;
    for (int64_t t = t0; t < t1; t += VX_SCAN_AT_ONCE) {
        if (per > VX_SCAN_AT_ONCE)   // else the loads above still stand in v
#pragma unroll
            for (int k = 0; k < VX_SCAN_AT_ONCE; ++k) v[k] = t + k < t1 ? col[(t + k) * parts] : 0u;
#pragma unroll
        for (int k = 0; k < VX_SCAN_AT_ONCE; ++k) {
            if (t + k < t1) col[(t + k) * parts] = run;
            run += v[k];
        }
    }
}

// exclusive sum over the work-group's threads
__device__ __forceinline__ uint32_t vx_block_scan(uint32_t v, uint32_t* total) {
    __shared__ uint32_t wsum[VX_WAVES];
    const int lane = threadIdx.x % PTV3_WAVE, wave = threadIdx.x / PTV3_WAVE;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < PTV3_WAVE; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, PTV3_WAVE);
        if (lane >= off) x += y;
    }
    if (lane == PTV3_WAVE - 1) wsum[wave] = x;
    __syncthreads();
    uint32_t base = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < VX_WAVES; ++k) {
        const uint32_t c = wsum[k];
        if (k < wave) base += c;
        tot += c;
    }
    *total = tot;
    __syncthreads();
    return x + base - v;
}

// A tile's pairs are put in part order in LDS first: runs of four or more go out together.
__global__ __launch_bounds__(VX_THREADS) void vx_split_kernel(const float* __restrict__ coord, int64_t n,
                                                              const int64_t* __restrict__ offset, int nb, float grid_size,
                                                              VoxWs w) {
    extern __shared__ uint64_t lds[];
    const int parts = 1 << w.part_bits;
    uint64_t* skey = lds;                                // [VX_TILE]
    uint32_t* sitem = (uint32_t*)(skey + VX_TILE);       // [VX_TILE] part << 16 | place in the tile
    uint32_t* start = sitem + VX_TILE;                   // [parts] first place of the part within the tile
    uint32_t* dest = start + parts;                      // [parts] where that place goes, less the place
    const VoxTile t = vx_tile(offset, nb, n);
    for (int b = threadIdx.x; b < parts; b += VX_THREADS) start[b] = 0;
    __syncthreads();
    uint64_t key[VX_ITEMS];
    uint32_t part[VX_ITEMS], nth[VX_ITEMS];
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int at = k * VX_THREADS + (int)threadIdx.x;
        if (at < t.count) {
            bool fits;
            key[k] = vx_key(coord, t.base + at, offset, t, w, grid_size, &fits);
            part[k] = vx_part(vh_mix(key[k]), w.part_bits);
            nth[k] = atomicAdd(&start[part[k]], 1u);
        }
    }
    __syncthreads();
    const int per = (parts + VX_THREADS - 1) / VX_THREADS;   // consecutive parts of a thread
    const int b0 = min(parts, (int)threadIdx.x * per), b1 = min(parts, b0 + per);
    uint32_t mine = 0, all = 0, total;
    for (int b = b0; b < b1; ++b) {
        mine += start[b];
        all += w.part_size[b];
    }
    uint32_t run = vx_block_scan(mine, &total), first = vx_block_scan(all, &total);
    for (int b = b0; b < b1; ++b) {
        const uint32_t c = start[b];
        start[b] = run;
        dest[b] = first + w.tile_parts[(int64_t)blockIdx.x * parts + b] - run;
        run += c;
        first += w.part_size[b];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int at = k * VX_THREADS + (int)threadIdx.x;
        if (at < t.count) {
            const uint32_t to = start[part[k]] + nth[k];
            skey[to] = key[k];
            sitem[to] = part[k] << 16 | (uint32_t)at;
        }
    }
    __syncthreads();
    for (int at = threadIdx.x; at < t.count; at += VX_THREADS) {
        const uint32_t item = sitem[at];
        const int64_t to = (int64_t)(dest[item >> 16] + (uint32_t)at);   // modulo 2^32: exact
        w.keys[to] = skey[at];
        w.point[to] = (int32_t)(t.base + (item & 0xffffu));
    }
}

// Rank of point i among the points of its voxel: the point with the lowest rank is kept. Seed 0: the
// index itself (the first point in input order, GridSample's test mode). Otherwise a bijection of the
// 32-bit index keyed by the seed (odd multiplications and xor-shifts, each invertible), so ranks never tie
// and the lowest belongs to a member drawn uniformly -- GridSample's train mode, which takes a random
// member of every voxel.
constexpr uint32_t vx_inverse_of(uint32_t a) {   // modulo 2^32, a odd: every step doubles the bits that are right
    uint32_t x = a;
    for (int i = 0; i < 5; ++i) x *= 2u - a * x;
    return x;
}

__device__ __forceinline__ int32_t vx_rank(int64_t i, uint32_t seed) {
    uint32_t x = (uint32_t)i;
    if (seed != 0u) {
        x ^= seed;
        x *= 0x9E3779B1u;
        x ^= x >> 15;
        x *= 0x85EBCA77u;
        x ^= x >> 13;
        x *= 0xC2B2AE3Du;
        x ^= x >> 16;
        x += seed * 0x27D4EB2Fu;
    }
    return (int32_t)x;
}

// the point of a rank
__device__ __forceinline__ int32_t vx_unrank(int32_t rank, uint32_t seed) {
    uint32_t x = (uint32_t)rank;
    if (seed != 0u) {
        x -= seed * 0x27D4EB2Fu;
        x ^= x >> 16;
        x *= vx_inverse_of(0xC2B2AE3Du);
        x ^= x >> 13 ^ x >> 26;
        x *= vx_inverse_of(0x85EBCA77u);
        x ^= x >> 15 ^ x >> 30;
        x *= vx_inverse_of(0x9E3779B1u);
        x ^= seed;
    }
    return (int32_t)x;
}

// Two passes over a part's pairs with its table: lowest rank of every voxel, then the point it stands for to every
// member. The table lies in LDS, or in memory that this work-group alone uses (relaxed atomic accesses, which no stale
// line of the CU's own cache can serve). False: more than `fill` voxels, nothing was written.
__device__ __forceinline__ bool vx_part_table(const VoxWs& w, int64_t base, uint32_t count, uint64_t* keys, int32_t* first,
                                              uint32_t slots, uint32_t fill, uint32_t* voxels, uint32_t seed) {
    for (uint32_t j = threadIdx.x; j < slots; j += VX_THREADS) {
        __hip_atomic_store(&keys[j], VX_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&first[j], 0x7fffffff, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < count; j += VX_THREADS) {
        const uint64_t key = w.keys[base + j];
        const int32_t rank = vx_rank(w.point[base + j], seed);
        uint32_t slot = (uint32_t)(((vh_mix(key) & 0xffffffffull) * slots) >> 32);
        for (uint32_t probe = 0; probe < slots; ++probe) {
            const uint64_t prev = atomicCAS((unsigned long long*)&keys[slot], (unsigned long long)VX_EMPTY, (unsigned long long)key);
            if (prev == VX_EMPTY || prev == key) {
                atomicMin(&first[slot], rank);
                if (prev == VX_EMPTY && count > fill) atomicAdd(voxels, 1u);
                break;
            }
            slot = slot + 1 == slots ? 0 : slot + 1;
        }
        // (a thread adds one voxel at most after the count is over `fill`: an empty slot is left)
        if (count > fill && __hip_atomic_load(voxels, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > fill) break;
    }
    __syncthreads();
    if (*voxels > fill) return false;
    for (uint32_t j = threadIdx.x; j < count; j += VX_THREADS) {
        const uint64_t key = w.keys[base + j];
        uint32_t slot = (uint32_t)(((vh_mix(key) & 0xffffffffull) * slots) >> 32);
        for (uint32_t probe = 0; probe < slots; ++probe) {
            if (__hip_atomic_load(&keys[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == key) break;
            slot = slot + 1 == slots ? 0 : slot + 1;
        }
        w.rep[w.point[base + j]] = vx_unrank(__hip_atomic_load(&first[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), seed);
    }
    return true;
}

__global__ __launch_bounds__(VX_THREADS) void vx_part_kernel(VoxWs w, uint32_t seed) {
    __shared__ uint64_t keys[VX_SLOTS];
    __shared__ int32_t first[VX_SLOTS];
    __shared__ uint32_t voxels;
    const int p = blockIdx.x;
    uint32_t before = 0, base;
    for (int b = threadIdx.x; b < p; b += VX_THREADS) before += w.part_size[b];
    vx_block_scan(before, &base);
    const uint32_t count = w.part_size[p];
    if (threadIdx.x == 0) voxels = 0;   // (visible behind the barrier that follows the clearing of the table)
    if (vx_part_table(w, base, count, keys, first, VX_SLOTS, VX_FILL, &voxels, seed)) return;
    __syncthreads();
    if (threadIdx.x == 0) voxels = 0;
    vx_part_table(w, base, count, w.table + 2 * (int64_t)base, w.table_first + 2 * (int64_t)base, 2 * count, 2 * count, &voxels, seed);
}

__global__ __launch_bounds__(VX_THREADS) void vx_count_kernel(int64_t n, VoxWs w) {
    const int64_t base = (int64_t)blockIdx.x * VX_TILE;
    uint32_t kept = 0, total;
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int64_t i = base + k * VX_THREADS + threadIdx.x;
        if (i < n && w.rep[i] == (int32_t)i) ++kept;
    }
    vx_block_scan(kept, &total);
    if (threadIdx.x == 0) w.tile_kept[blockIdx.x] = total;
}

// one block: exclusive scan of the tiles' counts in place; total and status to the host, which waits for them
__global__ __launch_bounds__(VX_THREADS) void vx_scan_kernel(VoxWs w, int64_t* host_slot, int64_t seq) {
    uint32_t carry = 0;
    for (int64_t b0 = 0; b0 < w.tiles; b0 += VX_THREADS) {
        const int64_t b = b0 + threadIdx.x;
        const uint32_t v = b < w.tiles ? w.tile_kept[b] : 0u;
        uint32_t total;
        const uint32_t ex = vx_block_scan(v, &total);
        if (b < w.tiles) w.tile_kept[b] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) {
        host_slot[PTV3_SLOT_DATA] = (int64_t)carry;
        host_slot[PTV3_SLOT_DATA + 1] = (int64_t)w.status[0];
        __threadfence_system();
        __hip_atomic_store(&host_slot[0], seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ __launch_bounds__(VX_THREADS) void vx_assign_kernel(const float* __restrict__ coord, int64_t n,
                                                               const int64_t* __restrict__ offset, int nb,
                                                               float grid_size, VoxWs w, int32_t* __restrict__ grid_out,
                                                               int64_t* __restrict__ index_out,
                                                               int64_t* __restrict__ offset_out) {
    __shared__ uint32_t wcnt[VX_ITEMS * VX_WAVES];
    const int lane = threadIdx.x % PTV3_WAVE, wave = threadIdx.x / PTV3_WAVE;
    const VoxTile t = vx_tile(offset, nb, n);
    uint64_t votes[VX_ITEMS];
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int at = k * VX_THREADS + (int)threadIdx.x;
        votes[k] = __ballot(at < t.count && w.rep[t.base + min(at, t.count - 1)] == (int32_t)(t.base + at));
        if (lane == 0) wcnt[k * VX_WAVES + wave] = (uint32_t)__popcll(votes[k]);
    }
    __syncthreads();
    static_assert(VX_FILL + VX_THREADS < VX_SLOTS, "room for one more voxel per thread");
    static_assert(VX_ITEMS * VX_WAVES == PTV3_WAVE, "one lane per step and wave");
    uint32_t before = wcnt[lane];   // of every step and wave: the kept points in front of it
    {
        const uint32_t own = before;
#pragma unroll
        for (int off = 1; off < PTV3_WAVE; off <<= 1) {
            const uint32_t y = __shfl_up(before, off, PTV3_WAVE);
            if (lane >= off) before += y;
        }
        before += w.tile_kept[blockIdx.x] - own;
    }
    const bool ends = offset[t.lo] <= t.base + t.count;   // a scene ends inside the tile
#pragma unroll
    for (int k = 0; k < VX_ITEMS; ++k) {
        const int at = k * VX_THREADS + (int)threadIdx.x;
        const int64_t i = t.base + at;
        const uint32_t pos = __shfl(before, k * VX_WAVES + wave, PTV3_WAVE) + (uint32_t)__popcll(votes[k] & ((1ull << lane) - 1));
        const bool keep = votes[k] >> lane & 1;
        if (keep) {
            int32_t g[3];
            vx_grid(coord, i, scene_in(offset, t.lo, t.hi, i), w, grid_size, g);
#pragma unroll
            for (int a = 0; a < 3; ++a) grid_out[3 * (int64_t)pos + a] = g[a];
            index_out[pos] = i;
            w.pos[i] = (int32_t)pos;
        }
        // the scenes that end with point i (several when empty scenes follow) end with the points kept up to it
        if (ends && at < t.count) {
            int b = scene_in(offset, t.lo, t.hi, i);
            while (b < nb && offset[b] == i + 1) offset_out[b++] = (int64_t)pos + (keep ? 1 : 0);
        }
    }
}

__global__ __launch_bounds__(256) void vx_inverse_kernel(int64_t n, VoxWs w, int64_t* __restrict__ inverse) {
    const int64_t i0 = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    int32_t p[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) p[k] = i0 + k * 256 < n ? w.rep[i0 + k * 256] : 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (i0 + k * 256 < n) inverse[i0 + k * 256] = w.pos[p[k]];
}

// ---- rows of several arrays, picked by one index ----------------------------------------------------------------------

struct GatherJobs {
    const char* src[PTV3_GATHER_MAX];
    char* dst[PTV3_GATHER_MAX];
    int32_t words[PTV3_GATHER_MAX], width[PTV3_GATHER_MAX];   // a row: `words` words of `width` bytes
    uint32_t magic[PTV3_GATHER_MAX];                          // t * magic >> 32 = t / words for t below 256 rows' words
};

constexpr int GATHER_ROWS = 256;

template <typename W>
__device__ __forceinline__ void gather_rows(const W* __restrict__ src, W* __restrict__ dst, const int64_t* __restrict__ index,
                                            int rows, int words, uint32_t magic) {
    for (int t = threadIdx.x; t < rows * words; t += 256) {
        const int r = words == 1 ? t : (int)__umulhi((uint32_t)t, magic);
        dst[t] = src[index[r] * words + (t - r * words)];
    }
}

// One array per blockIdx.y. A work-group's index entries stay in its first-level cache; writes are contiguous.
__global__ __launch_bounds__(256) void gather_rows_kernel(GatherJobs j, const int64_t* __restrict__ index, int64_t m) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const int a = blockIdx.y;
    const int64_t r0 = (int64_t)blockIdx.x * GATHER_ROWS;
    const int rows = (int)min((int64_t)GATHER_ROWS, m - r0), words = j.words[a];
    const char* src = j.src[a];
    char* dst = j.dst[a] + r0 * words * j.width[a];
    switch (j.width[a]) {
        case 16: return gather_rows((const u32x4*)src, (u32x4*)dst, index + r0, rows, words, j.magic[a]);
        case 8: return gather_rows((const u32x2*)src, (u32x2*)dst, index + r0, rows, words, j.magic[a]);
        case 4: return gather_rows((const uint32_t*)src, (uint32_t*)dst, index + r0, rows, words, j.magic[a]);
        case 2: return gather_rows((const uint16_t*)src, (uint16_t*)dst, index + r0, rows, words, j.magic[a]);
        default: return gather_rows((const uint8_t*)src, (uint8_t*)dst, index + r0, rows, words, j.magic[a]);
    }
}

}  // namespace

extern "C" size_t ptv3_voxelize_workspace_bytes(int64_t n, int n_scenes) {
    if (n < 0 || n_scenes < 1) return 0;
    return vx_carve(nullptr, n, n_scenes).bytes;
}

extern "C" int ptv3_voxelize(const float* coord, int64_t n, const int64_t* offset, int n_scenes, float grid_size,
                             int32_t* grid_coord, int64_t* index, int64_t* inverse, int64_t* offset_out,
                             int64_t* host_slot, int64_t seq, uint32_t pick_seed, void* workspace, size_t workspace_bytes,
                             void* stream_) {
    if (n < 1 || n >= (1ll << 30) || n_scenes < 1 || n_scenes > 65535 || !(grid_size > 0.f)) return PTV3_EINVAL;
    if (!coord || !offset || !grid_coord || !index || !offset_out || !host_slot || !workspace) return PTV3_EINVAL;
    VoxWs w = vx_carve(workspace, n, n_scenes);
    if (workspace_bytes < w.bytes) return PTV3_EWORKSPACE;
    hipStream_t stream = (hipStream_t)stream_;
    const size_t parts = (size_t)1 << w.part_bits;
    const size_t split_lds = VX_TILE * 12 + parts * 8;
    static LdsGrant grant;
    const int rc = ptv3_allow_lds((const void*)vx_split_kernel, split_lds, grant);
    if (rc) return rc;
    const dim3 tiles((unsigned)w.tiles), threads(VX_THREADS);
    hipLaunchKernelGGL(vx_init_kernel, dim3((unsigned)ptv3_ceil_div(3 * (int64_t)n_scenes, 256)), dim3(256), 0, stream, w, n_scenes, offset_out);
    hipLaunchKernelGGL(vx_scene_min_kernel, tiles, threads, 0, stream, coord, n, offset, n_scenes, w);
    hipLaunchKernelGGL(vx_split_count_kernel, tiles, threads, parts * 4, stream, coord, n, offset, n_scenes, grid_size, w);
    if (w.tiles <= 16 * VX_SCAN_AT_ONCE)
        hipLaunchKernelGGL(vx_split_scan_kernel<16>, dim3((unsigned)(parts * 16 / VX_SCAN_THREADS)), dim3(VX_SCAN_THREADS), 0, stream, w);
    else
        hipLaunchKernelGGL(vx_split_scan_kernel<64>, dim3((unsigned)(parts * 64 / VX_SCAN_THREADS)), dim3(VX_SCAN_THREADS), 0, stream, w);
    hipLaunchKernelGGL(vx_split_kernel, tiles, threads, split_lds, stream, coord, n, offset, n_scenes, grid_size, w);
    hipLaunchKernelGGL(vx_part_kernel, dim3((unsigned)parts), threads, 0, stream, w, pick_seed);
    hipLaunchKernelGGL(vx_count_kernel, tiles, threads, 0, stream, n, w);
    hipLaunchKernelGGL(vx_scan_kernel, dim3(1), threads, 0, stream, w, host_slot, seq);
    hipLaunchKernelGGL(vx_assign_kernel, tiles, threads, 0, stream, coord, n, offset, n_scenes, grid_size, w, grid_coord, index, offset_out);
    if (inverse)
        hipLaunchKernelGGL(vx_inverse_kernel, dim3((unsigned)ptv3_ceil_div(n, 1024)), dim3(256), 0, stream, n, w, inverse);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_gather_rows(const void* const* src, void* const* dst, const int64_t* row_bytes, int count,
                                const int64_t* index, int64_t m, void* stream) {
    if (count < 0 || count > PTV3_GATHER_MAX || m < 0 || m >= (1ll << 31) || (count && (!src || !dst || !row_bytes))) return PTV3_EINVAL;
    if (count == 0 || m == 0) return PTV3_OK;
    if (!index) return PTV3_EINVAL;
    GatherJobs j;
    for (int a = 0; a < count; ++a) {
        if (!src[a] || !dst[a] || row_bytes[a] < 1 || row_bytes[a] > PTV3_GATHER_MAX_ROW) return PTV3_EINVAL;
        const uintptr_t at = (uintptr_t)src[a] | (uintptr_t)dst[a] | (uintptr_t)row_bytes[a];
        int width = 16;
        while (at & (uintptr_t)(width - 1)) width >>= 1;
        const int words = (int)(row_bytes[a] / width);
        j.src[a] = (const char*)src[a];
        j.dst[a] = (char*)dst[a];
        j.words[a] = words;
        j.width[a] = width;
        // 256 * words * words < 2^32: the rounded-up reciprocal divides every word number of a work-group exactly
        j.magic[a] = (uint32_t)(((1ull << 32) + words - 1) / words);
    }
    hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)ptv3_ceil_div(m, GATHER_ROWS), (unsigned)count), dim3(256), 0,
                       (hipStream_t)stream, j, index, m);
    PTV3_RETURN_LAUNCH();
}
