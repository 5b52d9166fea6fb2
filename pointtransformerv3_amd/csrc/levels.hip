// The index of a whole forward: everything that follows from the coordinates alone, for every level of the encoder at
// once. Level by level this is a chain of some 170 small launches and eleven read-backs (curve codes and sort; then per
// level clusters, pooled tables and orders, voxel hash, pair counts and lists, tile lists, padding and slot tables); on
// scans of up to 100k points the launches and the waits cost more than the kernels. Here it is about 24 launches and
// three read-backs, because
//   * pooled levels do not wait for each other: a cell of level j is a run of equal `code >> shift_j` along EVERY curve
//     of level 0 (a curve's codes are hierarchical), so one pass over the sorted keys of level 0 counts the cells of all
//     levels, and another writes the pooled tables of all levels: a cell's number is its rank along the curve that is row
//     0 of the level above, its position along another curve is its rank there;
//   * the pair lists of all levels share their launches (hash, count, scan, fill): a work-group finds its level in a
//     small table in the kernel's arguments. The 3x3x3 lists of level 0 come out of the 5x5x5 fill (the inner taps), and
//     tile lists are written by the fill itself: a work-group of the fill IS a tile;
//   * a read-back is a store to pinned host memory from the last kernel of a stage, behind a sequence number the host
//     waits for: no copy, no event.
// The results are those of the separate entry points bit for bit (ptv3_pool_*, ptv3_kmap_plan_*, ptv3_conv_plan_tiles_sized,
// ptv3_pad_index, ptv3_attn_slots), which callers of single operators keep using.
#include <string.h>
#include <time.h>

#include "voxelhash.h"

int ptv3_serialize_keys(const int32_t* grid_coord, const int64_t* batch, int64_t n, int depth, const int32_t* order_ids_host, int k,
                        int key_bits, int64_t* code, int64_t* order, int64_t* inverse, void* sorted_keys, void* workspace,
                        size_t workspace_bytes, hipStream_t stream);   // sort.hip

namespace {

constexpr int LV = PTV3_MAX_LEVELS, OR = PTV3_MAX_ORDERS;
constexpr int LB = 256;             // positions per block of the cell passes
constexpr int GT = 128;             // threads of a pair-list work-group: a tile of 128 or 96 voxels
constexpr int TAPS5 = 125, TAPS3 = 27;
constexpr int TILE_WORDS = 32;
constexpr int MAX_FACT_BLOCKS = 1024;

// ---- stage 1: scene ids, sparse indices, grid extent ---------------------------------------------------------------

__global__ __launch_bounds__(256) void facts_kernel(const int32_t* __restrict__ grid, const int64_t* __restrict__ batch_in,
                                                    const int64_t* __restrict__ offset, int nb, int64_t n,
                                                    int64_t* __restrict__ batch, int4* __restrict__ indices,
                                                    int32_t* __restrict__ part) {
    __shared__ int32_t red[4][3];
    int32_t m[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        int64_t b = 0;
        if (batch_in) {
            b = batch_in[i];
        } else if (batch) {
            int lo = 0, hi = nb;   // first scene whose end is > i
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (offset[mid] <= i) lo = mid + 1; else hi = mid;
            }
            b = lo;
            batch[i] = b;
        }
        const int32_t x = grid[3 * i], y = grid[3 * i + 1], z = grid[3 * i + 2];
        if (indices) indices[i] = make_int4((int32_t)b, x, y, z);
        m[0] = max(m[0], x);
        m[1] = max(m[1], y);
        m[2] = max(m[2], z);
    }
    const int wave = threadIdx.x / PTV3_WAVE, lane = threadIdx.x % PTV3_WAVE;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m[a] = max(m[a], __shfl_xor(m[a], off, PTV3_WAVE));
        if (lane == 0) red[wave][a] = m[a];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        part[blockIdx.x * 3 + a] = max(max(red[0][a], red[1][a]), max(red[2][a], red[3][a]));
    }
}

// what a stage hands to the host: data words first, then the sequence number (the host waits for it)
__device__ __forceinline__ void host_flag(int64_t* slot, int which, int64_t seq) {
    __threadfence_system();
    __hip_atomic_store(&slot[which], seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(256) void publish_facts_kernel(const int32_t* __restrict__ part, int blocks,
                                                            const int64_t* __restrict__ offset, int nb, int64_t* slot,
                                                            int64_t seq) {
    __shared__ int32_t red[4][3];
    int32_t m[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
    for (int b = threadIdx.x; b < blocks; b += 256)
#pragma unroll
        for (int a = 0; a < 3; ++a) m[a] = max(m[a], part[b * 3 + a]);
    const int wave = threadIdx.x / PTV3_WAVE, lane = threadIdx.x % PTV3_WAVE;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m[a] = max(m[a], __shfl_xor(m[a], off, PTV3_WAVE));
        if (lane == 0) red[wave][a] = m[a];
    }
    for (int b = threadIdx.x; b < nb; b += 256) slot[PTV3_SLOT_ENDS + b] = offset[b];
    __syncthreads();
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        slot[PTV3_SLOT_DATA + a] = max(max(red[0][a], red[1][a]), max(red[2][a], red[3][a]));
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) host_flag(slot, 0, seq);
}

// ---- stage 2: the cells of every pooled level from the sorted keys of level 0 ---------------------------------------

struct CellArgs {
    int64_t n;
    int blocks, levels, k;         // levels: pooled levels (1 .. levels)
    int shift[LV];                 // shift[j]: bits dropped at pooled level j (1-based)
    int scene_shift;               // 3 * depth
    int curve0[LV];                // level-0 row whose ranks number the cells of level j
    int row_of[LV][OR];            // row of level j's tables that level-0 row o becomes
    int depth[LV];                 // pooled depth of level j (sum)
    const int64_t* order;          // (k, n)
    uint32_t* blk;                 // [k][levels][blocks]
    uint32_t* totals;              // [k][levels]
    uint32_t* end_local;           // [levels][nb]
    int32_t* cid[LV];              // (n,) number of the cell of level j a point lies in
    const int32_t* grid;
    const int64_t* batch;
    int64_t m[LV];
    int64_t *code[LV], *order_out[LV], *inverse_out[LV], *batch_out[LV], *cluster[LV], *idx_ptr[LV];
    int32_t* grid_out[LV];
    int4* indices_out[LV];
};

// bit j - 1: position i starts a cell of level j (its key, shifted, differs from the one in front)
template <typename KT>
__device__ __forceinline__ uint32_t cell_starts(const CellArgs& a, KT key, KT prev, bool first) {
    uint32_t f = 0;
    for (int j = 1; j <= a.levels; ++j)
        if (first || (key >> a.shift[j]) != (prev >> a.shift[j])) f |= 1u << (j - 1);
    return f;
}

template <typename KT>
__global__ __launch_bounds__(LB) void cell_count_kernel(CellArgs a, const KT* __restrict__ keys, int nb) {
    __shared__ uint32_t wcnt[LB / PTV3_WAVE][LV];
    const int o = blockIdx.y, tid = threadIdx.x, lane = tid % PTV3_WAVE, wave = tid / PTV3_WAVE;
    const int64_t i = (int64_t)blockIdx.x * LB + tid;
    const KT* row = keys + (int64_t)o * a.n;
    const bool live = i < a.n;
    const KT key = live ? row[i] : (KT)0;
    const KT prev = live && i > 0 ? row[i - 1] : (KT)0;
    const uint32_t f = live ? cell_starts(a, key, prev, i == 0) : 0u;
    uint32_t mine[LV];
#pragma unroll
    for (int j = 0; j < LV; ++j) {
        if (j >= a.levels) continue;
        const uint64_t bal = __ballot((f >> j) & 1u);
        mine[j] = (uint32_t)__popcll(bal & ((2ull << lane) - 1ull));   // starts up to and with this lane
        if (lane == 0) wcnt[wave][j] = (uint32_t)__popcll(bal);
    }
    __syncthreads();
    if (tid < a.levels) {
        uint32_t t = 0;
        for (int w = 0; w < LB / PTV3_WAVE; ++w) t += wcnt[w][tid];
        a.blk[((int64_t)o * a.levels + tid) * a.blocks + blockIdx.x] = t;
    }
    if (o == 0 && live) {   // the last position of a scene notes how many cells the block has started by then
        const KT next = i + 1 < a.n ? row[i + 1] : (KT)0;
        if (i == a.n - 1 || (next >> a.scene_shift) != (key >> a.scene_shift)) {
            const int64_t scene = (int64_t)((uint64_t)key >> a.scene_shift);
            if (scene < nb)
#pragma unroll
                for (int j = 0; j < LV; ++j) {
                    if (j >= a.levels) continue;
                    uint32_t t = mine[j];
                    for (int w = 0; w < wave; ++w) t += wcnt[w][j];
                    a.end_local[(int64_t)j * nb + scene] = t;
                }
        }
    }
}

constexpr int SCAN_T = 1024;

// exclusive scan of `count` words with stride `step` in place by one work-group; the sum in every thread
__device__ __forceinline__ uint32_t column_scan(uint32_t* p, int64_t count, int64_t step) {
    __shared__ uint32_t wsum[SCAN_T / PTV3_WAVE];
    const int lane = threadIdx.x % PTV3_WAVE, wave = threadIdx.x / PTV3_WAVE, waves = blockDim.x / PTV3_WAVE;
    uint32_t carry = 0;
    for (int64_t b0 = 0; b0 < count; b0 += blockDim.x) {
        const int64_t b = b0 + threadIdx.x;
        const uint32_t v = b < count ? p[b * step] : 0u;
        uint32_t x = v;
#pragma unroll
        for (int off = 1; off < PTV3_WAVE; off <<= 1) {
            const uint32_t y = __shfl_up(x, off, PTV3_WAVE);
            if (lane >= off) x += y;
        }
        if (lane == PTV3_WAVE - 1) wsum[wave] = x;
        __syncthreads();
        uint32_t ws = lane < waves ? wsum[lane] : 0u;
#pragma unroll
        for (int off = 1; off < SCAN_T / PTV3_WAVE; off <<= 1) {
            const uint32_t y = __shfl_up(ws, off, PTV3_WAVE);
            if (lane >= off) ws += y;
        }
        const uint32_t total = __shfl(ws, waves - 1, PTV3_WAVE);
        const uint32_t base = wave == 0 ? 0u : __shfl(ws, wave - 1, PTV3_WAVE);
        if (b < count) p[b * step] = carry + base + x - v;
        carry += total;
        __syncthreads();
    }
    return carry;
}

__global__ __launch_bounds__(SCAN_T) void cell_scan_kernel(uint32_t* blk, int blocks, uint32_t* totals) {
    const uint32_t t = column_scan(blk + (int64_t)blockIdx.x * blocks, blocks, 1);
    if (threadIdx.x == 0) totals[blockIdx.x] = t;
}

struct PadArgs {
    int levels;                        // all levels, level 0 included
    int patch[LV];
    int64_t *offset[LV], *pad_start[LV], *seq_start[LV];   // offset[0] is the caller's
};

// one work-group: pooled scene ends of every level, on the device and to the host; padded starts of every level
__global__ __launch_bounds__(256) void publish_cells_kernel(CellArgs a, PadArgs p, int nb, int64_t* slot, int64_t seq) {
    for (int e = threadIdx.x; e < a.levels * nb; e += 256) {
        const int j = e / nb, b = e % nb;
        int s = b;   // an empty scene ends where the one in front of it does
        while (s >= 0 && p.offset[0][s] == (s ? p.offset[0][s - 1] : 0)) --s;
        int64_t end = 0;
        if (s >= 0) end = (int64_t)a.blk[(int64_t)j * a.blocks + (p.offset[0][s] - 1) / LB] + a.end_local[(int64_t)j * nb + s];
        p.offset[j + 1][b] = end;
        slot[PTV3_SLOT_ENDS + (int64_t)(j + 1) * nb + b] = end;
    }
    for (int j = threadIdx.x; j < a.levels; j += 256) slot[PTV3_SLOT_DATA + 4 + j] = a.totals[j];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) host_flag(slot, 1, seq);
    const int l = threadIdx.x;
    if (l < p.levels) {
        int64_t prev = 0, op = 0, sq = 0;
        for (int s = 0; s < nb; ++s) {
            const int64_t end = p.offset[l][s], cnt = end - prev, patch = p.patch[l];
            prev = end;
            const int64_t padded = cnt > patch ? ((cnt + patch - 1) / patch) * patch : cnt;
            p.pad_start[l][s] = op;
            p.seq_start[l][s] = sq;
            op += padded;
            sq += (padded + patch - 1) / patch;
        }
        p.pad_start[l][nb] = op;
        p.seq_start[l][nb] = sq;
    }
}

// per thread: starts of its level-j cells up to and with its own position inside the block, for every level
template <typename KT> struct CellScan {
    KT key;
    uint32_t flags;
    uint32_t incl[LV];
};
template <typename KT>
__device__ __forceinline__ CellScan<KT> cell_scan(const CellArgs& a, const KT* row, int64_t i,
                                                  uint32_t (*wcnt)[LV]) {
    const int lane = threadIdx.x % PTV3_WAVE, wave = threadIdx.x / PTV3_WAVE;
    CellScan<KT> c;
    const bool live = i < a.n;
    c.key = live ? row[i] : (KT)0;
    const KT prev = live && i > 0 ? row[i - 1] : (KT)0;
    c.flags = live ? cell_starts(a, c.key, prev, i == 0) : 0u;
#pragma unroll
    for (int j = 0; j < LV; ++j) {
        c.incl[j] = 0;
        if (j >= a.levels) continue;
        const uint64_t bal = __ballot((c.flags >> j) & 1u);
        c.incl[j] = (uint32_t)__popcll(bal & ((2ull << lane) - 1ull));
        if (lane == 0) wcnt[wave][j] = (uint32_t)__popcll(bal);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < LV; ++j) {
        if (j >= a.levels) continue;
        for (int w = 0; w < wave; ++w) c.incl[j] += wcnt[w][j];
    }
    return c;
}

// cid[j][point] = rank of the point's level-j cell along the curve that numbers the cells of level j; blockIdx.y = j - 1
template <typename KT>
__global__ __launch_bounds__(LB) void cell_number_kernel(CellArgs a, const KT* __restrict__ keys) {
    __shared__ uint32_t wcnt[LB / PTV3_WAVE][LV];
    const int j = blockIdx.y + 1, o = a.curve0[j];
    const int64_t i = (int64_t)blockIdx.x * LB + threadIdx.x;
    const KT* row = keys + (int64_t)o * a.n;
    const int lane = threadIdx.x % PTV3_WAVE, wave = threadIdx.x / PTV3_WAVE;
    const bool live = i < a.n;
    bool f = false;
    if (live) f = i == 0 || (row[i] >> a.shift[j]) != (row[i - 1] >> a.shift[j]);
    const uint64_t bal = __ballot(f);
    uint32_t incl = (uint32_t)__popcll(bal & ((2ull << lane) - 1ull));
    if (lane == 0) wcnt[wave][0] = (uint32_t)__popcll(bal);
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += wcnt[w][0];
    if (!live) return;
    const uint32_t c = a.blk[((int64_t)o * a.levels + j - 1) * a.blocks + blockIdx.x] + incl - 1;
    const int64_t pt = a.order[(int64_t)o * a.n + i];
    a.cid[j][pt] = (int32_t)c;
    if (j == 1) a.cluster[1][pt] = (int64_t)c;
}

// the pooled tables of every level; blockIdx.y = level-0 row
template <typename KT>
__global__ __launch_bounds__(LB) void cell_tables_kernel(CellArgs a, const KT* __restrict__ keys) {
    __shared__ uint32_t wcnt[LB / PTV3_WAVE][LV];
    const int o = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * LB + threadIdx.x;
    const CellScan<KT> c = cell_scan<KT>(a, keys + (int64_t)o * a.n, i, wcnt);
    if (i >= a.n) return;
    if (i == a.n - 1) {   // the member lists end here
#pragma unroll
        for (int j = 1; j < LV; ++j)
            if (j <= a.levels && o == a.curve0[j]) a.idx_ptr[j][a.m[j]] = j == 1 ? a.n : a.m[j - 1];
    }
    if (!c.flags) return;
    const int64_t pt = a.order[(int64_t)o * a.n + i];
    int64_t pos_above = i;   // position, along this curve, among the cells of the level above
    int32_t cell_above = 0;
#pragma unroll
    for (int j = 1; j < LV; ++j) {
        if (j > a.levels) break;
        const int64_t pos = (int64_t)a.blk[((int64_t)o * a.levels + j - 1) * a.blocks + blockIdx.x] + c.incl[j - 1] - 1;
        const bool numbers = o == a.curve0[j];
        // every cell of the level above (every run start there) belongs to the level-j cell this position lies in
        if (j > 1 && numbers && ((c.flags >> (j - 2)) & 1u)) a.cluster[j][cell_above] = pos;
        if (!((c.flags >> (j - 1)) & 1u)) {
            break;   // no start here, so none on any coarser level either: their shifts are larger
        }
        const int32_t cell = a.cid[j][pt];
        const int r = a.row_of[j][o];
        a.order_out[j][(int64_t)r * a.m[j] + pos] = cell;
        a.inverse_out[j][(int64_t)r * a.m[j] + cell] = pos;
        a.code[j][(int64_t)r * a.m[j] + cell] = (int64_t)((uint64_t)c.key >> a.shift[j]);
        if (numbers) {   // here cell == pos
            const int d = a.depth[j];
            const int64_t b = a.batch[pt];
            const int32_t x = a.grid[3 * pt] >> d, y = a.grid[3 * pt + 1] >> d, z = a.grid[3 * pt + 2] >> d;
            a.grid_out[j][3 * pos] = x;
            a.grid_out[j][3 * pos + 1] = y;
            a.grid_out[j][3 * pos + 2] = z;
            a.batch_out[j][pos] = b;
            a.indices_out[j][pos] = make_int4((int32_t)b, x, y, z);
            a.idx_ptr[j][pos] = pos_above;
        }
        pos_above = pos;
        cell_above = cell;
    }
}

// ---- padding and slot tables of every level ------------------------------------------------------------------------

struct SlotArgs {
    int levels, nb;
    int first_block[LV + 1];
    int patch[LV];
    int64_t n[LV], n_pad[LV], n_seq[LV];
    const int64_t *offset[LV], *pad_start[LV], *seq_start[LV], *order[LV];
    int64_t *pad[LV], *unpad[LV];                 // null: not wanted
    int32_t* cu[LV];
    int32_t *src[LV][OR], *dst[LV][OR];           // null: row not wanted
    int k;
};

__global__ __launch_bounds__(256) void slots_kernel(SlotArgs a) {
    int l = 0;
    while (l + 1 < a.levels && (int)blockIdx.x >= a.first_block[l + 1]) ++l;
    const int64_t j = (int64_t)((int)blockIdx.x - a.first_block[l]) * 256 + threadIdx.x;
    if (j == 0) a.cu[l][a.n_seq[l]] = (int32_t)a.n_pad[l];
    if (j >= a.n_pad[l]) return;
    const int64_t* ps = a.pad_start[l];
    int lo = 0, hi = a.nb;   // pad_start[lo] <= j < pad_start[hi]; empty scenes share a start and are skipped
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ps[mid] <= j) lo = mid; else hi = mid;
    }
    const int64_t first = lo ? a.offset[l][lo - 1] : 0, cnt = a.offset[l][lo] - first, local = j - ps[lo];
    const int64_t patch = a.patch[l];
    // filler slots of the last patch reuse the points one patch earlier (model.py:412-423)
    const bool own = local < cnt;
    const int64_t at = first + (own ? local : local - patch);
    if (a.pad[l]) {
        a.pad[l][j] = at;
        if (own) a.unpad[l][at] = j;
    }
    if (local % patch == 0) a.cu[l][a.seq_start[l][lo] + local / patch] = (int32_t)j;
    for (int r = 0; r < a.k; ++r) {
        if (!a.src[l][r]) continue;
        const int32_t row = (int32_t)a.order[l][(int64_t)r * a.n[l] + at];
        a.src[l][r][j] = row;
        a.dst[l][r][j] = own ? row : -1;
    }
}

// ---- pair lists of every level -------------------------------------------------------------------------------------

struct ListLevel {
    const int4* idx;
    int64_t n;
    int group;                  // voxels per work-group = per tile (128 or 96)
    int groups;
    int want;                   // PTV3_LISTS_*
    VoxelHash h;
    int64_t cap;
    uint32_t* slot;             // [8][n] header slots of a voxel's blocks
    uint64_t* found;            // [n] (3x3x3) or [2][n] (5x5x5): taps that exist
    uint32_t *tap, *row, *tap_total, *row_total;       // [groups][27], [groups], [27], [1]
    uint32_t *tap5, *row5, *tap_total5, *row_total5;   // 5x5x5, level 0 only
    int32_t *tap_ptr, *row_ptr, *pair_in, *pair_slot, *tile_tap;
    uint32_t *tile_pair, *vox_taps;
    int32_t *tap_ptr5, *row_ptr5, *pair_in5, *pair_slot5;
    int32_t *pair_out, *pair_out5;
};

struct ListArgs {
    int first, levels;           // levels first .. levels - 1 take part
    int first_block[LV + 1];
    ListLevel lv[LV];
};

__device__ __forceinline__ int list_level(const ListArgs& a) {
    int l = a.first;
    while (l + 1 < a.levels && (int)blockIdx.x >= a.first_block[l + 1]) ++l;
    return l;
}

__global__ __launch_bounds__(256) void hash_clear_kernel(ListArgs a) {
    const int l = list_level(a);
    const int64_t i = (int64_t)((int)blockIdx.x - a.first_block[l]) * 256 + threadIdx.x;
    if (i < a.lv[l].cap) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 empty = {~0u, ~0u, 0u, 0u};   // key VH_EMPTY, no cell
        *(u32x4*)&a.lv[l].h.blocks[i] = empty;
    }
}

__global__ __launch_bounds__(256) void hash_insert_kernel(ListArgs a) {
    const int l = list_level(a);
    const int64_t i = (int64_t)((int)blockIdx.x - a.first_block[l]) * 256 + threadIdx.x;
    if (i < a.lv[l].n) vh_insert(a.lv[l].idx, i, a.lv[l].h);
}

// index among the 125 taps of 3x3x3 tap t3
__device__ __forceinline__ int inner_tap(int t3) { return ((t3 / 9 + 1) * 5 + (t3 / 3) % 3 + 1) * 5 + t3 % 3 + 1; }

__device__ __forceinline__ uint32_t inner_taps(uint64_t lo, uint64_t hi) {
    uint32_t f = 0;
#pragma unroll
    for (int t3 = 0; t3 < TAPS3; ++t3) {
        const int t5 = inner_tap(t3);
        f |= (uint32_t)((t5 < 64 ? lo >> t5 : hi >> (t5 - 64)) & 1ull) << t3;
    }
    return f;
}

// taps that exist around every voxel; per work-group and tap their number
template <int KS>
__global__ __launch_bounds__(GT) void list_count_kernel(ListArgs a) {
    constexpr int R = KS / 2, TAPS = KS * KS * KS;
    __shared__ unsigned long long mask[2][KS == 5 ? 128 : 32];
    __shared__ uint32_t rows[2][2];
    const int l = list_level(a);
    const ListLevel& v = a.lv[l];
    const int g = (int)blockIdx.x - a.first_block[l], tid = threadIdx.x, lane = tid % PTV3_WAVE, wave = tid / PTV3_WAVE;
    const int64_t i = (int64_t)g * v.group + tid;
    for (int e = tid; e < 2 * (KS == 5 ? 128 : 32); e += GT) (&mask[0][0])[e] = 0;
    __syncthreads();
    uint64_t lo = 0, hi = 0;
    if (tid < v.group && i < v.n) {
        const int4 c = v.idx[i];
        uint32_t slot[8];
        vh_taps<R>(v.h, c.x, c.y, c.z, c.w, slot, lo, hi);
#pragma unroll
        for (int k = 0; k < 8; ++k) v.slot[(int64_t)k * v.n + i] = slot[k];
        uint64_t f = lo;
        while (f) { const int t = __builtin_ctzll(f); f &= f - 1; atomicOr(&mask[wave][t], 1ull << lane); }
        f = hi;
        while (f) { const int t = 64 + __builtin_ctzll(f); f &= f - 1; atomicOr(&mask[wave][t], 1ull << lane); }
        v.found[i] = lo;
        if (KS == 5) v.found[v.n + i] = hi;
    }
    uint32_t c3 = (uint32_t)(KS == 5 ? __popc(inner_taps(lo, hi)) : __popcll(lo)), c5 = (uint32_t)(__popcll(lo) + __popcll(hi));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        c3 += __shfl_xor(c3, off, PTV3_WAVE);
        c5 += __shfl_xor(c5, off, PTV3_WAVE);
    }
    if (lane == 0) {
        rows[0][wave] = c3;
        rows[1][wave] = c5;
    }
    __syncthreads();
    if (tid == 0) {
        v.row[g] = rows[0][0] + rows[0][1];
        if (KS == 5) v.row5[g] = rows[1][0] + rows[1][1];
    }
    auto count_of = [&](int t) { return (uint32_t)(__popcll(mask[0][t]) + __popcll(mask[1][t])); };
    if (tid < TAPS3) v.tap[(int64_t)g * TAPS3 + tid] = count_of(KS == 5 ? inner_tap(tid) : tid);
    if (KS == 5 && tid < TAPS) v.tap5[(int64_t)g * TAPS5 + tid] = count_of(tid);
}

// one work-group per column: exclusive scan over the work-groups of a level's per-tap (and per-row) counts
__global__ __launch_bounds__(SCAN_T) void list_scan_kernel(ListArgs a) {
    int l = 0, col = blockIdx.x;
    bool five = false;
    for (;;) {   // columns of level 0: 27 + 1, then 125 + 1 where it has 5x5x5 lists; other levels 27 + 1
        if (col < TAPS3 + 1) break;
        col -= TAPS3 + 1;
        if (a.lv[l].tap5) {
            if (col < TAPS5 + 1) { five = true; break; }
            col -= TAPS5 + 1;
        }
        ++l;
    }
    const ListLevel& v = a.lv[l];
    const int taps = five ? TAPS5 : TAPS3;
    uint32_t* p = five ? (col < taps ? v.tap5 + col : v.row5) : (col < taps ? v.tap + col : v.row);
    const uint32_t t = column_scan(p, v.groups, col < taps ? taps : 1);
    if (threadIdx.x == 0) {
        if (col < taps) (five ? v.tap_total5 : v.tap_total)[col] = t;
        else *(five ? v.row_total5 : v.row_total) = t;
    }
}

// tap_ptr of every list (a wave each) and the pair counts to the host
__global__ __launch_bounds__(1024) void publish_lists_kernel(ListArgs a, int64_t* slot, int64_t seq) {
    const int lane = threadIdx.x % PTV3_WAVE, wave = threadIdx.x / PTV3_WAVE;
    const int l = wave >> 1;
    const bool five = wave & 1;
    if (l < a.levels && (!five || a.lv[l].tap5)) {
        const ListLevel& v = a.lv[l];
        const int taps = five ? TAPS5 : TAPS3;
        const uint32_t* total = five ? v.tap_total5 : v.tap_total;
        int32_t* ptr = five ? v.tap_ptr5 : v.tap_ptr;
        uint32_t carry = 0;
        for (int t0 = 0; t0 < taps; t0 += PTV3_WAVE) {
            const int t = t0 + lane;
            const uint32_t c = t < taps ? total[t] : 0u;
            uint32_t x = c;
#pragma unroll
            for (int off = 1; off < PTV3_WAVE; off <<= 1) {
                const uint32_t y = __shfl_up(x, off, PTV3_WAVE);
                if (lane >= off) x += y;
            }
            if (t < taps) ptr[t] = (int32_t)(carry + x - c);
            carry += __shfl(x, PTV3_WAVE - 1, PTV3_WAVE);
        }
        if (lane == 0) {
            ptr[taps] = (int32_t)carry;
            slot[PTV3_SLOT_DATA + 4 + LV + 2 * l + five] = (int64_t)carry;
        }
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) host_flag(slot, 2, seq);
}

constexpr int STAGE = 2048;   // pairs of one work-group staged in LDS for coalesced writes

// Work-group = tile. Per list: row_ptr, then every pair at its tap-major place (pair_in, pair_slot: ranks from the lane
// masks) and at its place in the tile's own list (tap-major inside the tile). KS = 5: the 5x5x5 lists and the inner 3x3x3.
template <int KS>
__global__ __launch_bounds__(GT) void list_fill_kernel(ListArgs a) {
    constexpr int R = KS / 2;
    __shared__ unsigned long long mask[2][128];
    __shared__ uint32_t tap_base[128], tap_start[128], wrows[2];
    __shared__ uint32_t hslot[8][GT];
    __shared__ uint8_t first_cell[GT];   // 2 bits per axis: where a voxel's window starts in its first block
    __shared__ uint32_t stage_q[STAGE];
    __shared__ int32_t stage_slot[STAGE];
    __shared__ uint16_t stage_vt[STAGE];   // voxel << 7 | tap
    const int l = list_level(a);
    const ListLevel& v = a.lv[l];
    const int g = (int)blockIdx.x - a.first_block[l], tid = threadIdx.x, lane = tid % PTV3_WAVE, wave = tid / PTV3_WAVE;
    const int64_t i = (int64_t)g * v.group + tid;
    const bool live = tid < v.group && i < v.n;
    const uint64_t below = (1ull << lane) - 1ull;
    int4 c = {0, 0, 0, 0};
    uint64_t lo = 0, hi = 0;
    if (live) {
        c = v.idx[i];
        lo = v.found[i];
        if (KS == 5) hi = v.found[v.n + i];
#pragma unroll
        for (int k = 0; k < 8; ++k) hslot[k][tid] = v.slot[(int64_t)k * v.n + i];
    }
    first_cell[tid] = (uint8_t)(((c.y + VH_SHIFT - R) & 3) << 4 | ((c.z + VH_SHIFT - R) & 3) << 2 | ((c.w + VH_SHIFT - R) & 3));
    // row of the voxel at tap t (of edge^3) of the tile's voxel `vox`
    auto source = [&](int vox, int t, int edge) -> int32_t {
        if (t == edge * edge * edge / 2) return (int32_t)((int64_t)g * v.group + vox);
        const int at = first_cell[vox], in = R - edge / 2;
        const int cx = (at >> 4) + t / (edge * edge) + in, cy = (at >> 2 & 3) + t / edge % edge + in, cz = (at & 3) + t % edge + in;
        const int k = cx >> 2 << 2 | cy >> 2 << 1 | cz >> 2, bit = (cx & 3) << 4 | (cy & 3) << 2 | (cz & 3);
        return v.h.rows[(int64_t)hslot[k][vox] * 64 + bit];
    };

    auto make = [&](uint64_t flo, uint64_t fhi, int taps, int edge, const int32_t* tap_ptr, const uint32_t* tap_off,
                    const uint32_t* row_off, int32_t* row_ptr, int32_t* pair_in, int32_t* pair_slot, int32_t* pair_out, bool pairs, bool tiles) {
        for (int e = tid; e < 256; e += GT) (&mask[0][0])[e] = 0;
        for (int t = tid; t < taps; t += GT) tap_base[t] = pairs ? (uint32_t)tap_ptr[t] + tap_off[(int64_t)g * taps + t] : 0u;
        const uint32_t cnt = (uint32_t)(__popcll(flo) + __popcll(fhi));
        uint32_t incl = cnt;
#pragma unroll
        for (int off = 1; off < PTV3_WAVE; off <<= 1) {
            const uint32_t y = __shfl_up(incl, off, PTV3_WAVE);
            if (lane >= off) incl += y;
        }
        if (lane == PTV3_WAVE - 1) wrows[wave] = incl;
        __syncthreads();
        {
            uint64_t f = flo;
            while (f) { const int t = __builtin_ctzll(f); f &= f - 1; atomicOr(&mask[wave][t], 1ull << lane); }
            f = fhi;
            while (f) { const int t = 64 + __builtin_ctzll(f); f &= f - 1; atomicOr(&mask[wave][t], 1ull << lane); }
        }
        const uint32_t total = wrows[0] + wrows[1];
        const uint32_t base = row_off[g];
        const uint32_t slot0 = base + (wave ? wrows[0] : 0u) + incl - cnt;
        __syncthreads();
        if (wave == 0) {   // where every tap's pairs start inside the tile
            const uint32_t c0 = (uint32_t)(__popcll(mask[0][lane]) + __popcll(mask[1][lane]));
            const uint32_t c1 = (uint32_t)(__popcll(mask[0][lane + 64]) + __popcll(mask[1][lane + 64]));
            uint32_t x0 = c0, x1 = c1;
#pragma unroll
            for (int off = 1; off < PTV3_WAVE; off <<= 1) {
                const uint32_t y0 = __shfl_up(x0, off, PTV3_WAVE), y1 = __shfl_up(x1, off, PTV3_WAVE);
                if (lane >= off) { x0 += y0; x1 += y1; }
            }
            tap_start[lane] = x0 - c0;
            tap_start[lane + 64] = __shfl(x0, PTV3_WAVE - 1, PTV3_WAVE) + x1 - c1;
            if (tiles && lane < TILE_WORDS) v.tile_tap[(int64_t)g * TILE_WORDS + lane] = lane == 28 ? (int32_t)base : (int32_t)(x0 - c0);
        }
        __syncthreads();
        if (live) {
            if (row_ptr) {
                row_ptr[i] = (int32_t)slot0;
                if (i == v.n - 1) row_ptr[v.n] = (int32_t)(slot0 + cnt);
            }
            if (tiles && v.vox_taps) v.vox_taps[i] = (uint32_t)flo;
        }
        const bool staged = total <= (uint32_t)STAGE;
        uint32_t slot = slot0;
        uint64_t f0 = flo, f1 = fhi;
        while (f0 | f1) {
            int t;
            if (f0) { t = __builtin_ctzll(f0); f0 &= f0 - 1; }
            else { t = 64 + __builtin_ctzll(f1); f1 &= f1 - 1; }
            const uint32_t rank = (uint32_t)__popcll(mask[wave][t] & below) + (wave ? (uint32_t)__popcll(mask[0][t]) : 0u);
            const uint32_t q = tap_base[t] + rank, e = tap_start[t] + rank;
            if (staged) {
                stage_q[e] = q;
                stage_slot[e] = (int32_t)slot;
                stage_vt[e] = (uint16_t)(tid << 7 | t);
            } else {
                const int32_t src = source(tid, t, edge);
                if (pairs) {
                    pair_in[q] = src;
                    pair_slot[q] = (int32_t)slot;
                    if (pair_out) pair_out[q] = (int32_t)i;
                }
                if (tiles) v.tile_pair[base + e] = (uint32_t)tid << 24 | (uint32_t)src;
            }
            ++slot;
        }
        if (staged) {
            __syncthreads();
            // the rows are looked up here, four pairs of a thread at a time, not in the loop above, where every lane
            // waited for the fullest one's lookups one after the other
            for (uint32_t e0 = tid; e0 < total; e0 += 4 * GT) {
                int32_t src[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t e = min(e0 + u * GT, total - 1), vt = stage_vt[e];
                    src[u] = source((int)(vt >> 7), (int)(vt & 127), edge);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t e = e0 + u * GT;
                    if (e >= total) break;
                    const uint32_t vox = (uint32_t)stage_vt[e] >> 7;
                    if (pairs) {
                        const uint32_t q = stage_q[e];
                        pair_in[q] = src[u];
                        pair_slot[q] = stage_slot[e];
                        if (pair_out) pair_out[q] = (int32_t)((int64_t)g * v.group + vox);
                    }
                    if (tiles) v.tile_pair[base + e] = vox << 24 | (uint32_t)src[u];
                }
            }
        }
        __syncthreads();
    };
    if (KS == 5 && (v.want & PTV3_LISTS_PAIRS5))
        make(lo, hi, TAPS5, 5, v.tap_ptr5, v.tap5, v.row5, v.row_ptr5, v.pair_in5, v.pair_slot5,
             v.pair_out5, true, false);
    const bool pairs = v.want & PTV3_LISTS_PAIRS, tiles = v.want & PTV3_LISTS_TILES;
    if (pairs || tiles)
        make(KS == 5 ? (uint64_t)inner_taps(lo, hi) : lo, 0, TAPS3, 3, v.tap_ptr, v.tap, v.row, pairs ? v.row_ptr : nullptr,
             v.pair_in, v.pair_slot, pairs ? v.pair_out : nullptr, pairs, tiles);
}

// ---- host ----------------------------------------------------------------------------------------------------------

// hands out 256-byte aligned pieces of a buffer; with a null base it only adds up what is needed
struct Carver {
    char* base;
    size_t off = 0;
    explicit Carver(void* b) : base((char*)b) {}
    template <typename T> T* take(size_t count) {
        T* p = base ? (T*)(base + off) : nullptr;
        off += ptv3_align256((count ? count : 1) * sizeof(T));
        return p;
    }
};

struct State {
    ptv3_index_cfg cfg;
    hipStream_t stream;
    int64_t* slot;
    int64_t seq;
    int depth, key_bits;
    const int32_t* grid;
    const int64_t *batch, *offset;
    int32_t* part;
    uint32_t *blk, *totals, *end_local;
    void* keys;
    CellArgs cells;
    PadArgs pads;
    ListArgs lists;
    ptv3_level lv[LV];
};
static_assert(sizeof(State) <= PTV3_INDEX_STATE_BYTES, "state buffer size");

int list_blocks(ListArgs& a, int first, int levels, int kind) {   // kind 0: headers, 1: voxels, 2: work-groups of voxels
    a.first = first;
    a.levels = levels;
    int at = 0;
    for (int l = first; l < levels; ++l) {
        a.first_block[l] = at;
        const ListLevel& v = a.lv[l];
        at += (int)(kind == 0 ? ptv3_ceil_div(v.cap, 256) : kind == 1 ? ptv3_ceil_div(v.n, 256) : v.groups);
    }
    a.first_block[levels] = at;
    return at;
}

// c: what only the index stages read; kept: what the convolutions read as well
void carve_list_scratch(Carver& c, Carver& kept, ListLevel& v, bool five) {
    v.cap = vh_capacity(v.n);
    v.groups = (int)ptv3_ceil_div(v.n, v.group);
    v.h.blocks = c.take<VoxelBlock>(v.cap);
    v.h.rows = c.take<int32_t>(v.cap * 64);
    v.h.mask = (uint32_t)(v.cap - 1);
    v.slot = c.take<uint32_t>(8 * v.n);
    v.found = c.take<uint64_t>((five ? 2 : 1) * v.n);
    v.tap = c.take<uint32_t>((size_t)v.groups * TAPS3);
    v.row = c.take<uint32_t>(v.groups);
    v.tap_total = c.take<uint32_t>(TAPS3 + 1);
    v.row_total = c.take<uint32_t>(1);
    v.tap_ptr = kept.take<int32_t>(TAPS3 + 1);
    v.tap5 = v.row5 = v.tap_total5 = v.row_total5 = nullptr;
    v.tap_ptr5 = nullptr;
    if (five) {
        v.tap5 = c.take<uint32_t>((size_t)v.groups * TAPS5);
        v.row5 = c.take<uint32_t>(v.groups);
        v.tap_total5 = c.take<uint32_t>(TAPS5 + 1);
        v.row_total5 = c.take<uint32_t>(1);
        v.tap_ptr5 = kept.take<int32_t>(TAPS5 + 1);
    }
}

int launch_hash_count(State& s, int first, int levels, hipStream_t stream) {
    ListArgs& a = s.lists;
    hipLaunchKernelGGL(hash_clear_kernel, dim3((unsigned)list_blocks(a, first, levels, 0)), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(hash_insert_kernel, dim3((unsigned)list_blocks(a, first, levels, 1)), dim3(256), 0, stream, a);
    const unsigned groups = (unsigned)list_blocks(a, first, levels, 2);
    if (a.lv[first].tap5) hipLaunchKernelGGL(list_count_kernel<5>, dim3(groups), dim3(GT), 0, stream, a);
    else hipLaunchKernelGGL(list_count_kernel<3>, dim3(groups), dim3(GT), 0, stream, a);
    PTV3_RETURN_LAUNCH();
}

template <typename KT> int launch_cells_count(State& s, hipStream_t stream) {
    CellArgs& a = s.cells;
    hipLaunchKernelGGL(cell_count_kernel<KT>, dim3((unsigned)a.blocks, (unsigned)a.k), dim3(LB), 0, stream, a,
                       (const KT*)s.keys, s.cfg.n_scenes);
    PTV3_RETURN_LAUNCH();
}

template <typename KT> int launch_cells_tables(State& s, hipStream_t stream) {
    CellArgs& a = s.cells;
    hipLaunchKernelGGL(cell_number_kernel<KT>, dim3((unsigned)a.blocks, (unsigned)a.levels), dim3(LB), 0, stream, a,
                       (const KT*)s.keys);
    hipLaunchKernelGGL(cell_tables_kernel<KT>, dim3((unsigned)a.blocks, (unsigned)a.k), dim3(LB), 0, stream, a,
                       (const KT*)s.keys);
    PTV3_RETURN_LAUNCH();
}

// The tables are small (16 bytes a point) and what a caller keeps; the scratch is 650 - 800 bytes a point, most of it the
// voxel hash, and is free again once the lists are made. In one buffer the 6 MB of sparse indices in a returned Point
// held 0.3 GB of a 400k-point batch.
struct Bytes {
    size_t tables, scratch;
};

Bytes carve_begin(State& s, void* tables, void* scratch) {
    const ptv3_index_cfg& g = s.cfg;
    Carver kept(tables), c(scratch);
    const int64_t n = g.n;
    s.lv[0].indices = kept.take<int32_t>(4 * n);
    s.part = c.take<int32_t>(3 * MAX_FACT_BLOCKS);
    const int pooled = g.n_levels - 1;
    for (int l = 0; l < g.n_levels; ++l) {
        if (l > 0) s.lv[l].offset = kept.take<int64_t>(g.n_scenes);
        s.pads.pad_start[l] = c.take<int64_t>(g.n_scenes + 1);
        s.pads.seq_start[l] = c.take<int64_t>(g.n_scenes + 1);
    }
    s.cells.blocks = (int)ptv3_ceil_div(n, LB);
    s.blk = c.take<uint32_t>((size_t)g.n_orders * pooled * s.cells.blocks);
    s.totals = c.take<uint32_t>((size_t)g.n_orders * pooled);
    s.end_local = c.take<uint32_t>((size_t)pooled * g.n_scenes);
    s.keys = c.take<uint64_t>((size_t)g.n_orders * n);
    ListLevel& v = s.lists.lv[0];
    v.n = n;
    v.group = ptv3_conv_tile_voxels(n, g.only128[0] ? 128 : 64);
    carve_list_scratch(c, kept, v, g.stem5);
    v.idx = (const int4*)s.lv[0].indices;
    return {kept.off, c.off};
}

bool cfg_ok(const ptv3_index_cfg* g) {
    if (!g || g->n < 1 || g->n >= (1ll << 31) / 128 || g->n_levels < 1 || g->n_levels > LV || g->n_orders < 1 ||
        g->n_orders > OR || g->n_scenes < 1)
        return false;
    for (int l = 0; l < g->n_levels; ++l)
        if (g->patch[l] < 1) return false;
    return true;
}

}  // namespace

extern "C" int ptv3_index_begin_bytes(const ptv3_index_cfg* cfg, size_t* tables, size_t* scratch) {
    if (!cfg_ok(cfg) || !tables || !scratch) return PTV3_EINVAL;
    State s = {};
    s.cfg = *cfg;
    const Bytes need = carve_begin(s, nullptr, nullptr);
    *tables = need.tables;
    *scratch = need.scratch;
    return PTV3_OK;
}

extern "C" int64_t ptv3_index_slot_words(int n_levels, int n_scenes) {
    return n_levels < 1 || n_scenes < 1 ? 0 : PTV3_SLOT_ENDS + (int64_t)n_levels * n_scenes;
}

static int fact_blocks(int64_t n) {
    const int64_t want = ptv3_ceil_div(n, 256);
    return (int)(want < MAX_FACT_BLOCKS ? want : MAX_FACT_BLOCKS);
}

extern "C" int ptv3_index_begin(void* state, const ptv3_index_cfg* cfg, const int32_t* grid_coord, const int64_t* batch_in,
                                const int64_t* offset, int64_t* batch_out, void* tables, size_t tables_bytes, void* scratch,
                                size_t scratch_bytes, int64_t* host_slot, int64_t seq, void* stream_) {
    if (!state || !cfg_ok(cfg) || !grid_coord || !offset || (!batch_in && !batch_out) || !tables || !scratch || !host_slot)
        return PTV3_EINVAL;
    State& s = *(State*)state;
    memset(&s, 0, sizeof(State));
    s.cfg = *cfg;
    const Bytes need = carve_begin(s, nullptr, nullptr);
    if (tables_bytes < need.tables || scratch_bytes < need.scratch) return PTV3_EWORKSPACE;
    carve_begin(s, tables, scratch);
    hipStream_t stream = (hipStream_t)stream_;
    s.slot = host_slot;
    s.seq = seq;
    s.grid = grid_coord;
    s.batch = batch_in ? batch_in : batch_out;
    s.offset = offset;
    s.lv[0].n = cfg->n;
    s.lv[0].batch = (int64_t*)s.batch;
    s.lv[0].offset = (int64_t*)offset;
    s.lv[0].grid = (int32_t*)grid_coord;
    const int blocks = fact_blocks(cfg->n);
    hipLaunchKernelGGL(facts_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, grid_coord, batch_in, offset, cfg->n_scenes,
                       cfg->n, batch_out, (int4*)s.lv[0].indices, s.part);
    hipLaunchKernelGGL(publish_facts_kernel, dim3(1), dim3(256), 0, stream, (const int32_t*)s.part, blocks, offset,
                       cfg->n_scenes, host_slot, seq);
    // level 0's neighbour search needs the coordinates only: it runs while the host reads the extent
    return launch_hash_count(s, 0, 1, stream);
}

extern "C" size_t ptv3_scene_facts_bytes(int64_t n) {
    return 3 * (size_t)fact_blocks(n) * sizeof(int32_t);
}

extern "C" int ptv3_scene_facts(const int32_t* grid_coord, int64_t n, const int64_t* offset, int n_scenes, void* workspace,
                                size_t workspace_bytes, int64_t* host_slot, int64_t seq, void* stream_) {
    if (n < 1 || n_scenes < 1 || !grid_coord || !offset || !workspace || !host_slot) return PTV3_EINVAL;
    if (workspace_bytes < ptv3_scene_facts_bytes(n)) return PTV3_EWORKSPACE;
    const int blocks = fact_blocks(n);
    hipStream_t stream = (hipStream_t)stream_;
    hipLaunchKernelGGL(facts_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, grid_coord, nullptr, offset, n_scenes, n, nullptr,
                       nullptr, (int32_t*)workspace);
    hipLaunchKernelGGL(publish_facts_kernel, dim3(1), dim3(256), 0, stream, (const int32_t*)workspace, blocks, offset, n_scenes,
                       host_slot, seq);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_index_wait(const int64_t* host_slot, int which, int64_t seq, void* stream_) {
    if (!host_slot || which < 0 || which > 2) return PTV3_EINVAL;
    const volatile int64_t* flag = host_slot + which;
    timespec t0, t1;
    clock_gettime(CLOCK_MONOTONIC, &t0);
    for (int64_t spin = 0;; ++spin) {
        if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq) return PTV3_OK;
        if ((spin & 1023) == 1023) {
            clock_gettime(CLOCK_MONOTONIC, &t1);
            if (t1.tv_sec - t0.tv_sec > 2) break;
        }
        __builtin_ia32_pause();
    }
    // far too long for these kernels alone: the stream may hold other work, or have failed
    const hipError_t e = hipStreamSynchronize((hipStream_t)stream_);
    if (e != hipSuccess) return (int)e;
    return __atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq ? PTV3_OK : PTV3_EINVAL;
}

extern "C" size_t ptv3_index_sort_bytes(const void* state) {
    return state ? ptv3_argsort_workspace_bytes(((const State*)state)->cfg.n, ((const State*)state)->cfg.n_orders) : 0;
}

extern "C" int ptv3_index_sort(void* state, int depth, int key_bits, const int32_t* order_ids, int64_t* code, int64_t* order,
                               int64_t* inverse, void* workspace, size_t workspace_bytes, void* stream_) {
    if (!state || !order_ids || !code || !order || !inverse || !workspace) return PTV3_EINVAL;
    State& s = *(State*)state;
    const ptv3_index_cfg& g = s.cfg;
    hipStream_t stream = (hipStream_t)stream_;
    int rc = ptv3_serialize_keys(s.grid, s.batch, g.n, depth, order_ids, g.n_orders, key_bits, code, order, inverse, s.keys, workspace,
                                 workspace_bytes, stream);
    if (rc != PTV3_OK) return rc;
    s.depth = depth;
    s.key_bits = key_bits;
    s.lv[0].code = code;
    s.lv[0].order = order;
    s.lv[0].inverse = inverse;
    CellArgs& a = s.cells;
    a.n = g.n;
    a.levels = g.n_levels - 1;
    a.k = g.n_orders;
    a.scene_shift = 3 * depth;
    int left = depth;
    for (int j = 1; j <= a.levels; ++j) {
        const int d = g.pool_depth[j] > left ? 0 : g.pool_depth[j];
        left -= d;
        a.depth[j] = a.depth[j - 1] + d;
        a.shift[j] = 3 * a.depth[j];
        s.lv[j].depth = left;
    }
    s.lv[0].depth = depth;
    a.order = order;
    a.blk = s.blk;
    a.totals = s.totals;
    a.end_local = s.end_local;
    a.grid = s.grid;
    a.batch = s.batch;
    s.pads.levels = g.n_levels;
    for (int l = 0; l < g.n_levels; ++l) {
        s.pads.patch[l] = g.patch[l];
        s.pads.offset[l] = s.lv[l].offset;
    }
    if (a.levels > 0) {
        rc = key_bits <= 32 ? launch_cells_count<uint32_t>(s, stream) : launch_cells_count<uint64_t>(s, stream);
        if (rc != PTV3_OK) return rc;
        hipLaunchKernelGGL(cell_scan_kernel, dim3((unsigned)(a.k * a.levels)), dim3(SCAN_T), 0, stream, a.blk, a.blocks,
                           a.totals);
    }
    hipLaunchKernelGGL(publish_cells_kernel, dim3(1), dim3(256), 0, stream, a, s.pads, g.n_scenes, s.slot, s.seq);
    PTV3_RETURN_LAUNCH();
}

namespace {

// sizes of every level from the words the sort stage left in the slot
void read_sizes(State& s) {
    const ptv3_index_cfg& g = s.cfg;
    for (int l = 0; l < g.n_levels; ++l) {
        ptv3_level& v = s.lv[l];
        if (l > 0) v.n = s.slot[PTV3_SLOT_DATA + 4 + l - 1];
        const int64_t* ends = s.slot + PTV3_SLOT_ENDS + (int64_t)l * g.n_scenes;
        ptv3_pad_sizes(ends, g.n_scenes, g.patch[l], &v.n_pad, &v.n_seq);
    }
}

Bytes carve_pool(State& s, void* tables, void* scratch) {
    const ptv3_index_cfg& g = s.cfg;
    Carver c(tables), free(scratch);
    const int k = g.n_orders;
    for (int l = 0; l < g.n_levels; ++l) {
        ptv3_level& v = s.lv[l];
        if (l > 0) {
            v.code = c.take<int64_t>((size_t)k * v.n);
            v.order = c.take<int64_t>((size_t)k * v.n);
            v.inverse = c.take<int64_t>((size_t)k * v.n);
            v.grid = c.take<int32_t>(3 * v.n);
            v.batch = c.take<int64_t>(v.n);
            v.indices = c.take<int32_t>(4 * v.n);
            v.cluster = c.take<int64_t>(s.lv[l - 1].n);
            v.idx_ptr = c.take<int64_t>(v.n + 1);
        }
        v.cu = c.take<int32_t>(v.n_seq + 1);
        v.pad = v.unpad = nullptr;
        if (l == 0 || g.pads_all) {
            v.pad = c.take<int64_t>(v.n_pad);
            v.unpad = c.take<int64_t>(v.n);
        }
        for (int r = 0; r < OR; ++r) {
            v.slot_src[r] = v.slot_dst[r] = nullptr;
            if (r < k && ((g.slot_orders[l] >> r) & 1u)) {
                v.slot_src[r] = c.take<int32_t>(v.n_pad);
                v.slot_dst[r] = c.take<int32_t>(v.n_pad);
            }
        }
    }
    free.take<char>(1);   // never empty, also where there is no pooled level
    for (int l = 1; l < g.n_levels; ++l) {
        s.cells.cid[l] = free.take<int32_t>(g.n);
        ListLevel& v = s.lists.lv[l];
        v.n = s.lv[l].n;
        v.group = ptv3_conv_tile_voxels(v.n, g.only128[l] ? 128 : 64);
        carve_list_scratch(free, c, v, false);
    }
    return {c.off, free.off};
}

size_t carve_lists(State& s, const int32_t* want, void* base) {
    Carver c(base);
    for (int l = 0; l < s.cfg.n_levels; ++l) {
        ListLevel& v = s.lists.lv[l];
        ptv3_level& out = s.lv[l];
        v.want = want[l];
        v.row_ptr = v.pair_in = v.pair_slot = v.tile_tap = nullptr;
        v.tile_pair = v.vox_taps = nullptr;
        v.row_ptr5 = v.pair_in5 = v.pair_slot5 = v.pair_out = v.pair_out5 = nullptr;
        if (want[l] & PTV3_LISTS_PAIRS) {
            v.row_ptr = c.take<int32_t>(v.n + 1);
            v.pair_in = c.take<int32_t>(out.n_pairs);
            v.pair_slot = c.take<int32_t>(out.n_pairs);
            if (want[l] & PTV3_LISTS_PAIR_OUT) v.pair_out = c.take<int32_t>(out.n_pairs);
        }
        if (want[l] & PTV3_LISTS_TILES) {
            v.tile_tap = c.take<int32_t>((size_t)v.groups * TILE_WORDS);
            v.tile_pair = c.take<uint32_t>(out.n_pairs);
            v.vox_taps = c.take<uint32_t>(v.n);
        }
        if (v.tap5 && (want[l] & PTV3_LISTS_PAIRS5)) {
            v.row_ptr5 = c.take<int32_t>(v.n + 1);
            v.pair_in5 = c.take<int32_t>(out.n_pairs5);
            v.pair_slot5 = c.take<int32_t>(out.n_pairs5);
            if (want[l] & PTV3_LISTS_PAIR_OUT5) v.pair_out5 = c.take<int32_t>(out.n_pairs5);
        }
    }
    return c.off;
}

}  // namespace

extern "C" int ptv3_index_pool_bytes(void* state, size_t* tables, size_t* scratch) {
    if (!state || !tables || !scratch) return PTV3_EINVAL;
    State& s = *(State*)state;
    read_sizes(s);
    for (int l = 0; l < s.cfg.n_levels; ++l)
        if (s.lv[l].n < 1 || s.lv[l].n > s.cfg.n || s.lv[l].n_pad >= (1ll << 31)) return PTV3_EINVAL;
    const Bytes need = carve_pool(s, nullptr, nullptr);
    *tables = need.tables;
    *scratch = need.scratch;
    return PTV3_OK;
}

extern "C" int ptv3_index_pool(void* state, const int32_t* perms, void* tables, size_t tables_bytes, void* scratch,
                               size_t scratch_bytes, void* stream_) {
    if (!state || !tables || !scratch) return PTV3_EINVAL;
    State& s = *(State*)state;
    const ptv3_index_cfg& g = s.cfg;
    hipStream_t stream = (hipStream_t)stream_;
    const Bytes need = carve_pool(s, nullptr, nullptr);
    if (tables_bytes < need.tables || scratch_bytes < need.scratch) return PTV3_EWORKSPACE;
    carve_pool(s, tables, scratch);
    CellArgs& a = s.cells;
    const int k = g.n_orders;
    // rows of the tables are permuted at every pooling: row r of level j is row perms[j][r] of the level above
    int from[OR];   // level-0 row behind row r of the level above
    for (int r = 0; r < k; ++r) from[r] = r;
    for (int j = 1; j <= a.levels; ++j) {
        a.curve0[j] = from[0];
        int next[OR];
        uint32_t seen = 0;
        for (int r = 0; r < k; ++r) {
            const int p = perms ? perms[(j - 1) * k + r] : r;
            if (p < 0 || p >= k || (seen >> p & 1u)) return PTV3_EINVAL;
            seen |= 1u << p;
            next[r] = from[p];
            a.row_of[j][next[r]] = r;
        }
        for (int r = 0; r < k; ++r) from[r] = next[r];
        const ptv3_level& v = s.lv[j];
        a.m[j] = v.n;
        a.code[j] = v.code;
        a.order_out[j] = v.order;
        a.inverse_out[j] = v.inverse;
        a.batch_out[j] = v.batch;
        a.cluster[j] = v.cluster;
        a.idx_ptr[j] = v.idx_ptr;
        a.grid_out[j] = v.grid;
        a.indices_out[j] = (int4*)v.indices;
        s.lists.lv[j].idx = (const int4*)v.indices;
    }
    int rc = PTV3_OK;
    if (a.levels > 0) {
        rc = s.key_bits <= 32 ? launch_cells_tables<uint32_t>(s, stream) : launch_cells_tables<uint64_t>(s, stream);
        if (rc != PTV3_OK) return rc;
        rc = launch_hash_count(s, 1, g.n_levels, stream);
        if (rc != PTV3_OK) return rc;
    }
    list_blocks(s.lists, 0, g.n_levels, 2);
    int cols = 0;
    for (int l = 0; l < g.n_levels; ++l) cols += TAPS3 + 1 + (s.lists.lv[l].tap5 ? TAPS5 + 1 : 0);
    hipLaunchKernelGGL(list_scan_kernel, dim3((unsigned)cols), dim3(SCAN_T), 0, stream, s.lists);
    hipLaunchKernelGGL(publish_lists_kernel, dim3(1), dim3(1024), 0, stream, s.lists, s.slot, s.seq);
    SlotArgs t = {};
    t.levels = g.n_levels;
    t.nb = g.n_scenes;
    t.k = k;
    int at = 0;
    for (int l = 0; l < g.n_levels; ++l) {
        const ptv3_level& v = s.lv[l];
        t.first_block[l] = at;
        at += (int)ptv3_ceil_div(v.n_pad, 256);
        t.patch[l] = g.patch[l];
        t.n[l] = v.n;
        t.n_pad[l] = v.n_pad;
        t.n_seq[l] = v.n_seq;
        t.offset[l] = v.offset;
        t.pad_start[l] = s.pads.pad_start[l];
        t.seq_start[l] = s.pads.seq_start[l];
        t.order[l] = v.order;
        t.pad[l] = v.pad;
        t.unpad[l] = v.unpad;
        t.cu[l] = v.cu;
        for (int r = 0; r < k; ++r) {
            t.src[l][r] = v.slot_src[r];
            t.dst[l][r] = v.slot_dst[r];
        }
    }
    t.first_block[g.n_levels] = at;
    hipLaunchKernelGGL(slots_kernel, dim3((unsigned)at), dim3(256), 0, stream, t);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_index_lists_bytes(void* state, const int32_t* want, size_t* bytes) {
    if (!state || !want || !bytes) return PTV3_EINVAL;
    State& s = *(State*)state;
    for (int l = 0; l < s.cfg.n_levels; ++l) {
        const int64_t* p = s.slot + PTV3_SLOT_DATA + 4 + LV + 2 * l;
        s.lv[l].n_pairs = p[0];
        s.lv[l].n_pairs5 = s.lists.lv[l].tap5 ? p[1] : 0;
        if (p[0] < 0 || p[0] > s.lv[l].n * TAPS3) return PTV3_EINVAL;
    }
    *bytes = carve_lists(s, want, nullptr);
    return PTV3_OK;
}

extern "C" int ptv3_index_lists(void* state, const int32_t* want, void* lists, size_t lists_bytes, void* stream_) {
    if (!state || !want || !lists) return PTV3_EINVAL;
    State& s = *(State*)state;
    hipStream_t stream = (hipStream_t)stream_;
    if (lists_bytes < carve_lists(s, want, nullptr)) return PTV3_EWORKSPACE;
    carve_lists(s, want, lists);
    int first = 0;
    if (s.lists.lv[0].tap5) {
        hipLaunchKernelGGL(list_fill_kernel<5>, dim3((unsigned)list_blocks(s.lists, 0, 1, 2)), dim3(GT), 0, stream, s.lists);
        first = 1;
    }
    if (first < s.cfg.n_levels)
        hipLaunchKernelGGL(list_fill_kernel<3>, dim3((unsigned)list_blocks(s.lists, first, s.cfg.n_levels, 2)), dim3(GT), 0,
                           stream, s.lists);
    for (int l = 0; l < s.cfg.n_levels; ++l) {
        const ListLevel& v = s.lists.lv[l];
        ptv3_level& o = s.lv[l];
        o.tap_ptr = v.tap_ptr;
        o.row_ptr = v.row_ptr;
        o.pair_in = v.pair_in;
        o.pair_slot = v.pair_slot;
        o.tile_tap = v.tile_tap;
        o.tile_pair = (int32_t*)v.tile_pair;
        o.vox_taps = (int32_t*)v.vox_taps;
        o.tap_ptr5 = v.tap_ptr5;
        o.row_ptr5 = v.row_ptr5;
        o.pair_in5 = v.pair_in5;
        o.pair_slot5 = v.pair_slot5;
        o.pair_out = v.pair_out;
        o.pair_out5 = v.pair_out5;
        o.tile_voxels = v.group;
    }
    PTV3_RETURN_LAUNCH();
}

extern "C" const ptv3_level* ptv3_index_levels(const void* state) { return state ? ((const State*)state)->lv : nullptr; }
