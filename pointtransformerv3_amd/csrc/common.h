// Shared helpers for the gfx950 kernels of libptv3_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "ptv3_hip.h"

#define PTV3_WAVE 64

// Launch-error check: returns the hipError_t (> 0) to the C caller.
#define PTV3_RETURN_LAUNCH()                         \
    do {                                             \
        hipError_t e__ = hipGetLastError();          \
        return e__ == hipSuccess ? PTV3_OK : (int)e__; \
    } while (0)

static inline int64_t ptv3_ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
// A thread index split into (row, piece) by the pieces of a row. A power of two, which the model's widths make it, is a
// shift; the 64-bit division is some hundred instructions, as much as everything else a thread of a row kernel does. Kernels
// bound by memory do not show it (unpooling add of 1M rows 180 us either way), shorter and busier ones do: BatchNorm + GELU of
// a scene of 1M points 235 -> 209 us in five launches; see pair_segment_sum_kernel.
struct PieceDiv {
    int count, shift;   // shift < 0: divide
};
static inline PieceDiv ptv3_piece_div(int count) {
    int s = 0;
    while ((1 << s) < count) ++s;
    return PieceDiv{count, (1 << s) == count ? s : -1};
}
__device__ __forceinline__ int64_t ptv3_row_of(int64_t e, PieceDiv d) { return d.shift >= 0 ? e >> d.shift : e / d.count; }

// The job of this work-group: the last of a table (first_block ascending) that starts at or before it. A lane per job: one
// trip to memory, where a walk down the table is one per job (22 jobs of packing weights in a forward: 14 - 21 us, 10 - 14 so).
template <typename J>
__device__ __forceinline__ int ptv3_job_of_block(const J* __restrict__ jobs, int n_jobs) {
    const int lane = threadIdx.x % 64;
    int started = 0;
    for (int j = 0; j < n_jobs; j += 64)
        started += __popcll(__ballot(j + lane < n_jobs && jobs[min(j + lane, n_jobs - 1)].first_block <= (int64_t)blockIdx.x));
    return max(started - 1, 0);
}

// Rows that are read for the last time, or written for much later, go past the caches (the nontemporal hint) where they are more
// than those hold: what the next kernels read stays there. Of less than that the last kernel's rows are still in the L2. The
// choice is a template argument: the compiler makes one ordinary access of two behind a condition.
template <bool ONCE, typename V> __device__ __forceinline__ V ptv3_read(const V* p) {
    if constexpr (ONCE) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool ONCE, typename V> __device__ __forceinline__ void ptv3_write(V* p, V v) {
    if constexpr (ONCE) __builtin_nontemporal_store(v, p);
    else *p = v;
}

static inline size_t ptv3_align256(size_t v) { return (v + 255) & ~(size_t)255; }

// More than 64 KB of dynamic LDS has to be allowed per kernel, and the runtime keeps that attribute per device.
// A launcher keeps one LdsGrant per kernel instantiation (a function-local static): the largest size allowed so
// far on each device. ptv3_allow_lds raises it for the current device when `lds` exceeds it; 0 or a hipError_t.
constexpr int PTV3_MAX_DEVICES = 64;
struct LdsGrant {
    std::atomic<size_t> bytes[PTV3_MAX_DEVICES];
};
static inline int ptv3_allow_lds(const void* kern, size_t lds, LdsGrant& grant) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    const bool tracked = dev >= 0 && dev < PTV3_MAX_DEVICES;
    if (tracked && lds <= grant.bytes[dev].load(std::memory_order_acquire)) return 0;
    static std::mutex mu;   // the slow path: set the attribute and record it as one step
    std::lock_guard<std::mutex> lock(mu);
    if (tracked && lds <= grant.bytes[dev].load(std::memory_order_relaxed)) return 0;
    e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    if (tracked) grant.bytes[dev].store(lds, std::memory_order_release);
    return 0;
}

// CUs of the current device: what rules that fill the part go by. 256, the whole MI355X, where there is none to ask (a size
// asked for before a device is there, on the host alone).
static inline int ptv3_cus() {
    static std::atomic<int> known[PTV3_MAX_DEVICES];
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 256;
    if (dev < PTV3_MAX_DEVICES && (n = known[dev].load(std::memory_order_relaxed)) > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) return 256;
    if (dev < PTV3_MAX_DEVICES) known[dev].store(n, std::memory_order_relaxed);
    return n;
}

// What the device's L2s hold: 4 MB an XCD of 32 CUs
static inline int64_t ptv3_l2_bytes() { return (int64_t)(ptv3_cus() / 32 > 1 ? ptv3_cus() / 32 : 1) << 22; }

// Weights that every XCD reads whole in the launch behind this one: a kernel that leaves memory idle asks for them, and they are
// in its XCD's L2 by then. In a forward they come from HBM otherwise, and a kernel that streams them has few requests in flight.
struct Ahead {
    const uint8_t* at[2];
    uint32_t lines[2];   // of 128 bytes, each begun
};
static inline Ahead ptv3_ahead(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
    return Ahead{{(const uint8_t*)a, (const uint8_t*)b},
                 {a ? (uint32_t)ptv3_ceil_div(a_bytes, 128) : 0, b ? (uint32_t)ptv3_ceil_div(b_bytes, 128) : 0}};
}
// This work-group's share: the lines are dealt to the last AHEAD_GROUPS work-groups of each XCD, whose own traffic will not have
// replaced them (two a CU), at most four a thread. What comes back is used in ptv3_asked alone, at the kernel's end, and so waited for there.
constexpr uint32_t AHEAD_GROUPS = 64;
__device__ __forceinline__ uint32_t ptv3_ask(const Ahead& a, int tid, int threads) {
    const uint32_t total = a.lines[0] + a.lines[1], groups = gridDim.x >> 3, slot = blockIdx.x >> 3;
    const uint32_t askers = min(groups, AHEAD_GROUPS);
    uint32_t v = 0;
    if (total == 0 || slot >= groups || slot + askers < groups) return v;
    const uint32_t per = (total + askers - 1) / askers, first = (slot + askers - groups) * per;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uint32_t i = (uint32_t)(tid + u * threads), line = first + i;
        if (i < per && line < total)
            v |= line < a.lines[0] ? a.at[0][(size_t)line * 128] : a.at[1][(size_t)(line - a.lines[0]) * 128];
    }
    return v;
}
__device__ __forceinline__ void ptv3_asked(uint32_t v) { asm volatile("" ::"v"(v)); }

// ptv3_patch_attn_fwd where the number of slots, cu_seqlens[n_seq], is known: what ptv3_patch_attn_cut goes by.
int ptv3_patch_attn_fwd_slots(const void* qkv, int dtype, int64_t n_rows, int channels, int heads, const int32_t* slot_src,
                              const int32_t* slot_dst, const int32_t* cu_seqlens, int64_t n_seq, int64_t max_seqlen,
                              int64_t slots, float scale, void* out, const Ahead& ahead, void* stream);
// ptv3_subm_conv_pairs_fwd
int ptv3_conv_pairs_ahead(const void* feat, int dtype, int64_t n, int cin, int taps, int64_t n_pairs, const int32_t* tap_ptr,
                          const int32_t* row_ptr, const int32_t* pair_in, const int32_t* pair_slot, const void* weight,
                          const void* bias, int cout, void* y, void* out, const Ahead& ahead, void* stream);

// Work-groups are dealt to the 8 XCDs round-robin in launch order, and every XCD has an L2 of its own.
// Launch index (or persistent-loop index, with a grid that is a multiple of 8) -> item such that each XCD
// works through one contiguous eighth of the items: neighbours in item order, which read the same cache lines
// (the heads of a sequence, the column blocks of one row tile), meet in one L2 at about the same time.
__device__ __forceinline__ int xcd_chunked_id(int bid, int total) {
    const int xcd = bid & 7, slot = bid >> 3;
    const int per = total >> 3, rem = total & 7;
    return xcd * per + min(xcd, rem) + slot;
}
