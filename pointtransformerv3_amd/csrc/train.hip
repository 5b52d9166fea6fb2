// A training step's forward and backward as one call each: the modules' operators under half-precision autocast
// (modules.py, autograd.py: Block._forward_training, SerializedPooling, SerializedUnpooling, Embedding), queued natively over
// an index of ptv3_index_*. As autograd nodes the same work is some 250 Python functions each way, about 20 ms of host
// time per step whatever the batch; here the host takes about 2 us per launch.
//
// One layout function places every tensor that the backward reads in the caller's activation buffer (`Acts`); forward and
// backward run it over the same sizes and meet at the same addresses. Gradients go straight to their places in one flat
// float buffer. What the separate nodes did in several passes is one here: the residual sum and its half copy for the
// next convolution, the sum of a block's two output gradients with the stochastic-depth factor for its branch
// (ptv3_two_sums), the slab sums of a block's weight gradients (ptv3_slab_sums).
#include <string.h>

#include "common.h"
#include "outer.h"

namespace {

#define DO(call)                                   \
    do {                                           \
        if (!dry) {                                \
            const int rc__ = (call);               \
            if (rc__ != PTV3_OK) return rc__;      \
        }                                          \
    } while (0)
#define TRY(call)                         \
    do {                                  \
        const int rc__ = (call);          \
        if (rc__ != PTV3_OK) return rc__; \
    } while (0)

struct Space {
    char* base;
    size_t at = 0, top = 0;
    explicit Space(void* b) : base((char*)b) {}
    void* take(size_t bytes) {
        void* p = base ? base + at : nullptr;
        at += ptv3_align256(bytes ? bytes : 1);
        if (at > top) top = at;
        return p;
    }
};

struct BlockActs {
    const void* xs;             // what the convolution reads (half)
    void *conv, *cpe, *sum1, *y1, *qkv, *attn, *sum2, *y2, *pre, *act, *out16;
    float* lse;
};
struct BnActs {
    void *x, *y;                // its input and its result behind the GELU (half)
    float* stats;               // mean, rstd, biased variance
};
struct StageActs {
    BlockActs *enc, *dec;
    void *pool_in, *pooled;     // projected rows of the level above and their segment maxima (half)
    BnActs pool_bn, up_bn, skip_bn;
    void *up_sum;               // unpooled rows: skip projection + child (half)
};
constexpr int MAX_BLOCKS = 256;
// A group of weight gradients: what it holds before it is launched, and its lists. Every group is two events each way and
// launches of its own, so small blocks share one: a step of 2 x 15k voxels has 12 groups at 64 MB and 31 at one a block, and
// queueing its backward takes the host 1.3 ms and 2.3 ms. On the GPU the step takes 8.06 and 8.13 ms (8.38 without a second
// stream), one of 4 x 100k 38.6 and 38.5 ms (39.6), whose blocks are all larger; 160 MB: 8.11, 38.6.
constexpr size_t GROUP_BYTES = 64u << 20;
constexpr int GROUP_LINEARS = 64, GROUP_CONVS = 16;

__global__ __launch_bounds__(256) void zero_floats_kernel(float* __restrict__ out, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < count) out[i] = 0.f;
}
// the BatchNorms' places in the gradients, which their backward adds onto: a work-group each
struct BnPlaces {
    static constexpr int MAX = 1 + 3 * PTV3_MAX_LEVELS;
    int64_t at[MAX];
    int floats[MAX], count;
    void add(const ptv3_train_bn& b, int c) {
        at[count] = b.gg;
        floats[count++] = 2 * c;
    }
};
__global__ __launch_bounds__(256) void zero_places_kernel(float* __restrict__ base, BnPlaces places) {
    for (int i = threadIdx.x; i < places.floats[blockIdx.x]; i += 256) base[places.at[blockIdx.x] + i] = 0.f;
}
int zero_places(float* base, const BnPlaces& places, hipStream_t stream) {
    hipLaunchKernelGGL(zero_places_kernel, dim3((unsigned)places.count), dim3(256), 0, stream, base, places);
    PTV3_RETURN_LAUNCH();
}
int zero_floats(float* out, int64_t count, hipStream_t stream) {
    hipLaunchKernelGGL(zero_floats_kernel, dim3((unsigned)ptv3_ceil_div(count, 256)), dim3(256), 0, stream, out, count);
    PTV3_RETURN_LAUNCH();
}

struct Run {
    const ptv3_train_net& net;
    const ptv3_level* lv;
    void* stream;
    hipStream_t hs;
    const int dt;               // PTV3_F16 or PTV3_BF16
    bool dry = false;           // only the scratch is measured: nothing is queued
    void* final_out = nullptr;  // the model's rows (float)
    StageActs st[PTV3_MAX_LEVELS];
    BlockActs pool[MAX_BLOCKS];
    BnActs stem_bn;
    void *stem_in, *stem_x;     // padded input rows, the stem's rows
    int32_t *map3[PTV3_MAX_LEVELS] = {}, *map5 = nullptr;   // neighbour maps of levels whose convolutions take the dense form
    bool has_map3[PTV3_MAX_LEVELS] = {};
    Run(const ptv3_train_net& n, const ptv3_level* l, void* s) : net(n), lv(l), stream(s), hs((hipStream_t)s), dt(n.dtype) {}

    void place_bn(Space& m, BnActs& b, int64_t n, int c) {
        b.x = m.take((size_t)n * c * 2);
        b.y = m.take((size_t)n * c * 2);
        b.stats = (float*)m.take(3 * (size_t)c * 4);
    }
    void place_block(Space& m, BlockActs& a, const ptv3_train_block& b, const ptv3_level& v) {
        const size_t r = (size_t)v.n * b.channels;
        a.conv = m.take(2 * r);
        a.cpe = m.take(2 * r);
        a.sum1 = m.take(4 * r);
        a.y1 = m.take(2 * r);
        a.qkv = m.take(6 * r);
        a.attn = m.take(2 * r);
        a.lse = (float*)m.take((size_t)b.heads * v.n_pad * 4);
        a.sum2 = m.take(4 * r);
        a.y2 = m.take(2 * r);
        a.pre = m.take(8 * r);
        a.act = m.take(8 * r);
        a.out16 = m.take(2 * r);
    }
    // every tensor that the backward reads
    void place(Space& m) {
        const int S = net.n_stages;
        stem_in = m.take((size_t)lv[0].n * net.stem.cin_padded * 2);
        place_bn(m, stem_bn, lv[0].n, net.stage[0].channels);
        BlockActs* next = pool;
        for (int s = 0; s < S; ++s) {
            const ptv3_train_stage& g = net.stage[s];
            if (s > 0) {
                st[s].pool_in = m.take((size_t)lv[s - 1].n * g.channels * 2);
                place_bn(m, st[s].pool_bn, lv[s].n, g.channels);
                st[s].pooled = st[s].pool_bn.x;
            }
            st[s].enc = next;
            for (int i = 0; i < g.n_enc; ++i) place_block(m, *next++, g.enc[i], lv[s]);
        }
        for (int s = S - 2; s >= 0; --s) {
            const ptv3_train_stage& g = net.stage[s];
            place_bn(m, st[s].up_bn, lv[s + 1].n, g.dec_channels);
            place_bn(m, st[s].skip_bn, lv[s].n, g.dec_channels);
            st[s].up_sum = m.take((size_t)lv[s].n * g.dec_channels * 2);
            st[s].dec = next;
            for (int i = 0; i < g.n_dec; ++i) place_block(m, *next++, g.dec[i], lv[s]);
        }
        place_maps(m);
    }

    // what each block's convolution reads
    void link() {
        for (int s = 0; s < net.n_stages; ++s) {
            const ptv3_train_stage& g = net.stage[s];
            for (int i = 0; i < g.n_enc; ++i) st[s].enc[i].xs = i ? st[s].enc[i - 1].out16 : s ? st[s].pool_bn.y : stem_bn.y;
            for (int i = 0; i < g.n_dec; ++i) st[s].dec[i].xs = i ? st[s].dec[i - 1].out16 : st[s].skip_bn.y;
        }
    }

    // x W^T + b on the kernel that fits (in / out: the product's own, also for a transposed weight)
    int linear(const void* x, const void* w, const void* b, int in, int out, int64_t n, void* y) {
        if (dry) return PTV3_OK;
        const bool rows = in == 32 || in == 64 || in == 96 || in == 128 || in == 192 || in == 256 || in == 384 || in == 512;
        if (rows && out % 32 == 0 && (in <= 256 || out <= 2 * in)) {
            if (in == 256 && out % 256 == 0 && n >= 4096) return ptv3_linear_wide_fwd(x, w, b, dt, n, in, out, 0, y, stream);
            return ptv3_linear_fwd(x, w, b, dt, n, in, out, 0, y, stream);
        }
        return ptv3_linear_gemm_fwd(x, w, b, nullptr, dt, n, in, out, y, stream);
    }

    int conv(const ptv3_train_block& b, const ptv3_level& v, bool back, const void* x, Space& scratch, void* out) {
        const int c = b.channels, form = ptv3_conv_form(v.n, v.n_pairs, c);
        const void *w = back ? b.conv_mirror : b.conv_w, *packed = back ? b.conv_mirror_packed : b.conv_packed;
        const void* bias = back ? nullptr : b.conv_b;
        if (dry && form) return PTV3_OK;
        if (form == 1)
            return ptv3_subm_conv_sparse_fwd(x, dt, v.n, c, 27, packed, bias, v.tile_tap, v.tile_pair, out, stream);
        if (form == 2)
            return ptv3_subm_conv_tiles_fwd_sized(x, dt, v.n, c, 27, v.tile_voxels, packed, bias, v.tile_tap, v.tile_pair,
                                                  v.vox_taps, out, stream);
        return conv_rows((int)(&v - lv), 27, x, c, w, bias, c, out, scratch);
    }
    // one that no tile form takes, as in features.hip; the neighbour maps of the dense form lie beside the activations
    int pair_form(int s, int taps, int cin, int cout) const {
        const ptv3_level& v = lv[s];
        return ptv3_conv_pair_form(dt, v.n, taps == 27 ? v.n_pairs : v.n_pairs5, taps, cin, cout, net.max_pair_density);
    }
    int conv_rows(int s, int taps, const void* x, int cin, const void* w, const void* bias, int cout, void* out, Space& scratch) {
        const ptv3_level& v = lv[s];
        const bool inner = taps == 27;
        const int64_t n_pairs = inner ? v.n_pairs : v.n_pairs5;
        const int32_t *tap_ptr = inner ? v.tap_ptr : v.tap_ptr5, *row_ptr = inner ? v.row_ptr : v.row_ptr5;
        const int32_t *pair_in = inner ? v.pair_in : v.pair_in5, *pair_slot = inner ? v.pair_slot : v.pair_slot5;
        const int form = pair_form(s, taps, cin, cout);
        if (form == PTV3_CONV_DENSE) {
            DO(ptv3_subm_conv_fwd(x, dt, v.n, cin, inner ? map3[s] : map5, taps, 1, w, bias, cout, out, stream));
            return PTV3_OK;
        }
        const bool wide = form == PTV3_CONV_PAIRS_WIDE;
        const size_t mark = scratch.at;
        void* y = scratch.take((size_t)n_pairs * cout * (wide ? 4 : 2));
        scratch.at = mark;
        if (dry) return PTV3_OK;
        if (wide)
            return ptv3_subm_conv_pairs_wide_fwd(x, dt, v.n, cin, taps, n_pairs, tap_ptr, row_ptr, pair_in, pair_slot, w, bias, cout,
                                                 (float*)y, out, stream);
        return ptv3_subm_conv_pairs_fwd(x, dt, v.n, cin, taps, n_pairs, tap_ptr, row_ptr, pair_in, pair_slot, w, bias, cout, y, out,
                                        stream);
    }
    bool dense3(int s) const {
        const ptv3_train_stage& g = net.stage[s];
        for (int side = 0; side < 2; ++side) {
            const int c = side ? g.dec_channels : g.channels;
            if ((side ? g.n_dec : g.n_enc) && ptv3_conv_form(lv[s].n, lv[s].n_pairs, c) == 0 &&
                pair_form(s, 27, c, c) == PTV3_CONV_DENSE)
                return true;
        }
        return false;
    }
    void place_maps(Space& m) {
        if (pair_form(0, 125, net.stem.cin_padded, net.stage[0].channels) == PTV3_CONV_DENSE)
            map5 = (int32_t*)m.take((size_t)lv[0].n * 125 * 4);
        for (int s = 0; s < net.n_stages; ++s) {
            has_map3[s] = dense3(s);
            if (has_map3[s]) map3[s] = (int32_t*)m.take((size_t)lv[s].n * 27 * 4);
        }
    }
    int make_map(int s, int ks, int32_t* map, Space& scratch) {
        const size_t mark = scratch.at, bytes = ptv3_kmap_workspace_bytes(lv[s].n);
        void* ws = scratch.take(bytes);
        scratch.at = mark;
        DO(ptv3_kmap_build(lv[s].indices, lv[s].n, ks, 1, map, ws, bytes, stream));
        return PTV3_OK;
    }
    int make_maps(Space& scratch) {   // by the forward; the backward finds them where they were placed
        if (pair_form(0, 125, net.stem.cin_padded, net.stage[0].channels) == PTV3_CONV_DENSE) TRY(make_map(0, 5, map5, scratch));
        for (int s = 0; s < net.n_stages; ++s)
            if (has_map3[s]) TRY(make_map(s, 3, map3[s], scratch));
        return PTV3_OK;
    }

    float* bn_sums = nullptr;   // zeroed sums of the layers to come
    int bn_gelu(const ptv3_train_bn& b, BnActs& a, int64_t n, int c) {
        if (dry) return PTV3_OK;
        float* sums = bn_sums;
        bn_sums += 2 * c;
        TRY(ptv3_batch_norm_sums(a.x, dt, n, c, sums, hs));
        return ptv3_batch_norm_gelu_train(a.x, dt, n, c, sums, b.g16, b.b16, b.eps, b.momentum, b.running_mean, b.running_var, a.stats,
                                          a.y, hs);
    }

    // out: the block's rows in float, or null where only the half copy (out16) is read
    int block_fwd(const ptv3_train_block& b, const BlockActs& a, const ptv3_level& v, int patch, const void* mask1, const void* mask2,
                  const void* skip, int skip_dt, void* out, bool copy16, Space& scratch) {
        const int64_t n = v.n;
        const int c = b.channels;
        TRY(conv(b, v, false, a.xs, scratch, a.conv));
        TRY(linear(a.conv, b.cpe.w, b.cpe.b, c, c, n, a.cpe));
        DO(ptv3_add_layer_norm_fwd(skip, skip_dt, a.cpe, dt, nullptr, 0, b.ln1.g, b.ln1.b, PTV3_F32, n, c, b.ln1.eps, a.sum1,
                                    PTV3_F32, a.y1, dt, b.ln_cpe.g, b.ln_cpe.b, b.ln_cpe.eps, stream));
        TRY(linear(a.y1, b.qkv.w, b.qkv.b, c, 3 * c, n, a.qkv));
        DO(ptv3_patch_attn_fwd_lse(a.qkv, dt, n, c, b.heads, v.slot_src[b.row], v.slot_dst[b.row], v.cu, v.n_seq, patch, v.n_pad,
                                    b.scale, 0.f, 0, a.attn, a.lse, stream));
        const size_t mark = scratch.at;
        void* branch = scratch.take((size_t)n * c * 2);
        TRY(linear(a.attn, b.proj.w, b.proj.b, c, c, n, branch));
        DO(ptv3_add_layer_norm_fwd(a.sum1, PTV3_F32, branch, dt, mask1, dt, b.ln2.g, b.ln2.b, PTV3_F32, n, c, b.ln2.eps, a.sum2,
                                    PTV3_F32, a.y2, dt, nullptr, nullptr, 0.f, stream));
        DO(ptv3_linear_gelu_fwd(a.y2, b.fc1.w, b.fc1.b, dt, n, c, 4 * c, a.pre, a.act, stream));
        TRY(linear(a.act, b.fc2.w, b.fc2.b, 4 * c, c, n, branch));
        DO(ptv3_two_sums(a.sum2, PTV3_F32, branch, dt, mask2, nullptr, dt, n, c, out, copy16 ? a.out16 : nullptr, dt, hs));
        scratch.at = mark;
        return PTV3_OK;
    }

    // blocks of a stage: the first adds onto `skip` (half rows), the others onto the one in front. The last one's float
    // rows go to `out`, or nowhere when it is null: what follows reads the half copy.
    int stage_fwd(const ptv3_train_block* bs, const BlockActs* as, int count, int level, const void* skip, void* out,
                  const void* const*& masks, Space& scratch) {
        const size_t mark = scratch.at;
        void* turn[2];
        for (int i = 0; i < 2; ++i) turn[i] = scratch.take((size_t)lv[level].n * bs[0].channels * 4);
        int skip_dt = dt;
        for (int i = 0; i < count; ++i) {
            const bool last = i + 1 == count;
            void* to = last ? out : turn[i & 1];
            TRY(block_fwd(bs[i], as[i], lv[level], net.patch[level], masks[0], masks[1], skip, skip_dt, to, !last || !out, scratch));
            masks += 2;
            skip = to;
            skip_dt = PTV3_F32;
        }
        scratch.at = mark;
        return PTV3_OK;
    }

    int forward(const void* feat, int feat_dt, const void* const* masks, Space& scratch) {
        const int S = net.n_stages;
        const ptv3_level& v0 = lv[0];
        const int c0 = net.stage[0].channels;
        int64_t count = 2 * c0;
        for (int s = 0; s < S; ++s) count += 2 * (s > 0 ? net.stage[s].channels : 0) + 4 * (s < S - 1 ? net.stage[s].dec_channels : 0);
        bn_sums = (float*)scratch.take((size_t)count * 4);
        DO(zero_floats(bn_sums, count, hs));
        DO(ptv3_pad_rows(feat, feat_dt, v0.n, net.stem.cin, net.stem.cin_padded, stem_in, dt, stream));
        TRY(make_maps(scratch));
        TRY(conv_rows(0, 125, stem_in, net.stem.cin_padded, net.stem.w, nullptr, c0, stem_bn.x, scratch));
        TRY(bn_gelu(net.stem.bn, stem_bn, v0.n, c0));
        const void* x = stem_bn.y;
        for (int s = 0; s < S; ++s) {
            const ptv3_train_stage& g = net.stage[s];
            if (s > 0) {
                const ptv3_level &v = lv[s], &up = lv[s - 1];
                TRY(linear(st[s - 1].enc[net.stage[s - 1].n_enc - 1].out16, g.pool.w, g.pool.b, g.pool.in, g.pool.out, up.n,
                           st[s].pool_in));
                DO(ptv3_segment_reduce(st[s].pool_in, dt, up.n, g.channels, up.order, v.idx_ptr, v.n, g.pool_reduce, st[s].pooled,
                                        stream));
                TRY(bn_gelu(g.pool_bn, st[s].pool_bn, v.n, g.channels));
                x = st[s].pool_bn.y;
            }
            TRY(stage_fwd(g.enc, st[s].enc, g.n_enc, s, x, nullptr, masks, scratch));
        }
        const void* child = st[S - 1].enc[net.stage[S - 1].n_enc - 1].out16;
        for (int s = S - 2; s >= 0; --s) {
            const ptv3_train_stage& g = net.stage[s];
            const ptv3_level &v = lv[s], &below = lv[s + 1];
            const int c = g.dec_channels;
            TRY(linear(child, g.up.w, g.up.b, g.up.in, c, below.n, st[s].up_bn.x));
            TRY(bn_gelu(g.up_bn, st[s].up_bn, below.n, c));
            TRY(linear(st[s].enc[g.n_enc - 1].out16, g.up_skip.w, g.up_skip.b, g.up_skip.in, c, v.n, st[s].skip_bn.x));
            TRY(bn_gelu(g.up_skip_bn, st[s].skip_bn, v.n, c));
            DO(ptv3_unpool_add(st[s].skip_bn.y, st[s].up_bn.y, dt, v.n, c, below.cluster, below.n, st[s].up_sum, stream));
            // the first block's convolution reads the skip projection alone (model.py:746)
            TRY(stage_fwd(g.dec, st[s].dec, g.n_dec, s, st[s].up_sum, s ? nullptr : final_out, masks, scratch));
            child = st[s].dec[g.n_dec - 1].out16;
        }
        return PTV3_OK;
    }

    // ---- backward
    float* grads = nullptr;

    // Weight gradients are no part of the chain from dout to the first layer: nothing waits for them but the end of the
    // call. They are put down while a block's chain is queued and launched together behind it (flush), on net.side if the
    // caller gave one, beside the chain of the next blocks. What they read and their slabs lie in one of two arenas in
    // turn; a group of blocks begins with a wait for the group before last, and ends when it holds GROUP_BYTES. On one stream
    // one arena serves every group: 1.5 GiB of scratch at 4 x 100k voxels where two arenas make it 2.1.
    hipStream_t side = nullptr;
    hipEvent_t ready = nullptr, done[2] = {};
    bool busy[2] = {}, unmarked = false, closed = true;   // unmarked: work on the side that no event stands behind
    int turn = 0;
    Space arenas[2] = {Space(nullptr), Space(nullptr)};
    LinearGrad linears[GROUP_LINEARS];
    int n_linears = 0;
    struct ConvGrad {
        const void *x, *dy;
        const int32_t *pair_out, *tap_ptr, *pair_in;
        int64_t n;
        int cin, cout, taps;
        float *dweight, *dbias;
    } convs[GROUP_CONVS];
    int n_convs = 0;

    // descriptions of callers that do not know the field end in front of it, with a zero where the flag is
    bool two_streams() const { return net.has_side && net.side; }
    int open_side() {
        if (!two_streams() || (hipStream_t)net.side == hs) return PTV3_OK;
        hipError_t e = hipEventCreateWithFlags(&ready, hipEventDisableTiming);
        for (int i = 0; i < 2 && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&done[i], hipEventDisableTiming);
        side = e == hipSuccess ? (hipStream_t)net.side : nullptr;
        return (int)e;
    }
    // `stream` goes on behind the last group of arena i, which counts as busy until that is so
    int wait_for(int i) {
        if (!busy[i]) return PTV3_OK;
        const hipError_t e = hipStreamWaitEvent(hs, done[i], 0);
        busy[i] = e != hipSuccess;
        return (int)e;
    }
    // `stream` goes on behind everything queued on the side
    int join() {
        const int first = wait_for(0), second = wait_for(1);
        return first ? first : second;
    }
    // Also where a call has failed: the caller's buffers are free again behind this call's work. Where no event says when the
    // side is through with them, the host waits for it.
    int close_side() {
        int rc = join();
        if (unmarked || busy[0] || busy[1]) {
            const int waited = (int)hipStreamSynchronize(side);
            rc = rc ? rc : waited;
        }
        for (int i = 0; i < 2; ++i)
            if (done[i]) (void)hipEventDestroy(done[i]);
        if (ready) (void)hipEventDestroy(ready);
        return rc;
    }
    // the arena for what the weight gradients of the next block read
    int enter(Space** arena) {
        if (closed) {
            closed = false;
            if (two_streams()) turn ^= 1;
            arenas[turn].at = 0;
            TRY(wait_for(turn));
        }
        *arena = &arenas[turn];
        return PTV3_OK;
    }
    int leave() {   // a block's chain has written what they read
        const bool full = arenas[turn].at >= GROUP_BYTES || n_linears + 8 > GROUP_LINEARS || n_convs == GROUP_CONVS;
        return full ? flush() : PTV3_OK;
    }
    // the weight gradients put down since the last flush
    int flush() {
        closed = true;
        if (!n_linears && !n_convs) return PTV3_OK;
        const bool beside = side && !dry;
        if (beside) {
            TRY((int)hipEventRecord(ready, hs));
            TRY((int)hipStreamWaitEvent(side, ready, 0));
        }
        unmarked = beside;
        int rc = launch_wgrads(arenas[turn], beside ? side : hs);
        n_linears = n_convs = 0;
        if (beside) {
            const int rec = (int)hipEventRecord(done[turn], side);
            unmarked = rec != PTV3_OK;
            busy[turn] = !unmarked;
            rc = rc ? rc : rec;
        }
        return rc;
    }
    int launch_wgrads(Space& arena, hipStream_t on) {
        SlabJob jobs[GROUP_LINEARS + GROUP_CONVS];
        int n_jobs = 0;
        for (int first = 0, last; first < n_linears; first = last) {   // up to eight in a row with as many rows share a launch
            for (last = first + 1; last < n_linears && last < first + 8 && linears[last].n == linears[first].n;) ++last;
            const size_t bytes = ptv3_linear_wgrads_bytes(linears + first, last - first);
            void* ws = bytes ? arena.take(bytes) : nullptr;
            DO(ptv3_linear_wgrads_slabs(linears + first, last - first, dt, ws, bytes, jobs + n_jobs, on));
            n_jobs += last - first;
        }
        for (int i = 0; i < n_convs; ++i) {
            const ConvGrad& g = convs[i];
            const size_t bytes = ptv3_subm_conv_wgrad_workspace_bytes(dt, g.n, g.cin, g.cout, g.taps);
            void* ws = bytes ? arena.take(bytes) : nullptr;
            DO(ptv3_subm_conv_wgrad_slabs(g.x, g.dy, dt, g.n, g.cin, g.cout, g.pair_out, g.tap_ptr, g.pair_in, g.taps, g.dweight,
                                           g.dbias, ws, bytes, &jobs[n_jobs], on));
            ++n_jobs;
        }
        DO(ptv3_slab_sums(jobs, n_jobs, on));
        return PTV3_OK;
    }
    // x and dy stay until the arena's next turn
    int wgrad(const ptv3_train_linear& l, int in, int out, const void* x, const void* dy, int64_t n) {
        if (n_linears == GROUP_LINEARS) return PTV3_EINVAL;
        linears[n_linears++] = LinearGrad{x, dy, n, in, out, grads + l.gw, grads + l.gb};
        return PTV3_OK;
    }
    int conv_wgrad(const ptv3_train_block& b, const ptv3_level& v, const void* x, const void* dy) {
        if (n_convs == GROUP_CONVS) return PTV3_EINVAL;
        convs[n_convs++] = ConvGrad{x, dy, v.pair_out, v.tap_ptr, v.pair_in, v.n, b.channels, b.channels, 27, grads + b.g_conv_w,
                                    grads + b.g_conv_b};
        return PTV3_OK;
    }
    int bn_bwd(const ptv3_train_bn& b, const BnActs& a, int64_t n, int c, const void* dy, void* dx) {
        if (dry) return PTV3_OK;
        return ptv3_batch_norm_bwd_onto(a.x, dt, dy, dt, a.stats, b.g, b.b, PTV3_F32, n, c, 1, 1, dx, dt, grads + b.gg, hs);
    }

    // d32, d16: gradient of the block's output in float and, times mask2, in half (in the group's arena). Leaves the
    // gradients of its residual input in dskip (skip_out_dt) and of its convolution's rows in dxs (half); the weights' in
    // `grads`.
    int block_bwd(const ptv3_train_block& b, const BlockActs& a, const ptv3_level& v, int patch, const void* mask1, const void* d32,
                  const void* d16, void* dskip, int skip_out_dt, void* dxs, Space& scratch, Space& arena) {
        const int64_t n = v.n;
        const int c = b.channels;
        const size_t mark = scratch.at, half = (size_t)n * c * 2;
        void *h4 = arena.take(4 * half), *h3 = arena.take(3 * half), *hb = arena.take(half), *dcpe = arena.take(half);
        void* dconv = arena.take(half);
        void *h1 = scratch.take(half), *dsum2 = scratch.take(2 * half);
        // MLP
        DO(ptv3_linear_gelu_bwd(d16, b.fc2.wt, a.pre, dt, n, c, 4 * c, h4, stream));
        TRY(wgrad(b.fc2, 4 * c, c, a.act, d16, n));
        TRY(wgrad(b.fc1, c, 4 * c, a.y2, h4, n));
        TRY(linear(h4, b.fc1.wt, nullptr, 4 * c, c, n, h1));
        // second LayerNorm and residual
        DO(ptv3_add_layer_norm_bwd(a.sum2, PTV3_F32, h1, dt, d32, PTV3_F32, mask1, dt, b.ln2.g, PTV3_F32, n, c, b.ln2.eps, dsum2,
                                    PTV3_F32, hb, dt, grads + b.ln2.gg, grads + b.ln2.gb, nullptr, 0, nullptr, 0.f, nullptr, nullptr,
                                    stream));
        // projection and attention
        TRY(wgrad(b.proj, c, c, a.attn, hb, n));
        TRY(linear(hb, b.proj.wt, nullptr, c, c, n, h1));
        {
            const size_t m2 = scratch.at, bytes = ptv3_patch_attn_bwd_workspace_bytes(dt, v.n_pad, c, b.heads);
            void* ws = scratch.take(bytes);
            DO(ptv3_patch_attn_bwd(a.qkv, a.attn, h1, dt, n, c, b.heads, v.slot_src[b.row], v.slot_dst[b.row], v.cu, v.n_seq, patch,
                                    v.n_pad, b.scale, a.lse, 0.f, 0, h3, ws, bytes, stream));
            scratch.at = m2;
        }
        TRY(wgrad(b.qkv, c, 3 * c, a.y1, h3, n));
        TRY(linear(h3, b.qkv.wt, nullptr, 3 * c, c, n, h1));
        // first LayerNorm, residual and the xCPE's norm
        DO(ptv3_add_layer_norm_bwd(a.sum1, PTV3_F32, h1, dt, dsum2, PTV3_F32, nullptr, 0, b.ln1.g, PTV3_F32, n, c, b.ln1.eps, dskip,
                                    skip_out_dt, dcpe, dt, grads + b.ln1.gg, grads + b.ln1.gb, a.cpe, dt, b.ln_cpe.g, b.ln_cpe.eps,
                                    grads + b.ln_cpe.gg, grads + b.ln_cpe.gb, stream));
        TRY(wgrad(b.cpe, c, c, a.conv, dcpe, n));
        TRY(linear(dcpe, b.cpe.wt, nullptr, c, c, n, dconv));
        TRY(conv_wgrad(b, v, a.xs, dconv));
        TRY(leave());
        TRY(conv(b, v, true, dconv, scratch, dxs));
        scratch.at = mark;
        return PTV3_OK;
    }

    // blocks of a stage, last to first. (a, b): parts of the last block's output gradient; the first block's input
    // gradients end up in dskip (half) and dxs (half).
    int stage_bwd(const ptv3_train_block* bs, const BlockActs* as, int count, int level, const void* const* masks, const void* a, int a_dt,
                  const void* b, int b_dt, void* dskip, void* dxs, Space& scratch) {
        const ptv3_level& v = lv[level];
        const int c = bs[0].channels;
        const size_t mark = scratch.at;
        void *d32 = scratch.take((size_t)v.n * c * 4), *ds = scratch.take((size_t)v.n * c * 4);
        for (int i = count - 1; i >= 0; --i) {
            Space* arena;
            TRY(enter(&arena));
            void* d16 = arena->take((size_t)v.n * c * 2);
            DO(ptv3_two_sums(a, a_dt, b, b_dt, nullptr, masks[2 * i + 1], dt, v.n, c, d32, d16, dt, hs));
            TRY(block_bwd(bs[i], as[i], v, net.patch[level], masks[2 * i], d32, d16, i ? ds : dskip, i ? PTV3_F32 : dt, dxs, scratch,
                          *arena));
            a = ds;
            a_dt = PTV3_F32;
            b = dxs;
            b_dt = dt;
        }
        scratch.at = mark;
        return PTV3_OK;
    }

    int backward(const void* dout, int dout_dt, const void* const* masks, Space& scratch) {
        const int S = net.n_stages;
        DO(ptv3_zero_ranges(grads, net.zero, net.n_zero, net.zero_blocks, stream));
        BnPlaces places = {};
        places.add(net.stem.bn, net.stage[0].channels);
        for (int s = 0; s < S; ++s) {
            const ptv3_train_stage& g = net.stage[s];
            if (s > 0) places.add(g.pool_bn, g.channels);
            if (s < S - 1) {
                places.add(g.up_bn, g.dec_channels);
                places.add(g.up_skip_bn, g.dec_channels);
            }
        }
        DO(zero_places(grads, places, hs));
        // gradients of the encoder stages' rows from the skip projections and the poolings (half)
        void *from_skip[PTV3_MAX_LEVELS] = {}, *from_pool[PTV3_MAX_LEVELS] = {}, *from_up[PTV3_MAX_LEVELS] = {};
        for (int s = 0; s < S; ++s) {
            const size_t r = (size_t)lv[s].n * net.stage[s].channels * 2;
            from_skip[s] = scratch.take(r);
            from_pool[s] = scratch.take(r);
            // of the decoder stage's rows, from the unpooling above it
            if (s > 0 && s < S - 1) from_up[s] = scratch.take((size_t)lv[s].n * net.stage[s].dec_channels * 2);
        }
        const void* const* enc_masks[PTV3_MAX_LEVELS];
        const void* const* dec_masks[PTV3_MAX_LEVELS];
        for (int s = 0; s < S; ++s) { enc_masks[s] = masks; masks += 2 * net.stage[s].n_enc; }
        for (int s = S - 2; s >= 0; --s) { dec_masks[s] = masks; masks += 2 * net.stage[s].n_dec; }
        // ---- decoder, last stage first
        const void* d = dout;
        int d_dt = dout_dt;
        for (int s = 0; s < S - 1; ++s) {
            const ptv3_train_stage& g = net.stage[s];
            const ptv3_level &v = lv[s], &below = lv[s + 1];
            const int c = g.dec_channels;
            const size_t mark = scratch.at, half = (size_t)v.n * c * 2;
            void *dskip = scratch.take(half), *dxs = scratch.take(half), *dpar = scratch.take(half);
            void* dchild = scratch.take((size_t)below.n * c * 2);
            TRY(stage_bwd(g.dec, st[s].dec, g.n_dec, s, dec_masks[s], nullptr, dt, d, d_dt, dskip, dxs, scratch));
            Space* arena;
            TRY(enter(&arena));
            void *dlin = arena->take(half), *dlin2 = arena->take((size_t)below.n * c * 2);
            // unpooling: the sum's gradient goes to the skip projection (whose rows the first convolution reads too) and,
            // summed over a cell's members, to the child
            DO(ptv3_two_sums(dskip, dt, dxs, dt, nullptr, nullptr, dt, v.n, c, nullptr, dpar, dt, hs));
            DO(ptv3_segment_reduce(dskip, dt, v.n, c, v.order, below.idx_ptr, below.n, 2, dchild, stream));
            TRY(bn_bwd(g.up_skip_bn, st[s].skip_bn, v.n, c, dpar, dlin));
            TRY(wgrad(g.up_skip, g.up_skip.in, c, st[s].enc[g.n_enc - 1].out16, dlin, v.n));
            TRY(linear(dlin, g.up_skip.wt, nullptr, c, g.up_skip.in, v.n, from_skip[s]));
            TRY(bn_bwd(g.up_bn, st[s].up_bn, below.n, c, dchild, dlin2));
            const void* child_rows = s + 1 < S - 1 ? st[s + 1].dec[net.stage[s + 1].n_dec - 1].out16
                                                   : st[S - 1].enc[net.stage[S - 1].n_enc - 1].out16;
            TRY(wgrad(g.up, g.up.in, c, child_rows, dlin2, below.n));
            void* dnext = s + 1 < S - 1 ? from_up[s + 1] : from_skip[S - 1];
            TRY(leave());
            TRY(linear(dlin2, g.up.wt, nullptr, c, g.up.in, below.n, dnext));
            scratch.at = mark;
            d = dnext;
            d_dt = dt;
        }
        // ---- encoder, bottom first
        for (int s = S - 1; s >= 0; --s) {
            const ptv3_train_stage& g = net.stage[s];
            const ptv3_level& v = lv[s];
            const int c = g.channels;
            const size_t mark = scratch.at, half = (size_t)v.n * c * 2;
            void *dskip = scratch.take(half), *dxs = scratch.take(half), *dx = scratch.take(half);
            TRY(stage_bwd(g.enc, st[s].enc, g.n_enc, s, enc_masks[s], s < S - 1 ? from_pool[s] : nullptr, dt, from_skip[s], dt, dskip,
                          dxs, scratch));
            DO(ptv3_two_sums(dskip, dt, dxs, dt, nullptr, nullptr, dt, v.n, c, nullptr, dx, dt, hs));
            Space* arena;
            TRY(enter(&arena));
            void* dseg = arena->take(half);
            if (s > 0) {
                const ptv3_level& up = lv[s - 1];
                void* dproj = arena->take((size_t)up.n * c * 2);
                TRY(bn_bwd(g.pool_bn, st[s].pool_bn, v.n, c, dx, dseg));
                DO(ptv3_segment_reduce_bwd(st[s].pool_in, st[s].pooled, dseg, dt, up.n, c, up.order, v.idx_ptr, v.n, g.pool_reduce,
                                            dproj, stream));
                TRY(wgrad(g.pool, g.pool.in, c, st[s - 1].enc[net.stage[s - 1].n_enc - 1].out16, dproj, up.n));
                TRY(leave());
                TRY(linear(dproj, g.pool.wt, nullptr, c, g.pool.in, up.n, from_pool[s - 1]));
            } else {
                TRY(bn_bwd(net.stem.bn, stem_bn, v.n, c, dx, dseg));
                const int cp = net.stem.cin_padded;
                float* dw = (float*)arena->take((size_t)c * 125 * cp * 4);
                convs[n_convs++] = ConvGrad{stem_in, dseg, v.pair_out5, v.tap_ptr5, v.pair_in5, v.n, cp, c, 125, dw, nullptr};
                TRY(flush());
                TRY(join());
                DO(ptv3_cut_rows(dw, (int64_t)c * 125, cp, net.stem.cin, grads + net.stem.gw, stream));
            }
            scratch.at = mark;
        }
        return PTV3_OK;
    }
};

__global__ __launch_bounds__(256) void zero_ranges_kernel(float* __restrict__ base, const ptv3_zero_range* __restrict__ ranges, int count) {
    int lo = 0, hi = count;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ranges[mid].first_block <= (int64_t)blockIdx.x) lo = mid; else hi = mid;
    }
    const int64_t i = ((int64_t)blockIdx.x - ranges[lo].first_block) * 256 + threadIdx.x;
    if (i < ranges[lo].count) base[ranges[lo].at + i] = 0.f;
}

__global__ __launch_bounds__(256) void cut_rows_kernel(const float* __restrict__ x, int64_t rows, int from, int to, float* __restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= rows * to) return;
    const int64_t r = e / to;
    out[e] = x[r * from + (e - r * to)];
}

bool net_ok(const ptv3_train_net* net, const ptv3_level* lv) {
    if (!net || !lv || net->n_stages < 2 || net->n_stages > PTV3_MAX_LEVELS) return false;
    if ((net->dtype != PTV3_F16 && net->dtype != PTV3_BF16) || !(net->max_pair_density >= 0.f)) return false;
    int blocks = 0;
    for (int s = 0; s < net->n_stages; ++s) {
        const ptv3_train_stage& g = net->stage[s];
        if (lv[s].n < 2 || g.n_enc < 1 || !g.enc || (s < net->n_stages - 1 && (g.n_dec < 1 || !g.dec))) return false;
        blocks += g.n_enc + g.n_dec;
        for (int i = 0; i < g.n_enc + g.n_dec; ++i) {
            const ptv3_train_block& b = i < g.n_enc ? g.enc[i] : g.dec[i - g.n_enc];
            if (b.row < 0 || b.row >= PTV3_MAX_ORDERS || !lv[s].slot_src[b.row]) return false;
            if (b.channels != (i < g.n_enc ? g.channels : g.dec_channels)) return false;
        }
    }
    return blocks <= MAX_BLOCKS;
}

// scratch of a pass, from a run of its own code that queues nothing; `parts` (backward): what the chain and each arena take
size_t scratch_bytes(const ptv3_train_net& net, const ptv3_level* lv, bool back, size_t* parts = nullptr) {
    Run* r = new Run(net, lv, nullptr);
    Space acts(nullptr), m(nullptr);
    r->place(acts);
    r->link();
    r->dry = true;
    static const void* none[2 * MAX_BLOCKS] = {};
    const int rc = back ? r->backward(nullptr, PTV3_F32, none, m) : r->forward(nullptr, PTV3_F32, none, m);
    const size_t sizes[3] = {m.top, r->arenas[0].top, r->arenas[1].top};
    delete r;
    if (parts) memcpy(parts, sizes, sizeof(sizes));
    return rc == PTV3_OK ? sizes[0] + sizes[1] + sizes[2] + 256 : 0;
}

}  // namespace

extern "C" int ptv3_zero_ranges(float* base, const ptv3_zero_range* ranges, int count, int64_t blocks, void* stream_) {
    if (count < 0 || blocks < 0 || blocks >= (1ll << 31)) return PTV3_EINVAL;
    if (!count || !blocks) return PTV3_OK;
    if (!base || !ranges) return PTV3_EINVAL;
    hipLaunchKernelGGL(zero_ranges_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream_, base, ranges, count);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_cut_rows(const float* x, int64_t rows, int from, int to, float* out, void* stream_) {
    if (rows < 0 || to < 1 || from < to) return PTV3_EINVAL;
    if (rows == 0) return PTV3_OK;
    if (!x || !out) return PTV3_EINVAL;
    hipLaunchKernelGGL(cut_rows_kernel, dim3((unsigned)ptv3_ceil_div(rows * to, 256)), dim3(256), 0, (hipStream_t)stream_, x, rows, from,
                       to, out);
    PTV3_RETURN_LAUNCH();
}

extern "C" int ptv3_train_bytes(const ptv3_train_net* net, const ptv3_level* levels, size_t* acts, size_t* fwd_scratch,
                                size_t* bwd_scratch) {
    if (!net_ok(net, levels) || !acts || !fwd_scratch || !bwd_scratch) return PTV3_EINVAL;
    Run* r = new Run(*net, levels, nullptr);
    Space m(nullptr);
    r->place(m);
    delete r;
    *acts = m.top;
    *fwd_scratch = scratch_bytes(*net, levels, false);
    *bwd_scratch = scratch_bytes(*net, levels, true);
    return PTV3_OK;
}

extern "C" int ptv3_train_fwd(const ptv3_train_net* net, const ptv3_level* levels, const void* feat, int feat_dtype,
                              const void* const* masks, void* acts, void* scratch, size_t scratch_size, float* out, void* stream) {
    if (!net_ok(net, levels) || !feat || !masks || !acts || !scratch || !out) return PTV3_EINVAL;
    if (scratch_size < scratch_bytes(*net, levels, false)) return PTV3_EWORKSPACE;
    Run* r = new Run(*net, levels, stream);
    Space a(acts), s(scratch);
    r->place(a);
    r->link();
    r->final_out = out;
    const int rc = r->forward(feat, feat_dtype, masks, s);
    delete r;
    return rc;
}

extern "C" int ptv3_train_bwd(const ptv3_train_net* net, const ptv3_level* levels, const void* dout, int dout_dtype,
                              const void* const* masks, const void* acts, void* scratch, size_t scratch_size, float* grads,
                              void* stream) {
    if (!net_ok(net, levels) || !dout || !masks || !acts || !scratch || !grads) return PTV3_EINVAL;
    size_t parts[3];
    if (scratch_size < scratch_bytes(*net, levels, true, parts)) return PTV3_EWORKSPACE;
    Run* r = new Run(*net, levels, stream);
    Space a(const_cast<void*>(acts)), s(scratch);
    r->place(a);
    r->link();
    r->grads = grads;
    r->arenas[0] = Space((char*)scratch + parts[0]);
    r->arenas[1] = Space((char*)scratch + parts[0] + parts[1]);
    int rc = r->open_side();
    if (rc == PTV3_OK) rc = r->backward(dout, dout_dtype, masks, s);
    const int joined = r->close_side();
    delete r;
    return rc ? rc : joined;
}
