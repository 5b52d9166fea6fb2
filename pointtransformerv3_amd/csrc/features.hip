// The feature side of a forward as one call: stem, encoder, decoder over an index made by ptv3_index_* (levels.hip), every
// launch queued from native code. Layer by layer from Python the same launches cost the host about 5 ms, more than the
// kernels themselves up to 100k points; from here about 2 us each. The kernels and the form each layer takes are those the
// modules would pick (modules.py, ops.py), so the results are the same bits.
#include <string.h>

#include "bnact.h"
#include "lintile.h"

namespace {

// bump allocator over the caller's workspace; a null base only measures
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

#define TRY(call)                        \
    do {                                 \
        const int rc__ = (call);         \
        if (rc__ != PTV3_OK) return rc__; \
    } while (0)

struct Run {
    const ptv3_net* net;
    const ptv3_level* lv;
    void* stream;
    Space mem;
    bool dry;
    int dt;          // dtype of the rows
    size_t es;
    int32_t *map3[PTV3_MAX_LEVELS] = {}, *map5 = nullptr;   // neighbour maps, where a convolution takes the dense form
    Run(const ptv3_net* n, const ptv3_level* l, void* s, void* ws)
        : net(n), lv(l), stream(s), mem(ws), dry(ws == nullptr), dt(n->dtype), es(n->dtype == PTV3_F32 ? 4 : 2) {}
    void* rows(int64_t n, int64_t c) { return mem.take((size_t)n * c * es); }
};

bool half_rows(int k) { return k == 32 || k == 64 || k == 128 || k == 256 || k == 512; }

// nn.Linear, the kernel ops.linear picks
int linear(Run& r, const void* x, const ptv3_linear_w& w, int64_t n, void* out) {
    if (r.dry) return PTV3_OK;
    if (r.dt == PTV3_F32)
        return ptv3_linear_f32_fwd(x, PTV3_F32, (const float*)w.w, (const float*)w.b, nullptr, n, w.in, w.out, 0, out, PTV3_F32,
                                   r.stream);
    if (half_rows(w.in) && w.out % 32 == 0 && (w.in <= 256 || w.out <= 2 * w.in)) {
        if (w.in == 256 && w.out % 256 == 0 && n >= 4096)
            return ptv3_linear_wide_fwd(x, w.w, w.b, r.dt, n, w.in, w.out, 0, out, r.stream);
        return ptv3_linear_fwd(x, w.w, w.b, r.dt, n, w.in, w.out, 0, out, r.stream);
    }
    if (w.in % 128 == 0 && w.out % 128 == 0)
        return ptv3_linear_gemm_fwd(x, w.w, w.b, nullptr, r.dt, n, w.in, w.out, out, r.stream);
    return ptv3_linear_any_fwd(x, w.w, w.b, nullptr, r.dt, n, w.in, w.out, 0, out, r.stream);
}

BnGelu bn_gelu(const ptv3_bn_w& bn) { return BnGelu{bn.mean, bn.var, bn.g, bn.b, bn.eps, bn.stats_f32}; }

// Linear -> BatchNorm1d (running statistics) -> GELU
int linear_bn_gelu(Run& r, const void* x, const ptv3_linear_w& w, const ptv3_bn_w& bn, int64_t n, void* out) {
    if (r.dt != PTV3_F32)
        return r.dry ? PTV3_OK
                     : ptv3_linear_bn_act_fwd(x, w.w, w.b, bn.mean, bn.var, bn.stats_f32, bn.g, bn.b, bn.eps, r.dt, n, w.in,
                                              w.out, 1, out, r.stream);
    const size_t mark = r.mem.at;
    void* y = r.rows(n, w.out);
    TRY(linear(r, x, w, n, y));
    r.mem.at = mark;
    return r.dry ? PTV3_OK
                 : ptv3_bn_act(y, bn.mean, bn.var, bn.stats_f32, bn.g, bn.b, r.dt, n, w.out, bn.eps, 1, out, r.stream);
}

// A convolution that no tile form takes: product rows, or the neighbour map where ptv3_conv_pair_form says so (then made
// in front of the forward, make_map).
int pair_form(const Run& r, int s, int taps, int cin, int cout) {
    const ptv3_level& v = r.lv[s];
    return ptv3_conv_pair_form(r.dt, v.n, taps == 27 ? v.n_pairs : v.n_pairs5, taps, cin, cout, r.net->max_pair_density);
}
int conv_rows(Run& r, int s, int taps, const void* x, int cin, const void* w, const void* bias, int cout, void* out,
              const Ahead& ahead = Ahead{}) {
    const ptv3_level& v = r.lv[s];
    const bool inner = taps == 27;
    const int64_t n_pairs = inner ? v.n_pairs : v.n_pairs5;
    const int32_t *tap_ptr = inner ? v.tap_ptr : v.tap_ptr5, *row_ptr = inner ? v.row_ptr : v.row_ptr5;
    const int32_t *pair_in = inner ? v.pair_in : v.pair_in5, *pair_slot = inner ? v.pair_slot : v.pair_slot5;
    const int form = pair_form(r, s, taps, cin, cout);
    if (form == PTV3_CONV_DENSE)
        return r.dry ? PTV3_OK
                     : ptv3_subm_conv_fwd(x, r.dt, v.n, cin, inner ? r.map3[s] : r.map5, taps, 1, w, bias, cout, out, r.stream);
    const bool wide = form == PTV3_CONV_PAIRS_WIDE;
    const size_t mark = r.mem.at;
    void* y = r.mem.take((size_t)n_pairs * cout * (wide ? 4 : r.es));
    r.mem.at = mark;
    if (r.dry) return PTV3_OK;
    if (wide)
        return ptv3_subm_conv_pairs_wide_fwd(x, r.dt, v.n, cin, taps, n_pairs, tap_ptr, row_ptr, pair_in, pair_slot, w, bias, cout,
                                             (float*)y, out, r.stream);
    return ptv3_conv_pairs_ahead(x, r.dt, v.n, cin, taps, n_pairs, tap_ptr, row_ptr, pair_in, pair_slot, w, bias, cout, y, out, ahead,
                                 r.stream);
}
// the tap-major neighbour map of level s, for the whole forward
int make_map(Run& r, int s, int ks, int32_t** map) {
    const ptv3_level& v = r.lv[s];
    *map = (int32_t*)r.mem.take((size_t)v.n * ks * ks * ks * sizeof(int32_t));
    const size_t mark = r.mem.at, bytes = ptv3_kmap_workspace_bytes(v.n);
    void* ws = r.mem.take(bytes);
    r.mem.at = mark;
    return r.dry ? PTV3_OK : ptv3_kmap_build(v.indices, v.n, ks, 1, *map, ws, bytes, r.stream);
}
int stem_inputs(const ptv3_net& net) { return net.dtype == PTV3_F32 ? net.stem_in : (net.stem_in + 15) / 16 * 16; }
int make_maps(Run& r) {
    const ptv3_net& net = *r.net;
    if (pair_form(r, 0, 125, stem_inputs(net), net.stage[0].channels) == PTV3_CONV_DENSE) TRY(make_map(r, 0, 5, &r.map5));
    for (int s = 0; s < net.n_stages; ++s) {
        const ptv3_stage_w& st = net.stage[s];
        bool need = false;
        for (int side = 0; side < 2; ++side) {
            const int c = side ? st.dec_channels : st.channels;
            if (!(side ? net.decoder && st.n_dec : st.n_enc)) continue;
            if (r.dt != PTV3_F32 && ptv3_conv_form(r.lv[s].n, r.lv[s].n_pairs, c) != 0) continue;
            need |= pair_form(r, s, 27, c, c) == PTV3_CONV_DENSE;
        }
        if (need) TRY(make_map(r, s, 3, &r.map3[s]));
    }
    return PTV3_OK;
}

// at 256 channels a caller may leave the packed copy out: the separate layers
bool head_wide(const ptv3_block_w& b, int64_t n) {
    return (b.channels == 128 || b.head_packed) && ptv3_block_head_wide_pays(n, b.channels);
}

int conv3(Run& r, const ptv3_block_w& b, int s, const void* x, void* out) {
    const int c = b.channels;
    const ptv3_level& v = r.lv[s];
    const int form = r.dt == PTV3_F32 ? 0 : ptv3_conv_form(v.n, v.n_pairs, c);
    if (form == 0) {
        Ahead ahead = {};   // what the first half streams through every work-group: 22.4 -> 19.9 us for 11.6k rows (see attention)
        if (r.dt != PTV3_F32 && c == 256 && head_wide(b, v.n)) ahead = ptv3_ahead(b.head_packed, 8ll * c * c, nullptr, 0);
        return conv_rows(r, s, 27, x, c, b.conv_w, b.conv_b, c, out, ahead);
    }
    if (r.dry) return PTV3_OK;
    if (form == 1)
        return ptv3_subm_conv_sparse_fwd(x, r.dt, v.n, c, 27, b.conv_packed, b.conv_b, v.tile_tap, v.tile_pair, out, r.stream);
    return ptv3_subm_conv_tiles_fwd_sized(x, r.dt, v.n, c, 27, v.tile_voxels, b.conv_packed, b.conv_b, v.tile_tap, v.tile_pair,
                                          v.vox_taps, out, r.stream);
}

int attention(Run& r, const ptv3_block_w& b, const ptv3_level& v, int patch, const void* qkv, int dt, void* out) {
    if (r.dry) return PTV3_OK;
    // 256 channels: the second half streams 1.2 MB through every work-group, 38.6 us of a room's 11.6k rows where they come from
    // HBM, 32.0 from the L2 (the attention 34.7 and 35.4). At 128 channels it is 0.3 MB and no faster; the layers of few rows
    // share their weights out over the work-groups.
    Ahead ahead = {};
    const int64_t square = (int64_t)b.channels * b.channels * 2;
    if (r.dt != PTV3_F32 && b.channels == 256 && !ptv3_block_tail_few_pays(v.n, 256))
        ahead = ptv3_ahead(b.proj_packed, square, b.mlp_packed, 8 * square);
    return ptv3_patch_attn_fwd_slots(qkv, dt, v.n, b.channels, b.heads, v.slot_src[b.row], v.slot_dst[b.row], v.cu, v.n_seq, patch,
                                     v.n_pad, b.scale, out, ahead, r.stream);
}

// A block (model.py:586-606): x its rows, xs what its convolution reads, out the new rows.
int block_half(Run& r, const ptv3_block_w& b, int s, const void* xs, const void* x, void* out) {
    const ptv3_level& v = r.lv[s];
    const int patch = r.net->patch[s];
    const int64_t n = v.n;
    const int c = b.channels;
    const size_t mark = r.mem.at;
    void *conv = r.rows(n, c), *feat = r.rows(n, c), *qkv = r.rows(n, 3 * c), *attn = r.rows(n, c), *normed = r.rows(n, c);
    const bool few = ptv3_block_tail_few_pays(n, c);
    const size_t few_bytes = few ? ptv3_block_tail_few_bytes(n, c) : 0;
    void* few_ws = few ? r.mem.take(few_bytes) : nullptr;
    TRY(conv3(r, b, s, xs, conv));
    if (!r.dry) {
        if (c <= 64) {
            TRY(ptv3_block_head_fused(conv, x, b.cpe.w, b.cpe.b, b.ln_cpe.g, b.ln_cpe.b, b.ln_cpe.eps, b.ln1.g, b.ln1.b, b.ln1.eps,
                                      b.qkv.w, b.qkv.b, r.dt, n, c, feat, qkv, r.stream));
        } else if (head_wide(b, n)) {
            TRY(ptv3_block_head_wide(conv, x, b.head_packed, b.cpe.b, b.ln_cpe.g, b.ln_cpe.b, b.ln_cpe.eps, b.ln1.g, b.ln1.b,
                                     b.ln1.eps, b.qkv.b, r.dt, n, c, feat, qkv, r.stream));
        } else {
            if (c == 256 && !few) {
                TRY(ptv3_linear_ln_fwd(conv, b.cpe.w, b.cpe.b, x, b.ln_cpe.g, b.ln_cpe.b, b.ln1.g, b.ln1.b, nullptr, r.dt, n, c, 3,
                                       b.ln_cpe.eps, feat, normed, r.stream));
            } else {
                TRY(linear(r, conv, b.cpe, n, attn));
                if (lin_front_pays(n, c, 3 * c)) {
                    LinArgs a = {};
                    LinFront f = {};
                    a.x = attn, a.w = b.qkv.w, a.bias = b.qkv.b, a.n = n, a.k = c, a.nout = 3 * c, a.out = qkv;
                    f.mode = LinFront::NORM_SUM_NORM, f.g = b.ln_cpe.g, f.b = b.ln_cpe.b, f.res = x, f.g2 = b.ln1.g, f.b2 = b.ln1.b;
                    f.eps = b.ln_cpe.eps, f.sum = feat;
                    TRY(lin_front(a, f, r.dt, (hipStream_t)r.stream));
                    normed = nullptr;
                } else {
                    TRY(ptv3_layer_norm(attn, x, b.ln_cpe.g, b.ln_cpe.b, b.ln1.g, b.ln1.b, nullptr, r.dt, n, c, b.ln_cpe.eps, 3,
                                        feat, normed, r.stream));
                }
            }
            if (normed) TRY(linear(r, normed, b.qkv, n, qkv));
        }
        TRY(attention(r, b, v, patch, qkv, r.dt, attn));
        if (few) {
            TRY(ptv3_block_tail_few(attn, feat, b.proj.w, b.proj.b, b.ln2.g, b.ln2.b, b.ln2.eps, b.fc1.w, b.fc1.b, b.fc2.w, b.fc2.b,
                                    r.dt, n, c, few_ws, few_bytes, out, r.stream));
        } else if (c <= 64) {
            TRY(ptv3_block_tail_fused(attn, feat, b.proj.w, b.proj.b, b.ln2.g, b.ln2.b, b.ln2.eps, b.fc1.w, b.fc1.b, b.fc2.w,
                                      b.fc2.b, r.dt, n, c, 4 * c, out, r.stream));
        } else if (c <= 256) {
            TRY(ptv3_block_tail_wide(attn, feat, b.proj_packed, b.proj.b, b.ln2.g, b.ln2.b, b.ln2.eps, b.mlp_packed, b.fc1.b,
                                     b.fc2.b, r.dt, n, c, out, r.stream));
        } else {
            TRY(linear(r, attn, b.proj, n, conv));
            TRY(ptv3_layer_norm(conv, feat, b.ln2.g, b.ln2.b, nullptr, nullptr, nullptr, r.dt, n, c, b.ln2.eps, 2, qkv, normed,
                                r.stream));
            TRY(ptv3_mlp_fused_packed(normed, qkv, b.mlp_packed, b.fc1.b, b.fc2.b, r.dt, n, c, out, r.stream));
        }
    }
    r.mem.at = mark;
    return PTV3_OK;
}

// the same in a float model: the attention works in half (model.py:477, :483), everything else in float
int block_float(Run& r, const ptv3_block_w& b, int s, const void* xs, const void* x, void* out) {
    const ptv3_level& v = r.lv[s];
    const int patch = r.net->patch[s];
    const int64_t n = v.n;
    const int c = b.channels;
    const size_t mark = r.mem.at;
    void *conv = r.rows(n, c), *feat = r.rows(n, c), *normed = r.rows(n, c), *hidden = r.rows(n, 4 * c);
    void* qkv = r.mem.take((size_t)n * 3 * c * 2);
    void* attn = r.mem.take((size_t)n * c * 2);
    TRY(conv3(r, b, s, xs, conv));
    if (!r.dry) {
        TRY(linear(r, conv, b.cpe, n, hidden));
        TRY(ptv3_layer_norm(hidden, x, b.ln_cpe.g, b.ln_cpe.b, b.ln1.g, b.ln1.b, nullptr, r.dt, n, c, b.ln_cpe.eps, 3, feat, normed,
                            r.stream));
        TRY(ptv3_linear_f32_fwd(normed, PTV3_F32, (const float*)b.qkv.w, (const float*)b.qkv.b, nullptr, n, c, 3 * c, 0, qkv,
                                PTV3_F16, r.stream));
        TRY(attention(r, b, v, patch, qkv, PTV3_F16, attn));
        TRY(ptv3_linear_f32_fwd(attn, PTV3_F16, (const float*)b.proj.w, (const float*)b.proj.b, nullptr, n, c, c, 0, conv, PTV3_F32,
                                r.stream));
        // the MLP accumulates onto the stored sum, so fc2's bias is added to that sum here
        TRY(ptv3_layer_norm(conv, feat, b.ln2.g, b.ln2.b, nullptr, nullptr, b.fc2.b, r.dt, n, c, b.ln2.eps, 2, out, normed,
                            r.stream));
        TRY(ptv3_linear_f32_fwd(normed, PTV3_F32, (const float*)b.fc1.w, (const float*)b.fc1.b, nullptr, n, c, 4 * c, 1, hidden,
                                PTV3_F32, r.stream));
        TRY(ptv3_linear_f32_fwd(hidden, PTV3_F32, (const float*)b.fc2.w, nullptr, (const float*)out, n, 4 * c, c, 0, out, PTV3_F32,
                                r.stream));
    }
    r.mem.at = mark;
    return PTV3_OK;
}

int block(Run& r, const ptv3_block_w& b, int s, const void* xs, const void* x, void* out) {
    return r.dt == PTV3_F32 ? block_float(r, b, s, xs, x, out) : block_half(r, b, s, xs, x, out);
}

// blocks of a stage from (xs, x); the last one writes `out` (n, channels)
int blocks(Run& r, const ptv3_block_w* bs, int count, int s, const void* xs, const void* x, void* out) {
    if (count == 0) return PTV3_OK;
    const size_t mark = r.mem.at;
    void* tmp[2] = {nullptr, nullptr};
    for (int i = 0; i < 2 && i < count - 1; ++i) tmp[i] = r.rows(r.lv[s].n, bs[0].channels);
    for (int i = 0; i < count; ++i) {
        void* to = i == count - 1 ? out : tmp[i & 1];
        TRY(block(r, bs[i], s, xs, x, to));
        xs = x = to;
    }
    r.mem.at = mark;
    return PTV3_OK;
}

int forward(Run& r, const void* feat, int feat_dtype, void* const* stage_out, void* out) {
    const ptv3_net& net = *r.net;
    const int S = net.n_stages;
    TRY(make_maps(r));
    // ---- stem: 5x5x5 convolution, BatchNorm, GELU (model.py:753-783)
    void* level_rows[PTV3_MAX_LEVELS] = {};
    for (int s = 0; s < S; ++s) {
        const ptv3_stage_w& st = net.stage[s];
        level_rows[s] = stage_out && stage_out[s] ? stage_out[s] : r.rows(r.lv[s].n, st.channels);
    }
    const int64_t n0 = r.lv[0].n;
    const int c0 = net.stage[0].channels;
    const size_t mark = r.mem.at;
    void* x = net.stage[0].n_enc > 0 ? r.rows(n0, c0) : level_rows[0];
    {
        const size_t m2 = r.mem.at;
        const void* in = feat;
        const int cin = stem_inputs(net);
        if (r.dt != PTV3_F32) {   // the matrix cores take input channels 16 at a time
            void* p = r.rows(n0, cin);
            if (!r.dry) TRY(ptv3_pad_rows(feat, feat_dtype, n0, net.stem_in, cin, p, r.dt, r.stream));
            in = p;
        }
        if (pair_form(r, 0, 125, cin, c0) == PTV3_CONV_PAIRS) {
            const ptv3_level& v = r.lv[0];
            void* y = r.rows(v.n_pairs5, c0);
            if (!r.dry)
                TRY(ptv3_conv_pairs_bn_gelu(in, r.dt, n0, cin, 125, v.n_pairs5, v.tap_ptr5, v.row_ptr5, v.pair_in5, v.pair_slot5,
                                            net.stem_w, c0, bn_gelu(net.stem_bn), y, x, (hipStream_t)r.stream));
        } else {
            void* z = r.rows(n0, c0);
            TRY(conv_rows(r, 0, 125, in, cin, net.stem_w, nullptr, c0, z));
            if (!r.dry)
                TRY(ptv3_bn_act(z, net.stem_bn.mean, net.stem_bn.var, net.stem_bn.stats_f32, net.stem_bn.g, net.stem_bn.b, r.dt, n0,
                                c0, net.stem_bn.eps, 1, x, r.stream));
        }
        r.mem.at = m2;
    }
    // ---- encoder
    for (int s = 0; s < S; ++s) {
        const ptv3_stage_w& st = net.stage[s];
        const ptv3_level& v = r.lv[s];
        if (s > 0) {   // grid pooling (model.py:609-712): projection, segment reduction, BatchNorm, GELU
            const ptv3_level& up = r.lv[s - 1];
            r.mem.at = mark;
            x = st.n_enc > 0 ? r.rows(v.n, st.channels) : level_rows[s];
            const size_t m2 = r.mem.at;
            void *p = r.rows(up.n, st.channels), *q = r.rows(v.n, st.channels);
            TRY(linear(r, level_rows[s - 1], st.pool, up.n, p));
            if (!r.dry) {
                TRY(ptv3_segment_reduce_bn_gelu(p, r.dt, up.n, st.channels, up.order, v.idx_ptr, v.n, st.pool_reduce,
                                                bn_gelu(st.pool_bn), q, x, (hipStream_t)r.stream));
            }
            r.mem.at = m2;
        }
        TRY(blocks(r, st.enc, st.n_enc, s, x, x, level_rows[s]));
    }
    r.mem.at = mark;
    if (!net.decoder) return PTV3_OK;
    // ---- decoder
    const void* child = level_rows[S - 1];
    void* child_buf[2] = {nullptr, nullptr};
    size_t need = 0;
    for (int s = 0; s < S - 1; ++s) {
        const size_t b = (size_t)r.lv[s].n * net.stage[s].dec_channels * r.es;
        need = b > need ? b : need;
    }
    for (int i = 0; i < 2; ++i) child_buf[i] = r.mem.take(need);
    for (int s = S - 2; s >= 0; --s) {
        const ptv3_stage_w& st = net.stage[s];
        const ptv3_level &v = r.lv[s], &below = r.lv[s + 1];
        const int c = st.dec_channels;
        const size_t m2 = r.mem.at;
        void *skip = r.rows(v.n, c), *p = r.rows(below.n, c), *sum = r.rows(v.n, c);
        TRY(linear_bn_gelu(r, child, st.up, st.up_bn, below.n, p));
        TRY(linear_bn_gelu(r, level_rows[s], st.up_skip, st.up_skip_bn, v.n, skip));
        void* to = s == 0 ? out : child_buf[s & 1];
        if (st.n_dec == 0) {
            if (!r.dry) TRY(ptv3_unpool_add(skip, p, r.dt, v.n, c, below.cluster, below.n, to, r.stream));
        } else {
            if (!r.dry) TRY(ptv3_unpool_add(skip, p, r.dt, v.n, c, below.cluster, below.n, sum, r.stream));
            // the first block's convolution reads the skip projection alone (model.py:746)
            TRY(blocks(r, st.dec, st.n_dec, s, skip, sum, to));
        }
        child = to;
        r.mem.at = m2;
    }
    return PTV3_OK;
}

}  // namespace

namespace {

// (n, c) rows in any dtype -> (n, padded) rows in dtype TO, zeros behind the c channels; a thread writes eight channels
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void pad_rows_kernel(const TI* __restrict__ x, int64_t n, int c, int padded,
                                                       PieceDiv pieces, TO* __restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t i = ptv3_row_of(e, pieces);
    if (i >= n) return;
    const int ch = (int)(e - i * pieces.count) * 8;
    typedef TO vec __attribute__((ext_vector_type(8)));
    vec v;
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = ch + k < c ? (TO)(float)x[i * c + ch + k] : (TO)0.f;
    *(vec*)(out + i * padded + ch) = v;
}

bool net_ok(const ptv3_net* net, const ptv3_level* lv) {
    if (!net || !lv || net->n_stages < 1 || net->n_stages > PTV3_MAX_LEVELS || net->stem_in < 1) return false;
    if (net->dtype < PTV3_F32 || net->dtype > PTV3_BF16 || !(net->max_pair_density >= 0.f)) return false;
    for (int s = 0; s < net->n_stages; ++s) {
        const ptv3_stage_w& st = net->stage[s];
        if (lv[s].n < 1 || st.n_enc < 0 || st.n_dec < 0 || (st.n_enc && !st.enc) || (st.n_dec && !st.dec)) return false;
        for (int i = 0; i < st.n_enc + st.n_dec; ++i) {
            const ptv3_block_w& b = i < st.n_enc ? st.enc[i] : st.dec[i - st.n_enc];
            if (!half_rows(b.channels) || b.channels != (i < st.n_enc ? st.channels : st.dec_channels)) return false;
            if (b.row < 0 || b.row >= PTV3_MAX_ORDERS || !lv[s].slot_src[b.row]) return false;
        }
    }
    return true;
}

}  // namespace

// 64 and 128 channels with few pairs: the pair form, its product rows in float. A tile form walks its taps one after the
// other however few tiles there are, while the pair form is two short launches that spread over the part. Float rows make its
// sums what the tile forms keep on chip, rounded once: the error against 64 bits is theirs (2.08e-4 in fp16; half rows
// 2.32e-4 at 1 - 4 us less). Measured in fp16, us, pair form with float rows / tile form / sparse tiles: 64 channels 11.7 /
// 13.8 / 20.7 at 6k pairs, 13.6 / 14.3 / 24.3 at 18k, 19.6 / 14.0 / 23.8 at 67k; 128 channels 12.9 / 19.0 at 8k, 20.2 / 19.5 at
// 36k, 25.2 / 20.4 at 92k, 40.5 / 26.6 at 167k. The lines are those of tiles that took 22 - 24 us (64) and 42 - 44 (128). By
// these figures tiles would pay from 20k and 35k pairs on: not taken yet, tests/test_gpu_small.py holds the route up to the lines.
extern "C" int ptv3_conv_few_pairs(int64_t n_pairs, int channels) {
    return (channels == 64 && n_pairs <= 70000) || (channels == 128 && n_pairs <= 185000);
}

// The form the 3x3x3 convolution of a half-precision level takes: 0 pair lists, 1 sparse tiles, 2 tiles. Above the few pairs
// of ptv3_conv_few_pairs the rule is on pairs per voxel: 32 and 64 channels take the sparse tile form up to 14 (work in
// proportion to the pairs; faster than both other forms from 2.5 to 10), 64 and 128 the tile form from 4 on (sums kept on
// chip, no pair matrix). At 64 channels the tile form is faster up to two of its work-groups a CU: 14.6 us against 18.9 at 20k
// voxels of 5.3 pairs, 20.8 against 22.9 at 55k, but 28.4 against 25.7 at 76k.
extern "C" int ptv3_conv_form(int64_t n, int64_t n_pairs, int channels) {
    if (n < 1 || n >= (1ll << 24)) return 0;
    if (ptv3_conv_few_pairs(n_pairs, channels)) return 0;
    const bool tiles = (channels == 64 || channels == 128) && n_pairs >= 4 * n;
    if (tiles && channels == 64 && n <= 2 * ptv3_cus() * 128) return 2;
    if ((channels == 32 || channels == 64) && n_pairs <= 14 * n) return 1;
    return tiles ? 2 : 0;
}

extern "C" int ptv3_pad_rows(const void* x, int x_dtype, int64_t n, int c, int padded, void* out, int out_dtype, void* stream_) {
    if (n < 0 || c < 1 || padded < c || padded % 8 != 0) return PTV3_EINVAL;
    if (x_dtype < PTV3_F32 || x_dtype > PTV3_BF16 || (out_dtype != PTV3_F16 && out_dtype != PTV3_BF16)) return PTV3_EINVAL;
    if (n == 0) return PTV3_OK;
    if (!x || !out) return PTV3_EINVAL;
    const dim3 grid((unsigned)ptv3_ceil_div(n * (padded / 8), 256)), block(256);
    hipStream_t stream = (hipStream_t)stream_;
#define PTV3_PAD(TI, TO) hipLaunchKernelGGL((pad_rows_kernel<TI, TO>), grid, block, 0, stream, (const TI*)x, n, c, padded, ptv3_piece_div(padded / 8), (TO*)out)
    if (out_dtype == PTV3_F16) {
        if (x_dtype == PTV3_F32) PTV3_PAD(float, _Float16);
        else if (x_dtype == PTV3_F16) PTV3_PAD(_Float16, _Float16);
        else PTV3_PAD(__bf16, _Float16);
    } else {
        if (x_dtype == PTV3_F32) PTV3_PAD(float, __bf16);
        else if (x_dtype == PTV3_F16) PTV3_PAD(_Float16, __bf16);
        else PTV3_PAD(__bf16, __bf16);
    }
#undef PTV3_PAD
    PTV3_RETURN_LAUNCH();
}

extern "C" size_t ptv3_features_bytes(const ptv3_net* net, const ptv3_level* levels, void* const* stage_out) {
    if (!net_ok(net, levels)) return 0;
    Run r(net, levels, nullptr, nullptr);
    return forward(r, nullptr, PTV3_F32, stage_out, nullptr) == PTV3_OK ? r.mem.top : 0;
}

extern "C" int ptv3_features_fwd(const ptv3_net* net, const ptv3_level* levels, const void* feat, int feat_dtype,
                                 void* const* stage_out, void* out, void* workspace, size_t workspace_bytes, void* stream) {
    if (!net_ok(net, levels) || !feat || !workspace || (net->decoder && !out)) return PTV3_EINVAL;
    if (net->dtype == PTV3_F32 && feat_dtype != PTV3_F32) return PTV3_EINVAL;
    if (workspace_bytes < ptv3_features_bytes(net, levels, stage_out)) return PTV3_EWORKSPACE;
    Run r(net, levels, stream, workspace);
    return forward(r, feat, feat_dtype, stage_out, out);
}

extern "C" int ptv3_net_refresh(const ptv3_refresh* f, void* stream) {
    if (!f) return PTV3_EINVAL;
    if (f->n_cast) TRY(ptv3_cast_params(f->cast, f->n_cast, f->cast_blocks, f->dtype, stream));
    if (f->stem_src) TRY(ptv3_pad_rows(f->stem_src, f->dtype, f->stem_rows, f->stem_in, f->stem_padded, f->stem_dst, f->dtype, stream));
    if (f->n_conv) TRY(ptv3_subm_conv_pack_weight_batch(f->conv, f->n_conv, f->conv_blocks, stream));
    if (f->n_mlp) TRY(ptv3_mlp_pack_weights_batch(f->mlp, f->n_mlp, f->mlp_blocks, stream));
    return PTV3_OK;
}
