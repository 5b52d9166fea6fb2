// Linear layers as tiles of the output (lintile.hip), for the layers' own files to hand small and long shapes to.
#pragma once
#include "common.h"

enum { ACT_NONE = 0, ACT_GELU = 1, ACT_GELU_KEEP = 2, ACT_GELU_GRAD = 3, ACT_BN = 4, ACT_BN_GELU = 5 };

struct LinArgs {
    const void *x, *w, *bias;                   // (n, k), (nout, k), (nout,) or NULL
    int64_t n;
    int k, nout, act;
    int row_tiles, col_tiles, order;            // filled in by the launch
    const void* resid;                          // ACT_NONE: added in fp32; may be out
    // ACT_GELU_KEEP: the value in front of the GELU, out; ACT_GELU_GRAD: in. Between the two lies the rest of the step: past the
    // caches both ways (4 rooms of 100k voxels 38.0 -> 37.8 ms)
    void* aux;
    const void *mean, *var, *gamma, *beta;      // ACT_BN, ACT_BN_GELU
    float bn_eps;
    int stats_f32;
    void* out;
};

// whether the tiled form takes the layer and is the faster one
bool lin_tiled_pays(int64_t n, int k, int nout, int act);
bool lin_tiled_takes(int k, int nout);
int lin_tiled(LinArgs& a, int dtype, hipStream_t stream);

// the GELU's training forms of a 256-input layer on the register-weight kernel (linearw.hip)
bool lin_wide_gelu_pays(int64_t n, int k, int nout);
int lin_wide_gelu(const void* x, const void* w, const void* bias, int dtype, int64_t n, int nout, int act, void* out, void* aux,
                  hipStream_t stream);

// The LayerNorm in front of a layer of few rows, formed by the layer itself instead of by a launch of its own.
struct LinFront {
    enum { NORM = 1, NORM_SUM_NORM = 2 };
    int mode;
    const void *g, *b;            // NORM: LayerNorm(x) is what is multiplied. NORM_SUM_NORM: the sum res + LayerNorm(x) goes
    const void *res, *g2, *b2;    // to `sum`, and its LayerNorm (g2, b2) is what is multiplied
    float eps;
    void* sum;
};
bool lin_front_pays(int64_t n, int k, int nout);
int lin_front(LinArgs& a, const LinFront& f, int dtype, hipStream_t stream);
