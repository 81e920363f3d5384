// xt_launch.h - the layer GEMM launchers as the engines call them: the entry points of the same kernels, with the number
// of lanes that run on the GPU at once as well (1 or 2; the entry points are lanes = 1). A tile that wins while a call
// has the chip to itself can lose beside the other lane's kernels, so the tile rules take it. Checks, results and errors
// are the entry points'. wx: the 2:4 indices (w their values), or NULL for dense weights.
#pragma once

#define XT_HIDDEN __attribute__((visibility("hidden")))

XT_HIDDEN int xt_qkv(const void *h8, const float *hs, int lds, const void *w, const void *wx, const float *ws,
                     const float *cs, void *q, void *k, void *vt, int rows, int lanes, void *stream);
XT_HIDDEN int xt_oproj(const void *a8, const float *as, int lds, const void *w, const void *wx, const float *ws, void *x,
                       int rows, int lanes, void *stream);
XT_HIDDEN int xt_fc2(const void *m8, const float *ms, int lds, const void *w, const void *wx, const float *ws,
                     const float *stat, const float *cn, const float *dn, void *x, int rows, int lanes, void *stream);
XT_HIDDEN int xt_px_proj(const void *a8, const float *as, int lds, const void *w, const float *ws, const float *bias,
                         void *x, int rows, int lanes, void *stream);
XT_HIDDEN int xt_px_fc1(const void *h8, const float *hs, int lds, const void *w, const float *ws, const float *bias,
                        const float *rs, void *m8, float *ms, int rows, int lanes, void *stream);
XT_HIDDEN int xt_px_fc2(const void *m8, const float *ms, int lds, const void *w, const float *ws, const float *bias,
                        void *x, int rows, int lanes, void *stream);
