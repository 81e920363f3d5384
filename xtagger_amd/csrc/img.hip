// img.hip - the patch-operand producer on the GPU: the reference's pi_ingest / pi_pyramid / pi_prep
// (src/core/procimg.h:592-969) for the wd model, from a decoded RGBA(X) image already in device memory to the fp16
// patch operand [(S/14)^2][592] the engine's input buffer holds (procimg.h:1606-1607), with no host round trip.
//
// Same arithmetic as the reference, element for element: the 2x2 pyramid and alpha-over-white in the same integer
// formulas, the axis weights in the same float operations (built without contraction; divisions IEEE), each output
// one fma per tap in tap order (vertical pass, then horizontal pass over RGBX), clamp to [-1, 1], fp16 by
// round-to-nearest-even. The outputs are therefore bit-identical to the reference's.
//
// One crop (eva_img_prep): the host picks the level and the rect on it (pi_level / pi_lsrc, scalar), then
// k_img_resample takes one 14-row band of 2 patches per block: both axes' tap tables (pi_axis) in shared memory, the
// vertical pass over the source columns the band takes (pi_vrow), the horizontal pass from there (pi_hrow), staged in
// shared memory in the operand's own layout and written out as contiguous 16-byte stores.
// A rect whose long side is S skips the resample (pi_idrow): k_img_ident normalises and white-pads the band directly.
#include "xt_abi.h"
#include "xtag_eva.h"

#define IMG_BAND_P 2                        // patches per band block (2 x 592 halves = 2368 contiguous bytes)
#define IMG_PATCH 592                       // halves per patch row of the operand (588 + 4 zero pad)

// ---- pi_row_rgbx with alpha (procimg.h:592-630): c -> (c a + 255 (255 - a)) / 255 rounded, X = 255, in place. Four
// pixels a thread (16 bytes at any pixel's alignment; a row's last pixels one by one); opaque pixels are left as they
// are by the formula ((255 c) / 255 = c, X = 255 already), so four of them are not written back. Bound by HBM. us for
// 3072 x 2048, one pixel a thread and every pixel written -> here, over 24 images in turn (4 images, which the caches
// hold): opaque 17.6 -> 6.7 (13.2 -> 5.2), a sixteenth translucent 17.6 -> 7.4 (13.2 -> 5.8), all of it 17.7 -> 12.1
// (13.2 -> 9.7).
typedef unsigned img_u4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ uint32_t img_white(uint32_t v)
{
    const uint32_t a = v >> 24, ia = 255u * (255u - a);
    uint32_t o = 0xFF000000u;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const uint32_t t = ((v >> (8 * c)) & 255u) * a + ia;
        o |= ((t + 128u + ((t + 128u) >> 8)) >> 8) << (8 * c);
    }
    return o;
}
__global__ void __launch_bounds__(256) k_img_over_white(uint8_t *__restrict__ p, size_t stride, uint32_t w, uint32_t h)
{
    const uint32_t x = 4 * (blockIdx.x * 64 + (threadIdx.x & 63)), y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= w || y >= h) return;
    uint32_t *px = (uint32_t *)(p + (size_t)y * stride) + x;
    if (w - x < 4) {
        for (uint32_t i = 0; i < w - x; i++) px[i] = img_white(px[i]);
        return;
    }
    const img_u4 v = *(const img_u4 *)px;
    if ((v[0] & v[1] & v[2] & v[3]) >> 24 == 255u) return;
    *(img_u4 *)px = img_u4{img_white(v[0]), img_white(v[1]), img_white(v[2]), img_white(v[3])};
}

// ---- pi_half (procimg.h:636-661): one level of the 2x2 box pyramid, per output pixel and channel
// ve = (a + c + 1) >> 1 over the two rows, then (ve + vo) >> 1 over the two columns
__global__ void __launch_bounds__(256) k_img_half(uint8_t *__restrict__ d, size_t ds, const uint8_t *__restrict__ s,
                                                  size_t ss, uint32_t wn, uint32_t hn)
{
    const uint32_t x = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y;
    if (x >= wn || y >= hn) return;
    const uint32_t *p0 = (const uint32_t *)(s + (size_t)(2 * y) * ss + 8 * (size_t)x);
    const uint32_t *p1 = (const uint32_t *)(s + (size_t)(2 * y + 1) * ss + 8 * (size_t)x);
    const uint2 r0 = {p0[0], p0[1]}, r1 = {p1[0], p1[1]};
    uint32_t o = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint32_t ve = (((r0.x >> (8 * c)) & 255u) + ((r1.x >> (8 * c)) & 255u) + 1u) >> 1;
        const uint32_t vo = (((r0.y >> (8 * c)) & 255u) + ((r1.y >> (8 * c)) & 255u) + 1u) >> 1;
        o |= ((ve + vo) >> 1) << (8 * c);
    }
    *(uint32_t *)(d + (size_t)y * ds + 4 * (size_t)x) = o;
}

// ---- pi_cubic / pi_axis (procimg.h:750-790), built per block in shared memory
__device__ __forceinline__ float img_cubic(float x)
{
    x = x < 0 ? -x : x;
    return x < 1.0f ? (1.5f * x - 2.5f) * x * x + 1.0f : x < 2.0f ? ((-0.5f * x + 2.5f) * x - 4.0f) * x + 2.0f : 0.0f;
}

// One axis: output index i of S over a virtual square of `side` with the content at [off, off + len); the weights
// come out scaled by sc, the constant offset by add (the x axis folds the [-1, 1] normalisation in).
struct ImgGeom {
    float scale, ss, support, sc, add;
    int32_t side, off, end;
};

__device__ __forceinline__ ImgGeom img_geom(uint32_t S, uint32_t side, uint32_t off, uint32_t len, float sc, float add)
{
    ImgGeom g;
    g.scale = (float)side / (float)S;
    const float fs = g.scale > 1.0f ? g.scale : 1.0f;
    g.support = 2.0f * fs;
    g.ss = 1.0f / fs;
    g.sc = sc;
    g.add = add;
    g.side = (int32_t)side;
    g.off = (int32_t)off;
    g.end = (int32_t)(off + len);
    return g;
}

// the taps [lo, hi) of output i and the content part [a, b) of them (pi_axis's integer bounds)
__device__ __forceinline__ void img_bounds(const ImgGeom &g, int32_t i, float &center, int32_t &lo, int32_t &hi,
                                           int32_t &a, int32_t &b)
{
    center = ((float)i + 0.5f) * g.scale;
    lo = (int32_t)(center - g.support + 0.5f);
    hi = (int32_t)(center + g.support + 0.5f);
    lo = lo < 0 ? 0 : lo;
    hi = hi > g.side ? g.side : hi;
    a = lo > g.off ? lo : g.off;
    b = hi < g.end ? hi : g.end;
    b = b < a ? a : b;
}

#define IMG_MT_MAX 24                       // taps per output for resample factors f < 5.5 (img_mt: 2 (int)(2 f + 1) + 2)
#define IMG_XN (14 * IMG_BAND_P)            // outputs of a block's two axes: 28 columns, then 14 rows
#define IMG_ON (IMG_XN + 14)
#define IMG_RT 512                          // threads of k_img_resample
#define IMG_SPAN 176                        // source columns of 28 outputs: 27 f between centres + 4 f + 2 < 172.5

// Tap tables (shared memory) of a block's outputs: columns x0 .. x0 + nx - 1 as outputs 0 .., rows y0 .. y0 + 13 as
// outputs IMG_XN ..: every raw weight in parallel (the same float expression as the reference), then one thread per
// output sums its taps in tap order (the reference's loop; taps past the last add an exact zero, so the loop has a
// fixed length and its reads overlap), then the content taps, scaled, in parallel again. w [output][mt] holds the
// content taps; s, n, k per output. Ends synchronised.
struct ImgTaps {
    float raw[IMG_ON * IMG_MT_MAX], w[IMG_ON * IMG_MT_MAX], k[IMG_ON], sum[IMG_ON];
    int32_t s[IMG_ON], n[IMG_ON], skip[IMG_ON];
};

// gy or gx, field by field (a reference to either would put both in scratch memory); the axes share the square
__device__ __forceinline__ ImgGeom img_axis(const ImgGeom &gx, const ImgGeom &gy, bool y)
{
    ImgGeom g = gx;
    g.sc = y ? gy.sc : gx.sc;
    g.add = y ? gy.add : gx.add;
    g.off = y ? gy.off : gx.off;
    g.end = y ? gy.end : gx.end;
    return g;
}

__device__ __forceinline__ void img_taps(const ImgGeom &gx, const ImgGeom &gy, int32_t x0, int32_t nx, int32_t y0,
                                         int32_t mt, ImgTaps &T)
{
    for (int32_t e = threadIdx.x; e < IMG_ON * IMG_MT_MAX; e += blockDim.x) {
        const int32_t c = e / IMG_MT_MAX, t = e - c * IMG_MT_MAX;
        const bool y = c >= IMG_XN;
        float wt = 0.0f;
        if (t < mt && (y || c < nx)) {
            const ImgGeom g = img_axis(gx, gy, y);
            float center;
            int32_t lo, hi, a, b;
            img_bounds(g, y ? y0 + c - IMG_XN : x0 + c, center, lo, hi, a, b);
            wt = lo + t < hi ? img_cubic(((float)(lo + t) - center + 0.5f) * g.ss) : 0.0f;
        }
        T.raw[e] = wt;
    }
    __syncthreads();
    if (threadIdx.x < IMG_ON) {
        const int32_t c = threadIdx.x;
        const bool y = c >= IMG_XN;
        if (y || c < nx) {
            const ImgGeom g = img_axis(gx, gy, y);
            float center, sm = 0.0f, white = 0.0f;
            int32_t lo, hi, a, b;
            img_bounds(g, y ? y0 + c - IMG_XN : x0 + c, center, lo, hi, a, b);
#pragma unroll
            for (int32_t t = 0; t < IMG_MT_MAX; t++) {
                const float wt = T.raw[c * IMG_MT_MAX + t];
                sm += wt;
                white += lo + t < a || lo + t >= b ? wt : 0.0f;
            }
            sm = g.sc / sm;
            T.sum[c] = sm;
            T.s[c] = a - g.off;
            T.n[c] = b - a;
            T.skip[c] = a - lo;
            T.k[c] = 255.0f * white * sm + g.add;
        } else {
            T.s[c] = T.n[c] = T.skip[c] = 0;
            T.sum[c] = T.k[c] = 0.0f;
        }
    }
    __syncthreads();
    for (int32_t e = threadIdx.x; e < IMG_ON * IMG_MT_MAX; e += blockDim.x) {
        const int32_t c = e / IMG_MT_MAX, t = e - c * IMG_MT_MAX;
        T.w[e] = t < T.n[c] ? T.raw[e + T.skip[c]] * T.sum[c] : 0.0f;  // skip + n <= mt
    }
    __syncthreads();
}

__device__ __forceinline__ uint16_t img_f16(float v)
{
    return __builtin_bit_cast(uint16_t, (_Float16)v);  // v_cvt_f16_f32: round to nearest even
}

// Band staging: 14 rows x np patches of the operand, [patch][592] halves, pad halves zero; written out with 16-byte
// stores (the band's patches are contiguous in the operand).
__device__ __forceinline__ void img_band_store(uint16_t *band, uint16_t *__restrict__ out, uint32_t S, uint32_t np)
{
    __syncthreads();
    const uint32_t pr = S / 14, p0 = blockIdx.y * pr + blockIdx.x * IMG_BAND_P;
    uint4 *dst = (uint4 *)(out + (size_t)p0 * IMG_PATCH);
    const uint4 *sb = (const uint4 *)band;
    for (uint32_t q = threadIdx.x; q < np * IMG_PATCH / 8; q += blockDim.x) dst[q] = sb[q];
}

// ---- pi_vrow and pi_hrow (procimg.h:800-868) of one band: rows 14 blockIdx.y .., patches blockIdx.x * IMG_BAND_P ..
// The block resamples vertically only the source columns its 28 output columns take (14 rows x those columns, RGB in
// fp32, into shared memory: neighbouring blocks repeat the taps' overlap, about a seventh), then horizontally from
// there, one output pixel per thread. Each value is the constant plus one fma per tap in tap order, as in the
// reference's two passes over whole rows. Bound by the latency of its steps (tap tables, source reads, horizontal taps)
// at these sizes; 512 threads a block (392: 10% slower, 832: 40%). us a call, two kernels with the vertical result in
// an fp32 [S][cw] scratch in between -> here: 3072 x 2048 at level 1 17.6 -> 13.1, 1847 x 2048 13.4 -> 11.1, 900 x 900
// at level 0 12.4 -> 9.7, 440 x 300 8.9 -> 7.4.
__global__ void __launch_bounds__(IMG_RT) k_img_resample(const uint8_t *__restrict__ src, size_t stride,
                                                                     uint32_t cw, uint32_t ch, uint32_t S,
                                                                     uint32_t side, uint32_t mt,
                                                                     uint16_t *__restrict__ out)
{
    __shared__ __attribute__((aligned(16))) uint16_t band[IMG_BAND_P * IMG_PATCH];
    __shared__ ImgTaps T;
    __shared__ float v[3][14 * IMG_SPAN];
    __shared__ int32_t span[2];
    const uint32_t pr = S / 14, pc0 = blockIdx.x * IMG_BAND_P;
    const uint32_t np = pr - pc0 < IMG_BAND_P ? pr - pc0 : IMG_BAND_P;
    const int32_t nx = (int32_t)(14 * np);
    if (threadIdx.x < np) *(uint2 *)(band + threadIdx.x * IMG_PATCH + 588) = uint2{0u, 0u};
    if (threadIdx.x == 0) span[0] = 0x7fffffff, span[1] = 0;
    img_taps(img_geom(S, side, (side - cw) >> 1, cw, 1.0f / 127.5f, -1.0f), img_geom(S, side, (side - ch) >> 1, ch, 1.0f, 0.0f),
             (int32_t)(pc0 * 14), nx, (int32_t)(blockIdx.y * 14), (int32_t)mt, T);
    if (threadIdx.x < IMG_XN && T.n[threadIdx.x]) {  // source columns [span[0], span[1]) that any output takes
        atomicMin(&span[0], T.s[threadIdx.x]);
        atomicMax(&span[1], T.s[threadIdx.x] + T.n[threadIdx.x]);
    }
    __syncthreads();
    const int32_t x0 = span[0], nc = span[1] - x0, nw = nc < 0 ? 0 : nc < IMG_SPAN ? nc : IMG_SPAN;
    for (int32_t e = threadIdx.x; e < 14 * nw; e += blockDim.x) {
        const int32_t ky = e / nw, x = e - ky * nw, c = IMG_XN + ky, n = T.n[c];
        const float *wj = T.w + c * IMG_MT_MAX;
        float a0 = T.k[c], a1 = a0, a2 = a0;
        const uint8_t *p = src + (size_t)T.s[c] * stride + 4 * (size_t)(x0 + x);
        // eight source pixels in flight; past the last tap its row again, with weight 0 (adds an exact zero)
        for (int32_t j0 = 0; j0 < n; j0 += 8) {
            uint32_t u[8];
#pragma unroll
            for (int32_t j = 0; j < 8; j++) u[j] = *(const uint32_t *)(p + (size_t)(j0 + j < n ? j0 + j : n - 1) * stride);
#pragma unroll
            for (int32_t j = 0; j < 8; j++) {
                const float w = wj[j0 + j];
                a0 = __builtin_fmaf(w, (float)(u[j] & 255u), a0);
                a1 = __builtin_fmaf(w, (float)((u[j] >> 8) & 255u), a1);
                a2 = __builtin_fmaf(w, (float)((u[j] >> 16) & 255u), a2);
            }
        }
        v[0][ky * IMG_SPAN + x] = a0;
        v[1][ky * IMG_SPAN + x] = a1;
        v[2][ky * IMG_SPAN + x] = a2;
    }
    __syncthreads();
    const uint32_t e = threadIdx.x;
    if (e < 14 * 14 * np) {
        const uint32_t ky = e / (14 * np), jj = e - ky * 14 * np;   // row in the band, column in the block
        const int32_t n = T.n[jj], o0 = (int32_t)ky * IMG_SPAN + (n ? T.s[jj] - x0 : 0);
        const float *wj = T.w + jj * IMG_MT_MAX;
        float r = T.k[jj], g = r, b = r;
#pragma unroll 8
        for (int32_t q = 0; q < n; q++) {
            const float wq = wj[q];
            r = __builtin_fmaf(wq, v[0][o0 + q], r);
            g = __builtin_fmaf(wq, v[1][o0 + q], g);
            b = __builtin_fmaf(wq, v[2][o0 + q], b);
        }
        uint16_t *o = band + (jj / 14) * IMG_PATCH + ky * 14 + jj % 14;
        o[0] = img_f16(__builtin_fminf(__builtin_fmaxf(b, -1.0f), 1.0f));
        o[196] = img_f16(__builtin_fminf(__builtin_fmaxf(g, -1.0f), 1.0f));
        o[392] = img_f16(__builtin_fminf(__builtin_fmaxf(r, -1.0f), 1.0f));
    }
    img_band_store(band, out, S, np);
}

// ---- pi_idrow (procimg.h:874-902): side == S, the identity: v / 127.5 - 1 as one fma, white (0x3C00) pad
__global__ void __launch_bounds__(256) k_img_ident(const uint8_t *__restrict__ src, size_t stride, uint32_t cw,
                                                   uint32_t ch, uint32_t S, uint16_t *__restrict__ out)
{
    __shared__ __attribute__((aligned(16))) uint16_t band[IMG_BAND_P * IMG_PATCH];
    const uint32_t pr = S / 14, pc0 = blockIdx.x * IMG_BAND_P, ox = (S - cw) >> 1, oy = (S - ch) >> 1;
    const uint32_t np = pr - pc0 < IMG_BAND_P ? pr - pc0 : IMG_BAND_P;
    const float sc = 1.0f / 127.5f;
    for (uint32_t q = threadIdx.x; q < np; q += blockDim.x) *(uint2 *)(band + q * IMG_PATCH + 588) = uint2{0u, 0u};
    for (uint32_t e = threadIdx.x; e < 14 * 14 * np; e += blockDim.x) {
        const uint32_t ky = e / (14 * np), jj = e - ky * 14 * np;
        const uint32_t i = blockIdx.y * 14 + ky, j = pc0 * 14 + jj;
        uint16_t *o = band + (jj / 14) * IMG_PATCH + ky * 14 + jj % 14;
        if (i - oy < ch && j - ox < cw) {
            const uint32_t v = *(const uint32_t *)(src + (size_t)(i - oy) * stride + 4 * (size_t)(j - ox));
            o[0] = img_f16(__builtin_fmaf((float)((v >> 16) & 255u), sc, -1.0f));
            o[196] = img_f16(__builtin_fmaf((float)((v >> 8) & 255u), sc, -1.0f));
            o[392] = img_f16(__builtin_fmaf((float)(v & 255u), sc, -1.0f));
        } else {
            o[0] = o[196] = o[392] = 0x3C00;
        }
    }
    img_band_store(band, out, S, np);
}

// ---------------------------------------------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------------------------------------------
static size_t img_a32(size_t n) { return (n + 31) & ~(size_t)31; }

static uint32_t img_mt(uint32_t side, uint32_t S)  // procimg.h:949
{
    return 2 * (uint32_t)(2.0f * (side > S ? (float)side / (float)S : 1.0f) + 1.0f) + 2;
}

extern "C" int eva_img_over_white(void *rgba, size_t stride, uint32_t w, uint32_t h, void *stream)
{
    if (!rgba || !w || !h || stride < (size_t)w * 4 || (stride & 3) || ((uintptr_t)rgba & 3))
        return xt_fail("eva_img_over_white", "bad image (4-byte aligned rows of w RGBA pixels)");
    hipLaunchKernelGGL(k_img_over_white, dim3((w + 255) / 256, (h + 3) / 4), dim3(256), 0, (hipStream_t)stream,
                       (uint8_t *)rgba, stride, w, h);
    return xt_check("eva_img_over_white");
}

// pi_pyramid's level sizes (procimg.h:665-681), PI_PYRMIN = 2 S: levels 1.. of p from p->lw[0], p->lh[0]
static uint32_t img_levels(eva_pyr *p, uint32_t S)
{
    uint32_t n;
    for (n = 1; n < EVA_PYR_LV; n++) {
        const uint32_t m = p->lw[n - 1] > p->lh[n - 1] ? p->lw[n - 1] : p->lh[n - 1];
        if ((m >> 1) < 2 * S || p->lw[n - 1] < 2 || p->lh[n - 1] < 2) break;
        p->lw[n] = p->lw[n - 1] >> 1;
        p->lh[n] = p->lh[n - 1] >> 1;
        p->ls[n] = img_a32((size_t)p->lw[n] * 4);
    }
    return n;
}

extern "C" size_t eva_img_pyramid_bytes(uint32_t w, uint32_t h, uint32_t S)
{
    eva_pyr p = {};
    p.lw[0] = w;
    p.lh[0] = h;
    const uint32_t n = img_levels(&p, S ? S : EVA_S);
    size_t total = 0;
    for (uint32_t L = 1; L < n; L++) total += p.ls[L] * p.lh[L];
    return total;
}

extern "C" int eva_img_pyramid(eva_pyr *p, void *levels, size_t bytes, uint32_t S, void *stream)
{
    if (!p || !p->lv[0] || !p->lw[0] || !p->lh[0] || p->ls[0] < (size_t)p->lw[0] * 4 || (p->ls[0] & 3) ||
        ((uintptr_t)p->lv[0] & 3))
        return xt_fail("eva_img_pyramid", "level 0 must be set (lv, lw, lh, ls: 4-byte aligned RGBX rows)");
    if (!S) S = EVA_S;
    const uint32_t n = img_levels(p, S);
    size_t total = 0;
    for (uint32_t L = 1; L < n; L++) total += p->ls[L] * p->lh[L];
    if (n > 1 && (!levels || bytes < total || ((uintptr_t)levels & 31)))
        return xt_fail("eva_img_pyramid", "levels must be 32-byte aligned and hold eva_img_pyramid_bytes()");
    uint8_t *blk = (uint8_t *)levels;
    for (uint32_t L = 1; L < n; L++) {
        p->lv[L] = blk;
        blk += p->ls[L] * p->lh[L];
        hipLaunchKernelGGL(k_img_half, dim3((p->lw[L] + 255) / 256, p->lh[L]), dim3(256), 0, (hipStream_t)stream,
                           p->lv[L], p->ls[L], (const uint8_t *)p->lv[L - 1], p->ls[L - 1], p->lw[L], p->lh[L]);
    }
    for (uint32_t L = n; L < EVA_PYR_LV; L++) {
        p->lv[L] = NULL;
        p->lw[L] = p->lh[L] = 0;
        p->ls[L] = 0;
    }
    p->nlv = n;
    return xt_check("eva_img_pyramid");
}

// scratch that the interface asks for: [S][cw] float4
static size_t img_scratch(uint32_t S, uint32_t cw) { return (size_t)S * cw * 16; }

extern "C" size_t eva_img_prep_bytes(uint32_t S, uint32_t max_side)
{
    if (!S) S = EVA_S;
    return img_scratch(S, max_side);
}

// A crop on its level: the host part of pi_prep (pi_level, pi_lsrc) and the limits that both entry points share. what
// names the entry point in errors; an S of 0 becomes the default side.
struct ImgRect {
    const uint8_t *src;
    size_t stride;
    uint32_t cw, ch, side, S;
};

static int img_rect(const char *what, const eva_pyr *p, uint32_t x0, uint32_t y0, uint32_t cw, uint32_t ch, uint32_t S,
                    const void *out, ImgRect &r)
{
    if (!S) S = EVA_S;
    if (!p || !p->nlv || p->nlv > EVA_PYR_LV || !p->lv[0]) return xt_fail(what, "no pyramid");
    if (S % 14 || S > 1008 || !out || ((uintptr_t)out & 15))
        return xt_fail(what, "S must be a multiple of 14 up to 1008; out 16-byte aligned");
    if (!cw || !ch || x0 >= p->lw[0] || y0 >= p->lh[0]) return xt_fail(what, "empty or outside rect");
    // pi_level + pi_lsrc (procimg.h:691-716)
    uint32_t L = 0;
    const uint32_t side0 = cw > ch ? cw : ch;
    while (L + 1 < p->nlv && (side0 >> (L + 1)) >= 2 * S) L++;
    uint32_t x1 = (x0 + cw) >> L, y1 = (y0 + ch) >> L;
    x1 = x1 < p->lw[L] ? x1 : p->lw[L];
    y1 = y1 < p->lh[L] ? y1 : p->lh[L];
    x0 >>= L;
    y0 >>= L;
    x0 = x0 < p->lw[L] ? x0 : p->lw[L] - 1;
    y0 = y0 < p->lh[L] ? y0 : p->lh[L] - 1;
    r.cw = x1 > x0 ? x1 - x0 : 1;
    r.ch = y1 > y0 ? y1 - y0 : 1;
    r.src = p->lv[L] + (size_t)y0 * p->ls[L] + (size_t)x0 * 4;
    r.stride = p->ls[L];
    r.side = r.cw > r.ch ? r.cw : r.ch;
    r.S = S;
    if (r.side != S && img_mt(r.side, S) > IMG_MT_MAX)
        return xt_fail(what, "rect more than 5x the model side on its level");  // from 5.5x on
    return 0;
}

// pi_prep of a checked rect: the identity where its long side is S, else the resample (which stages nothing in memory)
static int img_prep(const char *what, const ImgRect &r, void *out, void *stream)
{
    const uint32_t pr = r.S / 14;
    const dim3 bands((pr + IMG_BAND_P - 1) / IMG_BAND_P, pr);
    if (r.side == r.S)
        hipLaunchKernelGGL(k_img_ident, bands, dim3(256), 0, (hipStream_t)stream, r.src, r.stride, r.cw, r.ch, r.S,
                           (uint16_t *)out);
    else
        hipLaunchKernelGGL(k_img_resample, bands, dim3(IMG_RT), 0, (hipStream_t)stream, r.src, r.stride, r.cw, r.ch, r.S,
                           r.side, img_mt(r.side, r.S), (uint16_t *)out);
    return xt_check(what);
}

// The scratch of a resampled rect is checked as the interface says and passed no further.
extern "C" int eva_img_prep(const eva_pyr *p, uint32_t x0, uint32_t y0, uint32_t cw, uint32_t ch, uint32_t S,
                            void *scratch, size_t bytes, void *out, void *stream)
{
    ImgRect r;
    if (img_rect("eva_img_prep", p, x0, y0, cw, ch, S, out, r)) return -1;
    if (r.side != r.S && (!scratch || bytes < img_scratch(r.S, r.cw) || ((uintptr_t)scratch & 15)))
        return xt_fail("eva_img_prep", "scratch must be 16-byte aligned and hold S x (rect width on its level) x 16 "
                                       "bytes (eva_img_prep_bytes(S, side))");
    return img_prep("eva_img_prep", r, out, stream);
}

// ---- eva_img_prep without a scratch argument, for rects whose scratch would fit EVA_IMG_STATIC_BYTES
extern "C" int eva_img_prep_static(const eva_pyr *p, uint32_t x0, uint32_t y0, uint32_t cw, uint32_t ch, uint32_t S,
                                   void *out, void *stream)
{
    ImgRect r;
    if (img_rect("eva_img_prep_static", p, x0, y0, cw, ch, S, out, r)) return -1;
    if (r.side != r.S && img_scratch(r.S, r.cw) > EVA_IMG_STATIC_BYTES)
        return xt_fail("eva_img_prep_static", "rect too wide: S x (its width on its level) x 16 is more than "
                                              "EVA_IMG_STATIC_BYTES");
    return img_prep("eva_img_prep_static", r, out, stream);
}
