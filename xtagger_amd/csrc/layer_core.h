// layer_core.h - pieces shared by the block-GEMM kernels of the EVA02-L (wd) and ViTDet-L (PixAI) layers: the tile
// configuration, the shared-memory plan of the epilogues, the main-loop dispatch (dense or 2:4-sparse weights), the
// tile raster and the residual update of a wave tile.
#pragma once
#include "gemm_core.h"
#include "xt_abi.h"
#include "xt_launch.h"

typedef BsCfg<256, 256, 4, 2, 2> LayerCfg;  // 8 waves of 64 x 128: two heads (qkv) or 64 SwiGLU units (fc1) per wave
// Smaller tiles for grids that LayerCfg would leave mostly idle (with_res_cfg, and qkv's and fc1's own rules). Every
// output takes its K blocks in the same order whatever the tile, so the choice never changes a bit.
typedef BsCfg<128, 128, 4, 2, 2> LayerMid;  // 8 waves of 32 x 64, two blocks per CU
typedef BsCfg<64, 128, 2, 2, 3> LayerSml;   // 4 waves of 32 x 64, three stages, two blocks per CU

// Shared memory of the layer kernels: the main-loop stages, reused by the epilogues (one WM x 68 fp32 residual slice
// per wave, one [WN][WM + 4] bf16 transpose slice per wave, or the fc1 h tile), then the per-row statistics and
// per-column fold terms that k_fc2 fills while its first stages load.
template <class C>
struct LayerMem {
    static constexpr int PC = C::WN < 64 ? C::WN : 64;             // columns of a residual pass
    static constexpr int LD = PC + 4;                              // floats per row of a residual slice
    static constexpr int SLICE = C::WM * LD * 4;
    static constexpr int TRLD = C::WM + 4;                         // halves per row of a transpose slice
    static constexpr int TRSLICE = C::WN * TRLD * 2;
    static constexpr int EPI = C::NW * (SLICE > TRSLICE ? SLICE : TRSLICE);
    static constexpr int LOOP = C::LDS > C::LDS_SP ? C::LDS : C::LDS_SP;
    static constexpr int ROWSTAT = EPI > LOOP ? EPI : LOOP;        // byte offset of the per-row statistics
    static constexpr int SMEM = ROWSTAT + 8 * (C::BM + C::BN);     // row statistics, then column terms
    static_assert(SMEM <= 160 * 1024, "layer kernels fit the LDS");
};

__device__ __forceinline__ uint32_t pk_bf16(float a, float b)
{
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{a, b}), b2));
}

// two fp32 values rounded to fp16 (RNE) in one v_cvt_pk_f16_f32, a in the low half
__device__ __forceinline__ uint32_t pk_f16(float a, float b)
{
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    asm volatile("" : "+v"(a), "+v"(b));  // fp32 values: no fused fp32-op + fp16-round (v_fma_mix*) single rounding
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{a, b}), h2));
}

// The layer kernels take their weights dense (w, wx unused) or 2:4-sparse (SP: w = pack24 values, wx = indices).
// Nlive (default Npad): columns from Nlive on hold zero weights throughout, so waves that own only such columns skip
// their matrix work.
// TR (dense weights only): the tile transposed, as bs_mainloop's TR leaves it.
template <class C, bool SP, class Pre = BsNoPre, bool TR = false>
__device__ __forceinline__ void layer_mainloop(const uint8_t *A, int lda, const float *sa, int lds, const uint8_t *w,
                                               const uint32_t *wx, const float *ws, int rows, int Npad, int K, int m0,
                                               int n0, uint8_t *smem, v4f (&acc)[C::TM][C::TN], Pre pre = Pre(),
                                               int Nlive = -1)
{
    static_assert(!(SP && TR), "the sparse tile comes transposed from bs_mainloop_sp_t");
    if constexpr (SP) bs_mainloop_sp<C>(A, lda, sa, lds, w, wx, ws, rows, Npad, K, m0, n0, smem, acc, pre, Nlive);
    else bs_mainloop<C, Pre, true, TR>(A, lda, sa, lds, w, ws, rows, Npad, K, m0, n0, smem, acc, pre, Nlive);
}

template <class C>
__device__ __forceinline__ void layer_tile(int M, int N, int &m0, int &n0)
{
    int tm, tn;
    tile_of_block((M + C::BM - 1) / C::BM, (N + C::BN - 1) / C::BN, M % C::BM != 0, tm, tn);
    m0 = tm * C::BM;
    n0 = tn * C::BN;
}

typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v4f_e __attribute__((ext_vector_type(4), aligned(4)));     // 16 bytes of memory aligned to its elements
typedef unsigned v4u_e __attribute__((ext_vector_type(4), aligned(2)));  // only (fp32; 16-bit types)

// x + y for the fp16 x in the low (HI = 0) or high (HI = 1) half of a word and an fp32 y: one v_fma_mix_f32,
// fma(x, 1, y) with x widened exactly, which rounds once to fp32 as the conversion followed by v_add_f32 does
template <int HI>
__device__ __forceinline__ float h_add(uint32_t xw, float y)
{
    float r;
    if constexpr (HI) asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(xw), "v"(y));
    else asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(xw), "v"(y));
    return r;
}

// Residual update x = f16(x + y) of a wave's WM x WN tile, transposed as bs_mainloop's TR and the sparse main loop
// leave it: y(jn, im) gives the four values added to row mw + 16 im + (lane & 15), columns
// nw + 16 jn + 4 (lane >> 4) + r. In passes of PC = 64 columns (32 for a 32-column tile) the wave parks its y in its
// own LDS slice by one 16-byte store per (m tile, n tile) (rows of PC + 4 floats: the 16 rows of one store group start
// 4 banks apart), then each lane updates 8 consecutive halves with one 16-byte load and store, so one wave
// instruction covers whole rows of the pass. Every x load of the tile is issued before the first store (one memory
// round trip for the whole update), through a buffer descriptor that ends at row `rows`: rows past it load zero and
// their stores are dropped, with no branch between the loads.
template <class C, class Y>
__device__ __forceinline__ void residual_add_t(uint8_t *slices, Y y, uint16_t *__restrict__ x, int mw, int nw, int rows)
{
    using S = LayerMem<C>;
    constexpr int NP = C::WN / S::PC, LPR = S::PC / 8, RPI = 64 / LPR, NI = C::WM / RPI;  // lanes a row, rows a store
    float *tr = (float *)(slices + (threadIdx.x >> 6) * S::SLICE);
    const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const int rs = lane / LPR, ch = lane % LPR;
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(x, (uint32_t)rows * XT_D * 2u);
    const uint32_t off0 = (uint32_t)(((mw + rs) * XT_D + nw + 8 * ch) * 2);
    v4u xv[NP][NI];
#pragma unroll
    for (int pass = 0; pass < NP; pass++)
#pragma unroll
        for (int it = 0; it < NI; it++)
            xv[pass][it] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(off0 + (uint32_t)((RPI * it * XT_D + S::PC * pass) * 2)), 0, 0);
#pragma unroll
    for (int pass = 0; pass < NP; pass++) {
        if (pass) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the previous pass's slice reads are done
#pragma unroll
        for (int im = 0; im < C::TM; im++)
#pragma unroll
            for (int jq = 0; jq < S::PC / 16; jq++) {
                const v4f v = y(S::PC / 16 * pass + jq, im);
                *(float4 *)(tr + (16 * im + c16) * S::LD + 16 * jq + 4 * g) = make_float4(v[0], v[1], v[2], v[3]);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slice is the wave's own: no block barrier needed
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const int rr = RPI * it + rs;
            const float4 a = *(const float4 *)(tr + rr * S::LD + 8 * ch), b = *(const float4 *)(tr + rr * S::LD + 8 * ch + 4);
            const v4u v = xv[pass][it];
            v4u o;
            o[0] = pk_f16(h_add<0>(v[0], a.x), h_add<1>(v[0], a.y));
            o[1] = pk_f16(h_add<0>(v[1], a.z), h_add<1>(v[1], a.w));
            o[2] = pk_f16(h_add<0>(v[2], b.x), h_add<1>(v[2], b.y));
            o[3] = pk_f16(h_add<0>(v[3], b.z), h_add<1>(v[3], b.w));
            __builtin_amdgcn_raw_buffer_store_b128(o, rx, (int)(off0 + (uint32_t)((RPI * it * XT_D + S::PC * pass) * 2)), 0, 0);
        }
    }
}

template <class C>
static inline unsigned layer_grid(int rows, int N)
{
    return (unsigned)(((rows + C::BM - 1) / C::BM) * ((N + C::BN - 1) / C::BN));
}

// f(C{}) with the tile configuration C of a 1024-column GEMM (attention out-projection, fc2) over `rows` rows, K deep.
// 256 x 256 tiles read each operand least and win once they fill the CUs, but give only 4 tiles per 256 rows; a K step
// costs them about 1.35 us against 0.5-0.9 for the smaller ones, so a grid that leaves CUs idle is better cut finer.
//  - 64 x 128 while one round of two blocks per CU holds them (rows <= 4096). us, 256 x 256 -> 64 x 128:
//    K = 1024: 14.8 -> 5.3 at 1025 rows, 15.1 -> 6.9 at 2050; K = 2816: 32.6 -> 10.8 and 34.6 -> 15.4
//    (128 x 128: 6.9, 7.4; 19.4, 20.5);
//  - 128 x 128 while one round of two blocks per CU holds them (rows <= 8192): K = 2816 35.6 -> 22.5 at 4100 and
//    36.6 -> 25.3 at 6150 (64 x 128: 26.1, 33.1); K = 1024 15.7 -> 10.0 and 17.0 -> 11.9;
//  - above that 256 x 256 (K = 2816: 37.3 against 42.3 at 8200, 66.3 against 68.4 at 16400; K = 4736: 55.8 against
//    67.8 at 10368), except at K <= 1024 where the whole 256 x 256 tiles leave a last round at most half full (or fill
//    the rounds exactly and a partial row tile follows): 18.3 -> 16.9 at 8200, 31.9 -> 28.2 at 16400, 37.1 -> 34.5
//    at 20736, 52.2 -> 46.9 at 32800 (a last round fuller than that: 18.9 against 19.3 at 10250, 44.0 against 48.9 at
//    31104).
// Those are calls alone on the chip. Beside an engine's other lane, whose kernels take the CUs that a grid leaves idle,
// the 128 x 128 tiles' operand traffic costs more than they save: us per batch, the limits above (and qkv's) -> 256 x 256
// from 4353 rows a lane on: 5950 -> 5640 at 10 images, 7015 -> 6750 at 12, 7750 -> 7620 at 14, the same within 1% from 16
// to 64 (PixAI's proj: 30340 -> 30120 at 8). At 4100 rows 128 x 128 stays: 4300 against 4393 at 7 images, 4806 against
// 4839 at 8.
template <class F>
static inline void with_res_cfg(int rows, int K, int lanes, F f)
{
    const int tail = rows / LayerCfg::BM * (XT_D / LayerCfg::BN) % 256;  // whole 256 x 256 tiles of the last round
    if (rows <= 4096) f(LayerSml{});
    else if (lanes > 1 ? rows <= 4352 : rows <= 8192 || (K <= XT_D && tail <= 128 && (tail || rows % LayerCfg::BM)))
        f(LayerMid{});
    else f(LayerCfg{});
}

#define XT_ALIGNED(p) ((((uintptr_t)(p)) & 15) == 0)

// Token rows a layer launcher accepts: every 32-bit buffer offset (rows x 4736 bytes of the widest E4M3 activation,
// rows x 2048 of an fp16 residual or bf16 q / k, the XT_OOR = 2^31 sentinel of rows past the end) stays in range.
static inline int layer_rows_ok(const char *what, int rows, int lds)
{
    if (rows <= 0 || lds < rows || rows > (1 << 19)) return xt_fail(what, "bad shape (0 < rows <= 2^19, lds >= rows)");
    return 0;
}
