// layer.hip - the EVA02-L block GEMMs with their fused epilogues, all on the block-scaled main loop (gemm_core.h),
// plus the fp16 patch embedding. Reference roles (src/engine/eva_kernels.cu): k_qkv (41-114), k_oproj (134-162),
// k_fc1 (211-279), k_fc2 (286-334), k_pe + k_embed (126-130, 21-33), and the head k_headmv
// (src/engine/kern_common.cuh:679-727) as a block-scaled FP8 GEMM.
//
// Token rows: m = 1025 b + t for image b, token t (t = 0 is cls). Activations E4M3 [rows][K] with 1x128 scale
// planes [K/128][lds]; residual x fp16 [rows][1024].
#include "layer_core.h"


// ---------------------------------------------------------------------------------------------------------------
// k_qkv: h8 [rows][1024] x Wqkv [3072][1024] -> q, k bf16 [nb][16][1088][64] (RoPE on patch tokens), vt bf16
// [nb][16][64][1088]. A 256-column block is 4 heads of one of q | k | v; each wave owns two heads. The weight rows
// of q and k heads are stored quad-split (eva_k_prep_w perm 1): within a head, column tile j holds dim 4i + j for
// i = lane & 15, so a lane holds dims 4i .. 4i + 3, the rotary pairs 2i and 2i + 1 whole: their (cos, sin) come in one
// 16-byte load and the rotated dims leave in one 8-byte store. q rows carry log2(e)/8 (export_eva.py:71).
// ---------------------------------------------------------------------------------------------------------------
template <class C, bool SP>
__global__ void __launch_bounds__(C::NT) k_qkv(const uint8_t *__restrict__ h8, const float *__restrict__ hs,
                                                     int lds, const uint8_t *__restrict__ w,
                                                     const uint32_t *__restrict__ wx,
                                                     const float *__restrict__ ws, const float *__restrict__ cs,
                                                     uint16_t *__restrict__ q, uint16_t *__restrict__ k,
                                                     uint16_t *__restrict__ vt, int rows)
{
    constexpr int NH = C::TN / 4, TRLD = LayerMem<C>::TRLD;  // heads per wave
    __shared__ __attribute__((aligned(16))) uint8_t smem[LayerMem<C>::SMEM];
    v4f acc[C::TM][C::TN];
    int m0, n0, wm0, wn0;
    layer_tile<C>(rows, 3 * XT_D, m0, n0);
    args_resident(cs, q, k, vt, lds, rows);
    bs_wave_origin<C>(wm0, wn0);
    const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const int part = n0 >> 10, head0 = ((n0 & 1023) + wn0) >> 6;
    // v: the wave's rows x dims (one or two heads) are transposed through its own LDS slice ([WN dims][WM + 4] bf16,
    // padded rows), then lanes walk rows (consecutive tokens; two dims at a time where the wave has 32 rows, the lane's
    // own dim folded into its base pointers so that the loop steps both by constants). The slice takes the tile in
    // whichever layout the main loop leaves it: the sparse loop's transposed tile directly (no pass through the dense
    // layout first), the dense tile as one 8-byte write of four consecutive tokens per (row tile, column tile).
    uint16_t *tr = (uint16_t *)(smem + (threadIdx.x >> 6) * LayerMem<C>::TRSLICE);
    auto v_out = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        constexpr int DS = 64 / C::WM;  // dims per store instruction
        const int row = lane % C::WM, d0 = lane / C::WM, m = m0 + wm0 + row;
        if (m < rows) {
            const int b = m / XT_T, t = m - b * XT_T;
            const uint16_t *src = tr + d0 * TRLD + row;
#pragma unroll
            for (int hh = 0; hh < NH; hh++) {
                uint16_t *dst = vt + (((size_t)b * XT_NH + head0 + hh) * XT_HD + d0) * XT_TP + t;
#pragma unroll 8
                for (int d = 0; d < XT_HD; d += DS) dst[(size_t)d * XT_TP] = src[(64 * hh + d) * TRLD];
            }
        }
    };
    if constexpr (SP) {
        if (part == 2) {  // a separate copy of the sparse loop: its transposed tile goes straight into the slice
            v4f accT[C::TN][C::TM];  // accT[j][i][r]: dim 16 j + 4 g + r, row 16 i + c16 of the wave tile
            bs_mainloop_sp_t<C>(h8, XT_D, hs, lds, w, wx, ws, rows, 3 * XT_D, XT_D, m0, n0, smem, accT);
#pragma unroll
            for (int j = 0; j < C::TN; j++)
#pragma unroll
                for (int i = 0; i < C::TM; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        tr[(16 * j + 4 * g + r) * TRLD + 16 * i + c16] = (uint16_t)pk_bf16(accT[j][i][r], 0.f);
            v_out();
            return;
        }
    }
    layer_mainloop<C, SP>(h8, XT_D, hs, lds, w, wx, ws, rows, 3 * XT_D, XT_D, m0, n0, smem, acc);
    if (part < 2) {
        // every (cos, sin) pair of the tile is loaded before the first store: one memory round trip. Patch token t of
        // image b uses row t - 1 of the table (eva_kernels.cu:74-79); cls rows (t = 0) load an out-of-range offset
        // (zero) and are not rotated. Stores go through a descriptor that ends at image nb: rows past `rows` are
        // dropped without a branch.
        const int nbi = rows / XT_T;
        const __amdgpu_buffer_rsrc_t rc = buf_rsrc(cs, 1024u * 32u * 8u);
        const __amdgpu_buffer_rsrc_t rd = buf_rsrc(part ? k : q, (uint32_t)nbi * XT_NH * XT_TP * XT_HD * 2u);
        v4f rot[C::TM][4];  // (cos, sin) of pairs 2 c16 and 2 c16 + 1
        int tok[C::TM][4], img[C::TM][4];
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm0 + 16 * i + 4 * g + r, b = m / XT_T, t = m - b * XT_T;
                img[i][r] = b;
                tok[i][r] = t;
                rot[i][r] = __builtin_bit_cast(
                    v4f, __builtin_amdgcn_raw_buffer_load_b128(rc, (int)(((uint32_t)(t - 1) * 32u + 2 * c16) * 8u), 0, 0));
            }
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int b = img[i][r], t = tok[i][r];
#pragma unroll
                for (int hh = 0; hh < NH; hh++) {
                    uint32_t two[2];
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        float f0 = acc[i][4 * hh + 2 * p][r], f1 = acc[i][4 * hh + 2 * p + 1][r];
                        if (t) {  // one rounded product and one fma per rotated value
                            const float cr = rot[i][r][2 * p], sr = rot[i][r][2 * p + 1];
                            const float g0 = __builtin_fmaf(f0, cr, -(f1 * sr));
                            f1 = __builtin_fmaf(f1, cr, f0 * sr);
                            f0 = g0;
                        }
                        two[p] = pk_bf16(f0, f1);
                    }
                    const uint32_t off = (uint32_t)((((size_t)b * XT_NH + head0 + hh) * XT_TP + t) * XT_HD + 4 * c16) * 2u;
                    typedef unsigned v2u __attribute__((ext_vector_type(2)));
                    __builtin_amdgcn_raw_buffer_store_b64(v2u{two[0], two[1]}, rd, (int)off, 0, 0);
                }
            }
        return;
    }
    // v (dense tile): rows 16 i + 4 g + r of dim 16 j + c16 are four consecutive tokens of one slice row
#pragma unroll
    for (int i = 0; i < C::TM; i++)
#pragma unroll
        for (int j = 0; j < C::TN; j++) {
            typedef unsigned v2u __attribute__((ext_vector_type(2)));
            *(v2u *)(tr + (16 * j + c16) * TRLD + 16 * i + 4 * g) =
                v2u{pk_bf16(acc[i][j][0], acc[i][j][1]), pk_bf16(acc[i][j][2], acc[i][j][3])};
        }
    v_out();
}

// ---------------------------------------------------------------------------------------------------------------
// k_oproj: x [rows][1024] = f16(x + attn_out . Wo^T) (eva_kernels.cu:150-160, alpha folded into the block scales)
// ---------------------------------------------------------------------------------------------------------------
template <class C, bool SP>
__global__ void __launch_bounds__(C::NT) k_oproj(const uint8_t *__restrict__ a8, const float *__restrict__ as,
                                                       int lds, const uint8_t *__restrict__ w,
                                                       const uint32_t *__restrict__ wx,
                                                       const float *__restrict__ ws, uint16_t *__restrict__ x, int rows)
{
    __shared__ __attribute__((aligned(16))) uint8_t smem[LayerMem<C>::SMEM];
    v4f acc[C::TM][C::TN];
    int m0, n0, wm0, wn0;
    layer_tile<C>(rows, XT_D, m0, n0);
    args_resident(x, lds, rows);
    // the transposed tile (sparse: as the sparse main loop leaves it; dense: TR) goes straight into the residual update
    if constexpr (SP) {
        v4f accT[C::TN][C::TM];
        bs_mainloop_sp_t<C>(a8, XT_D, as, lds, w, wx, ws, rows, XT_D, XT_D, m0, n0, smem, accT);
        bs_wave_origin<C>(wm0, wn0);
        residual_add_t<C>(smem, [&](int jn, int im) { return accT[jn][im]; }, x, m0 + wm0, n0 + wn0, rows);
    } else {
        layer_mainloop<C, SP, BsNoPre, true>(a8, XT_D, as, lds, w, wx, ws, rows, XT_D, XT_D, m0, n0, smem, acc);
        bs_wave_origin<C>(wm0, wn0);
        residual_add_t<C>(smem, [&](int jn, int im) { return acc[im][jn]; }, x, m0 + wm0, n0 + wn0, rows);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// k_fc1: h8 [rows][1024] x W12 [5632][1024] -> SwiGLU h = silu(g) x (silu(g) = g / (1 + e^-g), the quotient by the
// hardware reciprocal, within 1 ulp), packed to
// m8 [rows][2816] E4M3 with 1x128 scales ms [22][lds], and per-(row, block) (sum h, sum h^2) of the unpacked h in
// stat [22][lds][2] for the folded MLP LayerNorm (eva_kernels.cu:211-279). W12 rows hold g and x of 16 units in
// alternate 16-row chunks (export_eva.py:60-62), so column tile 2c is g and 2c+1 is x of the same 16 units: a
// 256-column block is one 128-unit block of h; its rows are staged in LDS, where 8 threads per row take the |max|
// and the sums.
// Each (row, block) partial has one writer: no atomics, deterministic.
// ---------------------------------------------------------------------------------------------------------------
template <class C, bool SP, bool RS>
__global__ void __launch_bounds__(C::NT) k_fc1(const uint8_t *__restrict__ h8, const float *__restrict__ hs,
                                                     int lds, const uint8_t *__restrict__ w,
                                                     const uint32_t *__restrict__ wx,
                                                     const float *__restrict__ ws, uint8_t *__restrict__ m8,
                                                     float *__restrict__ ms, float *__restrict__ stat,
                                                     const float *__restrict__ rs, int rows)
{
    constexpr int NP = C::TN / 2;                        // SwiGLU tile pairs per wave (16 units each)
    __shared__ __attribute__((aligned(16))) uint8_t smem[LayerMem<C>::SMEM];
    static_assert(C::BN == 256 && C::BM * 8 % C::NT == 0, "packing items split evenly over the threads");
    int m0, n0, wm0, wn0;
    layer_tile<C>(rows, 2 * XT_HIDP, m0, n0);
    args_resident(m8, ms, stat, lds, rows);
    if constexpr (RS) args_resident(rs);
    // W12 rows past the last 16-unit chunk holding a real unit (2 x 2736) are zero padding
    constexpr int nlive = 2 * ((XT_HID + 15) / 16 * 16);
    // h tile [BM rows][128 units] fp32 in LDS, 16-byte chunk c of row r at chunk c ^ (r & 7)
    float *ht = (float *)smem;
    static_assert(C::BM * 128 * 4 <= LayerMem<C>::SMEM, "fc1 staging fits");
    static_assert(NP == 4 || NP == 2, "64 or 32 units per wave");
    const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const int ct = n0 >> 8;
    // silu(g) x, hardware reciprocal (1 ulp)
    auto swiglu = [](float gg, float xx) { return (gg * __builtin_amdgcn_rcpf(1.0f + __expf(-gg))) * xx; };
    // The transposed tile (sparse: as the sparse main loop leaves it; dense: TR): lane (g, c16) holds units
    // wn0 / 2 + 16 p + 4 g + r (r = 0..3) of row wm0 + 16 i + c16 for tile pair p (gate tile 2p, value tile 2p + 1: the
    // same unit in the same register), so each (i, p) is one 16-byte chunk, wn0 / 8 + 8 (p >> 1) + (4 (p & 1) + g), of a
    // row with row & 7 = c16 & 7: at tb[p & 1] + 2048 i + 32 (p >> 1) words.
    auto stage_h = [&](auto pair) {
        bs_wave_origin<C>(wm0, wn0);
        uint32_t tb[2];
#pragma unroll
        for (int ph = 0; ph < 2; ph++)
            tb[ph] = (uint32_t)((wm0 + c16) * 128 + (wn0 / 8 + ((4 * ph + g) ^ (c16 & 7))) * 4);
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
            for (int p = 0; p < NP; p++) {
                v4f gg, xx;
                pair(i, p, gg, xx);
                *(float4 *)(ht + tb[p & 1] + 2048 * i + 32 * (p >> 1)) =
                    make_float4(swiglu(gg[0], xx[0]), swiglu(gg[1], xx[1]), swiglu(gg[2], xx[2]), swiglu(gg[3], xx[3]));
            }
    };
    if constexpr (SP) {
        v4f accT[C::TN][C::TM];
        bs_mainloop_sp_t<C>(h8, XT_D, hs, lds, w, wx, ws, rows, 2 * XT_HIDP, XT_D, m0, n0, smem, accT, BsNoPre(),
                            nlive);
        stage_h([&](int i, int p, v4f &gg, v4f &xx) { gg = accT[2 * p][i]; xx = accT[2 * p + 1][i]; });
    } else {
        v4f acc[C::TM][C::TN];
        layer_mainloop<C, SP, BsNoPre, true>(h8, XT_D, hs, lds, w, wx, ws, rows, 2 * XT_HIDP, XT_D, m0, n0, smem, acc,
                                             BsNoPre(), nlive);
        stage_h([&](int i, int p, v4f &gg, v4f &xx) { gg = acc[i][2 * p]; xx = acc[i][2 * p + 1]; });
    }
    __syncthreads();
    // 8 consecutive threads per row, 16 consecutive units each: the row's |max| and sums over its 128 units meet in
    // a DPP tree over the 8 lanes; each thread packs its 16 units to E4M3 (one 16-byte store) and the first thread
    // of the row writes the block scale and the partial sums. Item it of a thread reads row
    // (tid >> 3) + 64 it, whose row & 7 does not depend on it: the four chunk addresses are bases plus 8192 it words.
    const __amdgpu_buffer_rsrc_t rm = buf_rsrc(m8, (uint32_t)rows * XT_HIDP);
    const int k8 = threadIdx.x & 7, r0 = threadIdx.x >> 3;
    uint32_t rb[4];
#pragma unroll
    for (int c = 0; c < 4; c++) rb[c] = (uint32_t)(r0 * 128 + ((((4 * k8 + c) ^ r0) & 7) | ((4 * k8 + c) & ~7)) * 4);
    float4 ru[4];  // RS: the per-unit multipliers of this thread's 16 units (the same units in every item)
    if constexpr (RS) {
#pragma unroll
        for (int c = 0; c < 4; c++) ru[c] = *(const float4 *)(rs + ct * 128 + 16 * k8 + 4 * c);
    }
#pragma unroll
    for (int it = 0; it < C::BM * 8 / C::NT; it++) {
        const int idx = threadIdx.x + it * C::NT, rr = idx >> 3, u0 = (idx & 7) * 16, m = m0 + rr;
        float4 v[4];
#pragma unroll
        for (int c = 0; c < 4; c++) v[c] = *(const float4 *)(ht + rb[c] + 128 * (C::NT / 8) * it);
        float amax = 0.f, s = 0.f, q = 0.f;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            s += (v[c].x + v[c].y) + (v[c].z + v[c].w);
            q = __builtin_fmaf(v[c].x, v[c].x, q);
            q = __builtin_fmaf(v[c].y, v[c].y, q);
            q = __builtin_fmaf(v[c].z, v[c].z, q);
            q = __builtin_fmaf(v[c].w, v[c].w, q);
            if constexpr (RS) {  // the sums are over h itself, the packed operand is h rs (eva_kernels.cu:258-264)
                v[c].x *= ru[c].x;
                v[c].y *= ru[c].y;
                v[c].z *= ru[c].z;
                v[c].w *= ru[c].w;
            }
            amax = __builtin_fmaxf(__builtin_fmaxf(amax, __builtin_fabsf(v[c].x)), __builtin_fabsf(v[c].y));  // v_max3
            amax = __builtin_fmaxf(__builtin_fmaxf(amax, __builtin_fabsf(v[c].z)), __builtin_fabsf(v[c].w));
        }
        amax = row8_absmax(amax);
        s = row8_sum(s);
        q = row8_sum(q);
        const float sc = block_scale(amax), inv = block_scale_inv(sc);
        uint32_t w4[4];
#pragma unroll
        for (int c = 0; c < 4; c++) w4[c] = e4_pack4_scaled(v[c].x * inv, v[c].y * inv, v[c].z * inv, v[c].w * inv);
        const v4u o = {w4[0], w4[1], w4[2], w4[3]};
        __builtin_amdgcn_raw_buffer_store_b128(o, rm, (int)((uint32_t)m * XT_HIDP + ct * 128 + u0), 0, 0);
        if ((idx & 7) == 0 && m < rows) {
            ms[(size_t)ct * lds + m] = sc;
            *(float2 *)(stat + ((size_t)ct * lds + m) * 2) = make_float2(s, q);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// k_fc2: x = f16(x + rstd (acc - mean c) + d) with acc = m8 . W~^T (W~ = W2 diag(gamma), c = W~ 1 from the packed
// W~, d = W2 beta), mean / rstd of the SwiGLU row over 2730 units from k_fc1's 22 partials summed in block order:
// mean = S / 2730, var = max(Q / 2730 - mean^2, 0), rstd = 1 / sqrt(var + 1e-6) (eva_kernels.cu:300-333).
// ---------------------------------------------------------------------------------------------------------------
template <class C, bool SP>
__global__ void __launch_bounds__(C::NT) k_fc2(const uint8_t *__restrict__ m8, const float *__restrict__ ms,
                                                     int lds, const uint8_t *__restrict__ w,
                                                     const uint32_t *__restrict__ wx,
                                                     const float *__restrict__ ws, const float *__restrict__ stat,
                                                     const float *__restrict__ cn, const float *__restrict__ dn,
                                                     uint16_t *__restrict__ x, int rows)
{
    using S = LayerMem<C>;
    __shared__ __attribute__((aligned(16))) uint8_t smem[S::SMEM];
    v4f acc[C::TM][C::TN];
    int m0, n0, wm0, wn0;
    layer_tile<C>(rows, XT_D, m0, n0);
    float2 *rs = (float2 *)(smem + S::ROWSTAT);              // [BM rows] (rstd, -mean * rstd)
    float2 *cd = (float2 *)(smem + S::ROWSTAT + 8 * C::BM);  // [BN columns] (c, d)
    auto rowstats = [&]() {
        if (threadIdx.x < C::BM) {
            const int m = m0 + threadIdx.x;
            float2 p[XT_HIDP / 128];
#pragma unroll
            for (int blk = 0; blk < XT_HIDP / 128; blk++)
                p[blk] = m < rows ? *(const float2 *)(stat + ((size_t)blk * lds + m) * 2) : make_float2(0.f, 0.f);
            float S = 0.f, Q = 0.f;
#pragma unroll
            for (int blk = 0; blk < XT_HIDP / 128; blk++) {
                S += p[blk].x;
                Q += p[blk].y;
            }
            const float mean = S / (float)XT_HID;
            float var = Q / (float)XT_HID - mean * mean;
            var = __builtin_fmaxf(var, 0.f);
            const float rstd = 1.0f / __builtin_sqrtf(var + XT_EPS);
            rs[threadIdx.x] = make_float2(rstd, -mean * rstd);
        } else if (threadIdx.x < C::BM + C::BN) {
            const int n = n0 + threadIdx.x - C::BM;
            cd[threadIdx.x - C::BM] = make_float2(cn[n], dn[n]);
        }
    };
    args_resident(x, stat, cn, dn, lds, rows);
    static_assert(C::BM + C::BN <= C::NT, "one thread per row statistic and per column term");
    const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    // The transposed tile (sparse: as the sparse main loop leaves it; dense: TR): lane (g, c16) holds row
    // wm0 + 16 im + c16 (one row statistic per m tile) and columns wn0 + 16 jn + 4 g + r (four column terms, 32 bytes
    // of cd, per n tile). The fold is applied as the residual update parks the tile.
    float2 st[C::TM];
    auto fold = [&](v4f v, int jn, int im) {
        const float4 *cq = (const float4 *)(cd + wn0 + 16 * jn + 4 * g);
        const float4 c01 = cq[0], c23 = cq[1];  // (c, d) of columns 4 g + 0 .. 3
        v[0] = __builtin_fmaf(st[im].x, v[0], __builtin_fmaf(st[im].y, c01.x, c01.y));
        v[1] = __builtin_fmaf(st[im].x, v[1], __builtin_fmaf(st[im].y, c01.z, c01.w));
        v[2] = __builtin_fmaf(st[im].x, v[2], __builtin_fmaf(st[im].y, c23.x, c23.y));
        v[3] = __builtin_fmaf(st[im].x, v[3], __builtin_fmaf(st[im].y, c23.z, c23.w));
        return v;
    };
    if constexpr (SP) {
        v4f accT[C::TN][C::TM];
        bs_mainloop_sp_t<C>(m8, XT_HIDP, ms, lds, w, wx, ws, rows, XT_D, XT_HIDP, m0, n0, smem, accT, rowstats);
        bs_wave_origin<C>(wm0, wn0);
#pragma unroll
        for (int im = 0; im < C::TM; im++) st[im] = rs[wm0 + 16 * im + c16];
        residual_add_t<C>(smem, [&](int jn, int im) { return fold(accT[jn][im], jn, im); }, x, m0 + wm0, n0 + wn0,
                          rows);
    } else {
        layer_mainloop<C, SP, decltype(rowstats), true>(m8, XT_HIDP, ms, lds, w, wx, ws, rows, XT_D, XT_HIDP, m0, n0,
                                                       smem, acc, rowstats);
        bs_wave_origin<C>(wm0, wn0);
#pragma unroll
        for (int im = 0; im < C::TM; im++) st[im] = rs[wm0 + 16 * im + c16];
        residual_add_t<C>(smem, [&](int jn, int im) { return fold(acc[im][jn], jn, im); }, x, m0 + wm0, n0 + wn0,
                          rows);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// k_head: out [nb][nt] = sigmoid(hb[n] + sum_kb ps[kb][m] hs[kb][n] sum_{k in kb} pq[m][k] hq[n][k])
// (kern_common.cuh:679-727 k_headmv, here an FP8 GEMM). The head rows carry 1x128 scales of their own (planes
// hs [8][ldh], as activations do), so every row is packed, and repacked by eva_head_put, independently of all others.
// The head is a weight stream (nt x 1 KB) against at most 128 input rows: one block per 64 output columns and 64 rows,
// 4 waves, wave w owning columns n0 + 16 w .. + 15. A wave issues the loads of all eight K blocks' weight fragments
// and scales before its first matrix instruction (one memory round trip for the stream instead of eight), then runs
// only the row tiles of 16 that hold input rows (a batch of 16 runs one of the four). Fragments come straight from L2
// into registers; descriptors that end at row nb of pq and row nt of hq load zero past them. Each output's K blocks
// are promoted in order, so a row's scores do not depend on the batch around it.
// ---------------------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_head(const uint8_t *__restrict__ pq, const float *__restrict__ ps, int lds,
                                              const uint8_t *__restrict__ hq, const float *__restrict__ hs, int ldh,
                                              const float *__restrict__ hb, float *__restrict__ out, int nb, int nt)
{
    constexpr int KB = XT_D / 128;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const int n0 = blockIdx.x * 64 + 16 * w, m0 = blockIdx.y * 64;
    const __amdgpu_buffer_rsrc_t ra = buf_rsrc(pq, (uint32_t)nb * XT_D), rw = buf_rsrc(hq, (uint32_t)nt * XT_D);
    const int nl = n0 + c16;                                  // weight row of this lane's B fragment, output column
    const int ncl = nl < nt ? nl : nt - 1;                    // clamped for the scale and bias reads
    v8i b[KB];
    float swv[KB];
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
        const uint32_t ko = (uint32_t)kb * 128u + 16u * g;
        const v4u blo = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)((uint32_t)nl * XT_D + ko), 0, 0);
        const v4u bhi = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)((uint32_t)nl * XT_D + ko + 64u), 0, 0);
        b[kb] = v8i{(int)blo[0], (int)blo[1], (int)blo[2], (int)blo[3], (int)bhi[0], (int)bhi[1], (int)bhi[2], (int)bhi[3]};
        swv[kb] = hs[(size_t)kb * ldh + ncl];
    }
    const int ntile = (nb - m0 + 15) >> 4;                    // row tiles holding input rows (block-uniform, >= 1)
    const float bias = hb[ncl];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (i >= ntile) break;
        v8i a[KB];
        float sa[KB][4];
        const uint32_t ar = (uint32_t)(m0 + 16 * i + c16) * XT_D;
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
            const uint32_t ko = (uint32_t)kb * 128u + 16u * g;
            const v4u alo = __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(ar + ko), 0, 0);
            const v4u ahi = __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(ar + ko + 64u), 0, 0);
            a[kb] = v8i{(int)alo[0], (int)alo[1], (int)alo[2], (int)alo[3], (int)ahi[0], (int)ahi[1], (int)ahi[2], (int)ahi[3]};
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + 16 * i + 4 * g + r;
                sa[kb][r] = m < nb ? ps[(size_t)kb * lds + m] : 0.f;
            }
        }
        v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
            const v4f p = mfma_e4m3_16x16x128(a[kb], b[kb]);
#pragma unroll
            for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(p[r], sa[kb][r] * swv[kb], acc[r]);
        }
        if (nl < nt)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + 16 * i + 4 * g + r;
                if (m < nb) out[(size_t)m * nt + nl] = 1.0f / (1.0f + __expf(-(acc[r] + bias)));
            }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// k_pe: patch embedding in fp16 with fp32 accumulation (v_mfma_f32_16x16x32_f16) and the position add fused
// (k_pe + k_embed, eva_kernels.cu:21-33, 126-130): x[1025 b + 1 + p] = f16(in[1024 b + p] . pe^T + pos[1 + p]),
// x[1025 b] = f16(pos[0]) (pos carries cls and the conv bias, export_eva.py:76-80). K = 592 in steps of 64 halves:
// rows of 128 bytes, as the E4M3 operands of the layer GEMMs, brought into LDS the same way (16-byte chunk c of row r
// at (c + r) & 7, C::NS stages, counted waits); the last step holds 16 halves, and the lanes whose chunk lies past
// them load an out-of-range offset (zero). The tile is transposed (weights as the MFMA's A operand), parked in the
// wave's slice of shared memory and leaves as whole 128-byte rows. Tile sizes: with_pe_cfg.
// PX: the PixAI patch GEMM (px_kernels.cu:133-138 k_ppe) instead: x[m] = f16(in[m] . pe^T) for window-major token rows
// m (no cls, no position: k_px_pembed adds it before its LayerNorm), rows a multiple of 128.
// ---------------------------------------------------------------------------------------------------------------
template <class C, bool PX>
__global__ void __launch_bounds__(C::NT) k_pe(const uint16_t *__restrict__ in, const uint16_t *__restrict__ pe,
                                              const float *__restrict__ pos, uint16_t *__restrict__ x, int rows)
{
    using S = LayerMem<C>;
    constexpr int STAGE = C::A_BYTES + C::B_BYTES, KB = (XT_K0P + 63) / 64, LPS = C::LA + C::LB;
    constexpr int LAST = XT_K0P % 64 / 8;  // 16-byte chunks of the last K step
    constexpr uint32_t LDB = XT_K0P * 2;
    constexpr int SLICES = C::NW * S::SLICE;
    static_assert(LAST > 0 && C::BM <= 128, "a partial last step; row tiles divide the 128-row granule of every caller");
    __shared__ __attribute__((aligned(16))) uint8_t smem[SLICES > C::NS * STAGE ? SLICES : C::NS * STAGE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int m0, n0, wm0, wn0;
    layer_tile<C>(rows, XT_D, m0, n0);  // XCD-aware: an XCD's blocks share their rows of `in` in its L2
    bs_wave_origin<C>(wm0, wn0);
    args_resident(pos, x);
    const v4i ra = buf_desc(in + (size_t)m0 * XT_K0P, C::BM * LDB), rb = buf_desc(pe + (size_t)n0 * XT_K0P, C::BN * LDB);
    const uint32_t base = lds_addr(smem);
    uint32_t off[LPS];
    bool tail[LPS];  // this lane's chunk lies past the last step's
#pragma unroll
    for (int i = 0; i < LPS; i++) {
        const int rl = 8 * (i < C::LA ? w * C::LA + i : w * C::LB + i - C::LA) + (lane >> 3), ch = ((lane & 7) - rl) & 7;
        off[i] = (uint32_t)rl * LDB + 16u * ch;
        tail[i] = ch >= LAST;
    }
    auto issue = [&](int stage, int kb) {
        const uint32_t st = base + (uint32_t)stage * STAGE;
#pragma unroll
        for (int i = 0; i < LPS; i++) {
            const uint32_t o = kb == KB - 1 && tail[i] ? XT_OOR : off[i];
            if (i < C::LA) dma16(ra, st + 1024u * (w * C::LA + i), o, (uint32_t)kb * 128u);
            else dma16(rb, st + C::A_BYTES + 1024u * (w * C::LB + i - C::LA), o, (uint32_t)kb * 128u);
        }
    };
    v4f acc[C::TM][C::TN];
#pragma unroll
    for (int i = 0; i < C::TM; i++)
#pragma unroll
        for (int j = 0; j < C::TN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    static_assert(C::NS - 1 <= KB, "the prologue issues whole steps");
#pragma unroll
    for (int k = 0; k < C::NS - 1; k++) issue(k, k);
    int cs = 0, is = C::NS - 1;
    for (int kb = 0; kb < KB; kb++) {
        wait_stages<C::NS - 2, LPS>(KB - 1 - kb);
        lds_barrier();
        if (kb + C::NS - 1 < KB) issue(is, kb + C::NS - 1);
        const uint8_t *ta = smem + cs * STAGE, *tb = ta + C::A_BYTES;
        typedef int v4w __attribute__((ext_vector_type(4)));
        v8i a[C::TM];
#pragma unroll
        for (int i = 0; i < C::TM; i++) a[i] = ld_frag(ta, wm0 + 16 * i);
#pragma unroll
        for (int j = 0; j < C::TN; j++) {
            const v8i b = ld_frag(tb, wn0 + 16 * j);
            const v8h blo = __builtin_bit_cast(v8h, v4w{b[0], b[1], b[2], b[3]});
            const v8h bhi = __builtin_bit_cast(v8h, v4w{b[4], b[5], b[6], b[7]});
#pragma unroll
            for (int i = 0; i < C::TM; i++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    blo, __builtin_bit_cast(v8h, v4w{a[i][0], a[i][1], a[i][2], a[i][3]}), acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < C::TM; i++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    bhi, __builtin_bit_cast(v8h, v4w{a[i][4], a[i][5], a[i][6], a[i][7]}), acc[i][j], 0, 0, 0);
        }
        cs = cs == C::NS - 1 ? 0 : cs + 1;
        is = is == C::NS - 1 ? 0 : is + 1;
    }
    lds_barrier();
    // acc[i][j][r]: row wm0 + 16 i + (lane & 15), column wn0 + 16 j + 4 (lane >> 4) + r
    constexpr int NP = C::WN / S::PC, LPR = S::PC / 8, RPI = 64 / LPR, NI = C::WM / RPI;  // lanes a row, rows a store
    float *tr = (float *)(smem + w * S::SLICE);
    const int g = lane >> 4, c16 = lane & 15, rs = lane / LPR, ch = lane % LPR;
#pragma unroll
    for (int pass = 0; pass < NP; pass++) {
        const int n = n0 + wn0 + S::PC * pass + 8 * ch;
        if (pass) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the previous pass's slice reads are done
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
            for (int jq = 0; jq < S::PC / 16; jq++) {
                const v4f v = acc[i][S::PC / 16 * pass + jq];
                *(float4 *)(tr + (16 * i + c16) * S::LD + 16 * jq + 4 * g) = make_float4(v[0], v[1], v[2], v[3]);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slice is the wave's own: no block barrier needed
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const int rr = RPI * it + rs, m = m0 + wm0 + rr;
            float4 a = *(const float4 *)(tr + rr * S::LD + 8 * ch), b = *(const float4 *)(tr + rr * S::LD + 8 * ch + 4);
            size_t row = m;
            if constexpr (!PX) {
                const int img = m >> 10, p = m & 1023;
                row = (size_t)img * XT_T + 1 + p;
                const float *pr = pos + (size_t)(1 + p) * XT_D + n;
                const v4f_e pa = *(const v4f_e *)pr, pb = *(const v4f_e *)(pr + 4);
                a = make_float4(a.x + pa[0], a.y + pa[1], a.z + pa[2], a.w + pa[3]);
                b = make_float4(b.x + pb[0], b.y + pb[1], b.z + pb[2], b.w + pb[3]);
            }
            *(v4u_e *)(x + row * XT_D + n) = v4u_e{pk_f16(a.x, a.y), pk_f16(a.z, a.w), pk_f16(b.x, b.y), pk_f16(b.z, b.w)};
        }
    }
    if constexpr (!PX)
        if ((m0 & 1023) == 0 && threadIdx.x < C::BN) {  // the first patch tile of an image also writes its cls row
            const int n = n0 + threadIdx.x;
            x[(size_t)(m0 >> 10) * XT_T * XT_D + n] = f2h(pos[n]);
        }
}

// ---------------------------------------------------------------------------------------------------------------
// C-ABI launchers
// ---------------------------------------------------------------------------------------------------------------
// qkv's tiles: 128 x 128 while one round of two blocks per CU holds them (rows <= 2688: 17.2 -> 8.4 us at 1025 rows,
// 18.5 -> 12.7 at 2050), and where 256 x 256 tiles would run a second round less than a quarter full (6150 rows: 34.3
// -> 30.0 us; not beside an engine's other lane, which takes the CUs of that round: 6725 -> 6950 us a batch of 12
// images); 256 x 256 elsewhere (20.6 against 22.1 us at 4100, 34.8 against 38.8 at 8200).
template <class F>
static void with_qkv_cfg(int rows, int lanes, F f)
{
    const unsigned big = layer_grid<LayerCfg>(rows, 3 * XT_D);
    if (rows <= 2688 || (lanes == 1 && big > 256 && big <= 320)) f(LayerMid{});
    else f(LayerCfg{});
}

// fc1's tiles (a block holds all 256 columns of a 128-unit scale block): 128 x 256, 16 waves of 32 x 64, while they
// fit the 256 CUs at once (rows <= 1408: 16.6 -> 10.2 us at 1025 rows); beyond that 256 x 256 (18.0 against 19.2 us at
// 2050 rows, 50.4 against 58.3 at 8200).
typedef BsCfg<128, 256, 4, 4, 3> Fc1Mid;
template <class F>
static void with_fc1_cfg(int rows, F f)
{
    if (rows <= 1408) f(Fc1Mid{});
    else f(LayerCfg{});
}

template <bool SP>
static int qkv_launch(const char *what, const void *h8, const float *hs, int lds, const void *w, const void *wx,
                      const float *ws, const float *cs, void *q, void *k, void *vt, int rows, int lanes, void *stream)
{
    if (layer_rows_ok(what, rows, lds)) return -1;
    if (rows % XT_T) return xt_fail(what, "rows must be nb * 1025");
    if (!XT_ALIGNED(h8) || !XT_ALIGNED(w) || (SP && !wx)) return xt_fail(what, "h8 and w must be 16-byte aligned");
    with_qkv_cfg(rows, lanes, [&](auto c) {
        using C = decltype(c);
        hipLaunchKernelGGL((k_qkv<C, SP>), dim3(layer_grid<C>(rows, 3 * XT_D)), dim3(C::NT), 0, (hipStream_t)stream,
                           (const uint8_t *)h8, hs, lds, (const uint8_t *)w, (const uint32_t *)wx, ws, cs,
                           (uint16_t *)q, (uint16_t *)k, (uint16_t *)vt, rows);
    });
    return xt_check(what);
}

template <bool SP>
static int oproj_launch(const char *what, const void *a8, const float *as, int lds, const void *w, const void *wx,
                        const float *ws, void *x, int rows, int lanes, void *stream)
{
    if (layer_rows_ok(what, rows, lds)) return -1;
    if (!XT_ALIGNED(a8) || !XT_ALIGNED(w) || (SP && !wx)) return xt_fail(what, "a8 and w must be 16-byte aligned");
    with_res_cfg(rows, XT_D, lanes, [&](auto c) {
        using C = decltype(c);
        hipLaunchKernelGGL((k_oproj<C, SP>), dim3(layer_grid<C>(rows, XT_D)), dim3(C::NT), 0, (hipStream_t)stream,
                           (const uint8_t *)a8, as, lds, (const uint8_t *)w, (const uint32_t *)wx, ws, (uint16_t *)x,
                           rows);
    });
    return xt_check(what);
}

template <bool SP>
static int fc1_launch(const char *what, const void *h8, const float *hs, int lds, const void *w, const void *wx,
                      const float *ws, void *m8, float *ms, float *stat, const float *rs, int rows, void *stream)
{
    if (layer_rows_ok(what, rows, lds)) return -1;
    if (!XT_ALIGNED(h8) || !XT_ALIGNED(w) || !XT_ALIGNED(m8) || !XT_ALIGNED(rs) || (SP && !wx))
        return xt_fail(what, "h8, w, m8, rs must be 16-byte aligned");
    with_fc1_cfg(rows, [&](auto c) {
        using C = decltype(c);
        const dim3 grid(layer_grid<C>(rows, 2 * XT_HIDP));
        if (rs)
            hipLaunchKernelGGL((k_fc1<C, SP, true>), grid, dim3(C::NT), 0, (hipStream_t)stream, (const uint8_t *)h8, hs,
                               lds, (const uint8_t *)w, (const uint32_t *)wx, ws, (uint8_t *)m8, ms, stat, rs, rows);
        else
            hipLaunchKernelGGL((k_fc1<C, SP, false>), grid, dim3(C::NT), 0, (hipStream_t)stream, (const uint8_t *)h8,
                               hs, lds, (const uint8_t *)w, (const uint32_t *)wx, ws, (uint8_t *)m8, ms, stat, rs, rows);
    });
    return xt_check(what);
}

template <bool SP>
static int fc2_launch(const char *what, const void *m8, const float *ms, int lds, const void *w, const void *wx,
                      const float *ws, const float *stat, const float *cn, const float *dn, void *x, int rows,
                      int lanes, void *stream)
{
    if (layer_rows_ok(what, rows, lds)) return -1;
    if (!XT_ALIGNED(m8) || !XT_ALIGNED(w) || (SP && !wx)) return xt_fail(what, "m8 and w must be 16-byte aligned");
    with_res_cfg(rows, XT_HIDP, lanes, [&](auto c) {
        using C = decltype(c);
        hipLaunchKernelGGL((k_fc2<C, SP>), dim3(layer_grid<C>(rows, XT_D)), dim3(C::NT), 0, (hipStream_t)stream,
                           (const uint8_t *)m8, ms, lds, (const uint8_t *)w, (const uint32_t *)wx, ws, stat, cn, dn,
                           (uint16_t *)x, rows);
    });
    return xt_check(what);
}

int xt_qkv(const void *h8, const float *hs, int lds, const void *w, const void *wx, const float *ws, const float *cs,
           void *q, void *k, void *vt, int rows, int lanes, void *stream)
{
    return wx ? qkv_launch<true>("eva_k_qkv_sp", h8, hs, lds, w, wx, ws, cs, q, k, vt, rows, lanes, stream)
              : qkv_launch<false>("eva_k_qkv", h8, hs, lds, w, wx, ws, cs, q, k, vt, rows, lanes, stream);
}

int xt_oproj(const void *a8, const float *as, int lds, const void *w, const void *wx, const float *ws, void *x, int rows,
             int lanes, void *stream)
{
    return wx ? oproj_launch<true>("eva_k_oproj_sp", a8, as, lds, w, wx, ws, x, rows, lanes, stream)
              : oproj_launch<false>("eva_k_oproj", a8, as, lds, w, wx, ws, x, rows, lanes, stream);
}

int xt_fc2(const void *m8, const float *ms, int lds, const void *w, const void *wx, const float *ws, const float *stat,
           const float *cn, const float *dn, void *x, int rows, int lanes, void *stream)
{
    return wx ? fc2_launch<true>("eva_k_fc2_sp", m8, ms, lds, w, wx, ws, stat, cn, dn, x, rows, lanes, stream)
              : fc2_launch<false>("eva_k_fc2", m8, ms, lds, w, wx, ws, stat, cn, dn, x, rows, lanes, stream);
}

extern "C" int eva_k_qkv(const void *h8, const float *hs, int lds, const void *w, const float *ws, const float *cs,
                         void *q, void *k, void *vt, int rows, void *stream)
{
    return qkv_launch<false>("eva_k_qkv", h8, hs, lds, w, nullptr, ws, cs, q, k, vt, rows, 1, stream);
}

extern "C" int eva_k_oproj(const void *a8, const float *as, int lds, const void *w, const float *ws, void *x, int rows,
                           void *stream)
{
    return oproj_launch<false>("eva_k_oproj", a8, as, lds, w, nullptr, ws, x, rows, 1, stream);
}

extern "C" int eva_k_fc1(const void *h8, const float *hs, int lds, const void *w, const float *ws, void *m8, float *ms,
                         float *stat, int rows, void *stream)
{
    return fc1_launch<false>("eva_k_fc1", h8, hs, lds, w, nullptr, ws, m8, ms, stat, nullptr, rows, stream);
}

extern "C" int eva_k_fc1_rs(const void *h8, const float *hs, int lds, const void *w, const float *ws, void *m8,
                            float *ms, float *stat, const float *rs, int rows, void *stream)
{
    if (!rs) return xt_fail("eva_k_fc1_rs", "rs must not be NULL");
    return fc1_launch<false>("eva_k_fc1_rs", h8, hs, lds, w, nullptr, ws, m8, ms, stat, rs, rows, stream);
}

extern "C" int eva_k_fc2(const void *m8, const float *ms, int lds, const void *w, const float *ws, const float *stat,
                         const float *cn, const float *dn, void *x, int rows, void *stream)
{
    return fc2_launch<false>("eva_k_fc2", m8, ms, lds, w, nullptr, ws, stat, cn, dn, x, rows, 1, stream);
}

extern "C" int eva_k_qkv_sp(const void *h8, const float *hs, int lds, const void *vals, const void *idx,
                            const float *ws, const float *cs, void *q, void *k, void *vt, int rows, void *stream)
{
    return qkv_launch<true>("eva_k_qkv_sp", h8, hs, lds, vals, idx, ws, cs, q, k, vt, rows, 1, stream);
}

extern "C" int eva_k_oproj_sp(const void *a8, const float *as, int lds, const void *vals, const void *idx,
                              const float *ws, void *x, int rows, void *stream)
{
    return oproj_launch<true>("eva_k_oproj_sp", a8, as, lds, vals, idx, ws, x, rows, 1, stream);
}

extern "C" int eva_k_fc1_sp(const void *h8, const float *hs, int lds, const void *vals, const void *idx,
                            const float *ws, void *m8, float *ms, float *stat, int rows, void *stream)
{
    return fc1_launch<true>("eva_k_fc1_sp", h8, hs, lds, vals, idx, ws, m8, ms, stat, nullptr, rows, stream);
}

extern "C" int eva_k_fc1_rs_sp(const void *h8, const float *hs, int lds, const void *vals, const void *idx,
                               const float *ws, void *m8, float *ms, float *stat, const float *rs, int rows,
                               void *stream)
{
    if (!rs) return xt_fail("eva_k_fc1_rs_sp", "rs must not be NULL");
    return fc1_launch<true>("eva_k_fc1_rs_sp", h8, hs, lds, vals, idx, ws, m8, ms, stat, rs, rows, stream);
}

extern "C" int eva_k_fc2_sp(const void *m8, const float *ms, int lds, const void *vals, const void *idx,
                            const float *ws, const float *stat, const float *cn, const float *dn, void *x, int rows,
                            void *stream)
{
    return fc2_launch<true>("eva_k_fc2_sp", m8, ms, lds, vals, idx, ws, stat, cn, dn, x, rows, 1, stream);
}

extern "C" int eva_k_head(const void *pq, const float *ps, int lds, const void *w, const float *ws, int ldw,
                          const float *hb, float *out, int nb, int nt, void *stream)
{
    if (nb <= 0 || nt <= 0 || lds < nb || ldw < nt || nb > EVA_NBMAX || nt > (1 << 20))
        return xt_fail("eva_k_head", "bad shape (0 < nb <= 128, 0 < nt <= 2^20, lds >= nb, ldw >= nt)");
    if (!XT_ALIGNED(pq) || !XT_ALIGNED(w)) return xt_fail("eva_k_head", "pq and w must be 16-byte aligned");
    hipLaunchKernelGGL(k_head, dim3((nt + 63) / 64, (nb + 63) / 64), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t *)pq, ps, lds, (const uint8_t *)w, ws, ldw, hb, out, nb, nt);
    return xt_check("eva_k_head");
}

// k_pe's tiles: 64 x 64 for up to 2048 patches (256 blocks for one image: 15.7 -> 5.0 us against the register-staged
// 128 x 128 tiles of the version before, whose ten K steps each waited out a load; 128 x 128 tiles here 7.6), 128 x 128
// in 8 waves beyond (us, before -> now: 22.4 -> 12.0 at 4 images, 52 -> 36 at 16, 102 -> 68 at 32; 10368 PixAI patches
// 27.1 -> 22.2, 41472: 94 -> 74; 64 x 64: 13.6, 47.5, 89, 28.3, 101). Bound there by LDS reads (one 1 KB fragment per
// two matrix instructions) and the 2 B store and 4 B position read per output.
typedef BsCfg<64, 64, 2, 2, 3> PeSml;
template <class F>
static void with_pe_cfg(int rows, F f)
{
    if (rows <= 2048) f(PeSml{});
    else f(LayerMid{});
}

extern "C" int eva_k_pe(const void *in, const void *pe, const float *pos, void *x, int nb, void *stream)
{
    if (nb <= 0) return xt_fail("eva_k_pe", "nb must be positive");
    if (!XT_ALIGNED(in) || !XT_ALIGNED(pe)) return xt_fail("eva_k_pe", "in and pe must be 16-byte aligned");
    if (nb > (1 << 19)) return xt_fail("eva_k_pe", "at most 2^19 images");
    with_pe_cfg(nb * XT_NP, [&](auto c) {
        using C = decltype(c);
        hipLaunchKernelGGL((k_pe<C, false>), dim3(layer_grid<C>(nb * XT_NP, XT_D)), dim3(C::NT), 0, (hipStream_t)stream,
                           (const uint16_t *)in, (const uint16_t *)pe, pos, (uint16_t *)x, nb * XT_NP);
    });
    return xt_check("eva_k_pe");
}

extern "C" int px_k_pe(const void *in, const void *pe, void *x, int rows, void *stream)
{
    if (rows <= 0 || rows % 128) return xt_fail("px_k_pe", "rows must be a positive multiple of 128 (an even batch)");
    if (!XT_ALIGNED(in) || !XT_ALIGNED(pe)) return xt_fail("px_k_pe", "in and pe must be 16-byte aligned");
    with_pe_cfg(rows, [&](auto c) {
        using C = decltype(c);
        hipLaunchKernelGGL((k_pe<C, true>), dim3(layer_grid<C>(rows, XT_D)), dim3(C::NT), 0, (hipStream_t)stream,
                           (const uint16_t *)in, (const uint16_t *)pe, (const float *)nullptr, (uint16_t *)x, rows);
    });
    return xt_check("px_k_pe");
}
