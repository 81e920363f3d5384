// quant.hip - E4M3 packing with per-block fp32 scales (activations 1x128, weights 128x128) and the standalone
// block-scaled GEMM. Reference roles: q2 / st4 / st8h (src/engine/kern_common.cuh:97-128) for activations,
// fp8() (src/tools/export_eva.py:64-66) for weights, gemm8 (kern_common.cuh:271-356) for the GEMM.
#include <type_traits>

#include "layer_core.h"

// ---- activations: x [M][ldx] (bf16, fp32 or fp16) -> q [M][ldq] E4M3, s [K/128][lds] ----
// One thread per 8 consecutive elements; the 16 threads of one 128-element block are 16 aligned lanes.
template <typename TIn>
__device__ __forceinline__ void load8(const TIn *p, float *v);
template <>
__device__ __forceinline__ void load8<uint16_t>(const uint16_t *p, float *v)
{
    const uint4 u = *(const uint4 *)p;
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
template <>
__device__ __forceinline__ void load8<_Float16>(const _Float16 *p, float *v)
{
    const v8h h = *(const v8h *)p;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = (float)h[i];
}
template <>
__device__ __forceinline__ void load8<float>(const float *p, float *v)
{
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

template <typename TIn>
__global__ void __launch_bounds__(256) k_quant_act(const TIn *__restrict__ x, int ldx, int M, int K,
                                                   uint8_t *__restrict__ q, int ldq, float *__restrict__ s, int lds)
{
    const int cpr = K >> 3;  // 8-element chunks per row
    const long total = (long)M * cpr;
    for (long t = (long)blockIdx.x * 256 + threadIdx.x; t < total; t += (long)gridDim.x * 256) {
        // the 16 lanes of a block share every trip: total and the stride are multiples of 16
        const int row = (int)(t / cpr), ch = (int)(t - (long)row * cpr);
        float v[8], amax = 0.f;
        load8<TIn>(x + (size_t)row * ldx + ch * 8, v);
#pragma unroll
        for (int i = 0; i < 8; i++) amax = __builtin_fmaxf(amax, __builtin_fabsf(v[i]));
        amax = row16_absmax(amax);  // the 16 lanes of the block: one DPP row, all active together
        const float sc = block_scale(amax), inv = block_scale_inv(sc);
        uint2 o;
        o.x = e4_pack4_scaled(v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv);
        o.y = e4_pack4_scaled(v[4] * inv, v[5] * inv, v[6] * inv, v[7] * inv);
        *(uint2 *)(q + (size_t)row * ldq + ch * 8) = o;
        if ((ch & 15) == 0) s[(size_t)(ch >> 4) * lds + row] = sc;
    }
}

// ---- weights: w [N][K] fp32 -> q [ceil(N/128)*128][K] E4M3 (pad rows zero), s [ceil(N/128)][K/128] ----
// One 256-thread block per 128 x 128 block: 64 elements per thread, |max| through LDS, then q = sat_rne(w / s).
__global__ void __launch_bounds__(256) k_quant_w(const float *__restrict__ w, int N, int K, uint8_t *__restrict__ q,
                                                 float *__restrict__ s)
{
    __shared__ float red[4];
    const int kb = blockIdx.x, nb = blockIdx.y, KB = K >> 7;
    const int t = threadIdx.x, c = t & 15, r0 = t >> 4;  // 16 threads x 8 columns cover a 128-wide row
    float amax = 0.f;
    for (int r = r0; r < 128; r += 16) {
        const int n = nb * 128 + r;
        if (n < N) {
            float v[8];
            load8<float>(w + (size_t)n * K + kb * 128 + c * 8, v);
#pragma unroll
            for (int i = 0; i < 8; i++) amax = __builtin_fmaxf(amax, __builtin_fabsf(v[i]));
        }
    }
    amax = wave_max(amax);
    if ((t & 63) == 0) red[t >> 6] = amax;
    __syncthreads();
    amax = __builtin_fmaxf(__builtin_fmaxf(red[0], red[1]), __builtin_fmaxf(red[2], red[3]));
    const float sc = block_scale(amax);
    if (t == 0) s[(size_t)nb * KB + kb] = sc;
    for (int r = r0; r < 128; r += 16) {
        const int n = nb * 128 + r;
        uint2 o = make_uint2(0, 0);
        if (n < N) {
            float v[8];
            load8<float>(w + (size_t)n * K + kb * 128 + c * 8, v);
            o.x = e4_pack4(v[0] / sc, v[1] / sc, v[2] / sc, v[3] / sc);
            o.y = e4_pack4(v[4] / sc, v[5] / sc, v[6] / sc, v[7] / sc);
        }
        *(uint2 *)(q + (size_t)n * K + kb * 128 + c * 8) = o;
    }
}

// ---- encoder check: E4M3 of the fp32 bit patterns first .. first + count - 1 ----
__global__ void __launch_bounds__(256) k_e4m3_bits(uint32_t first, uint32_t count, uint8_t *__restrict__ out)
{
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < count; i += gridDim.x * 256u)
        out[i] = (uint8_t)e4_pack2(__uint_as_float(first + i), 0.f);
}

// ---- block-scale rule check: block_scale (which 0) or block_scale_inv (which 1) of the fp32 bit patterns
// first .. first + count - 1, as bit patterns ----
__global__ void __launch_bounds__(256) k_scale_bits(uint32_t first, uint32_t count, int which, uint32_t *__restrict__ out)
{
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < count; i += gridDim.x * 256u) {
        const float x = __uint_as_float(first + i);
        out[i] = __float_as_uint(which ? block_scale_inv(x) : block_scale(x));
    }
}

// ---- standalone block-scaled GEMM: C [M][ldc] = bf16 or fp32 of the block-scaled product ----
// bf16: each wave parks its rows x 64 (or 32) fp32 of its tile in its own LDS slice (padded rows, conflict-free), then
// every lane rounds 8 consecutive columns to bf16 (RNE) and writes them with one 16-byte store, whatever the row's
// alignment (the hardware takes 16-byte stores at any element address; two-byte stores for an odd ldc or N, as before,
// took 242 us for 8200 x 13461 x 1024). Columns of a store that reaches past N go one by one. In the tiles of
// 64-row waves an aligned C (ldc and N multiples of 8, 16-byte aligned) has a kernel of its own that stores through a
// descriptor ending at row M, without 64-bit addresses and row compares: 4100 x 13456 x 1024 77.9 -> 76.0 us, 8200 x 5632
// x 1024 58.7 -> 57.6 (with 32-row waves slower: 4100 x 2048 x 256 8.9 -> 9.5). fp32 stores 16 bytes straight from the
// accumulators.
// SP: W holds the 2:4 values and WX the indices of the pack24 layout (bs_mainloop_sp); otherwise W is dense, WX unused.
template <class C, int OUT, bool SP>  // OUT 0: bf16, 1: fp32, 2: bf16 of an aligned C
__global__ void __launch_bounds__(C::NT) k_gemm(const uint8_t *__restrict__ A, int lda, const float *__restrict__ sa,
                                               int lds, const uint8_t *__restrict__ W, const uint32_t *__restrict__ WX,
                                               const float *__restrict__ sw, void *__restrict__ Cp, int ldc, int M,
                                               int N, int K)
{
    __shared__ __attribute__((aligned(16))) uint8_t smem[LayerMem<C>::ROWSTAT];
    v4f acc[C::TM][C::TN];
    int tm, tn;
    tile_of_block((M + C::BM - 1) / C::BM, (N + C::BN - 1) / C::BN, M % C::BM != 0, tm, tn);
    const int m0 = tm * C::BM, n0 = tn * C::BN, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const int Npad = (N + 127) & ~127;
    args_resident(Cp, ldc, N, M, lds);
    // the tile transposed (acc[i][j][r]: row m0 + wm0 + 16 i + c16, column n0 + wn0 + 16 j + 4 g + r): the sparse
    // loop's own layout, and the dense loop's with TR
    if constexpr (SP) {
        v4f accT[C::TN][C::TM];
        bs_mainloop_sp_t<C, BsNoPre, false>(A, lda, sa, lds, W, WX, sw, M, Npad, K, m0, n0, smem, accT);
#pragma unroll
        for (int i = 0; i < C::TM; i++)
#pragma unroll
            for (int j = 0; j < C::TN; j++) acc[i][j] = accT[j][i];
    } else {
        bs_mainloop<C, BsNoPre, C::BM < 256, true>(A, lda, sa, lds, W, sw, M, Npad, K, m0, n0, smem, acc);
    }
    int wm0, wn0;
    bs_wave_origin<C>(wm0, wn0);
    if constexpr (OUT == 1) {
#pragma unroll
        for (int i = 0; i < C::TM; i++) {
            const int row = m0 + wm0 + 16 * i + c16;
            if (row >= M) continue;
            float *crow = (float *)Cp + (size_t)row * ldc;
#pragma unroll
            for (int j = 0; j < C::TN; j++) {
                const int col = n0 + wn0 + 16 * j + 4 * g;
                if (col + 4 <= N) {
                    *(v4f_e *)(crow + col) = acc[i][j];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (col + r < N) crow[col + r] = acc[i][j][r];
                }
            }
        }
    } else {
        using S = LayerMem<C>;
        constexpr int LPR = S::PC / 8, RPI = 64 / LPR;  // lanes a row, rows a store
        float *tr = (float *)(smem + (threadIdx.x >> 6) * S::SLICE);
        const int rs = lane / LPR, ch = lane % LPR;
        auto park = [&](int pass) {
            if (pass) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the previous pass's slice reads are done
#pragma unroll
            for (int i = 0; i < C::TM; i++)
#pragma unroll
                for (int j = 0; j < S::PC / 16; j++) {
                    const v4f v = acc[i][S::PC / 16 * pass + j];
                    *(float4 *)(tr + (16 * i + c16) * S::LD + 16 * j + 4 * g) = make_float4(v[0], v[1], v[2], v[3]);
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slice is the wave's own: no block barrier needed
        };
        auto packed = [&](int rr) {
            const float *t = tr + rr * S::LD + 8 * ch;
            const float4 a = *(const float4 *)t, b = *(const float4 *)(t + 4);
            return v4u{f2bf(a.x) | (uint32_t)f2bf(a.y) << 16, f2bf(a.z) | (uint32_t)f2bf(a.w) << 16,
                       f2bf(b.x) | (uint32_t)f2bf(b.y) << 16, f2bf(b.z) | (uint32_t)f2bf(b.w) << 16};
        };
        if constexpr (OUT == 2) {
            const __amdgpu_buffer_rsrc_t rc = buf_rsrc(Cp, (uint32_t)M * (uint32_t)ldc * 2u);
#pragma unroll
            for (int pass = 0; pass < C::WN / S::PC; pass++) {
                park(pass);
                const int col = n0 + wn0 + S::PC * pass + 8 * ch;
#pragma unroll
                for (int it = 0; it < C::WM / RPI; it++) {
                    const int rr = RPI * it + rs;
                    const v4u o = packed(rr);
                    if (col < N)
                        __builtin_amdgcn_raw_buffer_store_b128(
                            o, rc, (int)(((uint32_t)(m0 + wm0 + rr) * (uint32_t)ldc + (uint32_t)col) * 2u), 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int pass = 0; pass < C::WN / S::PC; pass++) {
                park(pass);
                const int col = n0 + wn0 + S::PC * pass + 8 * ch;
#pragma unroll
                for (int it = 0; it < C::WM / RPI; it++) {
                    const int rr = RPI * it + rs, row = m0 + wm0 + rr;
                    const float *t = tr + rr * S::LD + 8 * ch;
                    uint16_t *c = (uint16_t *)Cp + (size_t)row * ldc + col;
                    if (row < M && col + 8 <= N) {
                        *(v4u_e *)c = packed(rr);
                    } else if (row < M) {
                        for (int e = 0; col + e < N; e++) c[e] = f2bf(t[e]);
                    }
                }
            }
        }
    }
}

// Tiles by how many there are (us; bf16 output, dense unless said; M x N x K):
//  - 64 x 64 while one round of two blocks per CU holds them: 128 x 128 -> 64 x 64 at 1 x 1000 x 4736 22.5 -> 12.0,
//    100 x 13461 x 1024 10.9 -> 7.3, 1025 x 1024 x 1024 7.8 -> 6.1 (64 x 128: 16.5, 8.7, 6.6);
//  - 64 x 128 likewise: 1025 x 3072 x 1024 9.05 -> 8.7, x 4736 31.9 -> 25.1 (64 x 64: 10.4, 32.2);
//  - 256 x 256 from 1.6 rounds of one block per CU on, and for one round where 128 x 128 would take more than 1.5 rounds
//    of two per CU: 3584 x 3584 x 1024 21.7 -> 20.4, 4096 x 3840 x 512 14.5 -> 13.2, 2:4-sparse 5000 x 2560 x 1024 21.6
//    -> 19.6; dense from K = 2048 on also at those 1.5 rounds (3000 x 4096 x 2048 33.0 -> 30.5; x 512 13.4 -> 13.8) and
//    past the next 1.5 (8200 x 3072 x 3072 92.4 -> 81.2; x 512 23.4 -> 24.6);
//  - 128 x 128 elsewhere, in 8 waves (LayerMid) where the last round holds at most one block per CU, which then has two
//    waves per SIMD (4 waves: 8200 x 2048 x 1024 27.5 against 25.9, 8100 x 3000 x 2048 with a full last round 58.8
//    against 60.5), and for 2:4-sparse weights past the K below (4 waves: 2050 x 3072 x 3072 28.6 against 26.7, x 128
//    6.4 against 6.6); in 4 waves (GemmMid) where two blocks per CU run to the end: 8 -> 4 waves 2050 x 3072 x 512 8.9
//    -> 8.5, 1143 x 6768 x 1536 17.5 -> 16.5, 4896 x 840 x 3072 26.2 -> 24.6; not for a bf16 C that is not aligned (1877
//    x 12690 x 128 15.1 against 16.3).
typedef BsCfg<64, 64, 2, 2, 3> GemmSml;
typedef BsCfg<128, 128, 2, 2, 2> GemmMid;
template <bool SP, class F>
static void with_gemm_cfg(int M, int N, int K, int out, F f)  // out as k_gemm's OUT
{
    auto tiles = [&](auto c) { return (long)((M + c.BM - 1) / c.BM) * ((N + c.BN - 1) / c.BN); };
    const long big = tiles(LayerCfg{}), last = tiles(LayerMid{}) % 512;
    const bool deep = !SP && K >= 2048;
    if (tiles(GemmSml{}) <= 512) f(GemmSml{});
    else if (tiles(LayerSml{}) <= 512) f(LayerSml{});
    else if (big >= (deep ? 385 : 410) || (big >= (deep ? 192 : 193) && big <= 256)) f(LayerCfg{});
    else if ((last > 0 && last < 256) || (SP && K > (out == 1 ? 896 : 128)) || !out) f(LayerMid{});
    else f(GemmMid{});
}

// ---------------------------------------------------------------------------------------------------------------
// C-ABI launchers
// ---------------------------------------------------------------------------------------------------------------
static int grid_for(long threads)
{
    long b = (threads + 255) / 256;
    return (int)(b < 1 ? 1 : b > 65535 ? 65535 : b);
}

extern "C" int eva_k_quant_act(const void *x, int in_kind, int ldx, int M, int K, void *q, int ldq, float *s, int lds,
                               void *stream)
{
    if (M < 0 || K % 128 || ldx < K || ldq < K || lds < M || in_kind < 0 || in_kind > 2 || ldx % 8 || ldq % 8)
        return xt_fail("eva_k_quant_act",
                       "bad shape (K % 128, ldx >= K, ldq >= K, lds >= M, ldx and ldq multiples of 8, in_kind 0..2)");
    if (((uintptr_t)x | (uintptr_t)q) & 15) return xt_fail("eva_k_quant_act", "x and q must be 16-byte aligned");
    if (!M) return 0;
    const long thr = (long)M * (K / 8);
    if (in_kind == 0)
        hipLaunchKernelGGL(k_quant_act<uint16_t>, dim3(grid_for(thr)), dim3(256), 0, (hipStream_t)stream,
                           (const uint16_t *)x, ldx, M, K, (uint8_t *)q, ldq, s, lds);
    else if (in_kind == 1)
        hipLaunchKernelGGL(k_quant_act<float>, dim3(grid_for(thr)), dim3(256), 0, (hipStream_t)stream, (const float *)x,
                           ldx, M, K, (uint8_t *)q, ldq, s, lds);
    else
        hipLaunchKernelGGL(k_quant_act<_Float16>, dim3(grid_for(thr)), dim3(256), 0, (hipStream_t)stream,
                           (const _Float16 *)x, ldx, M, K, (uint8_t *)q, ldq, s, lds);
    return xt_check("eva_k_quant_act");
}

extern "C" int eva_k_quant_w(const float *w, int N, int K, void *q, float *s, void *stream)
{
    if (N <= 0 || K <= 0 || K % 128) return xt_fail("eva_k_quant_w", "bad shape (N > 0, K % 128 == 0)");
    if (((uintptr_t)w | (uintptr_t)q) & 15) return xt_fail("eva_k_quant_w", "w and q must be 16-byte aligned");
    hipLaunchKernelGGL(k_quant_w, dim3(K / 128, (N + 127) / 128), dim3(256), 0, (hipStream_t)stream, w, N, K,
                       (uint8_t *)q, s);
    return xt_check("eva_k_quant_w");
}

extern "C" int eva_k_e4m3_bits(uint32_t first, uint32_t count, void *out, void *stream)
{
    if (!count) return 0;
    hipLaunchKernelGGL(k_e4m3_bits, dim3(grid_for(count)), dim3(256), 0, (hipStream_t)stream, first, count,
                       (uint8_t *)out);
    return xt_check("eva_k_e4m3_bits");
}

extern "C" int eva_k_scale_bits(uint32_t first, uint32_t count, int which, void *out, void *stream)
{
    if (which != 0 && which != 1) return xt_fail("eva_k_scale_bits", "which must be 0 (scale) or 1 (inverse)");
    if (!count) return 0;
    hipLaunchKernelGGL(k_scale_bits, dim3(grid_for(count)), dim3(256), 0, (hipStream_t)stream, first, count, which,
                       (uint32_t *)out);
    return xt_check("eva_k_scale_bits");
}

template <bool SP>
static int gemm_launch(const char *what, const void *qa, int lda, const float *sa, int lds, const void *qw,
                       const void *qx, const float *sw, int M, int N, int K, void *c, int ldc, int out_kind,
                       void *stream)
{
    if (M < 0 || N <= 0 || K <= 0 || K % 128 || lda < K || lda % 16 || lds < M || ldc < N ||
        (out_kind != 0 && out_kind != 1))
        return xt_fail(what, "bad shape (K % 128, lda >= K and a multiple of 16, lds >= M, ldc >= N, out_kind 0 or 1)");
    if (((uintptr_t)qa | (uintptr_t)qw) & 15) return xt_fail(what, "qa and qw must be 16-byte aligned");
    // buffer descriptors and row offsets are 32-bit: operands and output must stay below 2 GiB (the A-row sentinel
    // XT_OOR = 2^31 must lie past every valid offset) and 4 GiB
    const size_t Np = ((size_t)N + 255) / 256 * 256;
    if ((size_t)M * lda >= (1u << 31) || Np * K >= (1u << 31) || (size_t)M * ldc * (out_kind ? 4 : 2) >= (1ull << 32) ||
        (size_t)lds * (K / 128) * 4 >= (1u << 31))
        return xt_fail(what, "operands too large for 32-bit offsets (M * lda, N * K < 2^31 bytes, C < 4 GiB)");
    if (SP && (N % 16 || !qx || ((uintptr_t)qx & 3))) return xt_fail(what, "sparse weights: N % 16 == 0, 4-byte aligned indices");
    if (!M) return 0;
    const uint8_t *A = (const uint8_t *)qa, *W = (const uint8_t *)qw;
    const uint32_t *X = (const uint32_t *)qx;
    hipStream_t st = (hipStream_t)stream;
    // the descriptor's 32-bit offsets must not wrap for the rows of the last tile past M
    const bool aligned = ((ldc | N) & 7) == 0 && ((uintptr_t)c & 15) == 0 && ((size_t)M + 256) * ldc * 2 < (1ull << 32);
    const int out = out_kind ? 1 : aligned ? 2 : 0;
    with_gemm_cfg<SP>(M, N, K, out, [&](auto c_) {
        using T = decltype(c_);
        const dim3 grid((unsigned)(((M + T::BM - 1) / T::BM) * ((N + T::BN - 1) / T::BN)));
        constexpr bool wide = T::TM == 4;  // the tiles with a kernel for an aligned C
        auto run = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(T::NT), 0, st, A, lda, sa, lds, W, X, sw, c, ldc, M, N, K);
        };
        if (out == 1) run(k_gemm<T, 1, SP>);
        else if (wide && out == 2) run(k_gemm<T, wide ? 2 : 0, SP>);
        else run(k_gemm<T, std::is_same_v<T, GemmMid> ? 2 : 0, SP>);  // GemmMid: out is never 0
    });
    return xt_check(what);
}

extern "C" int eva_k_gemm(const void *qa, int lda, const float *sa, int lds, const void *qw, const float *sw, int M,
                          int N, int K, void *c, int ldc, int out_kind, void *stream)
{
    return gemm_launch<false>("eva_k_gemm", qa, lda, sa, lds, qw, nullptr, sw, M, N, K, c, ldc, out_kind, stream);
}

extern "C" int eva_k_gemm_sp(const void *qa, int lda, const float *sa, int lds, const void *vals, const void *idx,
                             const float *sw, int M, int N, int K, void *c, int ldc, int out_kind, void *stream)
{
    return gemm_launch<true>("eva_k_gemm_sp", qa, lda, sa, lds, vals, idx, sw, M, N, K, c, ldc, out_kind, stream);
}
