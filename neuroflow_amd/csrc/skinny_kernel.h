// skinny_kernel.h -- a quantised layer on a few rows (a GEMV or nearly one) in
// one launch.  Bound by latency: with one row the 1024 x 1024 layer reads 1 MB
// of weights, 0.2 us of HBM time, so what counts is how many dependent steps a
// block takes.  A block owns 16 rows x 16 columns and splits K over its
// waves: every wave loads its share of the rows (fp32) and of the 16 weight
// rows at once, straight into the MFMA operand layout (lane (r, g): row or
// column r, k = 16 g .. 16 g + 15 of a 64-wide block), quantises in registers,
// and one exchange through LDS sums the waves' 16 x 16 products.  The per-token
// formats add one LDS exchange for the row maxima.  Measured on MI355X (us):
// static 1 x 1024 -> 1024 148 (quantise launch + one thread per output) ->
// 12.6 (one-pass kernel, 16 rows, K in sequence) -> 5.2.
#pragma once

#include <type_traits>

#include "common.h"
#include "token_gemm_kernel.h"

namespace nfq {

// PER: 64-wide K blocks per wave; K <= 64 NW PER.
template <int NW, int PER, int FMT, int ACT>
__global__ __launch_bounds__(64 * NW) void k_skinny(RowsArgs a) {
    constexpr bool FP8 = FMT == TG_FP8;
    typedef typename TokenAcc<FP8>::type Acc;
    typedef std::conditional_t<FP8, float, int32_t> Sum;
    __shared__ __attribute__((aligned(16))) Sum part[NW][256];
    __shared__ float mx_s[NW][16], scale_s[16];
    __shared__ int32_t sa_s[NW][16], ws_s[NW][16], wd_s[NW][16];
    // Wave-uniform to the compiler too: an MFMA ignores EXEC, so the branch on
    // kb below must be a scalar one.
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int K = a.K, N = a.N;
    const int n0 = 16 * blockIdx.x;
    const int64_t m0 = 16 * static_cast<int64_t>(blockIdx.y);
    const bool live = m0 + r < a.M;

    // All the loads: PER x (16 floats of row m0 + r, 16 bytes of W row n0 + r).
    const float* row = a.A + (live ? m0 + r : m0) * K;
    const int n = n0 + r < N ? n0 + r : N - 1;
    const int last = K - 4;
    const int64_t w_total = static_cast<int64_t>(N) * K;
    v4f x[PER][4];
    v4i wv[PER];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int k0 = 64 * (wid + NW * p) + 16 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + 4 * j;
            x[p][j] = *reinterpret_cast<const v4f_u*>(row + (k < last ? k : last));
        }
        wv[p] = token_w16(a.W, static_cast<int64_t>(n) * K + k0, K - k0, w_total);
    }
    // Values past K (and rows past M) become 0.
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int k0 = 64 * (wid + NW * p) + 16 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int sh = live ? k0 + 4 * j - last : 4;
            if (sh > 0) {
                const v4f t = x[p][j];
                x[p][j][0] = sh == 1 ? t[1] : sh == 2 ? t[2] : sh == 3 ? t[3] : 0.0f;
                x[p][j][1] = sh == 1 ? t[2] : sh == 2 ? t[3] : 0.0f;
                x[p][j][2] = sh == 1 ? t[3] : 0.0f;
                x[p][j][3] = 0.0f;
            }
        }
    }

    float s = a.scale_A;
    if constexpr (FMT != TG_I8_FIXED) {
        float mx = 0.0f;
#pragma unroll
        for (int p = 0; p < PER; ++p)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                mx = fmaxf(fmaxf(mx, fmaxf(fabsf(x[p][j][0]), fabsf(x[p][j][1]))),
                           fmaxf(fabsf(x[p][j][2]), fabsf(x[p][j][3])));
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (g == 0) mx_s[wid][r] = mx;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NW; ++w) mx = fmaxf(mx, mx_s[w][r]);
        s = (mx == 0.0f) ? 1.0f : mx / (FP8 ? 448.0f : 127.0f);
    }

    Acc acc = {0, 0, 0, 0};
    int32_t sa = 0, wsum = 0, wdot = 0;
    const float inv = FP8 ? ((s == 0.0f) ? 1.0f : 1.0f / s) : 1.0f / s;
    const bool fast = s >= 0x1p-120f && s <= 0x1p120f;   // the fixed scale's reciprocal path
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int kb = wid + NW * p;
        const int k0 = 64 * kb + 16 * g;
        v4i xv;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t v;
            if constexpr (FP8) {
                v = fp8_pack4(x[p][j], inv);
            } else if constexpr (FMT == TG_I8_FIXED) {
                v = quant_i8_fixed4(x[p][j], s, inv, a.zp_A, fast);
            } else {
                v = pack4(quant_i8_token(x[p][j][0], s, inv), quant_i8_token(x[p][j][1], s, inv),
                          quant_i8_token(x[p][j][2], s, inv), quant_i8_token(x[p][j][3], s, inv));
            }
            if constexpr (FMT != TG_I8_TOKEN) v = token_mask_codes(v, K - (k0 + 4 * j));
            xv[j] = live ? static_cast<int>(v) : 0;
        }
        if constexpr (FP8) {
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16(wv[p][0], wv[p][1]),
                                                          fp8x8_to_bf16(xv[0], xv[1]), acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16(wv[p][2], wv[p][3]),
                                                          fp8x8_to_bf16(xv[2], xv[3]), acc, 0, 0, 0);
        } else {
            int32_t ws = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sa = sum_bytes_i8(static_cast<uint32_t>(xv[j]), sa);
                ws = sum_bytes_i8(static_cast<uint32_t>(wv[p][j]), ws);
            }
            wsum += ws;
            // The row-VNNI formula's dot stops at the last whole 64-wide
            // block (int8_gemm.cpp:366); the byte sums do not.
            if (kb < a.kb_dot) {
                wdot += ws;
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[p], xv, acc, 0, 0, 0);
            }
        }
    }
    *reinterpret_cast<Acc*>(&part[wid][4 * lane]) = acc;
    if constexpr (!FP8) {
        sa = row_sum4(sa);
        wsum = row_sum4(wsum);
        wdot = row_sum4(wdot);
        if (g == 0) {
            sa_s[wid][r] = sa;
            ws_s[wid][r] = wsum;
            wd_s[wid][r] = wdot;
        }
    }
    if constexpr (FMT != TG_I8_FIXED) {
        if (wid == 0 && g == 0) scale_s[r] = s;
    }
    __syncthreads();
    // Thread t (of 256): value t % 4 of lane t / 4's accumulator, row
    // (t / 4) % 16, column 4 (t / 64) + t % 4.
    for (int t = threadIdx.x; t < 256; t += 64 * NW) {
        const int rr = (t >> 2) & 15, c = 4 * (t >> 6) + (t & 3);
        const int64_t m = m0 + rr;
        const int col = n0 + c;
        if (m >= a.M || col >= N) continue;
        Sum D = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) D += part[w][t];
        float tv;
        if constexpr (FP8) {
            tv = D;
        } else {
            int32_t SA = 0, Sf = 0, Sd = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                SA += sa_s[w][rr];
                Sf += ws_s[w][c];
                Sd += wd_s[w][c];
            }
            if constexpr (FMT == TG_I8_TOKEN) SA += token_sum_past_k(scale_s[rr], 64 * NW * PER - K);
            const IntEpi e = int_epi_consts(a.formula, K, a.zp_A, a.zpW ? a.zpW[col] : 0, a.sumW ? a.sumW[col] : 0,
                                            a.sumW != nullptr, Sf, Sd);
            tv = int_epi_value_of<FMT == TG_I8_FIXED>(e, D, SA);
        }
        const float srow = FMT == TG_I8_FIXED ? a.scale_A : scale_s[rr];
        const float y = activate<ACT>(dequant_bias(a.sW[col], srow, tv, a.bias ? a.bias[col] : 0.0f));
        static_cast<float*>(a.C)[m * N + col] = y;
        if (FMT != TG_I8_FIXED && a.scale_out && col == 0) a.scale_out[m] = srow;
    }
}

}  // namespace nfq
