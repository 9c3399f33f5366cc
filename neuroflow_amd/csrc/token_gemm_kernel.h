// token_gemm_kernel.h -- a quantised layer in one pass for K <= 1024: a block
// quantises a tile of 64 or 16 rows of fp32 activations into codes held in LDS, then
// runs the whole N range from them with MFMAs, dequantise + bias +
// activation in the epilogue.  The activations are read once and the codes
// never reach HBM: the layer costs one fp32 read and one fp32 write, where
// the split form (quantise launch, codes to HBM, tiled GEMM) adds a launch
// and 2 MK bytes of code traffic and re-reads the codes per column block.
//
// Formats (FMT):
//   TG_I8_TOKEN  per-token INT8 (scale absmax / 127, the reference's correctly
//                rounded codes, int8_gemm.cpp:231-240), v_mfma_i32_16x16x64_i8
//   TG_I8_FIXED  one scale_A / zp_A for every row (int8_gemm.cpp:507-520, as
//                LinearForward and LinearForwardBatched run it)
//   TG_FP8       per-token E4M3 (scale absmax / 448); codes and weights stay
//                bytes in LDS and L2 and become bf16 in registers
//                (v_cvt_scalef32_pk_bf16_fp8), v_mfma_f32_16x16x32_bf16
//
// What bounds it: the fp32 read and write of HBM for large M, the chain of
// one tile's quantise and product for small M.  Measured on MI355X before
// (the row-tile kernel re-reading W per 16 rows, or one thread per output)
// and with this kernel: FP8 32768 x 256 -> 768 221 -> 27.9 us (4.8 TB/s), FP8
// 20011 x 101 -> 128 315 -> 10 us, static INT8 8192 x 512 -> 2048 27.2 ms ->
// 38 us, FP8 4096 x 1024 -> 1024 847 -> 43 us, INT8 200000 x 64 -> 46 1121 ->
// 39 us.
//
// k_token_gemm<KB, FMT, ACT, CT, RT, RAG>: K <= 64 KB, tiles of 16 RT rows
// (64, or 16 where few tiles leave the chip idle).  4 waves, 2 to 4 blocks per CU,
// each block quantising a tile and then running its product, persistent over
// (tile, column share) pairs.  RAG = false: K = 64 KB, N a multiple of 64 and
// 16-byte aligned buffers; without the masks and clamps, N <= 128 at large M runs
// at two thirds of the time (per-token INT8 60000 x 256 -> 128 25.1 -> 16.0 us,
// 40000 x 512 -> 64 35.5 -> 24.1).  RAG = true: any K up to 64 KB, any N, any
// alignment the types allow: loads are masked at K (rows of K % 4 != 0
// floats start 4-byte aligned, which the 16-byte loads accept), codes past K
// are 0, weight bytes past K are masked to 0, columns past N are not stored.
//
// Tile quantise: a wave quantises 4 RT rows, 4 at a time with 16 lanes per row
// (the reductions are DPP row steps), codes into LDS rows of 64 KB + 16
// bytes (the pad spreads the 16 rows of an operand read over the banks).
// Tile product: the N range is walked in chunks of 64 CT columns; wave w
// takes 16 CT columns of the chunk for all the rows: RT x CT tiles of 16 x 16
// accumulators (CT = 2 serves N <= 128, where CT = 4 leaves two of the four
// waves without columns).  Weights come from L2 (16 contiguous bytes of one
// weight row per lane and K step), codes from LDS.  As in the other kernels
// the weight tile is the MFMA's A operand, so a lane's four results are four
// adjacent output columns of one row, and lane group g takes k = 16 g ..
// 16 g + 15 of each 64-wide step in both operands (the product is a
// permutation of the K-sum, exact in int32).  The epilogue passes each
// 16-row strip of a wave's 16 x 16 CT outputs through a per-wave LDS strip,
// and the strip leaves as row-contiguous segments.
// Column constants: lane L of a wave owns column nw0 + L of its columns.  It
// loads that column's weight scale, bias, zero point and given sum_W before
// the K loop (one coalesced load each, whose latency the K loop covers),
// forms the INT8 epilogue constants from the weight bytes summed during the K
// loop (as in the row-tile kernels) and files everything in the wave's LDS
// tables, which the epilogue reads as 16-byte vectors per lane.  Loading them
// per output lane after the K loop instead puts a chain of dependent global
// loads -- each also waiting for the previous chunk's stores -- between
// every product and its stores.
#pragma once

#include "common.h"
#include "rows_kernel.h"

namespace nfq {

// Output stores carry the nt (non-temporal) policy: the streamed output then
// leaves the L2 to the weights the K loops re-read (measured at C4, six
// blocks of qkv + proj on 32768 tokens: 25.35 -> 22.3 us per layer; sc1
// 24.2 us).
constexpr int kTokenStoreCpol = 2;

enum TokenFmt { TG_I8_TOKEN = 0, TG_I8_FIXED = 1, TG_FP8 = 2 };

template <int KB, int CT, int RT>
struct TokenGemmShape {
    static constexpr int K = 64 * KB;
    static constexpr int ROW = K + 16;            // LDS code row stride (bytes)
    static constexpr int ROWS = 16 * RT;          // rows per tile
    static constexpr int CODES = ROWS * ROW;      // code tile bytes
    static constexpr int WCOLS = 16 * CT;         // columns per wave
    static constexpr int STRIP_W = WCOLS + 4;     // per-wave output strip row stride (floats)
    static constexpr int STRIP = 16 * STRIP_W * 4;
    static constexpr int ETAB = 64 * static_cast<int>(sizeof(IntEpi)) + 2 * 64 * 4;  // per-wave column consts
    static constexpr int ROWQ = 64 * 4 + 64 * 4;  // row scales, row code sums
    static constexpr int LDS = CODES + 4 * STRIP + 4 * ETAB + ROWQ;
};

typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));
typedef int v4i_u __attribute__((ext_vector_type(4), aligned(1)));

// Activations of 4 rows (row m of this lane's group g; rows past M read row
// M - 1 and are not used): float4 r + 16 j of the row, j < J, 0 past K.
// RAG: every lane loads, at an address clamped inside the row, and the loaded
// values are moved or cleared by selects: branches around the loads would
// put a wait at each (measured at 1500 x 320: 16 us against 8).
template <int J, bool RAG>
__device__ __forceinline__ void token_load4(const RowsArgs& a, int64_t m, int r, v4f (&x)[J]) {
    const int64_t M = a.M;
    const int K = RAG ? a.K : 64 * J;
    const float* row = a.A + (m < M ? m : M - 1) * static_cast<int64_t>(K);
    if constexpr (!RAG) {
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(row + 4 * r + 64 * j));
        return;
    }
    const int last = K < 4 ? 0 : K - 4;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int k = 4 * r + 64 * j;
        x[j] = __builtin_nontemporal_load(reinterpret_cast<const v4f_u*>(row + (k < last ? k : last)));
    }
    if (K % 4 == 0) {
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = 4 * r + 64 * j < K ? x[j] : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    } else {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int sh = 4 * r + 64 * j - last;    // elements the clamped load starts early by
            const v4f t = x[j];
            if (sh > 0) {
                x[j][0] = sh == 1 ? t[1] : sh == 2 ? t[2] : sh == 3 ? t[3] : 0.0f;
                x[j][1] = sh == 1 ? t[2] : sh == 2 ? t[3] : 0.0f;
                x[j][2] = sh == 1 ? t[3] : 0.0f;
                x[j][3] = 0.0f;
            }
        }
    }
}

// The four codes of a dword with those past K (left <= 3 remain) cleared: a
// zero activation's code is zp_A with a fixed scale, and NaN in FP8 when the
// row's scale is subnormal (0 * inf).
__device__ __forceinline__ uint32_t token_mask_codes(uint32_t v, int left) {
    return left <= 0 ? 0u : (left < 4 ? v & ((1u << (8 * left)) - 1u) : v);
}

// Per-token INT8 codes past K are 0 (and meet weights of 0) except in a row
// whose scale rounded to 0: there every code is that of x / 0 or 0 / 0, -128, and
// the row's code sum takes back the ones past K.
__device__ __forceinline__ int32_t token_sum_past_k(float s, int past) { return s == 0.0f ? 128 * past : 0; }

// Codes of local row lr (= 4 q + g of the wave's rows) from x into the tile
// and, for INT8, their byte sum; row scale and sum to lds_s / lds_sa (and
// the per-token scale to scale_out for rows < M).
template <int J, int FMT, bool RAG>
__device__ __forceinline__ void token_quantise_row(const RowsArgs& a, const v4f (&x)[J], int64_t m0, int lr,
                                                   int r, uint8_t* codes, int row_bytes, float* lds_s,
                                                   int32_t* lds_sa) {
    const bool live = m0 + lr < a.M;
    float s = a.scale_A;
    if constexpr (FMT != TG_I8_FIXED) {
        float mx = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j)
            mx = fmaxf(fmaxf(mx, fmaxf(fabsf(x[j][0]), fabsf(x[j][1]))), fmaxf(fabsf(x[j][2]), fabsf(x[j][3])));
        mx = fmaxf(mx, dpp_mov<0xB1>(mx));   // quad_perm [1,0,3,2]
        mx = fmaxf(mx, dpp_mov<0x4E>(mx));   // quad_perm [2,3,0,1]
        mx = fmaxf(mx, dpp_mov<0x141>(mx));  // row_half_mirror
        mx = fmaxf(mx, dpp_mov<0x140>(mx));  // row_mirror
        s = (mx == 0.0f) ? 1.0f : mx / (FMT == TG_FP8 ? 448.0f : 127.0f);
    }
    uint32_t* crow = reinterpret_cast<uint32_t*>(codes + lr * row_bytes);
    int32_t sa = 0;
    if constexpr (FMT == TG_FP8) {
        const float inv = (s == 0.0f) ? 1.0f : 1.0f / s;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            uint32_t v = fp8_pack4(x[j], inv);
            if constexpr (RAG) v = token_mask_codes(v, a.K - (4 * r + 64 * j));
            crow[r + 16 * j] = live ? v : 0u;
        }
    } else {
        const float inv = 1.0f / s;
        // Fixed scale: the reciprocal path needs a normal 1 / s.
        const bool fast = FMT == TG_I8_TOKEN || (s >= 0x1p-120f && s <= 0x1p120f);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            uint32_t v;
            if constexpr (FMT == TG_I8_TOKEN) {
                v = pack4(quant_i8_token(x[j][0], s, inv), quant_i8_token(x[j][1], s, inv),
                          quant_i8_token(x[j][2], s, inv), quant_i8_token(x[j][3], s, inv));
            } else {
                v = quant_i8_fixed4(x[j], s, inv, a.zp_A, fast);
                if constexpr (RAG) v = token_mask_codes(v, a.K - (4 * r + 64 * j));
            }
            v = live ? v : 0u;
            crow[r + 16 * j] = v;
            sa = sum_bytes_i8(v, sa);
        }
        sa += dpp_movi<0xB1>(sa);
        sa += dpp_movi<0x4E>(sa);
        sa += dpp_movi<0x141>(sa);
        sa += dpp_movi<0x140>(sa);
        if constexpr (RAG && FMT == TG_I8_TOKEN) sa += token_sum_past_k(s, 64 * J - a.K);
    }
    if (r == 0) {
        lds_s[lr] = s;
        lds_sa[lr] = sa;
        if (FMT != TG_I8_FIXED && a.scale_out && live) a.scale_out[m0 + lr] = s;
    }
}

// 16 weight bytes at byte `off` of the (N, K) matrix of `total` >= 16 bytes,
// of which the first `left` lie inside the row (the rest become 0).  Bytes
// past the row belong to the next one; a load that would pass the end of the
// matrix is moved back and its value shifted (the last rows' tails only).
__device__ __forceinline__ v4i token_w16(const uint8_t* W, int64_t off, int left, int64_t total) {
    const int64_t at = off < total - 16 ? off : total - 16;
    v4i v = *reinterpret_cast<const v4i_u*>(W + at);
    if (__any(at != off)) {
        const int sh = 8 * static_cast<int>(off - at < 16 ? off - at : 15);
        const uint64_t lo = static_cast<uint64_t>(static_cast<uint32_t>(v[0])) | (static_cast<uint64_t>(static_cast<uint32_t>(v[1])) << 32);
        const uint64_t hi = static_cast<uint64_t>(static_cast<uint32_t>(v[2])) | (static_cast<uint64_t>(static_cast<uint32_t>(v[3])) << 32);
        const uint64_t l = sh == 0 ? lo : sh < 64 ? (lo >> sh) | (hi << (64 - sh)) : hi >> (sh - 64);
        const uint64_t h = sh < 64 ? hi >> sh : 0;
        v = v4i{static_cast<int>(l), static_cast<int>(l >> 32), static_cast<int>(h), static_cast<int>(h >> 32)};
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int n = left - 4 * q;
        const uint32_t mask = n >= 4 ? 0xFFFFFFFFu : (n <= 0 ? 0u : (1u << (8 * n)) - 1u);
        v[q] = static_cast<int>(static_cast<uint32_t>(v[q]) & mask);
    }
    return v;
}

__device__ __forceinline__ void token_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool FP8>
struct TokenAcc { typedef v4i type; };
template <>
struct TokenAcc<true> { typedef v4f type; };

// The product of the code tile at m0 with the block's share of the
// column chunks (share, share + nshare, ...), by product wave `wid` (0..3).
// SUMS = false when every integer-epilogue term is zero whatever the weights
// (zp_A = 0, no weight zero points, no caller sum_W or the batched formula;
// and FP8): the weight byte sums and the epilogue constants are then skipped.
template <int KB, int FMT, int ACT, int CT, int RT, bool RAG, bool SUMS>
__device__ __forceinline__ void token_tile_gemm(const RowsArgs& a, const uint8_t* codes, const float* lds_s,
                                                const int32_t* lds_sa, float* strip, uint8_t* ctab, int64_t m0,
                                                int wid, int lane, int share, int nshare) {
    using S = TokenGemmShape<KB, CT, RT>;
    constexpr bool FP8 = FMT == TG_FP8;
    typedef typename TokenAcc<FP8>::type Acc;
    const int K = RAG ? a.K : S::K;
    const int r = lane & 15, g = lane >> 4;
    const int64_t M = a.M;
    const int N = a.N;
    int32_t* c0tab = reinterpret_cast<int32_t*>(ctab);                  // the wave's columns' INT8 constants
    int32_t* c1tab = c0tab + 64;
    int64_t* c2tab = reinterpret_cast<int64_t*>(c1tab + 64);
    float* swtab = reinterpret_cast<float*>(ctab + 64 * sizeof(IntEpi));  // weight scales
    float* btab = swtab + 64;                                             // biases
    const int64_t w_total = static_cast<int64_t>(N) * K;
    const int nkb = RAG ? (K + 63) / 64 : KB;
    const bool whole_k = !RAG || K % 64 == 0;   // no weight bytes to mask
    // 16-byte row segments need whole float4 columns; else dword stores.
    // Rows of whole 128-byte lines leave with the nt policy; other rows share
    // lines between blocks, which only the L2 can merge.
    const bool nt_store = !RAG || N % 32 == 0;
    const bool vec_store = !RAG || (N % 4 == 0 && (reinterpret_cast<uintptr_t>(a.C) & 15) == 0);

    // Row scales / code sums of the lane's rows 16 rt + r.
    float srow[RT];
    int32_t sarow[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        srow[rt] = lds_s[16 * rt + r];
        sarow[rt] = lds_sa[16 * rt + r];
    }

    for (int nc = share * (4 * S::WCOLS); nc < N; nc += nshare * (4 * S::WCOLS)) {
        const int nw0 = nc + S::WCOLS * wid;        // the wave's first column
        if (nw0 >= N) continue;                     // wave-uniform
        // This lane's column: constants loaded branch-free (an absent
        // array reads the scales and the value is replaced by 0).
        int cl = nw0 + (CT == 4 ? lane : lane & (S::WCOLS - 1));
        if constexpr (RAG) cl = cl < N ? cl : N - 1;
        const float my_sw = a.sW[cl];
        const float my_b0 = (a.bias ? a.bias : a.sW)[cl];
        int32_t my_zp0 = 0, my_sg0 = 0;
        if constexpr (SUMS) {
            my_zp0 = (a.zpW ? a.zpW : reinterpret_cast<const int32_t*>(a.sW))[cl];
            my_sg0 = (a.sumW ? a.sumW : reinterpret_cast<const int32_t*>(a.sW))[cl];
        }
        Acc acc[RT][CT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = Acc{0, 0, 0, 0};
        int32_t wsum[CT] = {}, wdot[CT] = {};
        // Two K steps per trip: unrolled further, the weight loads hoisted
        // ahead of the products push the kernel past 256 registers.
#pragma unroll 2
        for (int kb = 0; kb < nkb; ++kb) {
            v4i wv[CT], xv[RT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                int n = nw0 + 16 * ct + r;
                if constexpr (RAG) {
                    n = n < N ? n : N - 1;
                    const int k = 64 * kb + 16 * g;
                    const int64_t off = static_cast<int64_t>(n) * K + k;
                    if (whole_k) wv[ct] = *reinterpret_cast<const v4i_u*>(a.W + off);
                    else wv[ct] = token_w16(a.W, off, K - k, w_total);
                } else {
                    wv[ct] = *reinterpret_cast<const v4i*>(a.W + static_cast<int64_t>(n) * K + 64 * kb + 16 * g);
                }
                if constexpr (SUMS) {
                    int32_t s = 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) s = sum_bytes_i8(static_cast<uint32_t>(wv[ct][e]), s);
                    wsum[ct] += s;
                    if constexpr (RAG) wdot[ct] += kb < a.kb_dot ? s : 0;
                }
            }
            // The row-VNNI formula's dot stops at the last whole 64-wide
            // block (int8_gemm.cpp:366); the byte sums do not.
            if (RAG && !FP8 && kb >= a.kb_dot) continue;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                xv[rt] = *reinterpret_cast<const v4i*>(codes + (16 * rt + r) * S::ROW + 64 * kb + 16 * g);
            if constexpr (FP8) {
                v8bf wb[CT][2];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    wb[ct][0] = fp8x8_to_bf16(wv[ct][0], wv[ct][1]);
                    wb[ct][1] = fp8x8_to_bf16(wv[ct][2], wv[ct][3]);
                }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const v8bf x0 = fp8x8_to_bf16(xv[rt][0], xv[rt][1]);
                    const v8bf x1 = fp8x8_to_bf16(xv[rt][2], xv[rt][3]);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) {
                        acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[ct][0], x0, acc[rt][ct], 0, 0, 0);
                        acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[ct][1], x1, acc[rt][ct], 0, 0, 0);
                    }
                }
            } else {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
                        acc[rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wv[ct], xv[rt], acc[rt][ct], 0, 0, 0);
            }
        }
        // Weight byte sums of column 16 ct + r reduced over the lane groups;
        // lane (r, g) = column 16 g + r takes tile ct = g.
        bool trivial = true, small = true;
        if constexpr (SUMS) {
            int32_t wfull = 0, wd = 0;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const int32_t f = row_sum4(wsum[ct]);
                wfull = (g == ct) ? f : wfull;
                if constexpr (RAG) {
                    const int32_t d = row_sum4(wdot[ct]);
                    wd = (g == ct) ? d : wd;
                }
            }
            if constexpr (!RAG) wd = wfull;
            const int32_t my_zp = a.zpW ? my_zp0 : 0;
            const IntEpi mine = int_epi_consts(a.formula, K, a.zp_A, my_zp, a.sumW ? my_sg0 : 0,
                                               a.sumW != nullptr, wfull, wd);
            // Wave-uniform: all the columns' constants zero, the result is
            // (float)D; or no column's sum can leave 32 bits.
            trivial = !__any((mine.c0 != 0) | (mine.c1 != 0) | (mine.c2 != 0));
            small = !__any(!int_epi_small(mine, K));
            if (!trivial && lane < S::WCOLS) {
                c0tab[lane] = small ? mine.c0 + static_cast<int32_t>(mine.c2) : mine.c0;
                c1tab[lane] = mine.c1;
                c2tab[lane] = mine.c2;
            }
        }
        if (CT == 4 || lane < S::WCOLS) {
            swtab[lane] = my_sw;
            btab[lane] = a.bias ? my_b0 : 0.0f;
        }
        token_wave_sync();
        // Epilogue, one 16-row strip at a time through the wave's LDS strip.
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const int c0 = 16 * ct + 4 * g;          // the lane's first column in the wave
                float t[4];
                if (FP8 || trivial) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) t[v] = static_cast<float>(acc[rt][ct][v]);
                } else {
                    const v4i e0 = *reinterpret_cast<const v4i*>(c0tab + c0), e1 = *reinterpret_cast<const v4i*>(c1tab + c0);
                    if (small) {
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            t[v] = int_epi_value_small(e0[v], e1[v], static_cast<int32_t>(acc[rt][ct][v]), sarow[rt]);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            t[v] = int_epi_value_of<FMT == TG_I8_FIXED>(IntEpi{e0[v], e1[v], c2tab[c0 + v]},
                                                                        static_cast<int32_t>(acc[rt][ct][v]), sarow[rt]);
                    }
                }
                const v4f sw4 = *reinterpret_cast<const v4f*>(swtab + c0);
                const v4f b4 = *reinterpret_cast<const v4f*>(btab + c0);
                v4f y;
#pragma unroll
                for (int v = 0; v < 4; ++v) y[v] = activate<ACT>(dequant_bias(sw4[v], srow[rt], t[v], b4[v]));
                *reinterpret_cast<v4f*>(strip + r * S::STRIP_W + c0) = y;
            }
            token_wave_sync();
            // The strip's rows m0 + 16 rt .. + 15 as a buffer range clipped
            // at M: rows past it are dropped by the hardware.
            const int64_t r0 = m0 + 16 * rt;
            const int64_t left = M - r0 < 0 ? 0 : (M - r0 > 16 ? 16 : M - r0);
            const auto rs = __builtin_amdgcn_make_buffer_rsrc(static_cast<float*>(a.C) + r0 * N, 0,
                                                              static_cast<int>(left * N * 4), 0x00020000);
            if (vec_store) {
                constexpr int LPR = 4 * CT;              // lanes per row
#pragma unroll
                for (int q = 0; q < CT; ++q) {
                    const int sr = (64 / LPR) * q + lane / LPR;     // strip row
                    const int c = 4 * (lane % LPR);
                    const v4f v = *reinterpret_cast<const v4f*>(strip + sr * S::STRIP_W + c);
                    if (nt_store) {
                        if (!RAG || nw0 + c < N)
                            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), rs,
                                                                   (sr * N + nw0 + c) * 4, 0, kTokenStoreCpol);
                    } else if (nw0 + c < N) {
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), rs,
                                                               (sr * N + nw0 + c) * 4, 0, 0);
                    }
                }
            } else {
                constexpr int RPI = 64 / S::WCOLS;       // rows per instruction
                const int c = lane & (S::WCOLS - 1);
#pragma unroll 4
                for (int q = 0; q < 16 / RPI; ++q) {
                    const int sr = RPI * q + lane / S::WCOLS;
                    const float v = strip[sr * S::STRIP_W + c];
                    if (nw0 + c < N)
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rs, (sr * N + nw0 + c) * 4, 0, 0);
                }
            }
            token_wave_sync();
        }
    }
}

template <int KB, int FMT, int ACT, int CT, int RT, bool RAG>
__global__ __launch_bounds__(256, 2) void k_token_gemm(RowsArgs a, int nshare) {
    using S = TokenGemmShape<KB, CT, RT>;
    constexpr int J = KB;                        // float4 per lane per row in the quantise
    __shared__ __attribute__((aligned(16))) uint8_t lds[S::LDS];
    uint8_t* codes = lds;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* strip = reinterpret_cast<float*>(lds + S::CODES) + wid * (16 * S::STRIP_W);
    uint8_t* ctab = lds + S::CODES + 4 * S::STRIP + wid * S::ETAB;
    float* lds_s = reinterpret_cast<float*>(lds + S::CODES + 4 * S::STRIP + 4 * S::ETAB);
    int32_t* lds_sa = reinterpret_cast<int32_t*>(lds_s + 64);

    const int lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int64_t ntiles = (a.M + S::ROWS - 1) / S::ROWS;
    const int64_t nwork = ntiles * nshare;
    const bool zero_terms = FMT == TG_FP8 || (a.zp_A == 0 && !a.zpW && (!a.sumW || a.formula == F_BATCHED) &&
                                              (!RAG || a.formula == F_BATCHED || a.kb_dot * 64 >= a.K));

    for (int64_t work = blockIdx.x; work < nwork; work += gridDim.x) {
        // Shares of one tile are ntiles blocks apart (share-major).
        const int share = nshare == 1 ? 0 : static_cast<int>(work / ntiles);
        const int64_t m0 = (work - share * ntiles) * S::ROWS;
        // Quantise 4 RT rows per wave (rows 4 RT wid + 4 q + g, q < RT).
        {
            v4f x[RT][J];
            const int lr0 = 4 * RT * wid + g;
#pragma unroll
            for (int q = 0; q < RT; ++q) token_load4<J, RAG>(a, m0 + lr0 + 4 * q, r, x[q]);
#pragma unroll
            for (int q = 0; q < RT; ++q)
                token_quantise_row<J, FMT, RAG>(a, x[q], m0, lr0 + 4 * q, r, codes, S::ROW, lds_s, lds_sa);
        }
        __syncthreads();
        if (FMT == TG_FP8 || zero_terms)
            token_tile_gemm<KB, FMT, ACT, CT, RT, RAG, false>(a, codes, lds_s, lds_sa, strip, ctab, m0, wid, lane, share,
                                                          nshare);
        else
            token_tile_gemm<KB, FMT, ACT, CT, RT, RAG, FMT != TG_FP8>(a, codes, lds_s, lds_sa, strip, ctab, m0, wid,
                                                                  lane, share, nshare);
        __syncthreads();   // the next tile's quantise overwrites the codes
    }
}

}  // namespace nfq
