// launch_token.h -- the one-pass layer's launchers (token_gemm_kernel.h);
// included by the token_*.hip units, each instantiating one format.
#pragma once

#include "launch.h"
#include "token_gemm_kernel.h"

namespace nfq {

template <int KB, int FMT, int ACT, int CT, int RT, bool RAG>
static void launch_token_k(const RowsArgs& a, hipStream_t st) {
    auto kern = k_token_gemm<KB, FMT, ACT, CT, RT, RAG>;
    static const int per_cu = resident_blocks(kern);
    const int64_t tiles = (a.M + 16 * RT - 1) / (16 * RT);
    const int64_t slots = static_cast<int64_t>(num_cus()) * per_cu;
    // Fewer row tiles than resident blocks: the column chunks of a tile are
    // shared out over several blocks, each quantising the tile for itself (not
    // in place: one of them could write rows that another has yet to read).
    const int64_t chunks = in_place(a) ? 1 : (a.N + 64 * CT - 1) / (64 * CT);
    const int64_t share = std::max<int64_t>(1, std::min<int64_t>(chunks, slots / tiles));
    const int64_t grid = std::min<int64_t>(tiles * share, slots);
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(grid)), dim3(256), 0, st, a, static_cast<int>(share));
}

template <int KB, int FMT, int CT, int RT, bool RAG>
static void launch_token_act(const RowsArgs& a, int act, hipStream_t st) {
    if constexpr (FMT != TG_I8_FIXED) {
        if (act == ACT_RELU) return launch_token_k<KB, FMT, ACT_RELU, CT, RT, RAG>(a, st);
        if (act == ACT_GELU_TANH) return launch_token_k<KB, FMT, ACT_GELU_TANH, CT, RT, RAG>(a, st);
    }
    launch_token_k<KB, FMT, ACT_NONE, CT, RT, RAG>(a, st);
}

template <int FMT, int CT, int RT>
static void launch_token_rag(const RowsArgs& a, int act, hipStream_t st) {
    if (a.K <= 64) launch_token_act<1, FMT, CT, RT, true>(a, act, st);
    else if (a.K <= 128) launch_token_act<2, FMT, CT, RT, true>(a, act, st);
    else if (a.K <= 256) launch_token_act<4, FMT, CT, RT, true>(a, act, st);
    else if (RT == 4 || a.K <= 512) launch_token_act<8, FMT, CT, RT, true>(a, act, st);
    else if constexpr (RT == 1) launch_token_act<16, FMT, CT, RT, true>(a, act, st);
}

template <int FMT, int CT>
static void launch_token_whole(const RowsArgs& a, int act, hipStream_t st) {
    if (a.K == 128) launch_token_act<2, FMT, CT, 4, false>(a, act, st);
    else if (a.K == 256) launch_token_act<4, FMT, CT, 4, false>(a, act, st);
    else launch_token_act<8, FMT, CT, 4, false>(a, act, st);
}

// 64-row tiles: 32 columns per wave for N <= 128 (64 leave two waves without
// columns), and for K <= 64 up to N = 512, where the short K loop gains more from
// the third block per CU than from the wider strip (us, 64 columns / 32: fixed
// scale 200000 x 64 -> 132 62.6 / 50.1, -> 300 93.5 / 75.3, 40000 -> 512 29.0 / 22.1;
// FP8 and per-token alike; FP8 53783 x 48 -> 512, whose tiles just pass a round
// of three blocks, 28.4 / 32.8; wider, FP8 23854 x 64 -> 1268 84 / 94).
template <int FMT>
static void launch_token_fmt(const RowsArgs& a, int act, hipStream_t st) {
    if (token_small_tiles(a)) return launch_token_rag<FMT, 2, 1>(a, act, st);
    const bool narrow = a.N <= 128 || (a.K <= 64 && a.N <= 512);
    if (!token_whole(a)) return narrow ? launch_token_rag<FMT, 2, 4>(a, act, st) : launch_token_rag<FMT, 4, 4>(a, act, st);
    if (narrow) launch_token_whole<FMT, 2>(a, act, st);
    else launch_token_whole<FMT, 4>(a, act, st);
}

}  // namespace nfq
