// gemm_fp8.hip -- launchers of the tiled GEMM on E4M3 codes (gemm_kernel.h).
#include "gemm_kernel.h"
#include "launch.h"

namespace nfq {

template <int TM, int TN, int OUT, int ACT>
static void launch_pipe_fp8(const RowsArgs& a, hipStream_t st) {
    using S = GemmShape<TM, TN>;
    const int64_t blocks = ((a.M + S::BM - 1) / S::BM) * ((a.N + S::BN - 1) / S::BN);
    const int groups = num_cus() % 8 == 0 ? 8 : 1;
    hipLaunchKernelGGL((k_gemm_pipe<TM, TN, OUT, ACT, 16, true>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                       a, groups);
}

// 128 x 128 tiles when they give every CU a block, else 64 x 64 (a lone
// block's K steps take half the time each, and there are four times the
// blocks).  Measured on MI355X (whole layer, us, 64 x 64 / 128 x 128): 1000 x
// 1024 -> 1024 11.1 / 15.7, 4096 x 2048 -> 512 27.6 / 33.7, 4096 x 1024 -> 1024
// 22.2 / 21.5, 65536 x 1024 -> 1024 242 / 178 (0.8 PFLOP/s; a large bf16
// library product reaches 1.27 on this card); N = 64 72.5 / 75.2.  128 x 256
// tiles spill (the bf16 fragments beside 128 accumulators): 189.
template <int OUT, int ACT>
static void launch_fp8_act(const RowsArgs& a, hipStream_t st) {
    const int t = kernel_path().gemm_tile.load(std::memory_order_relaxed);
    const int64_t blocks = ((a.M + 127) / 128) * ((static_cast<int64_t>(a.N) + 127) / 128);
    const bool small = t == 22 || (t != 44 && (a.N <= 64 || blocks < num_cus()));
    if (small) launch_pipe_fp8<2, 2, OUT, ACT>(a, st);
    else launch_pipe_fp8<4, 4, OUT, ACT>(a, st);
}

template <int OUT>
void launch_gemm_fp8(const RowsArgs& a, int act, hipStream_t st) {
    if constexpr (OUT == OUT_RAW) {
        launch_fp8_act<OUT, ACT_NONE>(a, st);
    } else {
        if (act == ACT_RELU) launch_fp8_act<OUT, ACT_RELU>(a, st);
        else if (act == ACT_GELU_TANH) launch_fp8_act<OUT, ACT_GELU_TANH>(a, st);
        else launch_fp8_act<OUT, ACT_NONE>(a, st);
    }
}

template void launch_gemm_fp8<OUT_EPI>(const RowsArgs&, int, hipStream_t);
template void launch_gemm_fp8<OUT_RAW>(const RowsArgs&, int, hipStream_t);

}  // namespace nfq
