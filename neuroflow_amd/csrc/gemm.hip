// gemm.hip -- launchers of the tiled INT8 MFMA GEMM (gemm_kernel.h).
#include "gemm_kernel.h"
#include "launch.h"
#include "wide_kernel.h"

namespace nfq {

bool gemm_ok(const RowsArgs& a) {
    // K <= 65536 keeps a 256-row tile's byte count inside the 32-bit buffer
    // range, N <= 2^24 a 16-row output strip's.
    return a.K % 64 == 0 && a.K >= 128 && a.K <= 65536 && a.N % 4 == 0 && a.N <= (1 << 24) && a.kb_dot * 64 >= a.K &&
           aligned(a.Aq, 16) && aligned(a.W, 16) && aligned(a.C, 16);
}

template <int TM, int TN, int OUT, int ACT>
static void launch_gemm_t(const RowsArgs& a, hipStream_t st) {
    auto kern = k_gemm<TM, TN, OUT, ACT>;
    constexpr size_t lds = gemm_lds_bytes<TM, TN>();
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    (void)attr;  // a failure surfaces as a launch error
    using S = GemmShape<TM, TN>;
    const int64_t blocks = ((a.M + S::BM - 1) / S::BM) * ((a.N + S::BN - 1) / S::BN);
    // MI355X deals blocks round-robin to 8 XCDs of 32 CUs.
    const int groups = num_cus() % 8 == 0 ? 8 : 1;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(256), lds, st, a, groups);
}

// Tile shape: 128 x 256 for large M and N (two blocks per CU); 64 x 64 while
// there are at most two per CU (a lone block's K steps take half the time), two
// and a half where the epilogue has integer terms; then 128 x 128, but with at
// most one per CU (one and a half for K <= 256) 64 x 128, which gives more blocks, where K <
// 1024 or the epilogue has terms.  Measured on MI355X (us, 64 x 64 / 64 x 128 /
// 128 x 128): codes in, int32 out, 4096 x 3072 -> 256 8.5 / 9.9 / 14.4, 12000 x
// 1536 -> 256 (752 blocks of 64 x 64) 12.2 / 9.8 / 9.7, 9000 x 2048 -> 384 17.4 /
// 12.6 / 11.7; a symmetric per-token layer with its quantise 2000 x 960 -> 512
// 14.0 / 15.1 / 17.7, 4096 x 640 -> 768 14.8 / 14.3 / 15.6, 8192 x 640 -> 1024 27.0 /
// 24.8 / 23.8; fixed scale with zero points 9000 x 1536 -> 256 (564) 30.4 / 31.6 /
// 32.9, 4096 x 2048 -> 928 31.6 / 28.3 / 29.3.  256 x 256 (one wave per SIMD) never
// beats 128 x 256.
static int gemm_shape(const RowsArgs& a) {
    // A gemm_tile override of 88|48|44|24|22 forces a shape (for tile sweeps;
    // 22 and 24 only on the LDS-DMA kernel).
    const int t = kernel_path().gemm_tile.load(std::memory_order_relaxed);
    if (t == 88 || t == 48 || t == 44 || t == 22 || t == 24) return t;
    if (a.M >= 16384 && a.N >= 1024) return 48;
    const int64_t cus = num_cus();
    const bool terms = a.zpW || a.zp_A != 0 || (a.formula == F_ROW_VNNI && a.sumW);
    const int64_t b64 = ((a.M + 63) / 64) * ((static_cast<int64_t>(a.N) + 63) / 64);
    if (a.N <= 64 || 2 * b64 <= (terms ? 5 : 4) * cus) return 22;
    const int64_t b128 = ((a.M + 127) / 128) * ((static_cast<int64_t>(a.N) + 127) / 128);
    return (a.K < 1024 || terms) && 2 * b128 <= (a.K <= 256 ? 3 : 2) * cus ? 24 : 44;
}

template <int TM, int TN, int OUT, int ACT>
static void launch_pipe_t(const RowsArgs& a, hipStream_t st) {
    using S = GemmShape<TM, TN>;
    const int64_t blocks = ((a.M + S::BM - 1) / S::BM) * ((a.N + S::BN - 1) / S::BN);
    const int groups = num_cus() % 8 == 0 ? 8 : 1;
    const int mf = kernel_path().gemm_mfma.load(std::memory_order_relaxed);
    if (mf == 32)
        hipLaunchKernelGGL((k_gemm_pipe<TM, TN, OUT, ACT, 32>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                           a, groups);
    else
        hipLaunchKernelGGL((k_gemm_pipe<TM, TN, OUT, ACT, 16>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                           a, groups);
}

// Whether the formula's integer terms take the weight-row byte sums.
bool gemm_needs_colsum(const RowsArgs& a) {
    return (a.formula == F_ROW_VNNI && (a.sumW || a.zp_A != 0)) || (a.formula == F_ROW_SCALAR && a.zp_A != 0);
}

// The LDS-DMA kernel takes every case whose epilogue needs no byte sums of
// its own: row sums given when zero points may be nonzero, and weight-row
// sums given when the formula takes them.
bool gemm_pipe_ok(const RowsArgs& a, int out) {
    if (path_flag(kernel_path().gemm_reg)) return false;
    if (out == OUT_RAW) return true;
    return (!a.zpW || a.sum_in) && (!gemm_needs_colsum(a) || a.colsum_in);
}

// The persistent GEMM (wide_kernel.h): the fused epilogue with K = 512 or
// 1024, per-row scales given, and the byte sums the formula needs
// given (row code sums with zero points, weight-row sums with a caller's
// sum_W in the row-VNNI formula), as for the LDS-DMA kernel.
static bool wide_ok(const RowsArgs& a, int out) {
    if (out != OUT_EPI || path_flag(kernel_path().no_wide) || path_flag(kernel_path().gemm_reg))
        return false;
    if (kernel_path().gemm_tile.load(std::memory_order_relaxed) != 0) return false;
    if (a.zp_A < -1024 || a.zp_A > 1024) return false;   // the kernel's 64-bit term
    if ((a.K != 512 && a.K != 1024) || a.N % 4 != 0 || !a.scale_in) return false;
    if (a.formula == F_ROW_SCALAR || static_cast<int64_t>(128) * a.N * 4 >= (int64_t(1) << 31)) return false;
    return (!a.zpW || a.sum_in) && (!gemm_needs_colsum(a) || a.colsum_in) && aligned(a.Aq, 16) && aligned(a.W, 16) &&
           aligned(a.C, 4);
}

template <int ACT, int INT_EPI, int NK, int TJ>
static void launch_wide_t(const RowsArgs& a, hipStream_t st) {
    using Cf = WideCfg<TJ>;
    const int64_t ntiles = ((a.M + Cf::BM - 1) / Cf::BM) * ((a.N + Cf::BN - 1) / Cf::BN);
    const int grid = static_cast<int>(std::min<int64_t>(ntiles, num_cus()));
    const int c0_mode = gemm_needs_colsum(a) ? 1 : 0;
    hipLaunchKernelGGL((k_gemm_wide<ACT, INT_EPI, NK, TJ>), dim3(grid), dim3(kWideThreads), 0, st, a,
                       static_cast<int>(ntiles), c0_mode);
}

// 128 x 256 tiles when they give every CU at least two (fewer loads per
// product, and the epilogue of one tile overlaps the next); else 128 x 128.
// Measured on MI355X at K = N = 1024: M = 65536 91-110 us (128 x 128:
// 107-116), M = 4096 11.2 us (128 x 256: 14.2), M = 10000, N = 1000 23 us
// (31).
template <int ACT, int INT_EPI, int NK>
static void launch_wide_k(const RowsArgs& a, hipStream_t st) {
    const int64_t t256 = ((a.M + 127) / 128) * ((a.N + 255) / 256);
    if (t256 >= 2 * static_cast<int64_t>(num_cus())) launch_wide_t<ACT, INT_EPI, NK, 2>(a, st);
    else launch_wide_t<ACT, INT_EPI, NK, 1>(a, st);
}

template <int ACT>
static void launch_wide(const RowsArgs& a, hipStream_t st) {
    const bool int_epi = a.zpW || (a.formula == F_ROW_VNNI && a.sumW);
    if (a.zp_A != 0) {
        // Fixed-scale layers only, which have no activation.
        if constexpr (ACT == ACT_NONE) {
            RowsArgs b = a;
            if (!b.sumW && gemm_needs_colsum(a)) b.sumW = a.colsum_in;
            if (a.K == 1024) launch_wide_k<ACT, 2, 8>(b, st);
            else launch_wide_k<ACT, 2, 4>(b, st);
        }
    } else if (int_epi) {
        if (a.K == 1024) launch_wide_k<ACT, 1, 8>(a, st);
        else launch_wide_k<ACT, 1, 4>(a, st);
    } else {
        if (a.K == 1024) launch_wide_k<ACT, 0, 8>(a, st);
        else launch_wide_k<ACT, 0, 4>(a, st);
    }
}

template <int OUT, int ACT>
static void launch_gemm_act(const RowsArgs& a, hipStream_t st) {
    if constexpr (OUT == OUT_EPI) {
        if (wide_ok(a, OUT) && (a.zp_A == 0 || ACT == ACT_NONE)) {
            launch_wide<ACT>(a, st);
            return;
        }
    }
    const int shape = gemm_shape(a);
    if (shape != 88 && gemm_pipe_ok(a, OUT)) {
        if (shape == 48) launch_pipe_t<4, 8, OUT, ACT>(a, st);
        else if (shape == 22) launch_pipe_t<2, 2, OUT, ACT>(a, st);
        else if (shape == 24) launch_pipe_t<2, 4, OUT, ACT>(a, st);
        else launch_pipe_t<4, 4, OUT, ACT>(a, st);
        return;
    }
    switch (shape) {
        case 88: launch_gemm_t<8, 8, OUT, ACT>(a, st); break;
        case 48: launch_gemm_t<4, 8, OUT, ACT>(a, st); break;
        default: launch_gemm_t<4, 4, OUT, ACT>(a, st); break;
    }
}

template <int OUT>
void launch_gemm(const RowsArgs& a, int act, hipStream_t st) {
    if constexpr (OUT == OUT_RAW) {
        launch_gemm_act<OUT, ACT_NONE>(a, st);
    } else {
        if (act == ACT_RELU) launch_gemm_act<OUT, ACT_RELU>(a, st);
        else if (act == ACT_GELU_TANH) launch_gemm_act<OUT, ACT_GELU_TANH>(a, st);
        else launch_gemm_act<OUT, ACT_NONE>(a, st);
    }
}

template void launch_gemm<OUT_EPI>(const RowsArgs&, int, hipStream_t);
template void launch_gemm<OUT_RAW>(const RowsArgs&, int, hipStream_t);

}  // namespace nfq
