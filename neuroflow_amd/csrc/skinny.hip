// skinny.hip -- launchers of the few-row layer (skinny_kernel.h).
#include "launch.h"
#include "skinny_kernel.h"

namespace nfq {

// At most 4096 features (four 64-wide blocks per wave), K >= 4 and 16 bytes of
// weights (the clamped 16-byte loads).
bool skinny_ok(const RowsArgs& a) {
    return a.K >= 4 && a.K <= 4096 && a.N > 0 && static_cast<int64_t>(a.N) * a.K >= 16 &&
           (a.M + 15) / 16 <= 65535;
}

template <int FMT, int ACT>
static void launch_skinny_k(const RowsArgs& a, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((a.N + 15) / 16), static_cast<unsigned>((a.M + 15) / 16));
    if (a.K <= 256) hipLaunchKernelGGL((k_skinny<4, 1, FMT, ACT>), grid, dim3(256), 0, st, a);
    else if (a.K <= 1024) hipLaunchKernelGGL((k_skinny<16, 1, FMT, ACT>), grid, dim3(1024), 0, st, a);
    else if (a.K <= 2048) hipLaunchKernelGGL((k_skinny<16, 2, FMT, ACT>), grid, dim3(1024), 0, st, a);
    else hipLaunchKernelGGL((k_skinny<16, 4, FMT, ACT>), grid, dim3(1024), 0, st, a);
}

template <int FMT>
static void launch_skinny_act(const RowsArgs& a, int act, hipStream_t st) {
    if (act == ACT_RELU) launch_skinny_k<FMT, ACT_RELU>(a, st);
    else if (act == ACT_GELU_TANH) launch_skinny_k<FMT, ACT_GELU_TANH>(a, st);
    else launch_skinny_k<FMT, ACT_NONE>(a, st);
}

void launch_skinny_i8(const RowsArgs& a, int act, hipStream_t st) { launch_skinny_act<TG_I8_TOKEN>(a, act, st); }
void launch_skinny_i8_fixed(const RowsArgs& a, hipStream_t st) { launch_skinny_k<TG_I8_FIXED, ACT_NONE>(a, st); }
void launch_skinny_fp8(const RowsArgs& a, int act, hipStream_t st) { launch_skinny_act<TG_FP8>(a, act, st); }

}  // namespace nfq
