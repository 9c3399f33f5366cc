// token_i8.hip -- the one-pass layer (token_gemm_kernel.h), per-token INT8.
#include "launch_token.h"

namespace nfq {

bool token_gemm_ok(const RowsArgs& a) {
    // K >= 4 and 16 bytes of weights: the loads clamped inside a row or the
    // matrix read whole 16 bytes.  N <= 2^24 keeps a 16-row output strip's
    // byte count inside a buffer range.
    return a.K >= 4 && a.K <= 1024 && a.N > 0 && a.N <= (1 << 24) && static_cast<int64_t>(a.N) * a.K >= 16;
}

// 16-row tiles while their (row tile, 128-column chunk) pairs number at most
// 5 per CU: a 64-row tile's quantise and product chain (10 us at K = 256, 16
// us at K = 512, most CUs idle) is then the launch, and a quarter of it wins
// although each weight byte is read four times as often.  Measured on MI355X
// (us, 16-row / 64-row tiles): 1500 x 256 -> 256 6.2 / 9.9, 6000 x 320 -> 256
// 9.8 / 18, 20000 x 192 -> 128 9.3 / 12.2; past the line 6000 x 256 -> 512
// 11.5 / 10.8, 8192 x 512 -> 1024 36 / 22.  K of 257 to 384 pays for a 512-wide
// 64-row tile: there 16-row tiles hold to 8 pairs per CU (12000 x 320 -> 256
// 11.9 / 18).  K > 512 has 16-row tiles only (a 64-row tile's codes would
// leave one block per CU).
bool token_small_tiles(const RowsArgs& a) {
    const int force = kernel_path().token_rows.load(std::memory_order_relaxed);
    if (force) return force == 16 || a.K > 512;
    if (a.K > 512) return true;
    const int64_t pairs = ((a.M + 15) / 16) * ((static_cast<int64_t>(a.N) + 127) / 128);
    return pairs <= (a.K > 256 && a.K <= 384 ? 8 : 5) * static_cast<int64_t>(num_cus());
}

void launch_token_i8(const RowsArgs& a, int act, hipStream_t st) { launch_token_fmt<TG_I8_TOKEN>(a, act, st); }

}  // namespace nfq
