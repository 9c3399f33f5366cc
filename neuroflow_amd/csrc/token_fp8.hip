// token_fp8.hip -- the one-pass layer (token_gemm_kernel.h), per-token FP8 E4M3.
#include "launch_token.h"

namespace nfq {

void launch_token_fp8(const RowsArgs& a, int act, hipStream_t st) { launch_token_fmt<TG_FP8>(a, act, st); }

}  // namespace nfq
