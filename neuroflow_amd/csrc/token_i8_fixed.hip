// token_i8_fixed.hip -- the one-pass layer (token_gemm_kernel.h), INT8 with
// one scale and zero point for every row.
#include "launch_token.h"

namespace nfq {

void launch_token_i8_fixed(const RowsArgs& a, hipStream_t st) { launch_token_fmt<TG_I8_FIXED>(a, ACT_NONE, st); }

}  // namespace nfq
