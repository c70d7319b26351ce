// groupXtY instantiations of the MFMA kernels (gemm_mfma.hpp), a source of their own so that they compile beside the
// scatter2scatter ones.
#include "gemm_mfma.hpp"

namespace smoe {

int dispatch_xty_bf16(const XtYArgs& a, hipStream_t st) { return dispatch_xty<bf16_t>(a, st); }
int dispatch_xty_f16(const XtYArgs& a, hipStream_t st) { return dispatch_xty<f16_t>(a, st); }

}  // namespace smoe
