// groupXtY instantiations of the MFMA kernels (gemm_mfma.hpp), and scatter2scatter's tiles of 192 columns: a source of their own so
// that they compile beside the other scatter2scatter ones.
#include "gemm_mfma.hpp"

namespace smoe {

int dispatch_xty_bf16(const XtYArgs& a, hipStream_t st) { return dispatch_xty<bf16_t>(a, st); }
int dispatch_xty_f16(const XtYArgs& a, hipStream_t st) { return dispatch_xty<f16_t>(a, st); }

template <typename T>
int launch_narrow(const S2SArgs& a, bool b_tr, hipStream_t st) {
  return launch_s2s<T, Tile<256, 192, 2, 2, 2, true>>(a, b_tr, st);
}
template int launch_narrow<bf16_t>(const S2SArgs&, bool, hipStream_t);
template int launch_narrow<f16_t>(const S2SArgs&, bool, hipStream_t);

}  // namespace smoe
