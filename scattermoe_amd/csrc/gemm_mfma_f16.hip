// fp16 instantiation of the MFMA kernels (gemm_mfma.hpp).
#include "gemm_mfma.hpp"

namespace smoe {

int dispatch_s2s_f16(const S2SArgs& a, bool b_tr, hipStream_t st) { return dispatch_s2s<f16_t>(a, b_tr, st); }

}  // namespace smoe
