// fp16 instantiation of the MFMA kernels (gemm_mfma.hpp), N-contiguous weights.
#define SMOE_LAYOUTS 2
#include "gemm_mfma.hpp"

namespace smoe {

int dispatch_s2s_f16_n(const S2SArgs& a, hipStream_t st) { return dispatch_s2s<f16_t>(a, true, st); }

}  // namespace smoe
