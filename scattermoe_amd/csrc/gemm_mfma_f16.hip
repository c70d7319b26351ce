// fp16 instantiation of the MFMA kernels (gemm_mfma.hpp), K-contiguous weights; the others in gemm_mfma_f16_n.hip.
#define SMOE_LAYOUTS 1
#include "gemm_mfma.hpp"

namespace smoe {

int dispatch_s2s_f16_n(const S2SArgs& a, hipStream_t st);

int dispatch_s2s_f16(const S2SArgs& a, bool b_tr, hipStream_t st) {
  return b_tr ? dispatch_s2s_f16_n(a, st) : dispatch_s2s<f16_t>(a, false, st);
}

}  // namespace smoe
