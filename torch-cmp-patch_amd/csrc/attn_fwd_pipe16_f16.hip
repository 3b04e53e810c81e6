// Instantiations of the software-pipelined kernel (tile table in
// attn_fwd_pipe16_inst.h): fp16, scores scaled after the product.
#include "attn_fwd_pipe16_inst.h"

namespace cmpext3 {

hipError_t launch_pipe16_f16(const FwdParams& p, const SplitArgs& sa, int dk, bool causal, hipStream_t s) {
  return launch_pipe16_t<_Float16, false>(p, sa, dk, causal, s);
}

}  // namespace cmpext3
