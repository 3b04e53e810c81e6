// Instantiations of the software-pipelined kernel (tile table in
// attn_fwd_pipe16_inst.h): fp16, Q pre-scaled by scale * log2(e).
#include "attn_fwd_pipe16_inst.h"

namespace cmpext3 {

hipError_t launch_pipe16_f16ps(const FwdParams& p, const SplitArgs& sa, int dk, bool causal, hipStream_t s) {
  return launch_pipe16_t<_Float16, true>(p, sa, dk, causal, s);
}

}  // namespace cmpext3
