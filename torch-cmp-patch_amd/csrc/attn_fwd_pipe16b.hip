// Instantiations of the software-pipelined fp16/bf16 kernel (template in
// attn_fwd_pipe16.h) for bool masks in bit form (OPT bit 11; words and tile
// classes from attn_fwd_mask_bits.hip): non-causal inference launches of every
// head-dim bucket, K/V and the mask words straight into LDS.  Plan and
// dispatch in attn_fwd_plan16.hip.
#include "attn_fwd_pipe16.h"

namespace cmpext3 {

namespace {

// OPT 2: swizzled LDS rows where the bucket has them; OPT 8: K columns past D
// zeroed through the load offsets (free: they are fixed for the sweep)
template <typename T, int DK, bool PRESCALE>
hipError_t launch_bits_dk(const FwdParams& p, const SplitArgs& sa, hipStream_t s) {
  constexpr int occ = DK <= 64 ? 3 : DK <= 128 ? 2 : 1;
  constexpr int swz = DK == 32 || DK == 64 || DK == 128 ? 2 : 0;
  return launch_pipe16_cfg<T, DK, 4, 32, occ, false, PRESCALE, 1 | 8 | 256 | 2048 | swz>(p, sa, s);
}

template <typename T, bool PRESCALE>
hipError_t launch_bits(const FwdParams& p, const SplitArgs& sa, int dk, hipStream_t s) {
  switch (dk) {
    case 32: return launch_bits_dk<T, 32, PRESCALE>(p, sa, s);
    case 48: return launch_bits_dk<T, 48, PRESCALE>(p, sa, s);
    case 64: return launch_bits_dk<T, 64, PRESCALE>(p, sa, s);
    case 80: return launch_bits_dk<T, 80, PRESCALE>(p, sa, s);
    case 96: return launch_bits_dk<T, 96, PRESCALE>(p, sa, s);
    case 128: return launch_bits_dk<T, 128, PRESCALE>(p, sa, s);
    case 160: return launch_bits_dk<T, 160, PRESCALE>(p, sa, s);
    case 192: return launch_bits_dk<T, 192, PRESCALE>(p, sa, s);
    case 256: return launch_bits_dk<T, 256, PRESCALE>(p, sa, s);
  }
  return hipErrorNotSupported;
}

}  // namespace

hipError_t launch_pipe16_bits(const FwdParams& p, const SplitArgs& sa, int dk, bool bf16, bool prescale,
                              hipStream_t s) {
  if (bf16) return launch_bits<__bf16, false>(p, sa, dk, s);
  return prescale ? launch_bits<_Float16, true>(p, sa, dk, s) : launch_bits<_Float16, false>(p, sa, dk, s);
}

}  // namespace cmpext3
