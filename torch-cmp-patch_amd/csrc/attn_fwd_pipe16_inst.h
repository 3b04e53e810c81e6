// Tile table of the software-pipelined fp16/bf16 kernel (template in
// attn_fwd_pipe16.h) for head dims up to 128: which variant a planned launch
// runs.  Instantiated for one element type and Q scaling per source file
// (attn_fwd_pipe16_{f16,f16ps,bf16}.hip), which compile side by side.
//
// Like the v2 table in attn_fwd_mfma16.hip this replaces the reference's
// per-head-dim template table (src/cuda/fp16_flash_attention_hfma2.cu:278-285);
// entries come from an offline sweep on an MI355X.
#pragma once

#include "attn_fwd_pipe16.h"
#include "attn_fwd_plan16.h"

namespace cmpext3 {

// The mask is the same for every query row and is read in whole runs.
inline bool mask_bcast(const FwdParams& p) {
  return p.mask_kind != MASK_NONE && !p.mask_narrow && (p.m_q == 0 || p.Sq == 1);
}

template <typename T, int DK, bool CAUSAL, bool PRESCALE, int MOPT>
hipError_t launch_dk(const FwdParams& p, const SplitArgs& sa, hipStream_t s) {
  // OPT 1: s_setprio around the MFMA blocks; OPT 8: zero K columns past D;
  // OPT 16 (MOPT): attention mask
  constexpr int occ = MOPT ? pipe_occ_masked(DK) : pipe_occ(DK);
  // OPT 128: a single query block whose last waves hold no rows (decode,
  // packed query groups); those waves become the only K/V loaders and the
  // waves with rows only compute.  Taken with at least two rowless waves (the
  // loaders' chunk split assumes 128 or more loader threads); decode steps
  // run 0-20% faster than with every wave loading and computing.
  if constexpr (!CAUSAL && MOPT == 0) {
    if (p.Sq <= (kPipeNw - 2) * 32) {
      if (p.D == DK) return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 128>(p, sa, s);
      return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 8 | 128>(p, sa, s);
    }
  }
  // OPT 256 | 2: unmasked launches of the 32 / 64 / 128 buckets load K/V
  // tiles straight into swizzled LDS (no staging registers, one load
  // instruction per 2 KiB of tile, no bank conflicts; 3-4% faster on SDXL
  // self-attention, 6% on causal bf16 D = 128 than register staging).
  if constexpr (MOPT == 0 && (DK == 32 || DK == 64 || DK == 128)) {
    // OPT 512: stream-K (equal shares of the block-tile sequence; see
    // attn_fwd_pipe16.h), planned by launch_pipe16
    if constexpr (!CAUSAL) {
      if (sa.sk_wgs > 0) {
        if (p.D == DK) return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 256 | 512>(p, sa, s);
        return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 8 | 256 | 512>(p, sa, s);
      }
    }
    if (p.D == DK) return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 256>(p, sa, s);
    return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 8 | 256>(p, sa, s);
  }
  // masked launches of those buckets: the same LDS DMA, whose freed staging
  // registers the mask words use (masked fp16 D = 64 spilled 3-21 registers
  // with register staging; SDXL self-attention with a key-padding mask
  // 162 -> 121 us with the mask test of attn_fwd_pipe16.h)
  if constexpr (MOPT != 0 && (DK == 32 || DK == 64 || DK == 128)) {
    // OPT 1024: a query-broadcast mask read in runs (key padding [B,1,1,Sk]
    // and the like): its tile slices ride the DMA ring, no loads in the step
    if (mask_bcast(p)) {
      if (p.D == DK) return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 256 | 1024 | MOPT>(p, sa, s);
      return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 8 | 256 | 1024 | MOPT>(p, sa, s);
    }
    if (p.D == DK) return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 256 | MOPT>(p, sa, s);
    return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 2 | 8 | 256 | MOPT>(p, sa, s);
  }
  if (p.D == DK) return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | MOPT>(p, sa, s);
  return launch_pipe16_cfg<T, DK, kPipeNw, kPipeBk, occ, CAUSAL, PRESCALE, 1 | 8 | MOPT>(p, sa, s);
}

// Training forward (OPT 32: write the row log-sum-exp; MOPT 16: with an
// attention mask): buckets 64 and 128 only.
template <typename T, bool CAUSAL, bool PRESCALE, int MOPT>
hipError_t launch_lse_m(const FwdParams& p, const SplitArgs& sa, int dk, hipStream_t s) {
  // K/V straight into swizzled LDS, as for inference; query-broadcast masks
  // with K (OPT 1024)
  constexpr int LD = 2 | 256;
  if constexpr (MOPT != 0) {
    if (mask_bcast(p)) {
      if (dk == 64) {
        if (p.D == 64)
          return launch_pipe16_cfg<T, 64, kPipeNw, kPipeBk, pipe_occ(64), CAUSAL, PRESCALE, 1 | 32 | MOPT | LD | 1024>(p, sa, s);
        return launch_pipe16_cfg<T, 64, kPipeNw, kPipeBk, pipe_occ(64), CAUSAL, PRESCALE, 1 | 8 | 32 | MOPT | LD | 1024>(p, sa, s);
      }
      if (dk == 128) {
        if (p.D == 128)
          return launch_pipe16_cfg<T, 128, kPipeNw, kPipeBk, pipe_occ(128), CAUSAL, PRESCALE, 1 | 32 | MOPT | LD | 1024>(p, sa, s);
        return launch_pipe16_cfg<T, 128, kPipeNw, kPipeBk, pipe_occ(128), CAUSAL, PRESCALE, 1 | 8 | 32 | MOPT | LD | 1024>(p, sa, s);
      }
      return hipErrorNotSupported;
    }
  }
  if (dk == 64) {
    if (p.D == 64)
      return launch_pipe16_cfg<T, 64, kPipeNw, kPipeBk, pipe_occ(64), CAUSAL, PRESCALE, 1 | 32 | MOPT | LD>(p, sa, s);
    return launch_pipe16_cfg<T, 64, kPipeNw, kPipeBk, pipe_occ(64), CAUSAL, PRESCALE, 1 | 8 | 32 | MOPT | LD>(p, sa, s);
  }
  if (dk == 128) {
    if (p.D == 128)
      return launch_pipe16_cfg<T, 128, kPipeNw, kPipeBk, pipe_occ(128), CAUSAL, PRESCALE, 1 | 32 | MOPT | LD>(p, sa, s);
    return launch_pipe16_cfg<T, 128, kPipeNw, kPipeBk, pipe_occ(128), CAUSAL, PRESCALE, 1 | 8 | 32 | MOPT | LD>(p, sa, s);
  }
  return hipErrorNotSupported;
}

template <typename T, bool CAUSAL, bool PRESCALE>
hipError_t launch_lse(const FwdParams& p, const SplitArgs& sa, int dk, hipStream_t s) {
  return p.mask_kind != MASK_NONE ? launch_lse_m<T, CAUSAL, PRESCALE, 16>(p, sa, dk, s)
                                  : launch_lse_m<T, CAUSAL, PRESCALE, 0>(p, sa, dk, s);
}

// Narrow rows (OPT 64, FwdParams::elem_rows 4 or 8): inference, masked
// (MOPT 16) or not, buckets 64 and 128 only (other head dims are zero-padded
// up to them).
template <typename T, bool CAUSAL, int MOPT = 0>
hipError_t launch_narrow(const FwdParams& p, const SplitArgs& sa, int dk, hipStream_t s) {
  constexpr int occ64 = MOPT ? pipe_occ_masked(64) : pipe_occ(64);
  constexpr int occ128 = MOPT ? pipe_occ_masked(128) : pipe_occ(128);
  if (dk == 64)
    return launch_pipe16_cfg<T, 64, kPipeNw, kPipeBk, occ64, CAUSAL, false, 1 | 64 | MOPT>(p, sa, s);
  if (dk == 128)
    return launch_pipe16_cfg<T, 128, kPipeNw, kPipeBk, occ128, CAUSAL, false, 1 | 64 | MOPT>(p, sa, s);
  return hipErrorNotSupported;
}

template <typename T, bool CAUSAL, bool PRESCALE, int MOPT = 0>
hipError_t launch_bucket(const FwdParams& p, const SplitArgs& sa, int dk, hipStream_t s) {
  switch (dk) {
    case 32: return launch_dk<T, 32, CAUSAL, PRESCALE, MOPT>(p, sa, s);
    case 48: return launch_dk<T, 48, CAUSAL, PRESCALE, MOPT>(p, sa, s);
    case 64: return launch_dk<T, 64, CAUSAL, PRESCALE, MOPT>(p, sa, s);
    case 80: return launch_dk<T, 80, CAUSAL, PRESCALE, MOPT>(p, sa, s);
    case 96: return launch_dk<T, 96, CAUSAL, PRESCALE, MOPT>(p, sa, s);
    case 128: return launch_dk<T, 128, CAUSAL, PRESCALE, MOPT>(p, sa, s);
  }
  return hipErrorNotSupported;
}

// A planned launch of element type T: the training forward (masked or not),
// narrow rows (never pre-scaled: the narrow fp16 kernels then spill), masked
// (with causal, a pair must pass both rules) and plain launches.
template <typename T, bool PRESCALE>
hipError_t launch_pipe16_t(const FwdParams& p, const SplitArgs& sa, int dk, bool causal, hipStream_t s) {
  const bool masked = p.mask_kind != MASK_NONE;
  if (p.lse)
    return causal ? launch_lse<T, true, PRESCALE>(p, sa, dk, s) : launch_lse<T, false, PRESCALE>(p, sa, dk, s);
  if constexpr (!PRESCALE) {
    if (p.elem_rows) {
      if (masked) return causal ? launch_narrow<T, true, 16>(p, sa, dk, s) : launch_narrow<T, false, 16>(p, sa, dk, s);
      return causal ? launch_narrow<T, true>(p, sa, dk, s) : launch_narrow<T, false>(p, sa, dk, s);
    }
  }
  if (masked)
    return causal ? launch_bucket<T, true, PRESCALE, 16>(p, sa, dk, s)
                  : launch_bucket<T, false, PRESCALE, 16>(p, sa, dk, s);
  return causal ? launch_bucket<T, true, PRESCALE>(p, sa, dk, s) : launch_bucket<T, false, PRESCALE>(p, sa, dk, s);
}

}  // namespace cmpext3
