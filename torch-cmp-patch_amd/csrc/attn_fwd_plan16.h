// Tiles and occupancies of the software-pipelined fp16/bf16 kernel, shared by
// its instantiations (attn_fwd_pipe16_inst.h) and its launch plans
// (attn_fwd_plan16.hip).  All buckets use 4-wave workgroups and 32-key tiles;
// the waves per SIMD are the most the registers allow without spilling (D =
// 32: 4, D <= 64: 3, D <= 128: 2; above 128 one, with accumulation registers
// as the spill space).
#pragma once

#include "attn_common.h"

namespace cmpext3 {

constexpr int kPipeNw = 4;
constexpr int kPipeBk = 32;
constexpr int pipe_occ(int dk) { return dk <= 32 ? 4 : dk <= 64 ? 3 : dk <= 128 ? 2 : 1; }
// masked launches need a few more registers: D = 32 drops to 3 waves per SIMD
constexpr int pipe_occ_masked(int dk) { return dk <= 64 ? 3 : dk <= 128 ? 2 : 1; }

hipError_t launch_pipe16_f16(const FwdParams& p, const SplitArgs& sa, int dk, bool causal, hipStream_t s);
hipError_t launch_pipe16_f16ps(const FwdParams& p, const SplitArgs& sa, int dk, bool causal, hipStream_t s);
hipError_t launch_pipe16_bf16(const FwdParams& p, const SplitArgs& sa, int dk, bool causal, hipStream_t s);
hipError_t launch_pipe16_wide(const FwdParams& p, const SplitArgs& sa, int dk, bool bf16, bool causal,
                              bool prescale, hipStream_t s);
hipError_t launch_pipe16_bits(const FwdParams& p, const SplitArgs& sa, int dk, bool bf16, bool prescale,
                              hipStream_t s);

}  // namespace cmpext3
