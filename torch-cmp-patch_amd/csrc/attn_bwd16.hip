// Launch sequence of the attention backward (templates in attn_bwd16.h):
// Delta, then dK/dV over key blocks and dQ over query blocks in one launch, then
// the sums of what split sweeps left, all on the caller's stream.  Head dims up
// to 64 use the 64 bucket, up to 128 the 128 bucket, up to 192 and 256 those
// (columns past D are zero in every operand and never stored).
#include "attn_bwd16.h"

namespace cmpext3 {

namespace {

template <typename T, int DK, bool CAUSAL, bool MASK>
hipError_t launch_bwd_t(const BwdParams& p0, hipStream_t s) {
  BwdParams p = p0;
  const int64_t rows = (int64_t)p.B * p.H * p.Sq;
  hipLaunchKernelGGL(attn_bwd_delta<T>, dim3((unsigned)((rows + 31) / 32)), dim3(256), 0, s, p);
  p.n_blk = (p.Sk + 127) / 128;
  const int ns = p.nsplit > 1 && p.part ? p.nsplit : 1;
  p.nsplit = ns;
  if (ns == 1 || CAUSAL) p.nfull = 0;
  const int n_kv = p.B * p.Hkv * p.n_blk;
  p.n_wg = p.nfull > 0 ? p.nfull + (n_kv - p.nfull) * ns : n_kv * ns;
  p.n_blk_q = (p.Sq + 127) / 128;
  const int nsq = p.nsplit_q > 1 && p.part_q ? p.nsplit_q : 1;
  p.nsplit_q = nsq;
  if (nsq == 1 || CAUSAL) p.nfull_q = 0;
  const int n_q = p.B * p.H * p.n_blk_q;
  p.n_wg_q = p.nfull_q > 0 ? p.nfull_q + (n_q - p.nfull_q) * nsq : n_q * nsq;
  bool apart = false;
  if constexpr (DK == 64 && CAUSAL && MASK) {
    const int64_t slots = (int64_t)BwdDkdv<DK, CAUSAL, MASK>::OCC * device_cus();
    apart = last_round_full(n_kv, slots) && n_q >= 2 * slots && (n_kv >= 2 * slots || p.Sk >= 1792);
    if (apart) {
      hipLaunchKernelGGL((attn_bwd_grads<T, DK, CAUSAL, MASK, BWD_DKDV>), dim3(p.n_wg), dim3(256), 0, s, p);
      hipLaunchKernelGGL((attn_bwd_grads<T, DK, CAUSAL, MASK, BWD_DQ>), dim3(p.n_wg_q), dim3(256), 0, s, p);
    }
  }
  if (!apart) launch_both_sweeps(attn_bwd_grads<T, DK, CAUSAL, MASK, BWD_BOTH>, p, s);
  if (p.nfull > 0) {
    const int64_t n4 = (int64_t)(n_kv - p.nfull) * 128 * p.D / 4;
    hipLaunchKernelGGL((attn_bwd_tail_sum<T, true>), dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, p);
  }
  if (p.nfull_q > 0) {
    const int64_t n4 = (int64_t)(n_q - p.nfull_q) * 128 * p.D / 4;
    hipLaunchKernelGGL((attn_bwd_tail_sum<T, false>), dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, p);
  }
  launch_part_sums<T>(p, ns > 1 && p.nfull == 0, nsq > 1 && p.nfull_q == 0, s);
  return hipGetLastError();
}

template <typename T, bool MASK>
hipError_t launch_bwd_mask(const BwdParams& p, int dk, bool causal, hipStream_t s) {
  if (dk == 64) return causal ? launch_bwd_t<T, 64, true, MASK>(p, s) : launch_bwd_t<T, 64, false, MASK>(p, s);
  if (dk == 128) return causal ? launch_bwd_t<T, 128, true, MASK>(p, s) : launch_bwd_t<T, 128, false, MASK>(p, s);
  if (dk == 192) return causal ? launch_bwd_t<T, 192, true, MASK>(p, s) : launch_bwd_t<T, 192, false, MASK>(p, s);
  if (dk == 256) return causal ? launch_bwd_t<T, 256, true, MASK>(p, s) : launch_bwd_t<T, 256, false, MASK>(p, s);
  return hipErrorNotSupported;
}

template <typename T>
hipError_t launch_bwd_dtype(const BwdParams& p, int dk, bool causal, hipStream_t s) {
  return p.mask_kind != MASK_NONE ? launch_bwd_mask<T, true>(p, dk, causal, s)
                                  : launch_bwd_mask<T, false>(p, dk, causal, s);
}

}  // namespace

int bwd16_bucket(int D) { return D <= 0 ? -1 : D <= 64 ? 64 : D <= 128 ? 128 : D <= 192 ? 192 : D <= 256 ? 256 : -1; }

// Workgroups of the one launch that a CU holds.
template <int DK>
static int grads_occ(bool causal, bool masked) {
  if (masked) return causal ? bwd_occ<DK, true, true, BWD_BOTH>() : bwd_occ<DK, false, true, BWD_BOTH>();
  return causal ? bwd_occ<DK, true, false, BWD_BOTH>() : bwd_occ<DK, false, false, BWD_BOTH>();
}

// Split plan of the f16/bf16 gradient sweeps (split_sweep): dK/dV over
// 128-key blocks, each sweeping (query head of the group, 32-query tile);
// dQ over 128-query blocks, each sweeping 32-key tiles.
BwdSplit bwd16_split(int B, int H, int Hkv, int Sq, int Sk, int D, bool causal, bool masked, int cus) {
  BwdSplit sp;
  const int dk = bwd16_bucket(D);
  if (dk < 0 || (int64_t)B * H * Sq == 0 || Hkv < 1) return sp;
  const int occ = dk == 64    ? grads_occ<64>(causal, masked)
                  : dk == 128 ? grads_occ<128>(causal, masked)
                  : dk == 192 ? grads_occ<192>(causal, masked)
                              : grads_occ<256>(causal, masked);
  const int64_t n_kv = (int64_t)B * Hkv * ((Sk + 127) / 128), n_q = (int64_t)B * H * ((Sq + 127) / 128);
  const int64_t t_kv = (int64_t)(H / Hkv) * ((Sq + 31) / 32), t_q = (Sk + 31) / 32;
  // us per 32-row tile of one block, a CU to itself.  A mask costs dQ tiles more
  // than dK/dV ones (260 calls that both weighed 1.7, the dQ sweep of masked D <=
  // 64 at two workgroups per CU and a tail in any round planned otherwise: 7%
  // faster on average, 186 by over 3%, six slower by over 3%; dK/dV weighed 1, 22
  // slower by over 3%, some short grids of few heads by up to 20%)
  const float us_kv = (masked ? 1.25f : 1.f) * (dk <= 64 ? 0.74f : dk <= 128 ? 1.2f : dk <= 192 ? 2.f : 2.8f);
  const float us_q = (masked ? 1.7f : 1.f) * (dk <= 64 ? 0.49f : dk <= 128 ? 0.86f : dk <= 192 ? 1.35f : 1.83f);
  sp.ns_kv = split_sweep(n_kv, occ, cus, causal, t_kv, us_kv, 8e-6f * B * Hkv * Sk * D);
  sp.ns_q = split_sweep(n_q, occ, cus, causal, t_q, us_q, 4e-6f * B * H * Sq * D);
  // non-causal grids past one round: split only the last, partial round
  if (!causal && sp.ns_kv == 1) sp.ns_kv = split_tail(n_kv, occ, cus, t_kv, &sp.nfull_kv);
  if (!causal && sp.ns_q == 1) sp.ns_q = split_tail(n_q, occ, cus, t_q, &sp.nfull_q);
  return sp;
}

hipError_t launch_bwd16(const BwdParams& p, bool bf16, bool causal, hipStream_t s) {
  if ((int64_t)p.B * p.H * p.Sq == 0) return hipSuccess;
  const int dk = bwd16_bucket(p.D);
  return bf16 ? launch_bwd_dtype<__bf16>(p, dk, causal, s) : launch_bwd_dtype<_Float16>(p, dk, causal, s);
}

}  // namespace cmpext3
