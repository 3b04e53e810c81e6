// Launch plans of the software-pipelined fp16/bf16 kernel (attn_fwd_pipe16.h):
// which problems it takes, the key split, stream-K, the bit form of bool
// masks, and the exchange space of every split kernel.
//
// The key split (no counterpart in the reference) needs exchange space, and
// the library allocates none: the workspace entry points take it from the
// caller (cmpext3_attn_fwd_workspace_size says how much), the
// allocation-free entry point uses a fixed per-device array in this file
// (`scratch` below), and every other call runs unsplit.  bind_exchange, the
// one place a plan meets its space, serves all the split kernels.
#include <stdio.h>

#include <mutex>

#include "attn_fwd_plan16.h"

namespace cmpext3 {

namespace {

// Split plan limits: a part scans at least kMinPartTiles key tiles (shorter
// parts spend more on their prologue and merge than they save); with no
// whole round a CU holds at most kMaxPartsPerCu parts at once.
constexpr int kMinPartTiles = 8;
constexpr int kMaxPartsPerCu = 2;
constexpr int kMaxCausalParts = 8;       // parts per causal block at most
constexpr int kMinCausalPartTiles = 16;  // tiles of a causal block's longest part at least
constexpr int kMinManyCausalTiles = 24;  // the same with more than two parts
constexpr int kMinTailTiles = 32;        // tiles of a prefill block whose last half round is cut
constexpr int kLongCausalTiles = 64;     // a long causal sweep (the last block's tiles)
constexpr int kMi355xCus = 256;  // used when no device is visible (host-only calls)

int n_blocks(int B, int H, int Sq) { return B * H * ((Sq + kPipeNw * 32 - 1) / (kPipeNw * 32)); }
int n_key_tiles(int Sk) { return (Sk + kPipeBk - 1) / kPipeBk; }
// Key tiles of query block `nb - 1`'s sweep: all of them, or under causal
// those up to the block's last query row.
int causal_tiles(int Sk, int nb, bool causal) {
  const int64_t kend = causal ? (int64_t)nb * kPipeNw * 32 : Sk;
  return n_key_tiles(kend < Sk ? (int)kend : Sk);
}

// ---- Exchange storage of the allocation-free entry point
//
// One fixed array per device in the library's code object, zero-filled when
// the code object is loaded on a device and never allocated or freed by the
// library: the counters, then 16 MiB of partial (O, m, l) vectors (the
// layout of every exchange space, attn_common.h).  Every allocation-free
// call on a device shares it.  Host code never passes `scratch` itself to a
// kernel (in host code the name is only a stand-in for the device symbol):
// the device address comes from hipGetSymbolAddress, once per device.
constexpr size_t kScratchWsBytes = size_t(16) << 20;
constexpr size_t kScratchBytes = kExchangeCounterBytes + kScratchWsBytes;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// This device's scratch address, looked up on the first call with the device
// current (a failed lookup is retried on the next call; until one succeeds
// the allocation-free calls run unsplit).  Nothing is launched: the code
// object's zero fill is the counters' initial state.
void* scratch_ptr() {
  static std::mutex mu;
  static void* ptrs[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    ptrs[dev] = ptr;
  }
  return ptrs[dev];
}

// Waves per block that hold query rows: all of them unless the launch is a
// single block shorter than the workgroup (decode, packed grouped-query rows).
int exchange_waves(int n_qblk, int Sq) {
  return n_qblk > 1 ? kPipeNw : (Sq + 31) / 32 < kPipeNw ? (Sq + 31) / 32 : kPipeNw;
}

// What the plan weighs besides the grid: the head-dim bucket, the element type,
// and whether the block is short (decode, packed rows: at most 64 rows, a
// launch bound by the K/V stream).
struct PlanKind {
  int dk;
  bool f16, shortq;
};

// Whether two parts exchange O / l in fp16: fp16 launches whose grid and sweep
// allow two parts and no more (SDXL self-attention).  Where more would fit and
// the plan takes two because they are faster, as where fewer would, the
// exchange is fp32, as that of three and more: a second fp16 rounding of O
// would make the result less exact than the finer cut it replaces (rms
// error against 64 bits, N(0,1) inputs, [1,12,1024,1024,64]: 1.15 times the
// unsplit one with the fp16 exchange, 1.00 with fp32).
bool half_exchange(const PlanKind& k, int most) { return k.f16 && most == 2; }

// Cost of cutting a block's sweep in two, in key tiles of one block: the
// prologue, the exchange and the merge of one block (about 3 us) and each
// further block's share of the exchange's bytes.  Fitted on MI355X to
// [1,H,S,S,D] with 32 to 240 blocks (D = 48, 64, 128 and 256, S = 512 to
// 3072): where it exceeds the tiles a cut saves, the cut launch was the slower
// one, by up to half (bf16 [1,32,1024,1024,128], 256 blocks: 24 us whole, 37
// us cut), and with few exceptions only there.
float cut_cost(int dk, bool half, int n) {
  const float per_block = dk > 128 ? 0.057f : dk > 64 ? (half ? 0.063f : 0.114f) : (half ? 0.034f : 0.063f);
  const float base = !half || dk > 128 ? 6.f : dk > 64 ? 7.f : 8.f;
  return base + per_block * n;
}

// Parts of every block of a non-causal prefill with fewer blocks than CUs
// (half: two of them exchange in fp16).
// With a part to a CU, P parts save nt (1 - 1/P) tiles; two parts beyond that
// share CUs and save 0.38 nt (above D = 128 a CU holds one workgroup: nothing).
// Three parts and more all leave fp32 states, and from four on a launch pays
// another 5 (D > 128) or 12 tiles: bf16
// [1,8,1024,1024,D], 64 blocks, whole / in 2 / 3 / 4 parts, D = 64: 16.1 / 13.8
// / 12.8 / 17.2 us, D = 128: 21.5 / 19.9 / 19.4 / 23.1, D = 256: 46.7 / 37.5 /
// 34.3 / 37.1.
int prefill_parts(int dk, bool half, int n, int nt, int cus, int occ) {
  const float save2 = nt * (2 * n <= cus ? 0.5f : occ > 1 ? 0.38f : 0.f) - cut_cost(dk, half, n);
  int parts = save2 > 0.f ? 2 : 1;
  float best = save2 > 0.f ? save2 : 0.f;
  for (int p = 3; p <= nt / kMinPartTiles && n * p <= cus; ++p) {
    const float many = p > 3 ? (dk > 128 ? 5.f : 12.f) : dk > 64 && dk <= 128 ? 2.f : 0.f;
    const float save = nt * (1.f - 1.f / p) - cut_cost(dk, false, n * p / 2) - many;
    if (save > best) {
      best = save;
      parts = p;
    }
  }
  return parts;
}

// Which blocks run whole and how the rest are cut.  n blocks on `cus` CUs at
// `occ` workgroups per CU; the dispatcher hands workgroup i to CU i mod cus
// while all of them fit, so after the whole rounds each CU takes exactly one
// part.  ntiles: key tiles of a block (causal: of the longest block, whose
// sweep reaches the last query; ntiles_min those of the shortest, the first
// query block's).
//
// Causal launches keep their longest-first order.  Where the blocks fill at
// most half of the workgroup slots and either leave more than half of the
// CUs without a block or sweep long key ranges (at least kLongCausalTiles
// tiles for the last block), every block is cut into the same number of
// parts so that one round holds them all, the longest part keeping at least
// kMinCausalPartTiles tiles: each block's longest part, and so the launch,
// gets shorter.  Measured on MI355X (same run): [1,4,8192,128] bf16 135 ->
// 98 us, [1,8,2048,256] 85 -> 54 us, [1,8,1024,64] 17.2 -> 13.8 us; shorter
// sweeps on busy CUs lost to the parts' prologues and merges
// ([1,32,1024,128] 25 -> 28 us, [1,32,512,128] 16 -> 18 us) and stay whole.
// More than two parts want longer ones (kMinManyCausalTiles: bf16
// [1,16,2048,64] 29.2 whole, 23.1 in 2, 26.7 in 3; [1,8,2048,128] 39.2 / 27.1 /
// 27.9, 35.3 in 4), and where four would fill more than 3/4 of the slots three
// are better ([1,8,3072,64] 25.3 in 3, 32.1 in 4; below that [1,2,6000,64] 32.3
// in 3, 28.9 in 4).  Where the parts still have a CU each, shorter ones pay as
// well ([1,2,2048,64] 19.2 in 2, 14.7 in 4; [1,4,2048,128] 26.1 / 21.3;
// [1,2,2048,256] 52.8 / 38.3), and at three workgroups per CU three parts of up
// to half as many blocks as CUs ([1,6,2048,64] 19.8 in 2, 17.3 in 3, 18.5 in 4;
// [1,8,2048,64] 20.0 / 17.8).
// Every part of every block keeps at least one tile (a causal row sees a key in
// the first tile of a part, or none of the part's keys: its state then has no
// weight in the merge).
SplitArgs split_plan(int n, int ntiles, int occ, int cus, bool causal, int ntiles_min, const PlanKind& k) {
  SplitArgs sa = {n, 1, nullptr, nullptr, kPipeNw};
  if (cus <= 0) return sa;
  if (causal) {
    const int slots = occ * cus;
    if (n * 2 > slots || (n * 2 > cus && ntiles < kLongCausalTiles)) return sa;
    int most = slots / n;
    if (most > ntiles / kMinCausalPartTiles) most = ntiles / kMinCausalPartTiles;
    if (most > ntiles_min) most = ntiles_min;
    if (most > kMaxCausalParts) most = kMaxCausalParts;
    int parts = most;
    if (parts > 2 && parts > ntiles / kMinManyCausalTiles)
      parts = ntiles / kMinManyCausalTiles > 2 ? ntiles / kMinManyCausalTiles : 2;
    if (parts > 3 && n * 16 > slots * 3) parts = 3;
    int own = cus / n;  // parts that have a CU each
    if (occ >= 3 && own < 3 && n * 2 <= cus) own = 3;
    if (own > most) own = most;
    if (parts < own) parts = own;
    if (parts < 2) return sa;
    sa.nfull = 0;
    sa.nparts = parts;
    sa.half16 = half_exchange(k, most);
    return sa;
  }
  const int full = n / cus, rem = n - full * cus;
  if (rem == 0 || full + 1 > occ) return sa;  // whole rounds, or more than fits at once
  // After whole rounds each CU takes at most one part of the round that
  // remains.  With no whole round each CU can hold several parts at once: more
  // key ranges streamed side by side, more loads in flight (a decode step with
  // one part per CU reaches ~5.2 TB/s).
  const int per_cu = full == 0 ? (occ < kMaxPartsPerCu ? occ : kMaxPartsPerCu) : 1;
  int most = per_cu * cus / rem;
  if (most > ntiles / kMinPartTiles) most = ntiles / kMinPartTiles;
  int parts = most;
  if (full == 0 && !k.shortq) {
    parts = prefill_parts(k.dk, k.f16 && most <= 2, n, ntiles, cus, occ);
  } else if (full > 0 && !k.shortq) {
    // the tail of a prefill: two parts (bf16 [1,20,2048,2048,64], 64 blocks
    // left: whole 35.8 us, 2 parts 31.8, 3 32.2, 4 33.9), and where each CU
    // would take little less than a whole block more, only of long sweeps
    // ([1,64,768,768,64], 128 left: 17.9 whole, 18.2 cut; 1536: 29.8, 28.1)
    if (parts > 2) parts = 2;
    if (rem * 2 >= cus && ntiles < kMinTailTiles) parts = 1;
  }
  if (parts < 2) return sa;
  sa.nfull = full * cus;
  sa.nparts = parts;
  sa.half16 = half_exchange(k, most);
  return sa;
}

// Stream-K (OPT 512): for non-causal, unmasked inference launches of the
// LDS-DMA buckets whose blocks fill at least the CUs but not whole rounds of
// the occ * cus workgroup slots.  The launch is then ceil(n / slots) rounds
// of workgroups, each taking an equal share of the n * ntiles block-tile
// sequence (with the classic plan the CUs of the last round would idle once
// their half-blocks end: SDXL self-attention, 640 blocks on 768 slots).
// Shares of fewer than kMinPartTiles tiles would spend more on prologues and
// merges than they balance; the counters take 2 per (block, wave).
constexpr int kMaxStreamkWaves = kExchangeCounters / 2;

bool streamk_applies(const FwdParams& p, int n, int dk, int occ, int cus, bool causal, bool half) {
  if (causal || p.lse || p.elem_rows || p.mask_kind != MASK_NONE || p.pack_sq > 0) return false;
  if (!(dk == 32 || dk == 64 || dk == 128) || p.Sq <= (kPipeNw - 2) * 32) return false;
  const int slots = occ * cus;
  if (cus <= 0 || n < cus || n % slots == 0 || n * kPipeNw > kMaxStreamkWaves) return false;
  // Only where the classic plan leaves slots idle for the whole launch and the
  // sweeps are long enough to repay a second prologue per share and a merge
  // per block: one block per CU (no block left to split; D <= 64 fp16
  // [2,4,4096,4096,64] 48.9 -> 44.5 us, bf16 50.7 -> 46.7, but 28.1 -> 31.6 at
  // 2048 keys; D = 128 fp16 77.3 -> 74.0, bf16 72.9 -> 74.7), or, at two
  // workgroups per CU, a last round at most a quarter full (bf16
  // [2,10,4096,4096,128], 640 blocks, 187 -> 180; half full, 768 blocks of
  // [1,32,3072,3072,128], 153 -> 160).  Two blocks per CU of three lose on
  // shorter sweeps ([1,32,2048,2048,64] 41.4 -> 46.7).  Where the classic plan splits the
  // blocks past the whole CUs, it measured faster (SDXL self-attention 91.1 us
  // against 97.7 us stream-K, same run).
  const int nt = n_key_tiles(p.Sk);
  const bool idle_round = n < slots && n % cus == 0 && (dk > 64 ? half && nt >= 128 : nt >= (n == cus ? 72 : 128));
  const bool thin_tail = n > slots && occ == 2 && n % slots <= slots / 4 && nt >= 64;
  if (!idle_round && !thin_tail) return false;
  const int64_t rounds = (n + slots - 1) / slots;
  return (int64_t)n * nt / (rounds * slots) >= kMinPartTiles;
}

// The stream-K launch: workgroup count and part slots per block (an upper
// bound on the shares one block's tiles can touch).
SplitArgs streamk_plan(int n, int ntiles, int occ, int cus) {
  const int slots = occ * cus;
  const int W = (n + slots - 1) / slots * slots;
  const int share = (int)((int64_t)n * ntiles / W);  // tiles per share, rounded down
  SplitArgs sa = {0, ntiles / share + 2, nullptr, nullptr, kPipeNw, W};
  return sa;
}

}  // namespace

// The instantiation of a planned launch up to D = 128 (narrow rows are never
// pre-scaled).
static hipError_t launch_pipe16_kernel(const FwdParams& p, const SplitArgs& sa, int dk, bool bf16, bool causal,
                                       bool prescale, hipStream_t s) {
  if (bf16) return launch_pipe16_bf16(p, sa, dk, causal, s);
  return prescale && !p.elem_rows ? launch_pipe16_f16ps(p, sa, dk, causal, s) : launch_pipe16_f16(p, sa, dk, causal, s);
}

// A bool mask goes to bit form first (attn_fwd_mask_bits.hip) where that repays
// the extra launch (3-4 us).  Read element by element (narrow), it does from
// the shortest sweeps on: fp16 [2,10,4096,77,64] with a padding mask 23.4 ->
// 15.6 us, [1,12,77,77,64] 16.8 -> 9.5, bf16 [4,16,1531,1531,128] causal and
// padded 492 -> 61.  In whole runs: above D = 64 from 256 keys (bf16
// [4,16/8,S,S,128] at S = 256: 24.3 -> 17.0 us causal and padded, 20.6 -> 15.6
// key padding; at 2048: 198 -> 76 and 160 -> 141); up to D = 64 past 256 keys
// with a row for each query ([4,32,S,S,64] at S = 256: 13.5 -> 14.4, at 288:
// 17.5 -> 14.2), and, since one row for all queries rides the ring in runs for
// little, with that only from 768 (at 600: 25.8 -> 27.9, at 768: 33.5 -> 32.6).
bool mask_bits_applies(const FwdParams& p, bool causal) {
  MaskBits a;
  if (causal || p.lse || p.elem_rows || p.mask_kind != MASK_BOOL || !mask_bits_plan(p, &a)) return false;
  if (p.mask_narrow) return p.Sk >= 32;
  if (p.D > 64) return p.Sk >= 256;
  return a.rows > 1 ? p.Sk > 256 : p.Sk >= 768;
}

// The space for a mask's bit form: behind the `used` bytes of exchange of the
// caller's workspace (or the fixed scratch).  Null when it does not fit.
static char* bits_space(const FwdParams& p, size_t used, size_t bytes) {
  char* const base = p.fixed_exchange ? (char*)scratch_ptr() : (char*)p.workspace;
  const size_t room = p.fixed_exchange ? kScratchBytes : p.workspace_bytes;
  used = (used + 255) / 256 * 256;
  return base && used + bytes <= room ? base + used : nullptr;
}

// Compute units of the current device (256 on MI355X), cached per device.
int device_cus() {
  static int cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    return kMi355xCus;
  }
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
      (void)hipGetLastError();
      return kMi355xCus;
    }
    cus[dev] = n;
  }
  return cus[dev];
}

int bind_exchange(const FwdParams& p, int parts, size_t part_bytes, int ncnt, f32x4** ws, int** cnt) {
  *ws = nullptr;
  *cnt = nullptr;
  if (parts < 2) return 1;
  // the space this call may use: the fixed scratch, or the caller's workspace
  void* base = nullptr;
  size_t bytes = 0;
  if (p.dry) {
    p.dry->need = kExchangeCounterBytes + (size_t)parts * part_bytes;
    bytes = p.fixed_exchange ? kScratchBytes : p.workspace_bytes;
  } else if (p.fixed_exchange) {
    base = scratch_ptr();
    bytes = base ? kScratchBytes : 0;
  } else if (p.workspace) {
    base = p.workspace;
    bytes = p.workspace_bytes;
  }
  // as many key ranges as the partials room holds, if the counters fit
  int fit = 0;
  if (bytes > kExchangeCounterBytes && ncnt <= kExchangeCounters && part_bytes > 0) {
    const size_t room = (bytes - kExchangeCounterBytes) / part_bytes;
    fit = room < (size_t)parts ? (int)room : parts;
  }
  if (fit < 2) fit = 1;
  if (p.dry) {
    p.dry->parts = fit;
    return fit;
  }
  if (fit >= 2) {
    *cnt = (int*)base;
    *ws = (f32x4*)((char*)base + kExchangeCounterBytes);
  }
  return fit;
}

// True when the pipelined kernel takes this problem: head-dim bucket <= 128,
// a key sweep long enough for its prologue (four tiles in flight) to pay off
// (shorter sweeps run faster on the short-key and v2 kernels) unless an
// attention mask or the log-sum-exp output is asked for (up to D = 128 only
// this kernel has them), and K/V tiles addressable with 32-bit buffer
// offsets.  Above D = 128: launches with whole-chunk rows whose query
// blocks hold rows in at least three of their four waves (fewer rows: the
// decode and packed-row paths) and sweep at least kPipeMinSk keys, masked or
// not, inference or training.
constexpr int kPipeMinSk = 256;

bool pipe16_applies(const FwdParams& p, int dk) {
  if (dk > 128 && (p.elem_rows || p.Sq <= (kPipeNw - 2) * 32 || p.Sk < kPipeMinSk)) return false;
  if (p.Sk < kPipeMinSk && p.mask_kind == MASK_NONE && !p.lse) return false;
  const int64_t rs = p.k_s > p.v_s ? p.k_s : p.v_s;
  return (int64_t)(p.Sk + kPipeBk) * rs * 2 < (int64_t(1) << 31);
}

// `prescale` applies to fp16 (Q * scale * log2(e) must stay finite).  bf16
// never pre-scales: rounding Q*c to 8 mantissa bits moves each score by up to
// 2^-9 of its size, which at scale 1 (scores of tens of log2 units) breaks
// the 2e-2 bf16 bar, so bf16 scores get one FMA each instead.
// Grouped-query launches whose query heads hold less than one block of rows
// each (decode, short prefills) pack the G query heads of a K/V head into the
// rows of one problem: the K/V of that head is then streamed once for all of
// them, instead of once per query head with mostly empty blocks.  Non-causal
// inference launches only (the row position then does not matter), unmasked
// unless the kernel reads the mask by packed row (masked_rows: the decode
// kernel).
constexpr int kPackMaxSq = 64;

bool packs_query_heads(const FwdParams& p, bool causal, bool masked_rows) {
  return !causal && p.kv_group > 1 && p.Sq <= kPackMaxSq && (masked_rows || p.mask_kind == MASK_NONE) && !p.lse &&
         p.pack_sq == 0 && (int64_t)p.kv_group * p.Sq <= (int64_t)INT32_MAX / 2;
}

void pack_query_heads(FwdParams& p) {
  const int G = p.kv_group;
  p.pack_sq = p.Sq;
  p.q_g = p.q_h;
  p.o_g = p.o_h;
  p.m_g = p.m_h;
  p.m_h *= G;
  p.q_h *= G;  // packed head hk starts at query head hk * G
  p.o_h *= G;
  p.H /= G;
  p.Sq *= G;
  p.kv_group = 1;
}

hipError_t launch_pipe16(const FwdParams& p0, int dk0, bool bf16, bool causal, bool prescale, hipStream_t s) {
  FwdParams p = p0;
  if (packs_query_heads(p, causal, false)) pack_query_heads(p);
  // the training forward and the narrow-row variants have the 64 and 128
  // buckets only up to D = 128; above it the training forward has 192 and
  // 256, and neither it nor masked launches pre-scale Q (one instantiation
  // per dtype)
  const int dk = dk0 > 128 ? (p.lse && dk0 < 192 ? 192 : dk0)
                           : (p.lse || p.elem_rows) ? (dk0 <= 64 ? 64 : 128) : dk0;
  if (dk > 128 && (p.lse || p.mask_kind != MASK_NONE)) prescale = false;
  if (p.elem_rows && (p.elem_rows < 4 || p.lse)) return hipErrorNotSupported;
  // Without pre-scaling, masked keys enter as raw -inf and meet the multiplier
  // c in one FMA; scale 0 would make that 0 * -inf.  A multiplier of 1e-30
  // instead leaves every finite score's exp2 argument within 1e-22 of -m,
  // which rounds to the same probability as scale 0 gives, and keeps -inf.
  if ((!prescale || p.elem_rows) && p.c == 0.f) p.c = 1e-30f;
  const int cus = device_cus();
  const int occ = p.mask_kind != MASK_NONE ? pipe_occ_masked(dk) : pipe_occ(dk);
  const int n = n_blocks(p.B, p.H, p.Sq);
  const int dp = (dk + 31) / 32 * 32;
  // stream-K where it applies and its exchange fits the space this call has
  size_t sk_need = 0;
  if (streamk_applies(p, n, dk, occ, cus, causal, !bf16)) {
    SplitArgs sk = streamk_plan(n, n_key_tiles(p.Sk), occ, cus);
    const size_t part_bytes = (size_t)n * kPipeNw * split_vectors(dp) * 64 * sizeof(f32x4);
    const int fit = bind_exchange(p, sk.nparts, part_bytes, 2 * n * kPipeNw, &sk.ws, &sk.cnt);
    if (p.dry) sk_need = p.dry->need;
    if (fit == sk.nparts) {
      if (p.dry) return hipSuccess;
      return launch_pipe16_kernel(p, sk, dk, bf16, false, prescale, s);
    }
  }
  const int n_qblk = (p.Sq + kPipeNw * 32 - 1) / (kPipeNw * 32);
  SplitArgs sa = split_plan(n, causal_tiles(p.Sk, n_qblk, causal), occ, cus, causal, causal_tiles(p.Sk, 1, causal),
                            {dk, !bf16, p.Sq <= (kPipeNw - 2) * 32});
  sa.nwl = exchange_waves((p.Sq + kPipeNw * 32 - 1) / (kPipeNw * 32), p.Sq);
  if (p.dry) *p.dry = SplitInfo{0, 1};  // the stream-K attempt's record, if any, is not this plan
  if (sa.nparts > 1) {
    // Exchange space: the fixed scratch or the caller's workspace, cut to
    // fewer key ranges when the plan does not fit it (an unsplit launch needs
    // none, so no problem is ever refused for want of space).  The plan keeps
    // its whole blocks; only the split blocks' part count changes.
    const int nsplit = n - sa.nfull;
    const size_t part_bytes = (size_t)nsplit * sa.nwl * split_vectors(dp) * 64 * sizeof(f32x4);
    sa.nparts = bind_exchange(p, sa.nparts, part_bytes, 2 * nsplit * sa.nwl, &sa.ws, &sa.cnt);
    if (sa.nparts < 2) sa = SplitArgs{n, 1, nullptr, nullptr, sa.nwl};
  }
  if (p.dry) {
    // the size query reports the best plan's need (stream-K's, when it applies)
    if (sk_need > p.dry->need) p.dry->need = sk_need;
    MaskBits mb;
    if (mask_bits_applies(p, causal) && mask_bits_plan(p, &mb)) p.dry->bits = mb.bytes;
    return hipSuccess;
  }
  if (mask_bits_applies(p, causal)) {
    MaskBits mb;
    mask_bits_plan(p, &mb);
    const size_t nsplit = sa.nparts > 1 ? n - sa.nfull : 0;
    char* const at = bits_space(
        p, kExchangeCounterBytes + nsplit * sa.nparts * sa.nwl * split_vectors(dp) * 64 * sizeof(f32x4), mb.bytes);
    if (at) {
      mb.words = (uint32_t*)at;
      mb.cls = (unsigned char*)at + mb.words_bytes;
      const hipError_t err = launch_mask_bits(mb, s);
      if (err != hipSuccess) return err;
      const int64_t nblk = (mb.rows + kPipeNw * 32 - 1) / (kPipeNw * 32);
      p.bits = mb.words;
      p.bit_cls = mb.cls;
      p.bit_rows = mb.rows;
      p.bits_h = mb.heads > 1 ? (int64_t)mb.nt * mb.rows : 0;
      p.bits_b = mb.batch > 1 ? (int64_t)mb.heads * mb.nt * mb.rows : 0;
      p.cls_h = mb.heads > 1 ? nblk * mb.nt : 0;
      p.cls_b = mb.batch > 1 ? mb.heads * nblk * mb.nt : 0;
      return launch_pipe16_bits(p, sa, dk, bf16, prescale, s);
    }
  }
  if (dk > 128) return launch_pipe16_wide(p, sa, dk, bf16, causal, prescale, s);
  return launch_pipe16_kernel(p, sa, dk, bf16, causal, prescale, s);
}

void describe_pipe16(int dk, int B, int H, int Sq, int Sk, bool causal, bool narrow, bool bf16, char* buf, int len) {
  const int bq = kPipeNw * 32;
  const int n = n_blocks(B, H, Sq);
  const int n_qblk = (Sq + bq - 1) / bq;
  const SplitArgs sa = split_plan(n, causal_tiles(Sk, n_qblk, causal), pipe_occ(dk), device_cus(), causal,
                                  causal_tiles(Sk, 1, causal), {dk, !bf16, Sq <= (kPipeNw - 2) * 32});
  char split[96] = "";
  FwdParams p = {};
  p.Sq = Sq;
  p.Sk = Sk;
  p.mask_kind = MASK_NONE;
  p.elem_rows = narrow ? 4 : 0;
  if (streamk_applies(p, n, dk, pipe_occ(dk), device_cus(), causal, !bf16)) {
    const SplitArgs sk = streamk_plan(n, n_key_tiles(Sk), pipe_occ(dk), device_cus());
    snprintf(split, sizeof split, " stream-K: %d workgroups x %lld tiles of %d blocks (with a workspace)", sk.sk_wgs,
             (long long)n * n_key_tiles(Sk) / sk.sk_wgs, n);
  } else if (sa.nparts > 1) {
    snprintf(split, sizeof split, " key-split: %d whole + %d x %d parts", sa.nfull, n - sa.nfull, sa.nparts);
  }
  snprintf(buf, len,
           "pipe16 mfma 32x32x16 S^T-form, K one tile ahead of V: DK=%d DP=%d waves=%d BQ=%d BK=%d "
           "waves/SIMD=%d qtiles=%d%s",
           dk, (dk + 31) / 32 * 32, kPipeNw, bq, kPipeBk, pipe_occ(dk), (Sq + bq - 1) / bq, split);
}

}  // namespace cmpext3
