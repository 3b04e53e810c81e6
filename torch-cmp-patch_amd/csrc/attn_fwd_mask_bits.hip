// Bit form of a bool attention mask, made on the device before a masked
// prefill of the pipelined kernel (attn_fwd_pipe16.h, OPT bit 11).
//
// A bool mask costs the attention kernel a load per key where its rows are
// not whole aligned runs (a [B,1,1531,1531] mask: 32 byte loads per lane and
// tile), and says nothing about which key tiles a query block needs at all.
// One pass over the mask, read once for all the heads that share it, leaves
//   words  [mask batch][mask head][32-key tile][mask row]: bit i of a word is
//          set when key 32 t + i exists and is kept; 128 bytes per wave and
//          tile, which ride the K/V ring into LDS;
//   class  [mask batch][mask head][128-row block][32-key tile], one byte: 0 no
//          pair kept (the tile is skipped: neither loaded nor scored), 2
//          every pair kept (nothing to apply), 1 mixed.
// Dimensions the mask broadcasts over (stride 0) have size 1 here; a mask of
// one row for all queries has one block.  Both arrays live in the caller's
// workspace behind the key split's exchange, rewritten by every call.
//
// Bound: latency, not bytes.  A lane holds one row, so a load touches 64 lines,
// and a last tile that is not whole is read byte by byte in a loop: 13.7 us for
// the 9.4 MB of a [4,1,1531,1531] mask (0.7 TB/s, a seventh of a copy's rate),
// of which the last tile has 27 single bytes per row.  Small beside what it
// saves: bf16 [4,16/8,1531,1531,128] with that mask, causal and left-padded,
// 492 us with the mask read by the element, 61 us with this pass and the tiles
// it lets the sweep skip.
#include "attn_common.h"

namespace cmpext3 {

namespace {

constexpr int kBitRows = 128;   // rows per class block: a query block of the attention kernel
constexpr int kBitTiles = 8;    // 32-key tiles per workgroup

typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(1)));

// bit i of the result: byte i of w (4 bytes) is not zero
__device__ __forceinline__ uint32_t nonzero_bits(uint32_t w) {
  const uint32_t t = ((((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) >> 7) & 0x01010101u;
  return (t * 0x01020408u) >> 24;
}

// Workgroup: 128 rows x 8 tiles.  Thread: one row x 4 neighbouring tiles, a
// whole 128-byte line of an aligned row.
__global__ void __launch_bounds__(256) attn_mask_bits(const MaskBits a) {
  const int tid = thread_x(), lane = tid & 63, wave = tid >> 6;
  const int half = wave & 1, sub = wave >> 1;  // rows 64 half .., tiles 4 sub ..
  const int nch = (a.nt + kBitTiles - 1) / kBitTiles;
  const int blk = block_x() / nch, ch = block_x() - blk * nch;
  const int nblk = (a.rows + kBitRows - 1) / kBitRows;
  const int bh = blk / nblk, rb = blk - bh * nblk;
  const int b = bh / a.heads, h = bh - b * a.heads;
  const int row = rb * kBitRows + half * 64 + lane;
  const bool live = row < a.rows;
  const unsigned char* const src = (const unsigned char*)a.mask + b * a.m_b + h * a.m_h + (int64_t)(live ? row : 0) * a.m_q;
  uint32_t* const words = a.words + (int64_t)bh * a.nt * a.rows;
  __shared__ unsigned char part[2][kBitTiles];  // [half][tile]: 1 some kept, 2 all kept
  u32x4u x[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = ch * kBitTiles + 4 * sub + i;
    if (32 * (t + 1) <= a.Sk) {
      x[i][0] = *(const u32x4u*)(src + 32 * t);
      x[i][1] = *(const u32x4u*)(src + 32 * t + 16);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = ch * kBitTiles + 4 * sub + i;
    if (t >= a.nt) break;
    uint32_t w = 0;
    if (32 * (t + 1) <= a.Sk) {
#pragma unroll
      for (int j = 0; j < 8; ++j) w |= nonzero_bits(x[i][j >> 2][j & 3]) << (4 * j);
    } else {  // the last, partial tile: keys past Sk are not read
      for (int k = 32 * t; k < a.Sk; ++k) w |= (src[k] ? 1u : 0u) << (k - 32 * t);
    }
    if (live) words[(int64_t)t * a.rows + row] = w;
    const bool some = __builtin_amdgcn_ballot_w64(live && w != 0u) != 0;
    const bool all = __builtin_amdgcn_ballot_w64(live && w != 0xffffffffu) == 0;
    if (lane == 0) part[half][4 * sub + i] = (some ? 1 : 0) | (all ? 2 : 0);
  }
  __syncthreads();
  const int t = ch * kBitTiles + tid;
  if (tid < kBitTiles && t < a.nt) {
    const unsigned char p0 = part[0][tid], p1 = part[1][tid];
    const int cls = (p0 & p1 & 2) ? 2 : ((p0 | p1) & 1);
    a.cls[((int64_t)bh * nblk + rb) * a.nt + t] = (unsigned char)cls;
  }
}

}  // namespace

bool mask_bits_plan(const FwdParams& p, MaskBits* a) {
  if (p.mask_kind != MASK_BOOL) return false;
  a->mask = p.mask;
  a->m_b = p.m_b;
  a->m_h = p.m_h;
  a->m_q = p.m_q;
  a->batch = p.m_b == 0 ? 1 : p.B;
  a->heads = p.m_h == 0 ? 1 : p.H;
  a->rows = p.m_q == 0 ? 1 : p.Sq;
  a->Sk = p.Sk;
  a->nt = (p.Sk + 31) / 32;
  if (a->nt > kMaskBitsMaxTiles) return false;
  const int64_t nblk = (a->rows + kBitRows - 1) / kBitRows;
  const int64_t bh = (int64_t)a->batch * a->heads;
  const int64_t words = bh * a->nt * a->rows, cls = bh * nblk * a->nt;
  // 32-bit offsets inside one (batch, head), and a bounded workspace
  if (words * 4 + cls > kMaskBitsMaxBytes) return false;
  a->words_bytes = (size_t)((words * 4 + 255) / 256 * 256);
  a->bytes = a->words_bytes + (size_t)((cls + 255) / 256 * 256);
  return true;
}

hipError_t launch_mask_bits(const MaskBits& a, hipStream_t s) {
  const int nblk = (a.rows + kBitRows - 1) / kBitRows, nch = (a.nt + kBitTiles - 1) / kBitTiles;
  hipLaunchKernelGGL(attn_mask_bits, dim3((unsigned)(a.batch * a.heads * nblk * nch)), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace cmpext3
