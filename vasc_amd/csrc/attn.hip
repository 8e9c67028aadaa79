// Kernel 4: block-sparse flash attention forward for gfx950 (bf16 MFMA).
//
// Semantics follow SpargeAttn's block-sparse kernel
// (ZIP:csrc/qattn/qk_int_sv_f16_cuda_sm80.cuh:42-738): one workgroup per
// (128-row query block, head, batch) walks only the 64-key blocks named by
// its list, with a base-2 softmax and masking of keys past the end. The
// arithmetic is bf16 MFMA with fp32 accumulation instead of int8 QK^T + fp16
// PV, and the structure is CDNA4's:
//
//  * 4 waves x 32 query rows (two tiles of 16). S^T = K Q^T on
//    v_mfma_f32_16x16x32_bf16, so a lane owns one query row of each tile
//    (lane % 16) and 16 of the 64 keys of a block.
//  * The clock falls to a mean of 1.67 GHz of 2.4 under this kernel (counters
//    of a launch over 33312 keys, 16 heads and 132 blocks a row), so what a
//    block costs in energy counts. On random operands the 16x16x32 product
//    sustains 1.59 PFLOP/s at 2.06 GHz and the 32x32x16 one 1.50 at 1.89
//    (accumulators move half the register bytes per product). The change of
//    shape took that launch from 1.13 to 1.02 ms.
//  * O^T = Vt P^T on the same MFMA, so P feeds the B operand straight from
//    the S^T accumulators. Vt comes from vasc_pack_v with its keys permuted;
//    row i of S^T tile u of a 32-key group is key 8 u + 16 (i / 8) + i % 8 of
//    the group, which puts the probabilities in exactly that order.
//  * Row sums are products too: a ones operand against P, 4 of the block's 36
//    MFMAs. v_dot2 (the former row sum) shares the matrix pipe: 16 of them
//    beside 16 MFMAs and the exponentials cost a wave-block 350 cycles, the
//    products 47 (probe without memory, four waves per SIMD).
//  * The kernel is held to 128 VGPRs so four waves share each SIMD: MFMAs of
//    one wave overlap the exponentials of the others. In the launch above a
//    wave-block takes 943 cycles, 576 of them MFMA; in a probe without memory
//    770, where two waves of 64 rows per SIMD, which halve the LDS reads, took
//    980 (exposed latencies).
//  * Softmax is invariant to the exponent offset, which only has to keep the
//    probabilities inside fp32/bf16 range. The walk uses offset 0:
//    P = exp2(c S) on the exact fp32 logits, no max, no rescale, no branch.
//    Where c is 1 the product goes too. A row sum outside [2^-60, 2^120]
//    (looked at after blocks 0, 8, 24, 56, .. and at the end) sends the
//    workgroup through a second walk, whose offset follows the row maximum and
//    which also takes blocks outside the sequence; a walk that is about to leave
//    the range goes on in that form from where it stands. Checking and rescaling
//    per block cost 2 % of the launch. Both walks take Q from the registers and
//    only the last one stores, so the output may lie on Q's storage. Over 33312
//    keys, 16 heads, 132 blocks a row, q and k of std 1 / 4 / 8 take 1.05 /
//    1.15 / 1.12 ms (offset moved per block in the first walk: 1.17 / 1.20 /
//    1.60; second walk with a new maximum each block: 1.06 / 1.88 / 1.48). The
//    first walk ends a block after the look that failed: leaving at once, by a
//    break or an empty block, costs every launch 0.3 to 1 % (or spills).
//  * Keys past the sequence end (the partial last block) read the last key's
//    row: their V rows are zero and the ones operand is zeroed there.
//  * K and Vt tiles arrive by LDS DMA (global_load_lds_dwordx4) into a
//    double-buffered LDS tile one block ahead of the MFMAs. The 16-byte
//    chunks of a row are xor-swizzled so that the 16 rows of an operand read
//    fill all LDS banks: by (row/2)%8 in Vt; K operand rows are 0-7 and
//    16-23 (8-15, 24-31) of a group, so row bit 4 replaces bit 3 there. The
//    DMA is issued through asm without a memory clobber (the explicit waits
//    and barriers order it), so the compiler neither drains it before LDS
//    reads nor turns the uniform list reads into vector loads: the lists are
//    read through the constant address space on the scalar unit, and nothing
//    but the DMA counts in vmcnt inside the loop. Q is consumed before the
//    loop so that its load wait stays out of the loop body.
//  * workgroup ids are remapped so each XCD walks a contiguous range of
//    query blocks of the same head (K/V reuse in that XCD's L2).
//  * vasc_global_attn_fwd adds the layer's special-token queries, which
//    attend to every key (attention.py:8480-8484), to the same launch: their
//    workgroups take the first hardware ids, so they start first (each walks
//    every key block, about four times the work of a patch-query
//    workgroup), and they are remapped like the patch workgroups, so each
//    XCD takes the special queries of the heads whose patch queries it
//    walks and reads their K and V through the same L2.
#include <type_traits>

#include "common.h"

namespace vasc {
namespace {

constexpr int kBlockQ = 128;
constexpr int kBlockK = 64;
constexpr int kHeadDim = 64;
constexpr int kThreads = 256;
constexpr int kTile = kBlockK * kHeadDim;  // elements of one K or Vt tile

struct AttnParams {
  const uint16_t *q;
  int64_t q_sb, q_sh, q_st;
  const uint16_t *k;
  int64_t k_sb, k_sh, k_st;
  const uint16_t *vt;
  uint16_t *o;
  int64_t o_sb, o_sh, o_st;
  int64_t H, nq, nk, nqb, nkb;
  const int32_t *idx;
  int64_t idx_w;
  const int32_t *cnt;
  int32_t delta;
  float c;  // sm_scale * log2(e)
  int64_t num_wg;
  // special-token queries (dense over every key block), NULL when absent
  const uint16_t *q2;
  int64_t q2_sb, q2_sh, q2_st;
  uint16_t *o2;
  int64_t o2_sb, o2_sh, o2_st;
  int64_t nq2, nq2b, num_wg2, num_wg2_slots;
  // token-major output (tok_p > 0): query rows land on the frame-major token
  // rows of o (frames of tok_p tokens, tok_s special ones first)
  int64_t tok_p, tok_s;
  int32_t half_io;  // q and o are IEEE halves: q rounded to bf16 as it is read, o the bf16 result widened
  // 1: workgroups in hardware order, head-major (sequences whose K and V of
  // eight heads, one per XCD, would overflow the Infinity Cache); 0: each
  // XCD walks a contiguous range of query blocks
  int32_t head_major;
  // PV post-cut: per-head thresholds in log2 units and the
  // per-wave execution map [B, H, nqb * 4, pv_w] (written where PV ran)
  const float *pv_thr;
  int32_t *pv_map;
  int64_t pv_w;
  // key split of the special queries: nsplit workgroups walk split_blocks key
  // blocks each and leave float32 partial results, [num_wg2][nsplit][128 rows]
  // of 64 outputs of the part's keys alone, then of log2 of the row sums
  int32_t nsplit, split_blocks;
  float *part;
};

__device__ __forceinline__ floatx16 mfma32(u32x4 a, u32x4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Sum of a packed bf16 pair added to acc (v_dot2c_f32_bf16 with (1, 1)).
__device__ __forceinline__ float add_bf16_pair(uint32_t pair, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair),
                                         __builtin_bit_cast(bf16x2, 0x3f803f80u), acc, false);
}

// LDS chunk swizzle of tile row r (16-byte chunks, 8 per 128-byte row).
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

// Exact-path triggers: a lane's block sum above kHigh (a probability may be
// near overflow) or a running sum below kLow (the row's logits are so far
// below m that they lose precision).
constexpr float kHigh = 18446744073709551616.0f;  // 2^64
constexpr float kLow = 8.673617379884035e-19f;    // 2^-60
// Row sums at exponent offset 0 are good in [2^-60, 2^120]: below, products of
// small probabilities and small values would be flushed; above, the largest
// ones near overflow. The accumulated outputs are checked for finiteness beside
// them. A walk whose sums will leave the range is better left early: above 2^72
// after the first block (3.9 standard deviations, the largest of its 8192
// scores, where the walk's largest of a million lie at 4.9 to 5.2), later above
// 2^104. Sums still in the range then are kept and the second form goes on from
// them, 5 to 10 % slower a block; a walk left late starts again, at twice the time.
// Kept against started again, std 4: 17 blocks a row 193 -> 178 us, 9 blocks
// 19.1 -> 17.1, 34 blocks 103 -> 97 (offset moved per block: 184, 16.5, 100).
constexpr uint32_t kHighBits = 0x7b800000u, kLaterBits = 0x73800000u, kFirstBits = 0x63800000u, kLowBits = 0x21800000u;
// Second walk (see compute_online).
constexpr float kRaise = 64.f, kMargin = 32.f;
constexpr uint32_t kLeave = 1u, kRedo = 2u;

constexpr int kMaxSplit = 8;  // workgroups that share a special-query block's keys

// LDS DMA without a memory clobber (the waits and barriers that order it are
// explicit); uniform list reads then stay on the scalar unit.
__device__ __forceinline__ void dma16(const void *sbase, uint32_t voff_bytes, uint32_t lds_addr) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(lds_addr), "v"(voff_bytes), "s"(sbase));
}

__device__ __forceinline__ floatx4 mfma16(u32x4 a, u32x4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// LDS chunk swizzle of K tile row r in bsattn_fwd_kernel (see above).
__device__ __forceinline__ int swz_k(int r) { return ((r >> 1) & 3) | ((r >> 2) & 4); }


// Normalised results of a wave's two query tiles; a row without any
// probability is zero. sp: the special-query outputs.
__device__ __forceinline__ void store_rows(const AttnParams &p, bool sp, int64_t b, int64_t h, int64_t row0, int64_t nq,
                                           int lr, int g4, const floatx4 (&oacc)[2][4], const floatx4 (&lacc)[2]) {
  uint16_t *odst = sp ? p.o2 + b * p.o2_sb + h * p.o2_sh : p.o + b * p.o_sb + h * p.o_sh;
  const int64_t o_st = sp ? p.o2_st : p.o_st;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t qrow = row0 + 16 * i + lr;
    if (qrow >= nq) continue;
    int64_t orow = qrow;
    if (p.tok_p > 0) {
      const int64_t per = sp ? p.tok_s : p.tok_p - p.tok_s;  // queries per frame of this kind
      orow = (orow / per) * p.tok_p + (sp ? 0 : p.tok_s) + orow % per;
    }
    uint16_t *optr = odst + orow * o_st;
    const float ltot = lacc[i][0];
    const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      uint2 v;
      v.x = pack_bf16x2(oacc[i][t][0] * inv, oacc[i][t][1] * inv);
      v.y = pack_bf16x2(oacc[i][t][2] * inv, oacc[i][t][3] * inv);
      if (p.half_io) v = uint2{bf16x2_to_half2(v.x), bf16x2_to_half2(v.y)};
      *reinterpret_cast<uint2 *>(optr + 16 * t + 4 * g4) = v;
    }
  }
}

// kDense: every key block instead of a list. kUnit: c = 1 (sm_scale = ln 2:
// the queries hold log2(e) times the softmax scale, as the global layer packs
// them), so the probabilities are exp2(S) without a product per score: 690
// cycles a wave-block against 770 and 1.00 ms against 1.06 on lists of 132 of
// 521 blocks, 16 heads.
template <bool kDense, bool kUnit, bool kSplit>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void bsattn_fwd_kernel(const AttnParams p) {
  constexpr int CH = 512 / kThreads;  // 16-byte chunks per thread per tile
  constexpr uint32_t kBufBytes = 2 * kTile * 2;
  __shared__ __attribute__((aligned(2 * kBufBytes))) uint16_t smem[2][2][kTile];  // [buffer][K, Vt]
  __shared__ uint32_t redo;  // a wave's row sums are about to leave the range of offset 0 (kLeave) or have left it (kRedo)

  // Workgroups [0, num_wg2_slots) take the special-token queries (every key
  // block; the slot count is rounded up to a multiple of the 8 XCDs so that
  // both ranges start on XCD 0); the rest the patch queries of their lists.
  const bool dense = kDense || static_cast<int64_t>(blockIdx.x) < p.num_wg2_slots;
  const int64_t nqb = dense && !kDense ? p.nq2b : p.nqb;
  const int64_t hw = dense && !kDense ? static_cast<int64_t>(blockIdx.x)
                                      : static_cast<int64_t>(blockIdx.x) - p.num_wg2_slots;
  const int64_t wg = p.head_major ? hw : xcd_remap(hw, dense && !kDense ? p.num_wg2_slots : p.num_wg);
  const bool sp = dense && !kDense;  // a special-query workgroup
  if (sp && wg >= p.num_wg2 * (kSplit ? p.nsplit : 1)) return;  // padding of the special-query slots
  const int64_t unit = kSplit && sp ? wg / p.nsplit : wg;
  const int split = kSplit && sp ? static_cast<int>(wg % p.nsplit) : 0;
  const int qb = static_cast<int>(unit % nqb);
  const int64_t bh = unit / nqb;
  const int64_t h = bh % p.H;
  const int64_t b = bh / p.H;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave index, uniform
  // What depends on the lane alone is formed again after the walk instead of
  // kept through it, where every register is taken.
  int tid, lr, g4;
  auto lanes = [&]() __attribute__((always_inline)) {
    int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(l));
    tid = w * kWave + l;
    lr = l & 15;
    g4 = l >> 4;
  };
  lanes();

  int n;
  const int32_t *list = nullptr;
  const int blk0 = kSplit && sp ? split * p.split_blocks : 0;  // first block of a dense walk
  if (dense) {
    n = static_cast<int>(p.nkb) - blk0;
    if (kSplit && sp && n > p.split_blocks) n = p.split_blocks;
  } else {
    const int64_t row = bh * p.nqb + qb;
    list = p.idx + row * p.idx_w;
    n = p.cnt[row];
    n = n < 0 ? 0 : (n > p.idx_w ? static_cast<int>(p.idx_w) : n);
  }

  const uint16_t *qsrc = sp ? p.q2 : p.q;
  const int64_t q_sb = sp ? p.q2_sb : p.q_sb, q_sh = sp ? p.q2_sh : p.q_sh, q_st = sp ? p.q2_st : p.q_st;
  const int64_t nq = sp ? p.nq2 : p.nq;
  const int64_t row0 = static_cast<int64_t>(qb) * kBlockQ + w * 32;
  // a wave whose 32 rows all lie past the queries (the short last block of
  // the special queries) only stages its share of the tiles
  const bool idle = row0 >= nq;
  if (tid == 0) redo = 0;

  // Q as the B operand of S^T = K Q^T: lane holds row lr of tile i, d = 32s + 8 g4 .. +7.
  u32x4 qf[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t qrow = row0 + 16 * i + lr;
    const uint16_t *qptr = qsrc + b * q_sb + h * q_sh + (qrow < nq ? qrow : 0) * q_st;
#pragma unroll
    for (int s = 0; s < 2; ++s)
      qf[i][s] = qrow < nq ? *reinterpret_cast<const u32x4 *>(qptr + 32 * s + 8 * g4) : u32x4{0, 0, 0, 0};
  }
  if (p.half_io) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) qf[i][s] = half8_to_bf16(qf[i][s]);
  }
  // consume Q here so that the compiler's wait for these loads lands before
  // the loop instead of inside it
  asm volatile("" ::"v"(qf[0][0]), "v"(qf[0][1]), "v"(qf[1][0]), "v"(qf[1][1]));

  // Staging: LDS chunk ci = u*256 + tid lands at byte 16*ci (the DMA writes
  // lane i of a wave at base + 16*i); it holds tile row ci/8, logical chunk
  // (ci%8) ^ swizzle(row), so each lane fetches that global chunk. Both
  // swizzles are the same for row 32u + r as for r: a thread's byte offset
  // inside the block stays, and the row base (32u rows) goes into the scalar
  // base address.
  const uint16_t *kbase = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t *vbase = p.vt + (bh * p.nkb) * kTile;
  const int nk32 = static_cast<int>(p.nk);
  const int nkb32 = static_cast<int>(p.nkb);
  const int partial = (nk32 % kBlockK) ? nkb32 - 1 : -1;  // the partial last block, if any
  int r0, kc;
  uint32_t koff, voff;
  const uint32_t lds0 = lds_addr32(smem[0][0]);
  // K and Vt of block blk -> LDS buffer buf. Blocks outside [0, nkb) load
  // block 0 (the second walk masks them); rows of the partial block past the
  // sequence end read its last row.
  auto fetch = [&](int blk, int buf) __attribute__((always_inline)) {
    const int sb = (blk >= 0 && blk < nkb32) ? blk : 0;
    const uint16_t *kb = kbase + static_cast<int64_t>(sb) * kBlockK * p.k_st;
    const uint16_t *vb = vbase + static_cast<int64_t>(sb) * kTile;
    const uint32_t kd = lds0 + w * 64 * 16 + buf * kBufBytes, vd = kd + kTile * 2;
    if (sb == partial) {
      const int last_row = nk32 - 1 - partial * kBlockK;
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int r = 32 * u + r0;
        const int rr = r < last_row ? r : last_row;
        dma16(kb, static_cast<uint32_t>((static_cast<int64_t>(rr) * p.k_st + kc) * 2), kd + u * kThreads * 16);
      }
    } else {
#pragma unroll
      for (int u = 0; u < CH; ++u) dma16(kb + 32 * u * p.k_st, koff, kd + u * kThreads * 16);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) dma16(vb + 32 * u * kHeadDim, voff, vd + u * kThreads * 16);
  };
  // Keys of block blk that exist: 64, fewer for the partial last block, 0
  // for blocks outside [0, nkb).
  auto valid_keys = [&](int blk) __attribute__((always_inline)) {
    return (blk >= 0 && blk < nkb32) ? (blk == partial ? nk32 - blk * kBlockK : kBlockK) : 0;
  };

  const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};
  const float c = p.c;
  floatx4 oacc[2][4];  // O^T: [q tile][d tile]
  floatx4 lacc[2];     // row sums of the bf16 probabilities (every register of every lane group alike)
  float m[2];          // second walk: the row's exponent offset
  bool unset = true;   // second walk: no block has set the offset
  // operand addresses in the current buffer: row 16 (lr / 8) + lr % 8 of the
  // K tile and row lr of the Vt tile, chunk 4 s + g4
  typedef const __attribute__((address_space(3))) u32x4 *lds_ptr;
  uint32_t ka_addr[2], va_addr[2];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      lacc[i] = zero4;
      m[i] = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) oacc[i][t] = zero4;
    }
  };
  auto start = [&]() __attribute__((always_inline)) {
    r0 = tid >> 3;
    kc = ((tid & 7) ^ swz_k(r0)) * 8;
    koff = static_cast<uint32_t>((static_cast<int64_t>(r0) * p.k_st + kc) * 2);
    voff = static_cast<uint32_t>((r0 * kHeadDim + ((tid & 7) ^ swz(r0)) * 8) * 2);
    const int krow = 16 * (lr >> 3) + (lr & 7);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      ka_addr[s] = lds0 + krow * 128 + ((4 * s + g4) ^ swz_k(krow)) * 16;
      va_addr[s] = lds0 + kTile * 2 + lr * 128 + ((4 * s + g4) ^ swz(lr)) * 16;
    }
  };
  clear();
  start();
  auto k_op = [&](int kt, int s) {
    return *reinterpret_cast<lds_ptr>(ka_addr[s] + (32 * (kt >> 1) + 8 * (kt & 1)) * 128);
  };
  auto v_op = [&](int t, int s) { return *reinterpret_cast<lds_ptr>(va_addr[s] + 16 * t * 128); };
  // The A operand of the row sums: ones, zero at keys at or past lim.
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  u32x4 sum_a[2] = {ones, ones};
  auto set_ones = [&](int lim) __attribute__((always_inline)) {
    int lane_key = 16 * (g4 >> 1) + 4 * (g4 & 1);
    asm volatile("" : "+v"(lane_key));  // keeps the per-key compares out of the loop's registers
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int kk = 32 * s + 8 * (e >> 1) + lane_key + 2 * (e & 1);
        sum_a[s][e] = kk + 1 < lim ? 0x3f803f80u : (kk < lim ? 0x3f80u : 0u);
      }
  };
  // Probabilities at offset 0 and their products with Vt.
  auto compute = [&]() __attribute__((always_inline)) {
    floatx4 S[2][4];
    u32x4 ka[4][2];  // all K operands of the block, read before the first product
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int s = 0; s < 2; ++s) ka[kt][s] = k_op(kt, s);
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i) S[i][kt] = mfma16(ka[kt][s], qf[i][s], s == 0 ? zero4 : S[i][kt]);
    u32x4 pb[2][2];  // [q tile][32-key group]
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int kt = 2 * s + (e >> 1), r = 2 * (e & 1);
          pb[i][s][e] = pack_bf16x2(__builtin_amdgcn_exp2f(kUnit ? S[i][kt][r] : S[i][kt][r] * c),
                                    __builtin_amdgcn_exp2f(kUnit ? S[i][kt][r + 1] : S[i][kt][r + 1] * c));
        }
    u32x4 va[4][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) va[t][s] = v_op(t, s);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        lacc[i] = mfma16(sum_a[s], pb[i][s], lacc[i]);
#pragma unroll
        for (int t = 0; t < 4; ++t) oacc[i][t] = mfma16(va[t][s], pb[i][s], oacc[i][t]);
      }
    // every K read issued before the first score product, then the products,
    // the exponentials, the Vt reads and the products with them
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 16, 0);
    __builtin_amdgcn_sched_group_barrier(0x402, 80, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 20, 0);
  };
  // The second walk's block: probabilities relative to the row's offset m, which
  // follows the row maximum in steps: it moves where a score passes it by kRaise,
  // to kMargin above the block's maximum, so that few blocks move it (the first
  // block that has keys sets it). A whole number, so that the sums' rescaling is
  // exact. lim: the block's keys that exist (more than none).
  auto compute_online = [&](int lim) __attribute__((always_inline)) {
    floatx4 S[2][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4 a = k_op(kt, s);
#pragma unroll
        for (int i = 0; i < 2; ++i) S[i][kt] = mfma16(a, qf[i][s], s == 0 ? zero4 : S[i][kt]);
      }
    if (__builtin_expect(lim < kBlockK, 0)) {
      int lane_key = 16 * (g4 >> 1) + 4 * (g4 & 1);
      asm volatile("" : "+v"(lane_key));  // as in set_ones
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            S[i][kt][r] = 32 * (kt >> 1) + 8 * (kt & 1) + lane_key + r < lim ? S[i][kt][r] : -INFINITY;
    }
    float mx[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      mx[i] = S[i][0][0];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx[i] = fmaxf(mx[i], S[i][kt][r]);
    }
    const float over = fmaxf(fmaf(mx[0], c, -m[0]), fmaf(mx[1], c, -m[1]));
    if (__builtin_expect(unset || __ballot(over > kRaise) != 0, 0)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float top = fmaxf(mx[i], __shfl_xor(mx[i], 16));
        top = fmaxf(top, __shfl_xor(top, 32)) * c;
        float to = __builtin_rintf(top + kMargin);
        if ((!unset && top <= m[i]) || (__float_as_uint(top) & 0x7f800000u) == 0x7f800000u) to = m[i];
        const float alpha = unset ? 0.f : __builtin_amdgcn_exp2f(m[i] - to);
        m[i] = to;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          lacc[i][r] *= alpha;
#pragma unroll
          for (int t = 0; t < 4; ++t) oacc[i][t][r] *= alpha;
        }
      }
      unset = false;
    }
    u32x4 pb[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int kt = 2 * s + (e >> 1), r = 2 * (e & 1);
          // one rounding of c S - m, not one of c S before it
          pb[i][s][e] = pack_bf16x2(__builtin_amdgcn_exp2f(fmaf(S[i][kt][r], c, -m[i])),
                                    __builtin_amdgcn_exp2f(fmaf(S[i][kt][r + 1], c, -m[i])));
        }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < 2; ++i) lacc[i] = mfma16(ones, pb[i][s], lacc[i]);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const u32x4 a = v_op(t, s);
#pragma unroll
        for (int i = 0; i < 2; ++i) oacc[i][t] = mfma16(a, pb[i][s], oacc[i][t]);
      }
    }
  };
  // A row sum out of range, infinite or NaN (bit patterns, so that NaN
  // compares as well).
  auto sums_bad = [&](uint32_t high) __attribute__((always_inline)) {
    bool x = false;
#pragma unroll
    for (int i = 0; i < 2; ++i) x |= __float_as_uint(lacc[i][0]) - kLowBits > high - kLowBits;
    return __ballot(x) != 0;
  };

  // List entry j+1 is loaded during iteration j-1 (index clamped to the list)
  // so that reading it never waits on memory: the wait at the top of each
  // iteration already covers it.
  const __attribute__((address_space(4))) int32_t *clist =
      (const __attribute__((address_space(4))) int32_t *)(list);
  bool out_of_list = false;  // a block outside the sequence was listed
  int done = 0;              // blocks of the list that are in the sums
  // The walk: wait for a block's tiles, start the next block's DMA into the
  // other buffer, compute. kIdle: a wave without rows, which only stages its
  // share of the tiles and keeps the barriers. kOnline: the second walk.
  auto walk = [&](auto idle_wave, auto online) __attribute__((always_inline)) {
    constexpr bool kIdle = decltype(idle_wave)::value, kOnline = decltype(online)::value;
    const int j0 = kOnline ? done : 0;  // even: the walk is left a block after an even look
    int blk = dense ? blk0 + j0 : clist[j0];
    if (kOnline && !dense && p.delta)
      for (int i = 0; i < j0; ++i) blk += clist[i];  // not kept through the first walk, which has no registers to spare
    int32_t e_next = dense ? 0 : clist[j0 + 1 < n ? j0 + 1 : j0];
    fetch(blk, 0);
    int nw = n, look = 0;  // look: the block after which the row sums are looked at next (0, 8, 24, 56, ..)
#pragma clang loop unroll(disable)
    for (int j = j0; j < nw; ++j) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (!kOnline && __builtin_expect(j == look + 1, 0)) {
        if (__builtin_amdgcn_readfirstlane(redo)) nw = j + 1;  // ends after this block
        look = 2 * look + 8;
      }
      const int lim = valid_keys(blk);
      if (j + 1 < nw) {
        if (dense) {
          ++blk;
        } else {
          const int e = e_next;
          blk = p.delta ? blk + e : e;
          e_next = clist[j + 2 < n ? j + 2 : n - 1];
        }
        fetch(blk, (j & 1) ^ 1);
      }
      if constexpr (!kIdle) {
        if constexpr (kOnline) {
          if (lim > 0) compute_online(lim);
        } else {
          if (__builtin_expect(lim < kBlockK, 0)) {
            set_ones(lim);
            out_of_list |= lim == 0;
          }
          compute();
          if (__builtin_expect(lim < kBlockK, 0)) sum_a[0] = sum_a[1] = ones;
          if (__builtin_expect(j == look, 0) && sums_bad(look ? kLaterBits : kFirstBits)) atomicOr(&redo, kLeave);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          ka_addr[s] ^= kBufBytes;
          va_addr[s] ^= kBufBytes;
        }
      }
    }
    done = nw;
  };
  if (n > 0) {
    if (idle) {
      walk(std::true_type{}, std::false_type{});
    } else {
      walk(std::false_type{}, std::false_type{});
      uint32_t top = 0;  // largest magnitude of O, as bits
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const uint32_t o = __float_as_uint(oacc[i][t][r]) & 0x7fffffffu;
            top = o > top ? o : top;
          }
      if (sums_bad(kHighBits) || __ballot(top >= 0x7f800000u) != 0 || out_of_list) atomicOr(&redo, kRedo);
    }
  }

  __syncthreads();  // every wave is done with the tiles and with redo
  const uint32_t flags = __builtin_amdgcn_readfirstlane(redo);
  const bool again = (flags & kRedo) != 0;
  if (__builtin_expect(flags != 0, 0) && (again || done < n)) {
    // on from where the first walk ended, its sums being good at offset 0, or
    // again from the first block, with the queries still in registers: nothing is
    // stored before, so the output may lie on the queries' storage
    lanes();
    start();
    unset = again;
    if (again) {
      clear();
      done = 0;
    }
    if (idle)
      walk(std::true_type{}, std::true_type{});
    else
      walk(std::false_type{}, std::true_type{});
  }
  lanes();
  if (kSplit && sp) {
    float *part = p.part + wg * (kBlockQ * (kHeadDim + 1));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = w * 32 + 16 * i + lr;
      const float ltot = lacc[i][0];
      const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        *reinterpret_cast<floatx4 *>(part + r * kHeadDim + 16 * t + 4 * g4) =
            floatx4{oacc[i][t][0] * inv, oacc[i][t][1] * inv, oacc[i][t][2] * inv, oacc[i][t][3] * inv};
      if (g4 == 0) part[kBlockQ * kHeadDim + r] = m[i] + __builtin_amdgcn_logf(ltot);  // -inf for a sum of 0
    }
  } else {
    store_rows(p, sp, b, h, row0, nq, lr, g4, oacc, lacc);
  }
}

// Results of split special queries: the parts' outputs in split order, each
// weighted with its row sum (thread: row tid / 2, 32 features). The parts' sums
// come as logarithms, so parts of any exponent offset meet here.
__global__ __launch_bounds__(kThreads)
void combine_kernel(const AttnParams p) {
  const int64_t unit = blockIdx.x;
  const int64_t bh = unit / p.nq2b, h = bh % p.H, b = bh / p.H;
  const int r = threadIdx.x >> 1, d0 = (threadIdx.x & 1) * 32;
  const int64_t qrow = (unit % p.nq2b) * kBlockQ + r;
  if (qrow >= p.nq2) return;
  constexpr int64_t kPart = kBlockQ * (kHeadDim + 1);
  const float *part = p.part + unit * p.nsplit * kPart;
  float weight[kMaxSplit], top = -INFINITY;
#pragma unroll
  for (int s = 0; s < kMaxSplit; ++s)  // all loads in flight at once
    weight[s] = s < p.nsplit ? part[s * kPart + kBlockQ * kHeadDim + r] : -INFINITY;
#pragma unroll
  for (int s = 0; s < kMaxSplit; ++s) top = fmaxf(top, weight[s]);
  if (top == -INFINITY) top = 0.f;  // no part has a probability: weights 0
  floatx4 acc[8];
  float l = 0.f;
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kMaxSplit; ++s) {
    if (s >= p.nsplit) break;
    weight[s] = __builtin_amdgcn_exp2f(weight[s] - top);
    l += weight[s];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const floatx4 o = *reinterpret_cast<const floatx4 *>(part + s * kPart + r * kHeadDim + d0 + 4 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[c][e] = fmaf(weight[s], o[e], acc[c][e]);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t *optr = p.o2 + b * p.o2_sb + h * p.o2_sh +
                   (p.tok_p > 0 ? (qrow / p.tok_s) * p.tok_p + qrow % p.tok_s : qrow) * p.o2_st + d0;
#pragma unroll
  for (int c = 0; c < 8; c += 2) {
    const u32x4 v = {pack_bf16x2(acc[c][0] * inv, acc[c][1] * inv), pack_bf16x2(acc[c][2] * inv, acc[c][3] * inv),
                     pack_bf16x2(acc[c + 1][0] * inv, acc[c + 1][1] * inv),
                     pack_bf16x2(acc[c + 1][2] * inv, acc[c + 1][3] * inv)};
    *reinterpret_cast<u32x4 *>(optr + 4 * c) = v;
  }
}

// The PV post-cut (qk_int_sv_f16_cuda_sm80.cuh:291-381): 4 waves x 32 query
// rows on v_mfma_f32_32x32x16_bf16 (a lane owns row lane % 32 and 32 of the
// 64 keys), with the exponent offset m moved per block where its sums leave
// the range. Its execution map is kept per 32-row wave.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void bsattn_pv_kernel(const AttnParams p) {
  constexpr int CH = 512 / kThreads;  // 16-byte chunks per thread per tile
  __shared__ __attribute__((aligned(16))) uint16_t smem[2][2][kTile];  // [buffer][K, Vt]
  __shared__ float pv_gap[4];                                           // per-wave gap of the PV post-cut
  auto lds_u32 = [](const uint16_t *ptr) { return lds_addr32(ptr); };

  const int64_t nqb = p.nqb;
  const int64_t wg = p.head_major ? static_cast<int64_t>(blockIdx.x) : xcd_remap(blockIdx.x, p.num_wg);
  const int qb = static_cast<int>(wg % nqb);
  const int64_t bh = wg / nqb;
  const int64_t h = bh % p.H;
  const int64_t b = bh / p.H;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave index, uniform
  const int l = tid & 63, lr = l & 31, hf = l >> 5;

  const int64_t row = bh * p.nqb + qb;
  const int32_t *list = p.idx + row * p.idx_w;
  int n = p.cnt[row];
  n = n < 0 ? 0 : (n > p.idx_w ? static_cast<int>(p.idx_w) : n);

  const int64_t qrow = static_cast<int64_t>(qb) * kBlockQ + w * 32 + lr;
  const bool qvalid = qrow < p.nq;
  uint16_t *optr = p.o + b * p.o_sb + h * p.o_sh + (qvalid ? qrow : 0) * p.o_st;

  if (n == 0) {
    if (qvalid) {
#pragma unroll
      for (int c = hf; c < 8; c += 2) *reinterpret_cast<u32x4 *>(optr + c * 8) = u32x4{0, 0, 0, 0};
    }
    return;
  }

  // Q as the B operand of S^T = K Q^T: lane holds row lr, d = 16s + 8hf .. +7.
  u32x4 qf[4];
  {
    const uint16_t *qptr = p.q + b * p.q_sb + h * p.q_sh + (qvalid ? qrow : 0) * p.q_st;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      qf[s] = qvalid ? *reinterpret_cast<const u32x4 *>(qptr + 16 * s + 8 * hf) : u32x4{0, 0, 0, 0};
    // consume Q here so that the compiler's wait for these loads lands before
    // the loop instead of inside it
    asm volatile("" ::"v"(qf[0]), "v"(qf[1]), "v"(qf[2]), "v"(qf[3]));
  }

  // Staging: LDS chunk ci = u*256 + tid lands at byte 16*ci (the DMA writes
  // lane i of a wave at base + 16*i); it holds tile row ci/8, logical chunk
  // (ci%8) ^ swz(row), so each lane fetches that global chunk.
  const uint16_t *kbase = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t *vbase = p.vt + (bh * p.nkb) * kTile;
  const int nk32 = static_cast<int>(p.nk);
  const int nkb32 = static_cast<int>(p.nkb);
  const int partial = (nk32 % kBlockK) ? nkb32 - 1 : -1;  // the partial last block, if any
  // swz(32u + r) = swz(r): a thread's chunk column, and so its byte offset
  // inside the block, is the same for each of its CH chunks; only the row
  // base (32u rows) moves, and that goes into the scalar base address.
  const int r0 = tid >> 3;
  const int cc = (tid & 7) ^ swz(r0);
  const uint32_t koff = static_cast<uint32_t>((static_cast<int64_t>(r0) * p.k_st + cc * 8) * 2);
  const uint32_t voff = static_cast<uint32_t>((r0 * kHeadDim + cc * 8) * 2);
  const int last_row = partial >= 0 ? nk32 - 1 - partial * kBlockK : kBlockK - 1;
  // K and Vt of block blk -> LDS buffer buf. Blocks outside [0, nkb) load
  // block 0 (their scores are masked); rows of the partial block past the
  // sequence end read its last row.
  auto fetch = [&](int blk, int buf) {
    const int sb = (blk >= 0 && blk < nkb32) ? blk : 0;
    const uint16_t *kb = kbase + static_cast<int64_t>(sb) * kBlockK * p.k_st;
    const uint16_t *vb = vbase + static_cast<int64_t>(sb) * kTile;
    const uint32_t kd = lds_u32(smem[buf][0]) + w * 64 * 16, vd = lds_u32(smem[buf][1]) + w * 64 * 16;
    if (sb == partial) {
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int r = 32 * u + r0;
        const int rr = r < last_row ? r : last_row;
        dma16(kb, static_cast<uint32_t>((static_cast<int64_t>(rr) * p.k_st + cc * 8) * 2), kd + u * kThreads * 16);
      }
    } else {
#pragma unroll
      for (int u = 0; u < CH; ++u) dma16(kb + 32 * u * p.k_st, koff, kd + u * kThreads * 16);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) dma16(vb + 32 * u * kHeadDim, voff, vd + u * kThreads * 16);
  };
  // Keys of block blk that exist: 64, fewer for the partial last block, 0
  // for blocks outside [0, nkb).
  auto valid_keys = [&](int blk) {
    return (blk >= 0 && blk < nkb32) ? (blk == partial ? nk32 - blk * kBlockK : kBlockK) : 0;
  };

  const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  floatx16 oacc[2] = {zero16, zero16};
  float ls = 0.f;  // running sum of the bf16 probabilities (this lane's 32 keys per block)
  float m = 0.f;   // exponent offset of this lane's row (log2 units)
  const float c = p.c;
  float run_max = -5000000.0f;  // PV post-cut: running row max (log2 units)
  const float pv_threshold = p.pv_thr[h];

  // P = exp2(c S - m) for k-step s of the PV product (accumulators
  // 8(s%2)..+7 of tile s/2), packed to bf16; returns bs plus the sum of the
  // rounded pairs.
  auto exp_step = [&](const floatx16 (&S)[2], u32x4 (&pb)[4], int s, float bs) {
    const int t = s >> 1, r = 8 * (s & 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x0 = __builtin_amdgcn_exp2f(fmaf(S[t][r + 2 * e], c, -m));
      const float x1 = __builtin_amdgcn_exp2f(fmaf(S[t][r + 2 * e + 1], c, -m));
      pb[s][e] = pack_bf16x2(x0, x1);
      bs = add_bf16_pair(pb[s][e], bs);
    }
    return bs;
  };
  auto exp_block = [&](const floatx16 (&S)[2], u32x4 (&pb)[4]) {
    float bs0 = 0.f, bs1 = 0.f;  // two partial sums: shorter dependency chains
#pragma unroll
    for (int s = 0; s < 4; s += 2) {
      bs0 = exp_step(S, pb, s, bs0);
      bs1 = exp_step(S, pb, s + 1, bs1);
    }
    return bs0 + bs1;
  };
  // Scores of keys at or past lim (of the block's 64) to -inf. An opaque
  // copy of the lane's key offset keeps the 32 per-element key indices from
  // being hoisted out of the loop.
  auto mask_keys = [&](floatx16 (&S)[2], int lim) {
    int h4 = 4 * hf;
    asm volatile("" : "+v"(h4));
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kk = 32 * t + 8 * (r >> 2) + h4 + (r & 3);
        S[t][r] = kk < lim ? S[t][r] : -INFINITY;
      }
  };
  // Slow path for the current block (its missing keys already masked): move m to
  // the row max where the block left the fast path's range (both lanes of a
  // row agree), rescale O and the sum, redo P. Rows whose running sum is
  // negligible drop it (it holds no information relative to the new m)
  // instead of scaling it up.
  auto slow = [&](floatx16 (&S)[2], u32x4 (&pb)[4]) {
    float mx = S[0][0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, S[0][r]);
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, S[1][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    mx = mx == -INFINITY ? mx : mx * c - m;  // block max relative to m, log2 units
    const float lrow = ls + __shfl_xor(ls, 32);
    const bool tiny = !(lrow >= kLow);
    // g: how far m moves. Up to the block max when it is above m; down to it
    // only when the row so far is negligible (or empty).
    float g = 0.f;
    if (mx != -INFINITY) g = (mx > 0.f || tiny) ? mx : 0.f;
    const float alpha = tiny ? 0.f : __builtin_amdgcn_exp2f(-g);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      oacc[0][r] *= alpha;
      oacc[1][r] *= alpha;
    }
    ls *= alpha;
    m += g;
    return exp_block(S, pb);
  };

  // List entry j+1 is loaded during iteration j-1 (index clamped to the list)
  // so that reading it never waits on memory: the wait at the top of each
  // iteration already covers it.
  const __attribute__((address_space(4))) int32_t *clist =
      (const __attribute__((address_space(4))) int32_t *)(list);
  int blk = clist[0];
  int32_t e_next = clist[n > 1 ? 1 : 0];
  fetch(blk, 0);
  // One block: wait for its tiles, start the next block's DMA into the other
  // buffer, compute. The loop runs two blocks per trip so that each block's
  // buffer, and with it every LDS address, is a compile-time constant.
  auto step = [&](const int j, const int buf) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    const int cur = blk;
    if (j + 1 < n) {
      const int e = e_next;
      blk = p.delta ? blk + e : e;
      e_next = clist[j + 2 < n ? j + 2 : n - 1];
      fetch(blk, buf ^ 1);
    }
    const uint16_t *ks = smem[buf][0];
    const uint16_t *vs = smem[buf][1];

    // S^T tiles: keys 32t + [0,32) x this wave's 32 query rows.
    floatx16 S[2];
    u32x4 ka[4][2];  // all K operands of the block, read before the first product
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int row = 32 * t + lr;
        ka[s][t] = *reinterpret_cast<const u32x4 *>(ks + row * kHeadDim + ((2 * s + hf) ^ swz(row)) * 8);
      }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) S[t] = mfma32(ka[s][t], qf[s], s == 0 ? zero16 : S[t]);
    // every K read issued before the first score product
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 1);
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 1);

    // PV post-cut (qk_int_sv_f16_cuda_sm80.cuh:291-381 with update_mo,
    // attn_utils.cuh:419-466, per-block mode): gap = the largest over the
    // workgroup's rows of (block row max - running max) in log2 units; the
    // running max starts at -5e6 and follows every listed block, executed or
    // not; PV runs for the whole workgroup only when gap + threshold > 0.
    const int lim = valid_keys(cur);
    float mx = -5000000.0f;
    if (lim == kBlockK) {  // a whole block (the usual case): no per-key masks
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, S[t][r]);
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kk = 32 * t + 8 * (r >> 2) + 4 * hf + (r & 3);
          mx = kk < lim ? fmaxf(mx, S[t][r]) : mx;
        }
    }
    mx = fmaxf(mx, xor_lane(mx, 32)) * c;
    float gap = mx - run_max;  // the wave's largest, by VALU cross-lane moves (rows 0-31, both halves)
#pragma unroll
    for (int off = 16; off >= 1; off >>= 1) gap = fmaxf(gap, xor_lane(gap, off));
    run_max = fmaxf(run_max, mx);
    if (l == 0) pv_gap[w] = gap;

    // keys past the sequence end (partial or out-of-range blocks) are masked
    // before the exponentials, so such a block stays on the fast path unless
    // its sums leave the range
    if (lim < kBlockK) mask_keys(S, lim);
    u32x4 pb[4];
    float bs = exp_block(S, pb);  // changes no state: a skipped block drops it
    // the workgroup's decision, read after the exponentials so that the
    // barrier wait overlaps them
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const float g4 = fmaxf(fmaxf(pv_gap[0], pv_gap[1]), fmaxf(pv_gap[2], pv_gap[3]));
    if (!(g4 + pv_threshold > 0.f)) return;  // skipped: no sum, no PV
    if (l == 0 && p.pv_map && cur >= 0 && cur < nkb32)
      p.pv_map[((bh * p.nqb + qb) * 4 + w) * p.pv_w + cur] = 1;
    if (__ballot(!(bs <= kHigh) || !(ls + bs >= kLow))) bs = slow(S, pb);
    ls += bs;

    u32x4 va[4][2];  // all Vt operands of the block, read before the first product
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int n2 = 0; n2 < 2; ++n2) {
        const int row = 32 * n2 + lr;
        va[s][n2] = *reinterpret_cast<const u32x4 *>(vs + row * kHeadDim + ((2 * s + hf) ^ swz(row)) * 8);
      }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int n2 = 0; n2 < 2; ++n2) oacc[n2] = mfma32(va[s][n2], pb[s], oacc[n2]);
    // every Vt read issued before the first PV product
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
  };
  for (int j = 0; j < n; j += 2) {
    step(j, 0);
    if (j + 1 < n) step(j + 1, 1);
  }

  const float ltot = ls + __shfl_xor(ls, 32);
  const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
  if (qvalid) {
#pragma unroll
    for (int n2 = 0; n2 < 2; ++n2)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d0 = 32 * n2 + 8 * g + 4 * hf;
        uint2 v;
        v.x = pack_bf16x2(oacc[n2][4 * g + 0] * inv, oacc[n2][4 * g + 1] * inv);
        v.y = pack_bf16x2(oacc[n2][4 * g + 2] * inv, oacc[n2][4 * g + 3] * inv);
        *reinterpret_cast<uint2 *>(optr + d0) = v;
      }
  }
}

int check_bhtd(const char *name, const void *ptr, int64_t sb, int64_t sh, int64_t st) {
  VASC_REQUIRE(ptr != nullptr, "%s is NULL", name);
  VASC_REQUIRE((reinterpret_cast<uintptr_t>(ptr) & 15) == 0, "%s must be 16-byte aligned", name);
  VASC_REQUIRE(sb % 8 == 0 && sh % 8 == 0 && st % 8 == 0 && sb >= 0 && sh >= 0 && st > 0,
               "%s strides (%lld,%lld,%lld) must be non-negative multiples of 8 elements", name,
               (long long)sb, (long long)sh, (long long)st);
  return VASC_OK;
}

// Token-major output of vasc_global_attn_tokens_fwd (absent: P == 0).
struct OutTokens {
  int64_t P = 0, S = 0;
};

// How many workgroups share a special-query block's keys. Such a block walks
// every key block while a patch block walks its list (index_w entries), and the
// patch blocks keep the card (1024 resident workgroups) busy for about
// index_w * max(1, num_wg / 1024) of these steps: the special blocks are split to
// end with them, into parts of at least 32 key blocks. The host knows the width
// only: counts far below it, as a cdf threshold gives, leave a walk unsplit (8
// frames, counts a quarter of a full width: 117 us, split 98). Below 64 blocks
// the second launch and the workspace cost the host more than the split saves: at
// 2 frames of 1041 tokens the launch fell from 29 to 24 us and the layer, bound by
// the host, rose from 421 to 435. To the nearest part count: two parts for a walk
// that already ends with the patch blocks cost the 32-frame layer 0.4 to 1.1%.
// Unsplit, patch blocks alone and split, 16 heads, lists of a quarter: 56, 30 and
// 39 us at 4 frames; 120, 89 and 97 at 8; 300, 289 and 296 at 16.
int64_t special_splits(int64_t num_wg, int64_t nkb, int64_t index_w) {
  const int64_t busy = index_w * (num_wg > 1024 ? num_wg : 1024) / 1024;
  int64_t n = busy > 0 ? (nkb + busy / 2) / busy : 1;
  if (n > nkb / 32) n = nkb / 32;
  return n < 1 ? 1 : (n > kMaxSplit ? kMaxSplit : n);
}

// Special-token queries of vasc_global_attn_fwd (absent: q2 == NULL).
struct SpecialQueries {
  const uint16_t *q2 = nullptr;
  int64_t q2_sb = 0, q2_sh = 0, q2_st = 0;
  uint16_t *o2 = nullptr;
  int64_t o2_sb = 0, o2_sh = 0, o2_st = 0;
  int64_t nq2 = 0;
  float *part = nullptr;  // workspace of the key split (absent: no split)
};

int launch_attn(bool dense, const uint16_t *q, int64_t q_sb, int64_t q_sh, int64_t q_st,
                const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st, const uint16_t *vt,
                uint16_t *o, int64_t o_sb, int64_t o_sh, int64_t o_st, int64_t B, int64_t H,
                int64_t nq, int64_t nk, int64_t d, const int32_t *idx, int64_t idx_w,
                const int32_t *cnt, int32_t delta, float sm_scale, void *stream,
                const SpecialQueries &sq = SpecialQueries(), const float *pv_thr = nullptr,
                int32_t *pv_map = nullptr, const OutTokens &ot = OutTokens(), bool half_io = false) {
  VASC_SUPPORTED(d == kHeadDim, "head_dim %lld not built (built: 64)", (long long)d);
  VASC_REQUIRE(B > 0 && H > 0 && nq > 0 && nk > 0, "sizes must be positive");
  int rc;
  if ((rc = check_bhtd("q", q, q_sb, q_sh, q_st))) return rc;
  if ((rc = check_bhtd("k", k, k_sb, k_sh, k_st))) return rc;
  if ((rc = check_bhtd("o", o, o_sb, o_sh, o_st))) return rc;
  VASC_REQUIRE(vt != nullptr && (reinterpret_cast<uintptr_t>(vt) & 15) == 0, "vt must be a 16-byte aligned packed V");
  if (!dense) {
    VASC_REQUIRE(idx != nullptr && cnt != nullptr, "block_index and block_count are required");
    VASC_REQUIRE(idx_w > 0, "index_width must be positive");
  }
  VASC_REQUIRE(sm_scale > 0.f, "sm_scale must be positive");
  AttnParams p;
  p.q = q; p.q_sb = q_sb; p.q_sh = q_sh; p.q_st = q_st;
  p.k = k; p.k_sb = k_sb; p.k_sh = k_sh; p.k_st = k_st;
  p.vt = vt;
  p.o = o; p.o_sb = o_sb; p.o_sh = o_sh; p.o_st = o_st;
  p.H = H; p.nq = nq; p.nk = nk;
  p.nqb = cdiv(nq, kBlockQ);
  p.nkb = cdiv(nk, kBlockK);
  p.idx = idx; p.idx_w = idx_w; p.cnt = cnt; p.delta = delta;
  p.c = sm_scale * 1.4426950408889634f;
  p.num_wg = B * H * p.nqb;
  p.q2 = sq.q2; p.q2_sb = sq.q2_sb; p.q2_sh = sq.q2_sh; p.q2_st = sq.q2_st;
  p.o2 = sq.o2; p.o2_sb = sq.o2_sb; p.o2_sh = sq.o2_sh; p.o2_st = sq.o2_st;
  p.nq2 = sq.q2 ? sq.nq2 : 0;
  p.nq2b = cdiv(p.nq2, kBlockQ);
  p.num_wg2 = B * H * p.nq2b;
  const int64_t nsplit = p.num_wg2 && sq.part ? special_splits(p.num_wg, p.nkb, idx_w) : 1;
  p.nsplit = static_cast<int32_t>(nsplit);
  p.split_blocks = static_cast<int32_t>(cdiv(p.nkb, nsplit));
  p.part = sq.part;
  p.num_wg2_slots = (p.num_wg2 * nsplit + 7) / 8 * 8;
  // K and V of one head take 256 B per key token; from 192k tokens (48 MB a
  // head) the eight heads one per XCD that the contiguous mapping keeps in
  // flight exceed the 256 MB Infinity Cache by half, and walking the heads
  // one after another across all XCDs reads less from HBM (7 % faster at
  // 256k tokens, no change at 133k, 2 % slower at C2)
  p.head_major = nk >= 192 * 1024 ? 1 : 0;
  VASC_REQUIRE(p.num_wg + p.num_wg2_slots < (int64_t(1) << 31), "grid too large");
  VASC_SUPPORTED(nk < (int64_t(1) << 30) && nq < (int64_t(1) << 40), "sequence of %lld keys not built (< 2^30)",
                 (long long)nk);
  p.pv_thr = pv_thr;
  p.pv_map = pv_map;
  p.pv_w = p.nkb;
  p.tok_p = ot.P;
  p.tok_s = ot.S;
  p.half_io = half_io ? 1 : 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto kern = pv_thr ? bsattn_pv_kernel
              : dense      ? bsattn_fwd_kernel<true, false, false>
              : p.c == 1.f ? bsattn_fwd_kernel<false, true, false>
                           : bsattn_fwd_kernel<false, false, false>;
  if (nsplit > 1) kern = p.c == 1.f ? bsattn_fwd_kernel<false, true, true> : bsattn_fwd_kernel<false, false, true>;
  hipLaunchKernelGGL(kern, dim3(p.num_wg + p.num_wg2_slots), dim3(kThreads), 0, s, p);
  if ((rc = check_launch(dense ? "vasc_dense_attn_fwd" : "vasc_block_sparse_attn_fwd"))) return rc;
  if (nsplit == 1) return VASC_OK;
  hipLaunchKernelGGL(combine_kernel, dim3(p.num_wg2), dim3(kThreads), 0, s, p);
  return check_launch("vasc_global_attn/combine");
}

}  // namespace
}  // namespace vasc

extern "C" int vasc_block_sparse_attn_fwd(const uint16_t *q, int64_t q_sb, int64_t q_sh, int64_t q_st,
                                          const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                          const uint16_t *vt, uint16_t *o, int64_t o_sb, int64_t o_sh,
                                          int64_t o_st, int64_t B, int64_t H, int64_t nq, int64_t nk,
                                          int64_t d, const int32_t *block_index, int64_t index_width,
                                          const int32_t *block_count, int32_t index_is_delta,
                                          float sm_scale, void *stream) {
  return vasc::launch_attn(false, q, q_sb, q_sh, q_st, k, k_sb, k_sh, k_st, vt, o, o_sb, o_sh, o_st, B, H,
                           nq, nk, d, block_index, index_width, block_count, index_is_delta, sm_scale,
                           stream);
}

extern "C" int vasc_block_sparse_attn_f16_fwd(const uint16_t *q, int64_t q_sb, int64_t q_sh, int64_t q_st,
                                          const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                          const uint16_t *vt, uint16_t *o, int64_t o_sb, int64_t o_sh,
                                          int64_t o_st, int64_t B, int64_t H, int64_t nq, int64_t nk,
                                          int64_t d, const int32_t *block_index, int64_t index_width,
                                          const int32_t *block_count, int32_t index_is_delta,
                                          float sm_scale, void *stream) {
  return vasc::launch_attn(false, q, q_sb, q_sh, q_st, k, k_sb, k_sh, k_st, vt, o, o_sb, o_sh, o_st, B, H,
                           nq, nk, d, block_index, index_width, block_count, index_is_delta, sm_scale,
                           stream, vasc::SpecialQueries(), nullptr, nullptr, vasc::OutTokens(), true);
}

extern "C" int vasc_block_sparse_attn_pv_fwd(const uint16_t *q, int64_t q_sb, int64_t q_sh, int64_t q_st,
                                             const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                             const uint16_t *vt, uint16_t *o, int64_t o_sb, int64_t o_sh,
                                             int64_t o_st, int64_t B, int64_t H, int64_t nq, int64_t nk,
                                             int64_t d, const int32_t *block_index, int64_t index_width,
                                             const int32_t *block_count, int32_t index_is_delta, float sm_scale,
                                             const float *pv_threshold, int32_t *pv_map, void *stream) {
  VASC_REQUIRE(pv_threshold != nullptr, "pv_threshold ([H] float32, device) is required");
  return vasc::launch_attn(false, q, q_sb, q_sh, q_st, k, k_sb, k_sh, k_st, vt, o, o_sb, o_sh, o_st, B, H,
                           nq, nk, d, block_index, index_width, block_count, index_is_delta, sm_scale, stream,
                           vasc::SpecialQueries(), pv_threshold, pv_map);
}

extern "C" int vasc_dense_attn_fwd(const uint16_t *q, int64_t q_sb, int64_t q_sh, int64_t q_st,
                                   const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                   const uint16_t *vt, uint16_t *o, int64_t o_sb, int64_t o_sh, int64_t o_st,
                                   int64_t B, int64_t H, int64_t nq, int64_t nk, int64_t d, float sm_scale,
                                   void *stream) {
  return vasc::launch_attn(true, q, q_sb, q_sh, q_st, k, k_sb, k_sh, k_st, vt, o, o_sb, o_sh, o_st, B, H, nq,
                           nk, d, nullptr, 1, nullptr, 0, sm_scale, stream);
}

extern "C" int64_t vasc_global_attn_workspace_size(int64_t B, int64_t H, int64_t n_patch, int64_t n_special, int64_t nk,
                                                   int64_t index_width) {
  using namespace vasc;
  if (B <= 0 || H <= 0 || n_patch <= 0 || n_special <= 0 || nk <= 0 || index_width <= 0) return 0;
  const int64_t n = special_splits(B * H * cdiv(n_patch, kBlockQ), cdiv(nk, kBlockK), index_width);
  return n == 1 ? 0 : B * H * cdiv(n_special, kBlockQ) * n * kBlockQ * (kHeadDim + 1) * 4;
}

static int global_attn_impl(const uint16_t *q_patch, int64_t qp_sb, int64_t qp_sh, int64_t qp_st,
                            const uint16_t *q_special, int64_t qs_sb, int64_t qs_sh, int64_t qs_st,
                            const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st, const uint16_t *vt,
                            uint16_t *o_patch, int64_t op_sb, int64_t op_sh, int64_t op_st, uint16_t *o_special,
                            int64_t os_sb, int64_t os_sh, int64_t os_st, int64_t B, int64_t H, int64_t n_patch,
                            int64_t n_special, int64_t nk, int64_t d, const int32_t *block_index,
                            int64_t index_width, const int32_t *block_count, float sm_scale, void *workspace,
                            int64_t workspace_bytes, void *stream) {
  using namespace vasc;
  SpecialQueries sq;
  if (n_special > 0) {
    int rc;
    if ((rc = check_bhtd("q_special", q_special, qs_sb, qs_sh, qs_st))) return rc;
    if ((rc = check_bhtd("o_special", o_special, os_sb, os_sh, os_st))) return rc;
    sq.q2 = q_special; sq.q2_sb = qs_sb; sq.q2_sh = qs_sh; sq.q2_st = qs_st;
    sq.o2 = o_special; sq.o2_sb = os_sb; sq.o2_sh = os_sh; sq.o2_st = os_st;
    sq.nq2 = n_special;
    if (workspace) {
      VASC_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, "workspace must be 16-byte aligned");
      VASC_REQUIRE(workspace_bytes >= vasc_global_attn_workspace_size(B, H, n_patch, sq.nq2, nk, index_width),
                   "workspace of %lld bytes is too small", (long long)workspace_bytes);
      sq.part = static_cast<float *>(workspace);
    }
  }
  VASC_REQUIRE(n_special >= 0, "n_special must be non-negative");
  return launch_attn(false, q_patch, qp_sb, qp_sh, qp_st, k, k_sb, k_sh, k_st, vt, o_patch, op_sb, op_sh, op_st,
                     B, H, n_patch, nk, d, block_index, index_width, block_count, 0, sm_scale, stream, sq);
}

extern "C" int vasc_global_attn_fwd(const uint16_t *q_patch, int64_t qp_sb, int64_t qp_sh, int64_t qp_st,
                                    const uint16_t *q_special, int64_t qs_sb, int64_t qs_sh, int64_t qs_st,
                                    const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                    const uint16_t *vt, uint16_t *o_patch, int64_t op_sb, int64_t op_sh,
                                    int64_t op_st, uint16_t *o_special, int64_t os_sb, int64_t os_sh,
                                    int64_t os_st, int64_t B, int64_t H, int64_t n_patch, int64_t n_special,
                                    int64_t nk, int64_t d, const int32_t *block_index, int64_t index_width,
                                    const int32_t *block_count, float sm_scale, void *stream) {
  return global_attn_impl(q_patch, qp_sb, qp_sh, qp_st, q_special, qs_sb, qs_sh, qs_st, k, k_sb, k_sh, k_st, vt,
                          o_patch, op_sb, op_sh, op_st, o_special, os_sb, os_sh, os_st, B, H, n_patch, n_special,
                          nk, d, block_index, index_width, block_count, sm_scale, nullptr, 0, stream);
}

extern "C" int vasc_global_attn_ws_fwd(const uint16_t *q_patch, int64_t qp_sb, int64_t qp_sh, int64_t qp_st,
                                       const uint16_t *q_special, int64_t qs_sb, int64_t qs_sh, int64_t qs_st,
                                       const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                       const uint16_t *vt, uint16_t *o_patch, int64_t op_sb, int64_t op_sh,
                                       int64_t op_st, uint16_t *o_special, int64_t os_sb, int64_t os_sh,
                                       int64_t os_st, int64_t B, int64_t H, int64_t n_patch, int64_t n_special,
                                       int64_t nk, int64_t d, const int32_t *block_index, int64_t index_width,
                                       const int32_t *block_count, float sm_scale, void *workspace,
                                       int64_t workspace_bytes, void *stream) {
  return global_attn_impl(q_patch, qp_sb, qp_sh, qp_st, q_special, qs_sb, qs_sh, qs_st, k, k_sb, k_sh, k_st, vt,
                          o_patch, op_sb, op_sh, op_st, o_special, os_sb, os_sh, os_st, B, H, n_patch, n_special,
                          nk, d, block_index, index_width, block_count, sm_scale, workspace, workspace_bytes,
                          stream);
}

static int global_attn_tokens_impl(const uint16_t *q_patch, int64_t qp_sb, int64_t qp_sh, int64_t qp_st,
                                   const uint16_t *q_special, int64_t qs_sb, int64_t qs_sh, int64_t qs_st,
                                   const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st, const uint16_t *vt,
                                   uint16_t *out, int64_t B, int64_t H, int64_t N, int64_t P, int64_t S, int64_t nk,
                                   int64_t d, const int32_t *block_index, int64_t index_width,
                                   const int32_t *block_count, float sm_scale, void *workspace,
                                   int64_t workspace_bytes, void *stream) {
  using namespace vasc;
  VASC_REQUIRE(N > 0 && P > S && S >= 0, "invalid frame sizes N=%lld P=%lld S=%lld", (long long)N, (long long)P,
               (long long)S);
  VASC_REQUIRE(nk == N * P, "nk %lld must be N*P = %lld", (long long)nk, (long long)(N * P));
  VASC_REQUIRE(out != nullptr && (reinterpret_cast<uintptr_t>(out) & 15) == 0, "out must be a 16-byte aligned [B,N*P,H*d]");
  // out [B, N*P, H*d] contiguous: (b, h, token) strides
  const int64_t o_sb = N * P * H * d, o_sh = d, o_st = H * d;
  SpecialQueries sq;
  if (S > 0) {
    int rc;
    if ((rc = check_bhtd("q_special", q_special, qs_sb, qs_sh, qs_st))) return rc;
    sq.q2 = q_special; sq.q2_sb = qs_sb; sq.q2_sh = qs_sh; sq.q2_st = qs_st;
    sq.o2 = out; sq.o2_sb = o_sb; sq.o2_sh = o_sh; sq.o2_st = o_st;
    sq.nq2 = N * S;
    if (workspace) {
      VASC_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, "workspace must be 16-byte aligned");
      VASC_REQUIRE(workspace_bytes >= vasc_global_attn_workspace_size(B, H, N * (P - S), sq.nq2, nk, index_width),
                   "workspace of %lld bytes is too small", (long long)workspace_bytes);
      sq.part = static_cast<float *>(workspace);
    }
  }
  OutTokens ot;
  ot.P = P;
  ot.S = S;
  return launch_attn(false, q_patch, qp_sb, qp_sh, qp_st, k, k_sb, k_sh, k_st, vt, out, o_sb, o_sh, o_st, B, H,
                     N * (P - S), nk, d, block_index, index_width, block_count, 0, sm_scale, stream, sq, nullptr,
                     nullptr, ot);
}

extern "C" int vasc_global_attn_tokens_fwd(const uint16_t *q_patch, int64_t qp_sb, int64_t qp_sh, int64_t qp_st,
                                           const uint16_t *q_special, int64_t qs_sb, int64_t qs_sh, int64_t qs_st,
                                           const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                           const uint16_t *vt, uint16_t *out, int64_t B, int64_t H, int64_t N,
                                           int64_t P, int64_t S, int64_t nk, int64_t d,
                                           const int32_t *block_index, int64_t index_width,
                                           const int32_t *block_count, float sm_scale, void *stream) {
  return global_attn_tokens_impl(q_patch, qp_sb, qp_sh, qp_st, q_special, qs_sb, qs_sh, qs_st, k, k_sb, k_sh, k_st,
                                 vt, out, B, H, N, P, S, nk, d, block_index, index_width, block_count, sm_scale,
                                 nullptr, 0, stream);
}

extern "C" int vasc_global_attn_tokens_ws_fwd(const uint16_t *q_patch, int64_t qp_sb, int64_t qp_sh, int64_t qp_st,
                                              const uint16_t *q_special, int64_t qs_sb, int64_t qs_sh, int64_t qs_st,
                                              const uint16_t *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
                                              const uint16_t *vt, uint16_t *out, int64_t B, int64_t H, int64_t N,
                                              int64_t P, int64_t S, int64_t nk, int64_t d,
                                              const int32_t *block_index, int64_t index_width,
                                              const int32_t *block_count, float sm_scale, void *workspace,
                                              int64_t workspace_bytes, void *stream) {
  return global_attn_tokens_impl(q_patch, qp_sb, qp_sh, qp_st, q_special, qs_sb, qs_sh, qs_st, k, k_sb, k_sh, k_st,
                                 vt, out, B, H, N, P, S, nk, d, block_index, index_width, block_count, sm_scale,
                                 workspace, workspace_bytes, stream);
}
