// Grouped expert GEMMs for 16-bit data on gfx950, asynchronous-copy pipeline: the kernel template.
//
// Output tiles of BM x BN (256 x 256), 4 wavefronts 2x2, 32x32x16 MFMA, fp32 accumulate; operands never pass through
// vector registers on their way to LDS:
//
//  * Global -> LDS copies are `global_load_lds_dwordx4`: every lane names its own 16-byte source and
//    the 64 lanes of a wave fill 1 KB of LDS in lane order.  The contraction is cut into slabs of
//    32; the forward's weight slabs rotate through four buffers of 16 KB and are requested three to four
//    slabs (about 3000 MFMA cycles at 256 x 256) before they are consumed, which covers HBM latency with one wave
//    per SIMD; the activation rows rotate through two buffers of a slab pair (32 KB) each.
//  * An operand whose rows are k-contiguous in memory ([row][k]) keeps that layout in LDS and is read
//    with one 16-byte ds_read per MFMA operand.  Such operands are copied two slabs at a time (128
//    bytes of a row per copy), so that every request to L2 is a whole cache line: with 64-byte pieces
//    the same kernel makes 1.5 times the L2 requests and runs 10-15 % slower.
//  * [n][k] weights (the input-gradient products) are such an operand too: their B ring is three slab
//    pairs (160 KB of LDS with the A ring), the copies are spread four per wave over every k-step and
//    only every second slab needs a wait and a workgroup barrier.
//  * The forward weights are [k][n] in memory and stay [k][n] in LDS (512 bytes per k row);
//    MFMA operands are read with `ds_read_b64_tr_b16`, the LDS transpose read of gfx950, which
//    hands lane i of a 16-lane group column n0+i for 4 consecutive k.  No register transpose, no
//    LDS store instruction, no staging registers.
//  * LDS swizzles are applied on the global side (a lane picks which 16-byte piece it fetches), as
//    the LDS side of an asynchronous copy is fixed to lane order:
//        [row][k] tiles: piece c (0..7, two slabs) of row r sits at position c ^ ((r >> 1) & 7)
//        [k][n]  tiles: piece c of row k sits at position c ^ ((k & 3) << 2)
//    so that both kinds of MFMA operand reads touch every bank once.
//  * Software pipeline per slab (two k-steps of 16): the operands of the second k-step are read
//    while the MFMAs of the first run; then the wave waits for the next slab's copies, one
//    workgroup barrier, the freed buffer is re-filled with slab s+4, the first operands of slab
//    s+1 are read, and the MFMAs of the second k-step run.  All LDS and HBM latency sits behind
//    MFMAs; only the barrier itself is exposed.
//
// The MFMAs take the weights as their first operand, so that a lane's accumulators are one output row
// and runs of four consecutive columns: the interleaved (gate, up) columns of the clamped SwiGLU
// (csrc/moe.cpp:164-180) meet in one lane, and the staging stores are 4 or 8 bytes wide.
//
// Contraction lengths that are not whole slab pairs (multiples of 64): the copies of the last pair re-read valid data
// where the contraction has ended, and the wave that copied them overwrites what lies past the end with zeros in LDS, between
// the wait for those copies and the barrier in front of their first use: of both operands, because an infinite weight that
// is read again would make a NaN with the zero of the activations.  Only the last few steps of the
// pipeline know about it, in instantiations of their own (RAGGED): the even lengths keep their registers (with
// the clamps in one kernel for both, prefill at 4096 tokens ran 2 % slower).  A tensor-parallel rank's slice of a layer has
// such lengths, 720 of 2880: the down product of one, 8012 rows on 32 experts, takes 70 us this way and took 124 us on the
// register-staged kernel, the only one that allowed them.
//
// Requirements: contraction length and leading dimensions multiples of 8 elements.
#pragma once

#include <type_traits>

#include "stream_slab.h"

namespace yamoe {

namespace async {

constexpr int kBK = 32;
constexpr int kThreads = 256;
constexpr int kMostRounds = 8;  // up to this many rounds of tiles, no XCD takes more of them than it must (see gemm_async_kernel)
constexpr int kBandRows = 8;  // row tiles of one band of an expert with many row tiles (see gemm_async_kernel)

// LDS layout and copy shapes of a tile of BM rows x BN columns
template <int BM_, int BN_> struct Tile {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int kAStages = 2, kAStageBytes = BM * 128;  // A ring: pairs of slabs (BM rows x 128 B)
  static constexpr int kBStages = 4, kBStageBytes = BN * 64;   // B ring: single slabs (32 k rows x 2 BN bytes)
  static constexpr int kBRing = kAStages * kAStageBytes;       // byte offset of the B ring
  static constexpr int kRingBytes = kBRing + kBStages * kBStageBytes;
  static constexpr int kStagingBytes = BM * (BN * 2 + 16);     // output tile staged for the row-wise store
  static constexpr int kBiasOff = kStagingBytes > kRingBytes ? kStagingBytes : kRingBytes;  // the tile's bias values
  static constexpr int kLds = kBiasOff + BN * 2;
  // [n][k] weights (the input-gradient products) keep B in slab pairs as well, three of them
  static constexpr int kBPairStages = 3, kBPairBytes = BN * 128;
  static constexpr int kRingNk = kBRing + kBPairStages * kBPairBytes;
  static constexpr int kDotBytes = BM * BN * 2;                // the tile of the second tensor of a row dot
  static constexpr int kLdsNk = kRingNk > kStagingBytes ? kRingNk : kStagingBytes;
  static_assert(kDotBytes <= kLdsNk, "the dot's tile fits");
  // copies per wave (1 KB each): an A pair, a slab of B, a pair of [n][k] B; a B copy covers kBRows k rows
  static constexpr int kACopies = BM / 32, kBRows = 512 / BN, kBCopies = 8 / kBRows, kBPairCopies = BN / 32;
  static constexpr int kMi = BM / 64, kNi = BN / 64;           // 32-row and 32-column blocks of a wave
  static constexpr int kParts = kRowTile / BM;                 // tiles that a row tile of the schedule is cut into
  static constexpr int kPerSimd = BM * BN <= 128 * 128 ? 2 : 1;  // workgroups per CU that registers and LDS are kept small for
};

enum { EPI_STORE = 0, EPI_GLU = 1 };

struct Args {
  const void *A;        // [rows, lda], k-contiguous
  const void *B;        // [E, Kd, Nd] ([k][n] per expert)
  const void *bias;     // [E, Nd] or null
  void *C;              // EPI_STORE: [rows, ldc]; EPI_GLU: act [rows, Nd/2]
  void *C2;             // EPI_GLU: optional pre-activations [rows, Nd]
  const int *a_rows;    // optional gather of A rows: source row = a_rows[p] / a_div
  const int *sched;
  FastDiv a_div, n_col_div;  // divisions by the gather divisor and by n_col_tiles
  FastDiv band_div;          // division by kBandRows * n_col_tiles
  int Kd, Nd, lda, ldb, ldc, n_col_tiles;
  long long b_expert_stride;
  // EPI_STORE with [n][k] weights, optional: dot_part[row][2 * col_tile + wave column] = the fp32 accumulators of the
  // row times dot_with[row][same columns] (a [rows, ldc] tensor), summed over the wave column's half of the tile
  const void *dot_with;
  float *dot_part;
  // FORM_CARRIER: the schedule's streaming list is worked off by stream_wgs workgroups of every XCD in this launch
  const int *small;
  int stream_wgs, n_stream_slabs;
  bool carries_alone;  // also where there is no tile (otherwise streaming launches of their own do it then)
  // FORM_REGULAR: every expert has reg_rows rows, cut into reg_tiles tiles of reg_per_tile; reg_units = experts times column
  // tiles, reg_div and reg_tile_div divide by an expert's tiles of all columns and of one
  int reg_rows, reg_tiles, reg_per_tile, reg_units;
  FastDiv reg_div, reg_tile_div;
#ifdef YAMOE_TILE_STAMPS
  unsigned long long *stamps;  // [stamps_cap][8]: see yamoe_debug_tile_stamps
  int stamps_cap;
#endif
};

#ifdef YAMOE_TILE_STAMPS
// Diagnostic build (-DYAMOE_TILE_STAMPS, `python -m yamoe_amd.tile_stamps`): thread 0 of every tile of gemm_async_kernel
// leaves eight words at stamps[8 * flat tile index]: the shader clock (s_memtime) at workgroup entry, before the first
// copy, when the first slab has landed, after the contraction loop, before the row-wise stores and at the end, then
// valid rows | valid columns << 16, and where it ran (XCC id << 8 | SE, SH and CU id).
#define YAMOE_STAMP(i) if (tid == 0) stamp_reg[i] = __builtin_amdgcn_s_memtime()
#else
#define YAMOE_STAMP(i)
#endif

template <typename T> struct Mma;
template <> struct Mma<bf16_t> {
  __device__ static inline void run(const u32x4 &a, const u32x4 &b, f32x16 &c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma<f16_t> {
  __device__ static inline void run(const u32x4 &a, const u32x4 &b, f32x16 &c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

// two fp32 values rounded to T, packed low / high
template <typename T> __device__ inline uint32_t pack2(float lo, float hi) {
  typedef T T2 __attribute__((ext_vector_type(2)));
  T2 v = {ElemTraits<T>::from_f32(lo), ElemTraits<T>::from_f32(hi)};
  return __builtin_bit_cast(uint32_t, v);
}
// four consecutive elements of T (8-byte aligned) as fp32
template <typename T> __device__ inline void load4_f32(const T *p, float (&out)[4]) {
  typedef T T4 __attribute__((ext_vector_type(4)));
  T4 v = *(const T4 *)p;
#pragma unroll
  for (int i = 0; i < 4; ++i) out[i] = ElemTraits<T>::to_f32(v[i]);
}

template <int N> __device__ inline void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// what one slab step of the pipeline issues besides its MFMAs
// VM: which wait stands between its k-steps (see the pipeline comment in run_tile)
enum { VM_NONE, VM_EVEN, VM_ODD, VM_LAST_B, VM_NK, VM_ALL };
// LAST: where the copies of the two k-steps belong to the last slab pair (bit 0: A, bit 1: B of the first k-step, bit 2: B
// of the second); ZERO: what is cleared past the end of the contraction after the wait, by which it has landed
enum { ZERO_NONE, ZERO_PAIR, ZERO_A_AND_FIRST, ZERO_SECOND };  // the last pair; its A and its first B slab; its second B slab
template <bool P1A_, bool P1B_, bool P2A_, bool P2B_, bool NEXT_, int VM_, bool BAR_ = true, int LAST_ = 0, int ZERO_ = ZERO_NONE>
struct StepCfg {
  static constexpr bool P1A = P1A_, P1B = P1B_, P2A = P2A_, P2B = P2B_, NEXT = NEXT_, BAR = BAR_;
  static constexpr int ZERO = ZERO_;
  static constexpr bool LAST_A = LAST_ & 1, LAST_B1 = (LAST_ >> 1) & 1, LAST_B2 = (LAST_ >> 2) & 1;
  static constexpr int VM = VM_;
};

struct TileInfo {
  int expert, row0, rows_valid, n0;
#ifdef YAMOE_TILE_STAMPS
  int slot;
  unsigned long long t_entry, t_lookup;
#endif
};

// NMI / NNI: how many of this wave's 32-row and 32-column blocks of the tile (four each at 256 x 256) hold valid rows / columns.  The
// 32-column blocks alternate between the two wave columns (block cb belongs to wave column cb & 1), so a tile of 64
// or 128 valid columns (the last column tile of a 2880-wide matrix) gives both wave columns a quarter or half of the
// MFMAs instead of all of them to one.
// NAB: how many of the tile's 32-row blocks are copied (the others hold no valid row).
template <typename T, class S, int EPI, int NMI, bool BNK, bool RAGGED, int NNI = S::kNi, int NAB = S::kACopies>
__device__ __forceinline__ void run_tile(const Args &args, const TileInfo &ti, const int tid, const char *a_base,
                                const uint32_t (&a_off)[S::kACopies], const char *b_base,
                                const uint32_t (&b_off)[BNK ? S::kBPairCopies : S::kBCopies], long long b_slab_bytes) {
  constexpr int kBN = S::BN, kAStages = S::kAStages, kAStageBytes = S::kAStageBytes, kBStages = S::kBStages,
                kBStageBytes = S::kBStageBytes, kBRing = S::kBRing, kBPairStages = S::kBPairStages,
                kBPairBytes = S::kBPairBytes, kBiasOff = S::kBiasOff;
  constexpr int kHalfA = S::kACopies / 2, kHalfB = S::kBCopies / 2, kHalfBp = S::kBPairCopies / 2;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, kept in a scalar register
  const int wm = wave >> 1, wn = wave & 1;
  constexpr int NACC = NMI > 0 ? NMI : 1;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);  // LDS byte address of the A ring

  f32x16 acc[NACC][S::kNi];
#pragma unroll
  for (int mi = 0; mi < NACC; ++mi)
#pragma unroll
    for (int ni = 0; ni < S::kNi; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0.0f;

  const int n_pairs = RAGGED ? (args.Kd + 2 * kBK - 1) / (2 * kBK) : args.Kd / (2 * kBK), n_slabs = 2 * n_pairs;
#ifdef YAMOE_TILE_STAMPS
  unsigned long long stamp_reg[6] = {ti.t_entry, ti.t_lookup, 0, 0, 0, 0};
#endif

  // The tile's bias values, one per thread, requested before anything else: they are the oldest entry of the memory
  // queue, so the first wait of the pipeline covers them, and the epilogue finds them in a register instead of
  // paying a memory latency per column block.  ([n][k] weights are the input-gradient products: no bias.)
  const bool has_bias = !BNK && args.bias != nullptr;
  T bias_reg = ElemTraits<T>::from_f32(0.0f);
  if (has_bias) bias_reg = ((const T *)args.bias)[(long long)ti.expert * args.Nd + min(ti.n0 + (kBN < kThreads ? tid & (kBN - 1) : tid), args.Nd - 1)];

  // ---- copy issue ----------------------------------------------------------------------------------
  // A pair p (slabs 2p, 2p+1): copy c is the 32-row block c of the tile, this wave fills its rows 8*wave + (lane >> 3),
  // 128 bytes each.  Blocks without valid rows (c >= NAB) are not copied: nobody reads them, and a tile of 192 rows,
  // the common one, moves an eighth less through the L1 than a full one.  (The count is a template parameter: a
  // run-time test around every copy and a run-time wait count cost more than the copies saved.)
  // `last` (the copies of the last pair): where the contraction ends inside the pair, lanes past its end fetch the row's
  // first piece of the pair instead.
  const int a_piece = ((lane & 7) ^ ((4 * wave + (lane >> 4)) & 7)) * 16;  // byte of the pair this lane copies
  const int last_bytes = args.Kd * (int)sizeof(T) - (n_pairs - 1) * 128;   // bytes of a row in the last pair
  auto copy_a = [&](int pair, int c, bool last) {
    if (c < NAB)
      copy16_to_lds(a_base + (long long)pair * (2 * kBK * (int)sizeof(T)), a_off[c] - (RAGGED && last && a_piece >= last_bytes ? a_piece : 0),
                    lds0 + (uint32_t)(pair & (kAStages - 1)) * kAStageBytes + (uint32_t)(32 * c + 8 * wave) * 128u);
  };
  auto issue_a = [&](int pair) {
#pragma unroll
    for (int c = 0; c < S::kACopies; ++c) copy_a(pair, c, pair == n_pairs - 1);
  };
  // clears what this wave copied of the last A pair beyond the end of the contraction
  auto zero_a = [&]() {
    if constexpr (RAGGED) {
      int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
      asm volatile("" : "+v"(l));  // (the lane number once more: nothing of this is kept in registers through the loop)
      if (((l & 7) ^ ((4 * wave + (l >> 4)) & 7)) * 16 >= last_bytes) {
        char *at = lds + ((n_pairs - 1) & (kAStages - 1)) * kAStageBytes + 8 * wave * 128 + l * 16;
#pragma unroll
        for (int c = 0; c < NAB; ++c) *(u32x4 *)(at + 32 * 128 * c) = (u32x4){0, 0, 0, 0};
      }
    }
  };
  // B slab: this wave fills k rows 8*wave .. + 7, kBRows of them per copy.  In the last pair, k rows past the end re-read
  // the last one (and a slab that lies past the end as a whole is addressed from the one before it).
  auto copy_b = [&](int slab, int i, bool last) {
    uint32_t off = b_off[i];
    int src_slab = slab;
    if (RAGGED && last) {
      int kd = args.Kd;
      asm volatile("" : "+s"(kd));  // (evaluated here: kept from before the loop it would cost the loop registers)
      src_slab = min(slab, (kd - 1) / kBK);
      const int k = 8 * wave + S::kBRows * i + lane / (kBN / 8);
      off -= (uint32_t)((k - (min(slab * kBK + k, kd - 1) - src_slab * kBK)) * args.ldb * (int)sizeof(T));
    }
    copy16_to_lds(b_base + (long long)__builtin_amdgcn_readfirstlane(src_slab) * b_slab_bytes, off,
                  lds0 + kBRing + (uint32_t)(slab & (kBStages - 1)) * kBStageBytes + (uint32_t)(8 * wave + S::kBRows * i) * (2 * kBN));
  };
  auto issue_b = [&](int slab) {
#pragma unroll
    for (int i = 0; i < S::kBCopies; ++i) copy_b(slab, i, slab >= n_slabs - 2);
  };
  // [n][k] weights: copy c of B pair `pair`, rows BN/4*wave + 8*c + (lane >> 3) like A
  auto copy_bp = [&](int pair, int c, bool last) {
    const int piece = ((lane & 7) ^ ((4 * c + (lane >> 4)) & 7)) * 16;
    copy16_to_lds(b_base + (long long)pair * (2 * b_slab_bytes), b_off[c] - (RAGGED && last && piece >= last_bytes ? piece : 0),
                  lds0 + kBRing + (uint32_t)(pair % kBPairStages) * kBPairBytes + (uint32_t)(kBN / 4 * wave + 8 * c) * 128u);
  };
  auto issue_bp = [&](int pair) {
#pragma unroll
    for (int c = 0; c < S::kBPairCopies; ++c) copy_bp(pair, c, pair == n_pairs - 1);
  };
  // the same for what this wave copied of slab `n_slabs - 2 + second` of B, and of the last B pair
  auto zero_b = [&](int second) {
    if constexpr (RAGGED) {
      int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
      asm volatile("" : "+v"(l));
      const int slab = n_slabs - 2 + second, k0 = 8 * wave + l / (kBN / 8);
      char *at = lds + kBRing + (slab & (kBStages - 1)) * kBStageBytes + 8 * wave * (2 * kBN) + l * 16;
#pragma unroll
      for (int i = 0; i < S::kBCopies; ++i)
        if (slab * kBK + k0 + S::kBRows * i >= args.Kd) *(u32x4 *)(at + S::kBRows * i * (2 * kBN)) = (u32x4){0, 0, 0, 0};
    }
  };
  auto zero_bp = [&]() {
    if constexpr (RAGGED) {
      int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
      asm volatile("" : "+v"(l));
      char *at = lds + kBRing + ((n_pairs - 1) % kBPairStages) * kBPairBytes + kBN / 4 * wave * 128 + l * 16;
#pragma unroll
      for (int c = 0; c < S::kBPairCopies; ++c)
        if (((l & 7) ^ ((4 * c + (l >> 4)) & 7)) * 16 >= last_bytes) *(u32x4 *)(at + 8 * c * 128) = (u32x4){0, 0, 0, 0};
    }
  };
  auto zero_last = [&]() {
    zero_a();
    if constexpr (BNK) zero_bp();
    else { zero_b(0); zero_b(1); }
  };

  // ---- MFMA operand reads ----------------------------------------------------------------------------
  // A operand (block mi, slab parity par, k-step ks): row (mi*2+wm)*32 + lane%32, piece par*4 + ks*2 + lane/32
  // at position piece ^ ((row >> 1) & 7).
  const int rl = lane & 31, g = lane >> 5;
  int a_rd[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) a_rd[ks] = (wm * 32 + rl) * 128 + (((ks * 2 + g) ^ ((rl >> 1) & 7)) << 4);
  // B operand (column block ni, k-step ks, half h): k = ks*16 + g*8 + h*4 + j, 4 columns at
  // (ni*2+wn)*32 + 16*((lane>>4)&1) + 4*q, where j = (lane&15)>>2 and q = lane&3.
  const int j4 = (lane & 15) >> 2, q4 = lane & 3;
  int b_rd[S::kNi];
#pragma unroll
  for (int ni = 0; ni < S::kNi; ++ni) {
    int col = (ni * 2 + wn) * 32 + 16 * ((lane >> 4) & 1) + 4 * q4;
    int piece = (col >> 3) ^ (j4 << 2);
    b_rd[ni] = (g * 8 + j4) * (2 * kBN) + (piece << 4) + (col & 7) * 2;
  }
  // B operand of a [n][k] tile (BNK): stored like A, in slab pairs of 128-byte rows; row (ni*2+wn)*32 + lane%32,
  // one 16-byte read per operand.
  int b_rdk[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) b_rdk[ks] = (wn * 32 + rl) * 128 + (((ks * 2 + g) ^ ((rl >> 1) & 7)) << 4);

  u32x4 fa0[NACC], fa1[NACC], fb0[S::kNi], fb1[S::kNi];
  // Operand fragments of one k-step in the order the MFMAs want them: B0, A0, B1, B2, B3, A1, A2, A3.
  // Slab s sits in A pair buffer (s>>1)&1 (the odd slab of a pair 64 bytes further, by XOR) and B buffer s&3.
  constexpr int kFrags = NMI > 0 ? NNI + NMI : 0;
  auto read_frag = [&](int s, int ks, int f, u32x4 (&fa)[NACC], u32x4 (&fb)[S::kNi]) {
    if (f == 1 || f >= 1 + NNI) {
      const int mi = f == 1 ? 0 : f - NNI;
      const char *sa = lds + ((s >> 1) & (kAStages - 1)) * kAStageBytes;
      fa[mi] = *(const u32x4 *)(sa + (a_rd[ks] ^ ((s & 1) << 6)) + mi * 8192);
    } else {
      const int ni = f == 0 ? 0 : f - 1;
      if constexpr (BNK) {
        const char *sb = lds + kBRing + ((s >> 1) % kBPairStages) * kBPairBytes;
        fb[ni] = *(const u32x4 *)(sb + (b_rdk[ks] ^ ((s & 1) << 6)) + ni * 8192);
      } else {
        const char *sb = lds + kBRing + (s & (kBStages - 1)) * kBStageBytes;
        u32x2 lo = lds_read_tr16(sb + b_rd[ni] + ks * (32 * kBN));
        u32x2 hi = lds_read_tr16(sb + b_rd[ni] + ks * (32 * kBN) + 8 * kBN);
        fb[ni] = (u32x4){lo[0], lo[1], hi[0], hi[1]};
      }
    }
  };
  auto read_frags = [&](int s, int ks, u32x4 (&fa)[NACC], u32x4 (&fb)[S::kNi]) {
#pragma unroll
    for (int f = 0; f < kFrags; ++f) read_frag(s, ks, f, fa, fb);
  };
  auto mma = [&](const u32x4 (&fa)[NACC], const u32x4 (&fb)[S::kNi]) {
#pragma unroll
    for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NNI; ++ni) Mma<T>::run(fb[ni], fa[mi], acc[mi][ni]);
  };
  // ---- pipeline -----------------------------------------------------------------------------------------
  // A slab is two k-steps with one workgroup barrier between them; after the barrier of slab t nobody reads
  // slab t's buffers any more.  The L1 path moves 64 bytes per clock into LDS and a slab needs 32 KB of
  // copies against 1024 clocks of MFMAs, so the copies are spread as evenly as the buffer lifetimes allow:
  //   second k-step of slab t:  (t odd) first half of A pair (t+1)/2 + 1;  first half of B slab t + 4
  //   first k-step of slab t:   (t even) second half of A pair t/2 + 1;    second half of B slab t + 3
  // which is 6, 2, 2, 6 copies per wave over the four k-steps of a slab pair (256 x 256).  Copies retire in order, so
  // "slab s+1 has landed" is a bound on the number of younger copies in flight at the end of the first
  // k-step of slab s: for even s two B slabs and one A pair (VM_EVEN: 8 + the pair's copies, 16 for a full tile), for odd
  // s one and a half B slabs (VM_ODD: 6), then half a slab (VM_LAST_B: 2) and none for the last two waits.
  if constexpr (BNK) {
    // [n][k] weights, both operands in slab pairs.  After the barrier of an odd slab 2p+1 pair p is dead: A pair p+2
    // goes into its buffer during the next two k-steps and B pair p+3 during the two after those, four copies per wave
    // in every k-step.  Only odd slabs wait (VM_NK: for pair p+1, with the copies of B pair p+2 still in flight) and
    // only odd slabs need the workgroup barrier.
    issue_a(0);
    issue_bp(0);
    if (n_slabs > 2) { issue_a(1); issue_bp(1); }
    if (n_slabs >= 8) {
      wait_vmcnt<S::kBPairCopies + NAB>();  // pair 0 is there when only A pair 1 and B pair 1 are in flight
    } else {
      if (n_slabs > 4) issue_bp(2);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  } else {
    issue_b(0);
    issue_a(0);
    if (n_slabs > 1) issue_b(1);
    if (n_slabs > 2) { issue_b(2); issue_a(1); }
    if (n_slabs > 3) issue_b(3);
    // Only slab 0 (the first copies of B and of A) has to be there to start; the waits of the slab steps below bound the
    // number of younger copies in flight, and that bound holds for what is left of these as well.
    if (n_slabs >= 8) wait_vmcnt<3 * S::kBCopies + NAB>();  // B1, B2, B3 and A pair 1
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (RAGGED && n_pairs <= 2) zero_last();
  __syncthreads();
  YAMOE_STAMP(2);
  read_frags(0, 0, fa0, fb0);

  // The instruction order is fixed by hand, because one wave per SIMD has nobody to hide behind: every LDS
  // read and every copy is issued in the shadow of an MFMA (an MFMA occupies the matrix pipe for 8 issue
  // slots), a whole k-step before its result is needed.
  //   first k-step:  MFMAs on set 0 + its copies + the LDS reads of the second k-step into set 1
  //   wait for slab s+1's copies; workgroup barrier
  //   second k-step: MFMAs on set 1 + its copies + the LDS reads of slab s+1's first k-step into set 0
  constexpr int kMma = NNI * NMI;
  constexpr int kSlots = kMma > 2 ? kMma - 2 : 1;  // the last two MFMAs of a k-step carry nothing
  auto slab_step = [&](int s, auto cfg) {
    typedef decltype(cfg) C;
    __builtin_amdgcn_sched_barrier(0);
    {
      constexpr int kA = C::P1A ? kHalfA : 0, kB = C::P1B ? (BNK ? kHalfBp : kHalfB) : 0, kItems = kA + kB + kFrags;
#pragma unroll
      for (int j = 0; j < (kMma > 0 ? kMma : 1); ++j) {
        if (j < kMma) Mma<T>::run(fb0[j % NNI], fa0[j / NNI], acc[j / NNI][j % NNI]);
        if (j < kSlots) {
#pragma unroll
          for (int i = j * kItems / kSlots; i < (j + 1) * kItems / kSlots; ++i) {
            if (i < kA) copy_a(s / 2 + 1, kHalfA + i, C::LAST_A);
            else if (i < kA + kB) {
              if constexpr (BNK) copy_bp((s + 3) / 2, kHalfBp + i - kA, C::LAST_B1);
              else copy_b(s + 3, kHalfB + i - kA, C::LAST_B1);
            }
            else read_frag(s, 1, i - kA - kB, fa1, fb1);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (C::VM == VM_EVEN) wait_vmcnt<2 * S::kBCopies + NAB>();
    else if constexpr (C::VM == VM_ODD) wait_vmcnt<S::kBCopies + kHalfB>();
    else if constexpr (C::VM == VM_LAST_B) wait_vmcnt<kHalfB>();
    else if constexpr (C::VM == VM_NK) wait_vmcnt<S::kBPairCopies>();
    else if constexpr (C::VM == VM_ALL) wait_vmcnt<0>();
    if constexpr (C::ZERO == ZERO_PAIR) zero_last();
    else if constexpr (C::ZERO == ZERO_A_AND_FIRST) { zero_a(); zero_b(0); }
    else if constexpr (C::ZERO == ZERO_SECOND) zero_b(1);
    if constexpr (C::BAR) __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    {
      constexpr int kA = C::P2A ? kHalfA : 0, kB = C::P2B ? (BNK ? kHalfBp : kHalfB) : 0, kItems = kA + kB + (C::NEXT ? kFrags : 0);
#pragma unroll
      for (int j = 0; j < (kMma > 0 ? kMma : 1); ++j) {
        if (j < kMma) Mma<T>::run(fb1[j % NNI], fa1[j / NNI], acc[j / NNI][j % NNI]);
        if (j < kSlots) {
#pragma unroll
          for (int i = j * kItems / kSlots; i < (j + 1) * kItems / kSlots; ++i) {
            if (i < kA) copy_a((s + 1) / 2 + 1, i, C::LAST_A);
            else if (i < kA + kB) {
              if constexpr (BNK) copy_bp(s / 2 + 2, i - kA, C::LAST_B2);
              else copy_b(s + 4, i - kA, C::LAST_B2);
            }
            else read_frag(s + 1, 0, i - kA - kB, fa0, fb0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // the same with every decision taken at run time, for contractions shorter than 8 slabs
  auto slab_step_short = [&](int s, bool odd) {
    read_frags(s, 1, fa1, fb1);
    mma(fa0, fb0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (RAGGED && odd && s + 3 == n_slabs && n_pairs > 2) zero_last();
    __syncthreads();
    if (odd && s + 3 < n_slabs) issue_a((s + 1) / 2 + 1);
    if constexpr (!BNK) {
      if (s + kBStages < n_slabs) issue_b(s + kBStages);  // ([n][k]: at most three B pairs, all requested up front)
    }
    if (s + 1 < n_slabs) read_frags(s + 1, 0, fa0, fb0);
    mma(fa1, fb1);
  };
  if (BNK && n_slabs >= 8) {
    slab_step(0, StepCfg<false, false, false, true, true, VM_NONE, false>());
    slab_step(1, StepCfg<false, true, true, false, true, VM_NK>());
    int s = 2;
    for (; s + (RAGGED ? 7 : 5) < n_slabs; s += 2) {  // steady state: pair s/2 is consumed, A pair s/2 + 1 and B pair s/2 + 2 arrive
      slab_step(s, StepCfg<true, false, false, true, true, VM_NONE, false>());
      slab_step(s + 1, StepCfg<false, true, true, false, true, VM_NK>());
    }
    if constexpr (RAGGED) {
      // the same once more (s = n_slabs - 6): what it copies belongs to the last pair, but for the A half of its first step
      slab_step(s, StepCfg<true, false, false, true, true, VM_NONE, false, 4>());
      slab_step(s + 1, StepCfg<false, true, true, false, true, VM_NK, true, 1 | 2>());
      s += 2;
    }
    // the last two pairs (s = n_slabs - 4)
    slab_step(s, StepCfg<true, false, false, false, true, VM_NONE, false, 1>());
    slab_step(s + 1, StepCfg<false, false, false, false, true, VM_ALL, true, 0, ZERO_PAIR>());
    slab_step(s + 2, StepCfg<false, false, false, false, true, VM_NONE, false>());
    slab_step(s + 3, StepCfg<false, false, false, false, false, VM_NONE, false>());
  } else if (n_slabs >= 8) {
    // copies of the (first, second) k-step: A half, B half; whether slab s+1 is read; the wait
    slab_step(0, StepCfg<false, false, false, true, true, VM_EVEN>());
    slab_step(1, StepCfg<false, true, true, true, true, VM_ODD>());
    int s = 2;
    for (; s + 7 < n_slabs; s += 2) {  // steady state
      slab_step(s, StepCfg<true, true, false, true, true, VM_EVEN>());
      slab_step(s + 1, StepCfg<false, true, true, true, true, VM_ODD>());
    }
    // the last six slabs (s = n_slabs - 6): the last copies go out in the first k-step of slab n_slabs - 4
    slab_step(s, StepCfg<true, true, false, true, true, VM_EVEN, true, 4>());
    slab_step(s + 1, StepCfg<false, true, true, true, true, VM_ODD, true, 1 | 2 | 4>());
    slab_step(s + 2, StepCfg<true, true, false, false, true, VM_EVEN, true, 1 | 2>());
    slab_step(s + 3, StepCfg<false, false, false, false, true, VM_LAST_B, true, 0, ZERO_A_AND_FIRST>());
    slab_step(s + 4, StepCfg<false, false, false, false, true, VM_ALL, true, 0, ZERO_SECOND>());
    slab_step(s + 5, StepCfg<false, false, false, false, false, VM_NONE>());
  } else {
    for (int s = 0; s < n_slabs; s += 2) {
      slab_step_short(s, false);
      slab_step_short(s + 1, true);
    }
  }

  YAMOE_STAMP(3);
  // ---- epilogue -------------------------------------------------------------------------------------
  // The output tile is staged in LDS (the slab ring is dead by now) as [row][column] and then written
  // out row by row with 16 bytes per lane, so that a wave stores whole 512-byte (or 256-byte) row
  // segments instead of 2 bytes per lane.
  // The MFMAs run with the operands exchanged (weights as the A operand), so a lane holds one output row and four
  // consecutive columns per register quad:
  // acc[mi][ni][v]: tile row (mi*2+wm)*32 + lane%32, tile column (ni*2+wn)*32 + 8*(v/4) + 4*(lane/32) + v%4
  // which makes the staging stores 8 bytes wide and puts a (gate, up) pair into one lane.
  const int rows_valid = ti.rows_valid, n0 = ti.n0;
  const long long out_row0 = ti.row0;

  // rows of `width` elements, row stride width*2 + 16 bytes
  auto store_rows = [&](T *dst, long long ld, int col0, int width, int col_limit) {
    const int stride = width * 2 + 16;
    const int chunks = width >> 3, rows_per_pass = kThreads / chunks;
    const int c = tid % chunks;
    if (col0 + c * 8 >= col_limit) return;
    T *p = dst + out_row0 * ld + col0 + c * 8;
    for (int r = tid / chunks; r < rows_valid; r += rows_per_pass)
      *(u32x4 *)(p + (long long)r * ld) = *(const u32x4 *)(lds + r * stride + c * 16);
  };
  // the bias of this lane's 16 columns of column block ni, from the copy in LDS
  auto load_bias = [&](int ni, float (&b)[16]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (has_bias) load4_f32((const T *)(lds + kBiasOff) + (ni * 2 + wn) * 32 + 8 * q + 4 * g, t);
#pragma unroll
      for (int i = 0; i < 4; ++i) b[4 * q + i] = t[i];
    }
  };
  // natural column order: value = acc + bias[column]   (the plain product, or, with `pre`, the pre-activations as the
  // backward reads them: even columns gate, odd columns up)
  auto stage_biased = [&](auto pre) {
    constexpr int stride = kBN * 2 + 16;
    char *lp = lds + (wm * 32 + rl) * stride + (wn * 32 + 4 * g) * 2;  // one address per lane, the rest are constants
#pragma unroll
    for (int ni = 0; ni < NNI; ++ni) {
      float b[16];
      load_bias(ni, b);
#pragma unroll
      for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16 &a = acc[mi][ni];
          u32x2 v;
          if constexpr (decltype(pre)::value) {
            typedef T T2 __attribute__((ext_vector_type(2)));
            T2 lo = {pre_activation_store<T>(a[4 * q] + b[4 * q], false), pre_activation_store<T>(a[4 * q + 1] + b[4 * q + 1], true)};
            T2 hi = {pre_activation_store<T>(a[4 * q + 2] + b[4 * q + 2], false), pre_activation_store<T>(a[4 * q + 3] + b[4 * q + 3], true)};
            v = (u32x2){__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
          } else {
            v = (u32x2){pack2<T>(a[4 * q] + b[4 * q], a[4 * q + 1] + b[4 * q + 1]),
                        pack2<T>(a[4 * q + 2] + b[4 * q + 2], a[4 * q + 3] + b[4 * q + 3])};
          }
          *(u32x2 *)(lp + mi * 64 * stride + (ni * 64 + 8 * q) * 2) = v;
        }
    }
  };

  if (has_bias && (kBN >= kThreads || tid < kBN)) *(T *)(lds + kBiasOff + tid * 2) = bias_reg;  // (outside the ring and the staging area)
  __syncthreads();  // every wave has finished reading the slab ring
  if constexpr (EPI == EPI_STORE && BNK) {
    // Row dots of the product with a second tensor of the output's shape, taken from the fp32 accumulators before they
    // are rounded (the routing gradient <grad_out . W_down^T, act>, csrc/experts_backward.cu:83-88): every wave writes
    // one partial sum per valid row, over half of the tile's columns; whoever reads them adds 2 * n_col_tiles values
    // per row in a fixed order.  The tile of the second tensor comes in through LDS by asynchronous copies, all in
    // flight at once (the ring is dead): the 16-byte pieces of row r XOR-swizzled with r on the
    // global side, so that the 32 lanes that read the same columns of 32 consecutive rows touch every bank once.
    if (args.dot_part != nullptr) {
      {
        const uint32_t lds_tile = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
        const char *src = (const char *)((const T *)args.dot_with + out_row0 * args.ldc + n0);
        const long long ld_bytes = (long long)args.ldc * (long long)sizeof(T);
        constexpr int kPieces = kBN / 8;  // 16-byte pieces of a row
#pragma unroll 8
        for (int i = 0; i < S::BM / 4 / S::kBRows; ++i) {
          const int row = S::BM / 4 * wave + S::kBRows * i + lane / kPieces;
          int piece = (lane ^ row) & (kPieces - 1);
          if (n0 + piece * 8 >= args.Nd) piece = 0;  // columns past the end: re-read valid ones, never used
          const uint32_t off = (uint32_t)(min(row, rows_valid - 1) * ld_bytes + piece * 16);
          copy16_to_lds(src, off, lds_tile + (uint32_t)(S::BM / 4 * wave + S::kBRows * i) * (2 * kBN));
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      __syncthreads();
      const int n_part = 2 * args.n_col_tiles, part_col = 2 * (n0 / kBN) + wn;
      const char *lp = lds + (wm * 32 + rl) * (2 * kBN) + g * 8;
#pragma unroll
      for (int mi = 0; mi < NMI; ++mi) {
        const int r = (mi * 2 + wm) * 32 + rl;
        float part = 0.0f;
#pragma unroll
        for (int ni = 0; ni < NNI; ++ni)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            // a run of four columns is valid or invalid as a whole (the column count is a multiple of 8)
            if (n0 + (ni * 2 + wn) * 32 + 8 * q + 4 * g < args.Nd) {
              float w4[4];
              load4_f32((const T *)(lp + mi * 64 * (2 * kBN) + ((((ni * 2 + wn) * 4 + q) ^ (rl & (kBN / 8 - 1))) << 4)), w4);
#pragma unroll
              for (int i = 0; i < 4; ++i) part += acc[mi][ni][4 * q + i] * w4[i];
            }
          }
        part += __shfl_xor(part, 32);
        if (g == 0 && r < rows_valid) args.dot_part[(out_row0 + r) * n_part + part_col] = part;
      }
      __syncthreads();  // the staging area is about to be overwritten with the output tile
    }
  }
  if constexpr (EPI == EPI_STORE) {
    stage_biased(std::false_type());
    __syncthreads();
    YAMOE_STAMP(4);
    store_rows((T *)args.C, args.ldc, n0, kBN, args.Nd);
  } else {
    if (args.C2 != nullptr) {  // pre-activations for the backward: the biased product itself
      stage_biased(std::true_type());
      __syncthreads();
      store_rows((T *)args.C2, args.Nd, n0, kBN, args.Nd);
      __syncthreads();
    }
    // A register quad holds (gate, up, gate, up) of two neighbouring activations of one row.
    constexpr int stride = (kBN / 2) * 2 + 16;
    char *lp = lds + (wm * 32 + rl) * stride + (wn * 16 + 2 * g) * 2;
#pragma unroll
    for (int ni = 0; ni < NNI; ++ni) {
      float b[16];
      load_bias(ni, b);
#pragma unroll
      for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16 &a = acc[mi][ni];
          float h0 = glu_forward(a[4 * q] + b[4 * q], a[4 * q + 1] + b[4 * q + 1]);
          float h1 = glu_forward(a[4 * q + 2] + b[4 * q + 2], a[4 * q + 3] + b[4 * q + 3]);
          *(uint32_t *)(lp + mi * 64 * stride + (ni * 32 + 4 * q) * 2) = pack2<T>(h0, h1);
        }
    }
    __syncthreads();
    YAMOE_STAMP(4);
    store_rows((T *)args.C, args.ldc, n0 >> 1, kBN / 2, args.Nd >> 1);
  }
#ifdef YAMOE_TILE_STAMPS
  YAMOE_STAMP(5);
  if (tid == 0 && args.stamps != nullptr && ti.slot < args.stamps_cap) {
    unsigned long long *o = args.stamps + 8ll * ti.slot;
#pragma unroll
    for (int i = 0; i < 6; ++i) o[i] = stamp_reg[i];
    o[6] = (unsigned long long)(uint32_t)ti.rows_valid | ((unsigned long long)(uint32_t)min(kBN, args.Nd - ti.n0) << 16);
    const unsigned hw = __builtin_amdgcn_s_getreg((4 << 0) | (8 << 6) | (7 << 11));    // HW_ID bits 8..15: CU, SH and SE id
    const unsigned xcc = __builtin_amdgcn_s_getreg((20 << 0) | (0 << 6) | (3 << 11));  // XCC_ID
    o[7] = ((unsigned long long)xcc << 8) | hw;
  }
#endif
}

// One workgroup's part of the streaming list: items `first`, first + step, ...  An item is a slab of one expert, and
// neighbouring items, which different XCDs work on, are neighbouring slabs.  (17 to 32 rows as the last rows of an
// expert beside its tiles, or where invalid ids leave no expert more: a capacity that does keeps the tiles' launches away.)  Two
// launches less per layer: 2048 tokens x 2 on 16 experts, 1024 wide, whole layer 81.6 -> 78.1 us, 426 x 2: 42.4 -> 39.5.  In
// launches of many rounds these workgroups took the time of the streaming kernel to the microsecond, behind the tiles or
// between the first of them (Zipf routing, 16 384 tokens: gate_up 1794 + 266 and 2063 us); in short ones they are best behind
// the tiles (in front of them: 150 drawn calls 0.996 in the mean, single ones up to 1.24).
static_assert(kThreads == kStreamWaves * kWave, "a workgroup of the tile kernels is one of the streaming kernel");
template <typename T, int EPI, bool GATHER, int DEPTH> __device__ __forceinline__ void stream_items(const Args &args, int first, int step) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  StreamArgs a = {};
  a.A = args.A; a.B = args.B; a.bias = args.bias; a.C = args.C; a.C2 = args.C2; a.a_rows = args.a_rows; a.a_div = args.a_div;
  a.Kd = args.Kd; a.Nd = args.Nd; a.lda = args.lda; a.ldc = args.ldc;
  if (args.sched[0] == 0 && !args.carries_alone) return;
  const int items = args.sched[1] * args.n_stream_slabs;
  for (int it = first; it < items; it += step) {
    const int s = it / args.n_stream_slabs;
    const int *e = args.small + 4 * s;
    const int expert = __builtin_amdgcn_readfirstlane(e[0]), row0 = __builtin_amdgcn_readfirstlane(e[1]);
    const int rows = __builtin_amdgcn_readfirstlane(e[2]), slab = it - s * args.n_stream_slabs;
    if (rows > 16) stream_slab<T, EPI == EPI_GLU, GATHER, kStreamWaves, 2, 2>(a, (float *)lds, expert, row0, rows, slab);
    else stream_slab<T, EPI == EPI_GLU, GATHER, kStreamWaves, DEPTH, 1>(a, (float *)lds, expert, row0, rows, slab);
    __syncthreads();  // the next item's partial sums take the place of this one's
  }
}

// Where a launch's work comes from.  Instantiations of their own, because all forms in one kernel, told apart at run time, leave
// it short of scalar registers (19 to 42 spilled, none with the list alone): the gate_up product of 67 600 rows on 128 experts
// (Zipf routing, 720 x 5760, 29 rounds of tiles with a short contraction) took 744 us instead of 727.  150 drawn calls that carry
// streamed experts 0.993 in the mean, single ones 0.94 to 1.09: where their workgroups meet tiles on a CU changes with
// the time at which idle workgroups leave.
enum {
  FORM_LIST = 0,     // the schedule's row tiles
  FORM_CARRIER = 1,  // these and the schedule's streaming list, by stream_wgs workgroups of every XCD
  FORM_REGULAR = 2,  // every expert has reg_rows rows: no schedule
};

template <typename T, class S, int EPI, bool GATHER, bool BNK, bool RAGGED, int FORM>
__global__ __launch_bounds__(kThreads, S::kPerSimd) void gemm_async_kernel(const Args args) {
  constexpr int kBN = S::BN;

  // Workgroup b runs on XCD b % 8 and takes tile b / 8 of that XCD's share of the tile list.  The shares have
  // equal cost, not equal length, and are cut on (expert, column tile) boundaries, so the row tiles that read
  // the same weight slabs meet in one L2.  A share longer than its slots hands its excess to the workgroups that shorter
  // shares leave over.  An XCD has as many slots as the rounds that the whole list takes on 256 CUs have places on its
  // 32: shares of equal cost put 27 to 35 tiles of a 252-tile list on an XCD, and one tile over a round costs a round.
  // Whole forwards, us, slots for every workgroup / as here: 979 tokens x 2 on 16 experts, 2048 wide: 153 / 123; 3553 x 4 on 32,
  // 1024: 176 / 134; 3773 x 4 on 128, 2048: 728 / 687; 2003 x 4 on 32, 2880 x 720: 224 / 168 where the routing makes up to 256 gate_up
  // tiles, 225 / 225 where it makes 258 to 270.  130 drawn forwards, here over slots for everybody in the mean: 2 rounds 0.90,
  // 3 0.96, 4 0.97, 5 0.99, 6 0.99, 7 0.985, 8 0.985 (single ones 0.76 to 1.009), 9 to 21 1.000 (0.98 to 1.014).  Beyond kMostRounds a
  // round is little of a launch, and tiles of very different cost should stay where the cost puts them (29 rounds, Zipf
  // routing: 3250 / 3276); there only the grid bounds a share (it has at least as many workgroups as there are tiles).
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1;
#ifdef YAMOE_TILE_STAMPS
  const unsigned long long t_entry = __builtin_amdgcn_s_memtime();
#endif
  int L;
  const int place = blockIdx.x / kXcds;
  constexpr bool regular = FORM == FORM_REGULAR;
  const int stream_wgs = FORM == FORM_CARRIER ? args.stream_wgs : 0;
  auto cut_of = [&](int x) {
    return regular ? (int)((long long)x * args.reg_units / kXcds) * args.reg_tiles : sched_cut(args.sched, x, args.n_col_tiles);
  };
  {
    const int xcd = blockIdx.x % kXcds;
    const int first = cut_of(xcd), count = cut_of(xcd + 1) - first;
    const int total = regular ? args.reg_units * args.reg_tiles : sched_cut_row_tiles(args.sched, xcd) * args.n_col_tiles;
    const int rounds = ceil_div(total, kXcds * kXcdCus);
    if constexpr (FORM == FORM_CARRIER) {
      const int k = place - (int)(gridDim.x / kXcds - stream_wgs);  // behind the tiles
      if (k >= 0) {
        stream_items<T, EPI, GATHER, S::kPerSimd == 1 ? 3 : 2>(args, k * kXcds + xcd, stream_wgs * kXcds);
        return;
      }
    }
    const int i = place / S::kParts;
    int slots = (gridDim.x / kXcds - stream_wgs) / S::kParts;
    if (rounds <= kMostRounds) slots = min(slots, rounds * kXcdCus);
    if (i >= slots) return;
    if (i < count) {
      L = first + i;
    } else {
      int cut[kXcds + 1];
#pragma unroll
      for (int x = 0; x <= kXcds; ++x) cut[x] = cut_of(x);
      int rank = i - count;  // rank of this workgroup among the idle ones
#pragma unroll
      for (int x = 0; x < kXcds; ++x)
        if (x < xcd) rank += max(slots - (cut[x + 1] - cut[x]), 0);
      L = -1;
#pragma unroll
      for (int x = 0; x < kXcds; ++x) {
        int excess = max(cut[x + 1] - cut[x] - slots, 0);
        if (L < 0) {
          if (rank < excess) L = cut[x] + slots + rank;
          else rank -= excess;
        }
      }
      if (L < 0) return;
    }
  }
  TileInfo ti;
  {
    const int *tiles = args.sched + kSchedHeader;
    int gfirst, gcount, local;
    FastDiv by_gcount;
    if constexpr (regular) {
      gfirst = fast_div(L, args.reg_div);  // (the expert: it has no tiles in a list)
      gcount = args.reg_tiles;
      by_gcount = args.reg_tile_div;
      local = L - gfirst * gcount * args.n_col_tiles;
    } else {
      const int t0 = fast_div(L, args.n_col_div);
      gfirst = __builtin_amdgcn_readfirstlane(tiles[8 * t0 + 3]);
      gcount = __builtin_amdgcn_readfirstlane(tiles[8 * t0 + 4]);
      by_gcount = {(uint32_t)__builtin_amdgcn_readfirstlane(tiles[8 * t0 + 5]),
                   (uint32_t)__builtin_amdgcn_readfirstlane(tiles[8 * t0 + 6])};
      local = L - gfirst * args.n_col_tiles;
    }
    int col_tile, row_tile;
    if (gcount < 2 * kBandRows) {
      // the expert's tiles column by column: its few row tiles follow each other and share the column's weight slabs
      col_tile = fast_div(local, by_gcount);
      row_tile = local - col_tile * gcount;
    } else {
      // An expert with many row tiles, in bands of kBandRows row tiles (the last band takes the remainder), each band
      // column by column.  The 32 CUs of an XCD work on 32 consecutive tiles; column by column over the whole expert
      // those are 32 row tiles of one column, which share the weight slabs but fetch 32 different sets of rows, and
      // every row comes through the L2 once per column tile (measured at 8192 rows per expert: 12 times the
      // algorithmic bytes fetched, 4.4 TB/s, and the products 11 % slower than in bands).  In a band they are 4
      // columns of 8 row tiles: 8 sets of rows and 4 sets of slabs for the same 32 tiles.  Bands of 4 to 16 row tiles
      // measure within 1 % of each other; below 16 row tiles the column order is as good or better.
      const int bands = gcount / kBandRows;
      int band = min(fast_div(local, args.band_div), bands - 1);
      const int in_band = local - band * kBandRows * args.n_col_tiles;
      const int band_rows = band == bands - 1 ? gcount - band * kBandRows : kBandRows;
      col_tile = (int)((uint32_t)in_band / (uint32_t)band_rows);
      row_tile = band * kBandRows + in_band - col_tile * band_rows;
    }
    // (the same for every lane; said explicitly, so that the operand addresses built from them stay in scalar registers
    // whatever the compiler can prove about the work list's memory)
    if constexpr (regular) {
      ti.expert = gfirst;
      ti.row0 = gfirst * args.reg_rows + row_tile * args.reg_per_tile;
      ti.rows_valid = min(args.reg_per_tile, args.reg_rows - row_tile * args.reg_per_tile);
    } else {
      const int *te = tiles + 8 * (gfirst + row_tile);
      ti.expert = te[0];
      ti.row0 = te[1];
      ti.rows_valid = te[2];
    }
    ti.expert = __builtin_amdgcn_readfirstlane(ti.expert);
    ti.row0 = __builtin_amdgcn_readfirstlane(ti.row0);
    ti.rows_valid = __builtin_amdgcn_readfirstlane(ti.rows_valid);
    if constexpr (S::kParts == 2) {
      // The row tile's two halves are neighbours in the grid, on one XCD.  More than 128 rows are cut into two parts of
      // whole 32-row blocks as equal as they get; up to 128 rows are one part, and the other workgroup has nothing to do.
      const int first_rows = ti.rows_valid > S::BM ? ((ti.rows_valid + 63) >> 6) * 32 : ti.rows_valid;
      if (place & 1) {
        ti.row0 += first_rows;
        ti.rows_valid -= first_rows;
        if (ti.rows_valid <= 0) return;
      } else {
        ti.rows_valid = first_rows;
      }
    }
    ti.n0 = col_tile * kBN;
#ifdef YAMOE_TILE_STAMPS
    ti.slot = L; ti.t_entry = t_entry;
#endif
  }

  // A copies: copy i fetches rows 32*i + 8*wave + (lane >> 3); LDS position lane & 7 holds piece pos ^ ((row >> 1) & 7)
  // (a gathering instantiation without a row list reads its rows in order, like the others: the form the callers use
  // when the gathered tensor is too large for 32-bit byte offsets from its start and they have permuted it first)
  const bool gathers = GATHER && args.a_rows != nullptr;
  uint32_t a_off[S::kACopies];
#pragma unroll
  for (int i = 0; i < S::kACopies; ++i) {
    int row = 32 * i + 8 * wave + (lane >> 3);
    int piece = (lane & 7) ^ ((row >> 1) & 7);
    int r = min(row, ti.rows_valid - 1);
    long long src = r;
    if (gathers) src = fast_div(args.a_rows[ti.row0 + r], args.a_div);
    a_off[i] = (uint32_t)((src * args.lda + piece * 8) * (long long)sizeof(T));
  }
  const char *a_base = (const char *)((const T *)args.A + (gathers ? 0ll : (long long)ti.row0 * args.lda));

  const long long b_ld_bytes = (long long)args.ldb * (long long)sizeof(T);
  uint32_t b_off[BNK ? S::kBPairCopies : S::kBCopies];
  const char *b_base;
  long long b_slab_bytes;
  if constexpr (BNK) {
    // B is [n][k] (k-contiguous rows, one per output column), copied like A: rows BN/4*wave + 8*i + (lane >> 3), 128
    // bytes (two slabs) of each per copy, so that every request is a whole cache line; LDS position lane & 7 holds
    // piece pos ^ ((row >> 1) & 7)
#pragma unroll
    for (int i = 0; i < S::kBPairCopies; ++i) {
      int row = kBN / 4 * wave + 8 * i + (lane >> 3);
      int piece = (lane & 7) ^ ((row >> 1) & 7);
      int r = min(row, args.Nd - 1 - ti.n0);  // columns past the end re-read the last one; never stored
      b_off[i] = (uint32_t)(r * b_ld_bytes + piece * 16);
    }
    b_base = (const char *)((const T *)args.B + (long long)ti.expert * args.b_expert_stride + (long long)ti.n0 * args.ldb);
    b_slab_bytes = kBK * (long long)sizeof(T);
  } else {
    // B is [k][n]: k rows 8*wave + kBRows*i + lane / (BN/8); LDS position lane % (BN/8) holds piece pos ^ ((k & 3) << 2)
#pragma unroll
    for (int i = 0; i < S::kBCopies; ++i) {
      int k = 8 * wave + S::kBRows * i + lane / (kBN / 8);
      int piece = (lane & (kBN / 8 - 1)) ^ ((k & 3) << 2);
      int col = ti.n0 + piece * 8;
      if (col >= args.Nd) col = ti.n0;  // columns past the end re-read valid ones; never stored
      b_off[i] = (uint32_t)(k * b_ld_bytes + (long long)(col - ti.n0) * (long long)sizeof(T));
    }
    b_base = (const char *)((const T *)args.B + (long long)ti.expert * args.b_expert_stride + ti.n0);
    b_slab_bytes = kBK * b_ld_bytes;
  }

#ifdef YAMOE_TILE_STAMPS
  // (after the work-list look-ups and the gathered row numbers: a_off depends on both)
  asm volatile("s_waitcnt vmcnt(0)" : : "v"(a_off[0]), "v"(a_off[S::kACopies - 1]) : "memory");
  ti.t_lookup = __builtin_amdgcn_s_memtime();
#endif
  const int n_blocks32 = (ti.rows_valid + 31) >> 5;
  const int n_mi = (n_blocks32 - wm + 1) >> 1;
  // valid 32-column blocks of this wave column (they alternate between the two); tiles of 64 or 128 valid columns with
  // three or four row blocks per wave have instantiations of their own, everything else computes all four blocks
  const int wn = wave & 1;
  const int n_blocks32_n = (min(kBN, args.Nd - ti.n0) + 31) >> 5;
  const int n_ni = (n_blocks32_n - wn + 1) >> 1;
#define YAMOE_RUN(NMI_, NNI_) run_tile<T, S, EPI, NMI_, BNK, RAGGED, NNI_>(args, ti, tid, a_base, a_off, b_base, b_off, b_slab_bytes)
#define YAMOE_RUN6(NNI_) run_tile<T, S, EPI, 3, BNK, RAGGED, NNI_, 6>(args, ti, tid, a_base, a_off, b_base, b_off, b_slab_bytes)
  if constexpr (S::kMi == 4) {
    // six row blocks (161..192 rows, what an expert with a few rows more than two full tiles is cut into): both wave
    // rows have three, and only six of the eight blocks are copied
    const bool six = n_blocks32 == 6;
    if (n_ni <= 2 && n_mi >= 3) {
      if (n_ni <= 1) { if (n_mi == 4) YAMOE_RUN(4, 1); else if (six) YAMOE_RUN6(1); else YAMOE_RUN(3, 1); }
      else { if (n_mi == 4) YAMOE_RUN(4, 2); else if (six) YAMOE_RUN6(2); else YAMOE_RUN(3, 2); }
      return;
    }
    if (six) { YAMOE_RUN6(4); return; }
    switch (n_mi) {
      case 4: YAMOE_RUN(4, 4); break;
      case 3: YAMOE_RUN(3, 4); break;
      case 2: YAMOE_RUN(2, 4); break;
      case 1: YAMOE_RUN(1, 4); break;
      default: YAMOE_RUN(0, 4); break;
    }
  } else {
    if (n_ni <= 1) { if (n_mi == 2) YAMOE_RUN(2, 1); else if (n_mi == 1) YAMOE_RUN(1, 1); else YAMOE_RUN(0, 1); }
    else { if (n_mi == 2) YAMOE_RUN(2, 2); else if (n_mi == 1) YAMOE_RUN(1, 2); else YAMOE_RUN(0, 2); }
  }
#undef YAMOE_RUN
#undef YAMOE_RUN6
}

#ifdef YAMOE_TILE_STAMPS
static unsigned long long *g_tile_stamps = nullptr;
static int g_tile_stamps_cap = 0;
#endif

template <typename T, class S, int EPI, bool GATHER, bool BNK, bool RAGGED, int FORM>
static int launch(const Args &args, int max_row_tiles, hipStream_t stream) {
  auto kernel = gemm_async_kernel<T, S, EPI, GATHER, BNK, RAGGED, FORM>;
  constexpr int lds_bytes = BNK ? S::kLdsNk : S::kLds;
  static DeviceFlags attr_done;  // one per kernel instantiation
  if (int rc = ensure_dynamic_lds((const void *)kernel, lds_bytes, attr_done, "gemm_async_kernel")) return rc;
  long long total = (long long)max_row_tiles * args.n_col_tiles;
  if (total <= 0) return 0;
  total = (total + kXcds - 1) / kXcds * kXcds * S::kParts + args.stream_wgs * kXcds;
#ifdef YAMOE_TILE_STAMPS
  Args stamped = args;
  stamped.stamps = g_tile_stamps;
  stamped.stamps_cap = g_tile_stamps_cap;
  hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(kThreads), lds_bytes, stream, stamped);
#else
  hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(kThreads), lds_bytes, stream, args);
#endif
  return check_launch("gemm_async_kernel");
}

}  // namespace async

}  // namespace yamoe
