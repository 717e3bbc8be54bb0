// Grouped weight gradients for 16-bit data on gfx950, on the asynchronous-copy pipeline of gemm_async_tile.h.
#include "gemm_async_tile.h"

namespace yamoe {

namespace async {

constexpr int kBN = 256;

// ---- weight gradients: dW[e] = L[rows of e]^T * R[rows of e] -----------------------------------------------
// (csrc/experts_backward.cu:198, 311).  The contraction runs over the expert's kept rows, so both operands are
// [k][m] / [k][n] in memory: both stay that way in LDS (single-slab buffers of 32 k-rows) and both are read with
// the LDS transpose read.  The last slab of an expert is usually partial: the copies of its missing rows read
// whatever follows in memory (the caller keeps that readable) and the wave that issued them overwrites them with
// zeros in LDS before anybody reads the slab.
struct WgradArgs {
  const void *A;  // [N, Md] rows in expert order; with a_rows: [*, Md], sorted row p is row a_rows[p] / a_div of it
  const void *B;  // [N, Nd]
  void *C;        // [E, Md, Nd]
  const int *counts, *offsets;
  const int *a_rows;
  FastDiv a_div;
  FastDiv band_div;  // division by kWgradBand * n_n_tiles
  int a_rows_max;  // largest value a_rows may hold
  int capacity, E, Md, Nd, n_m_tiles, n_n_tiles;
  // optional: [E, Nd] column sums of the expert's rows of B (the bias gradient that goes with this weight gradient,
  // csrc/experts_backward.cu:277, 308)
  void *bias_grad;
};

template <bool P1_, bool P2_, bool NEXT_, bool ZERO_, int VM_> struct WStepCfg {
  static constexpr bool P1 = P1_, P2 = P2_, NEXT = NEXT_, ZERO = ZERO_;
  static constexpr int VM = VM_;
};

// 128 x 256 tiles with a three-slab ring (72 KB of LDS, at most 256 registers per lane), so that two workgroups
// share a CU: an expert's contraction is short (its kept rows), a tile spends a third of its time filling the ring
// and storing its result, and with a second workgroup on the same SIMDs the matrix pipe works through that.
constexpr int kSmallBM = 128, kSmallStages = 3;
constexpr int kSmallAStage = kBK * kSmallBM * 2, kSmallBStage = kBK * kBN * 2;  // 8 KB + 16 KB per slab
// From four slabs on (97 rows) a tile goes through the pipelined loop, which starts once one slab is there; shorter ones
// wait for everything they contract.  (With the line at six slabs, forward + backward of 32 experts of 128 rows, 2048 x 2048,
// took 882 us against 848; of 125 rows, 2880 x 2880, 1383 against 1334.)
constexpr int kSmallPipelined = kSmallStages + 1;
constexpr int kSmallBRing = kSmallStages * kSmallAStage;
constexpr int kSmallRing = kSmallStages * (kSmallAStage + kSmallBStage);
constexpr int kSmallStaging = kSmallBM * (kBN * 2 + 16);
constexpr int kSmallLds = kSmallRing > kSmallStaging ? kSmallRing : kSmallStaging;

// Adds up the eight values of a fragment of the right operand (a lane holds one column): what the bias gradient is made of.
template <typename T> __device__ inline float add_fragment(const u32x4 &f, float sum) {
  typedef T T8 __attribute__((ext_vector_type(8)));
  const T8 v = __builtin_bit_cast(T8, f);
#pragma unroll
  for (int i = 0; i < 8; ++i) sum += ElemTraits<T>::to_f32(v[i]);
  return sum;
}
// The lane's sum over its half of the contraction and the other half's: one column of the bias gradient.
template <typename T> __device__ inline void store_column_sum(const WgradArgs &args, int expert, int col, float sum, int g) {
  sum += __shfl_xor(sum, 32);
  if (g == 0 && col < args.Nd) ((T *)args.bias_grad)[(long long)expert * args.Nd + col] = ElemTraits<T>::from_f32(sum);
}

// The staged tile (rows of `stride` bytes in LDS) goes out row by row, 16 bytes a lane.  STREAMING: 1.6 GB of gradients per
// backward pass that nobody reads back soon would otherwise push the operand tiles out of L2.
template <typename T, int BN>
__device__ inline void store_tile(const WgradArgs &args, const char *lds, int stride, int tid, int expert, int m0, int n0, int rows_m,
                                  bool streaming) {
  constexpr int chunks = BN >> 3, rows_per_pass = kThreads / chunks;
  const int c = tid % chunks;
  if (n0 + c * 8 >= args.Nd) return;
  T *p = (T *)args.C + ((long long)expert * args.Md + m0) * args.Nd + n0 + c * 8;
  if (streaming) {
    for (int r = tid / chunks; r < rows_m; r += rows_per_pass)
      __builtin_nontemporal_store(*(const u32x4 *)(lds + r * stride + c * 16), (u32x4 *)(p + (long long)r * args.Nd));
  } else {
    for (int r = tid / chunks; r < rows_m; r += rows_per_pass)
      *(u32x4 *)(p + (long long)r * args.Nd) = *(const u32x4 *)(lds + r * stride + c * 16);
  }
}

// SUMS: this wave also leaves column sums of the expert's rows of the right operand (the bias gradient that goes with the
// weight gradient), from the fragments that it multiplies, 16 vector instructions per fragment beside two MFMAs: the waves of
// an expert's first row tile, those of wave row 0 (SUMS = 1) the first two of their column blocks, those of wave row 1 (SUMS =
// 2) the other two.
template <typename T, int NMI, bool GATHER, int SUMS>
__device__ inline void run_wgrad_tile_small(const WgradArgs &args, const int tid, const int expert, const int m0,
                                            const int n0, const int rows_m, const long long first, const int rows) {
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  constexpr int NACC = NMI > 0 ? NMI : 1;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);

  f32x16 acc[NACC][4];
#pragma unroll
  for (int mi = 0; mi < NACC; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0.0f;

  const int n_slabs = (rows + kBK - 1) / kBK;
  const long long lda_bytes = (long long)args.Md * (long long)sizeof(T), ldb_bytes = (long long)args.Nd * (long long)sizeof(T);

  // A copies: piece i (0..1) = k rows 4*(2*wave + i) + (lane >> 4) of the slab, 256 bytes each; LDS position lane & 15
  // holds piece pos ^ ((k & 3) << 2).  B copies: piece i (0..3) = k rows 8*wave + 2*i + (lane >> 5).
  uint32_t a_off[2], b_off[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int k = 4 * (2 * wave + i) + (lane >> 4);
    int piece = (lane & 15) ^ ((k & 3) << 2);
    int ca = m0 + piece * 8;
    if (ca >= args.Md) ca = m0;
    a_off[i] = (uint32_t)((GATHER ? 0ll : k * lda_bytes) + (long long)(ca - m0) * (long long)sizeof(T));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int k = 8 * wave + 2 * i + (lane >> 5);
    int piece = (lane & 31) ^ ((k & 3) << 2);
    int cb = n0 + piece * 8;
    if (cb >= args.Nd) cb = n0;
    b_off[i] = (uint32_t)(k * ldb_bytes + (long long)(cb - n0) * (long long)sizeof(T));
  }
  const char *a_base = (const char *)((const T *)args.A + (GATHER ? 0ll : first * args.Md) + m0);
  const char *b_base = (const char *)((const T *)args.B + first * args.Nd + n0);
  // Gathered A rows: the four k rows of piece i of a slab are rows a_rows[first + 32*slab + 4*(2*wave + i) + 0..3]
  // / a_div of A.  The positions are the same for the whole wave, so the look-ups are scalar loads (rows_of), issued
  // at the start of the half slab whose last slot issues the copy; there the lane picks its row and turns it into a
  // byte offset (row_bytes).  Positions past the expert's rows (up to 31 past the end of the list: the caller keeps
  // that readable) hold somebody else's row or anything at all: the value is clamped to the list's range, and what the
  // copy fetches is zeroed in LDS before use.  The list is read through the constant address space, which makes the loads scalar whatever the
  // compiler can prove about the memory in between (the list was written by an earlier launch).
  typedef const __attribute__((address_space(4))) int *ConstInts;
  ConstInts a_rows = GATHER ? (ConstInts)(uintptr_t)(args.a_rows + first) : (ConstInts)0;
  auto rows_of = [&](int slab, int i, int (&ix)[4]) {
    if constexpr (GATHER) {
      const int k0 = slab * kBK + 4 * (2 * wave + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) ix[j] = a_rows[k0 + j];
    }
  };
  auto row_bytes = [&](int (&ix)[4]) -> uint32_t {
    if constexpr (!GATHER) return 0u;
    // the four values pass through an empty statement: the loads stay where rows_of put them, all four of them, and
    // what follows is three selects rather than loads under branches
    int r0 = ix[0], r1 = ix[1], r2 = ix[2], r3 = ix[3];
    asm volatile("" : "+s"(r0), "+s"(r1), "+s"(r2), "+s"(r3));
    const bool odd = (lane & 16) != 0, high = (lane & 32) != 0;
    const int lo = odd ? r1 : r0, hi = odd ? r3 : r2;
    const uint32_t r = min((uint32_t)(high ? hi : lo), (uint32_t)args.a_rows_max);
    return (uint32_t)fast_div((int)r, args.a_div) * (uint32_t)lda_bytes;
  };
  auto copy_a = [&](int slab, int i, uint32_t row) {
    copy16_to_lds(a_base + (GATHER ? 0ll : (long long)slab * kBK * lda_bytes), a_off[i] + row,
                  lds0 + (uint32_t)(slab % kSmallStages) * kSmallAStage + (uint32_t)(4 * (2 * wave + i)) * 256u);
  };
  auto copy_a_now = [&](int slab, int i) {  // look-up and copy in one go: outside the pipelined loop
    int ix[4] = {0, 0, 0, 0};
    rows_of(slab, i, ix);
    copy_a(slab, i, row_bytes(ix));
  };
  auto copy_b = [&](int slab, int i) {
    copy16_to_lds(b_base + (long long)slab * kBK * ldb_bytes, b_off[i],
                  lds0 + kSmallBRing + (uint32_t)(slab % kSmallStages) * kSmallBStage + (uint32_t)(8 * wave + 2 * i) * 512u);
  };
  auto copy_slab = [&](int slab) {
    copy_a_now(slab, 0); copy_b(slab, 0); copy_b(slab, 1); copy_a_now(slab, 1); copy_b(slab, 2); copy_b(slab, 3);
  };
  auto zero_tail = [&](int slab) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      int k = 4 * (2 * wave + i) + (lane >> 4);
      if (slab * kBK + k >= rows)
        *(u32x4 *)(lds + (slab % kSmallStages) * kSmallAStage + 4 * (2 * wave + i) * 256 + lane * 16) = (u32x4){0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int k = 8 * wave + 2 * i + (lane >> 5);
      if (slab * kBK + k >= rows)
        *(u32x4 *)(lds + kSmallBRing + (slab % kSmallStages) * kSmallBStage + (8 * wave + 2 * i) * 512 + lane * 16) = (u32x4){0, 0, 0, 0};
    }
  };

  const int g = lane >> 5, rl = lane & 31, j4 = (lane & 15) >> 2, q4 = lane & 3;
  int a_rd[NACC], b_rd[4];
#pragma unroll
  for (int mi = 0; mi < NACC; ++mi) {
    int col = (mi * 2 + wm) * 32 + 16 * ((lane >> 4) & 1) + 4 * q4;
    a_rd[mi] = (g * 8 + j4) * 256 + ((((col >> 3) ^ (j4 << 2))) << 4) + (col & 7) * 2;
  }
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) {
    int col = wn * 128 + ni * 32 + 16 * ((lane >> 4) & 1) + 4 * q4;
    b_rd[ni] = (g * 8 + j4) * 512 + ((((col >> 3) ^ (j4 << 2))) << 4) + (col & 7) * 2;
  }
  u32x4 fa0[NACC], fa1[NACC], fb0[4], fb1[4];
  float colsum[2] = {0.0f, 0.0f};
  constexpr int kSumFrom = SUMS == 2 ? 2 : 0;
  constexpr int kFrags = NMI > 0 ? 4 + NMI : 0;
  // fragment order B0, A0, B1, B2, B3, A1
  auto read_frag = [&](int s, int ks, int f, u32x4 (&fa)[NACC], u32x4 (&fb)[4]) {
    const bool is_a = f == 1 || f >= 5;
    const int idx = is_a ? (f == 1 ? 0 : f - 4) : (f == 0 ? 0 : f - 1);
    const char *sp = is_a ? lds + (s % kSmallStages) * kSmallAStage + a_rd[idx] + ks * 4096
                          : lds + kSmallBRing + (s % kSmallStages) * kSmallBStage + b_rd[idx] + ks * 8192;
    u32x2 lo = lds_read_tr16(sp);
    u32x2 hi = lds_read_tr16(sp + (is_a ? 1024 : 2048));
    u32x4 v = (u32x4){lo[0], lo[1], hi[0], hi[1]};
    if (is_a) fa[idx] = v; else fb[idx] = v;
  };
  auto read_frags = [&](int s, int ks, u32x4 (&fa)[NACC], u32x4 (&fb)[4]) {
#pragma unroll
    for (int f = 0; f < kFrags; ++f) read_frag(s, ks, f, fa, fb);
  };

  // pipeline: slab t+3 goes into the buffer slab t leaves at its mid-slab barrier: first half of its copies
  // (A piece 0, B pieces 0-1) in the second k-step of slab t, second half in the first k-step of slab t+1; "slab
  // s+1 has landed" = at most 6 younger copies in flight
  constexpr int kMma = 4 * NMI;
  constexpr int kSlots = kMma > 2 ? kMma - 2 : 1;
  if (n_slabs > 0) {
#pragma unroll
    for (int s = 0; s < kSmallStages; ++s)
      if (s < n_slabs) copy_slab(s);
    if (n_slabs >= kSmallPipelined) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");  // slab 0 is enough to start with
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int s = 0; s < kSmallStages; ++s)
      if (n_slabs < kSmallPipelined && s < n_slabs && (s + 1) * kBK > rows) zero_tail(s);
    __syncthreads();
    read_frags(0, 0, fa0, fb0);
  }
  // In the pipelined loop the ring stage of every slab is a compile-time constant (the loop is unrolled by the ring
  // depth), so that an operand read is one ds_read with an immediate offset from a per-lane base and a copy's LDS
  // address one scalar add: with the stage computed per slab (a division by 3, then one vector add per read) the
  // loop carried 3.4 vector instructions per MFMA, 30 of them in a block ahead of each slab's first MFMA.
  const char *pa[NACC], *pb[4];
#pragma unroll
  for (int mi = 0; mi < NACC; ++mi) pa[mi] = lds + a_rd[mi];
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) pb[ni] = lds + kSmallBRing + b_rd[ni];
  const uint32_t lds_a_wave = lds0 + (uint32_t)(8 * wave) * 256u, lds_b_wave = lds0 + kSmallBRing + (uint32_t)(8 * wave) * 512u;
  auto read_frag_c = [&](auto stage, int ks, int f, u32x4 (&fa)[NACC], u32x4 (&fb)[4]) {
    constexpr int ST = decltype(stage)::value;
    const bool is_a = f == 1 || f >= 5;
    const int idx = is_a ? (f == 1 ? 0 : f - 4) : (f == 0 ? 0 : f - 1);
    const char *sp = is_a ? pa[idx] + ST * kSmallAStage + ks * 4096 : pb[idx] + ST * kSmallBStage + ks * 8192;
    u32x2 lo = lds_read_tr16(sp);
    u32x2 hi = lds_read_tr16(sp + (is_a ? 1024 : 2048));
    u32x4 v = (u32x4){lo[0], lo[1], hi[0], hi[1]};
    if (is_a) fa[idx] = v; else fb[idx] = v;
  };
  auto copy_a_c = [&](auto stage, int slab, int i, uint32_t row) {
    constexpr int ST = decltype(stage)::value;
    copy16_to_lds(a_base + (GATHER ? 0ll : (long long)slab * kBK * lda_bytes), a_off[i] + row,
                  lds_a_wave + (uint32_t)(ST * kSmallAStage + 4 * i * 256));
  };

  auto copy_b_c = [&](auto stage, int slab, int i) {
    constexpr int ST = decltype(stage)::value;
    copy16_to_lds(b_base + (long long)slab * kBK * ldb_bytes, b_off[i], lds_b_wave + (uint32_t)(ST * kSmallBStage + 2 * i * 512));
  };
  // slab s sits in ring stage ST
  auto slab_step = [&](int s, auto cfg, auto stage) {
    typedef decltype(cfg) C;
    constexpr int ST = decltype(stage)::value;
    typedef std::integral_constant<int, (ST + 1) % kSmallStages> Next;   // slab s + 1
    typedef std::integral_constant<int, (ST + 2) % kSmallStages> Next2;  // slab s + 2; slab s + 3 takes stage ST again
    __builtin_amdgcn_sched_barrier(0);
    {
      constexpr int kC = C::P1 ? 3 : 0, kItems = kC + kFrags;
      int ix[4] = {0, 0, 0, 0};  // gathered rows: the four rows of the A piece copied in this half slab
#pragma unroll
      for (int j = 0; j < (kMma > 0 ? kMma : 1); ++j) {
        if (j < kMma) Mma<T>::run(fb0[j & 3], fa0[j >> 2], acc[j >> 2][j & 3]);
        if (SUMS && (j & ~1) == kSumFrom) colsum[j & 1] = add_fragment<T>(fb0[j & 3], colsum[j & 1]);
        if (j < kSlots) {
#pragma unroll
          for (int i = j * kItems / kSlots; i < (j + 1) * kItems / kSlots; ++i) {
            if (i < kC) {
              if (i == 0) { if constexpr (GATHER) rows_of(s + 2, 1, ix); else copy_a_c(Next2(), s + 2, 1, 0u); }
              else copy_b_c(Next2(), s + 2, 1 + i);
            }
            else read_frag_c(stage, 1, i - kC, fa1, fb1);
          }
          if (GATHER && kC > 0 && j == kSlots - 1) copy_a_c(Next2(), s + 2, 1, row_bytes(ix));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (C::VM == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    else if constexpr (C::VM == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (C::ZERO) zero_tail(s + 1);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    {
      constexpr int kC = C::P2 ? 3 : 0, kItems = kC + (C::NEXT ? kFrags : 0);
      int ix[4] = {0, 0, 0, 0};  // gathered rows: the four rows of the A piece copied in this half slab
#pragma unroll
      for (int j = 0; j < (kMma > 0 ? kMma : 1); ++j) {
        if (j < kMma) Mma<T>::run(fb1[j & 3], fa1[j >> 2], acc[j >> 2][j & 3]);
        if (SUMS && (j & ~1) == kSumFrom) colsum[j & 1] = add_fragment<T>(fb1[j & 3], colsum[j & 1]);
        if (j < kSlots) {
#pragma unroll
          for (int i = j * kItems / kSlots; i < (j + 1) * kItems / kSlots; ++i) {
            if (i < kC) {
              if (i == 0) { if constexpr (GATHER) rows_of(s + 3, 0, ix); else copy_a_c(stage, s + 3, 0, 0u); }
              else copy_b_c(stage, s + 3, i - 1);
            }
            else read_frag_c(Next(), 0, i - kC, fa0, fb0);
          }
          if (GATHER && kC > 0 && j == kSlots - 1) copy_a_c(stage, s + 3, 0, row_bytes(ix));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // the same step with the ring stage taken from the slab number at run time: for the slabs the unrolled loop leaves
  // over and for the last three (the stage they start in depends on the slab count)
  auto slab_step_rt = [&](int s, auto cfg) {
    typedef decltype(cfg) C;
    __builtin_amdgcn_sched_barrier(0);
    {
      constexpr int kC = C::P1 ? 3 : 0, kItems = kC + kFrags;
      int ix[4] = {0, 0, 0, 0};  // gathered rows: the four rows of the A piece copied in this half slab
#pragma unroll
      for (int j = 0; j < (kMma > 0 ? kMma : 1); ++j) {
        if (j < kMma) Mma<T>::run(fb0[j & 3], fa0[j >> 2], acc[j >> 2][j & 3]);
        if (SUMS && (j & ~1) == kSumFrom) colsum[j & 1] = add_fragment<T>(fb0[j & 3], colsum[j & 1]);
        if (j < kSlots) {
#pragma unroll
          for (int i = j * kItems / kSlots; i < (j + 1) * kItems / kSlots; ++i) {
            if (i < kC) {
              if (i == 0) { if constexpr (GATHER) rows_of(s + 2, 1, ix); else copy_a(s + 2, 1, 0u); }
              else copy_b(s + 2, 1 + i);
            }
            else read_frag(s, 1, i - kC, fa1, fb1);
          }
          if (GATHER && kC > 0 && j == kSlots - 1) copy_a(s + 2, 1, row_bytes(ix));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (C::VM == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    else if constexpr (C::VM == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (C::ZERO) zero_tail(s + 1);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    {
      constexpr int kC = C::P2 ? 3 : 0, kItems = kC + (C::NEXT ? kFrags : 0);
      int ix[4] = {0, 0, 0, 0};  // gathered rows: the four rows of the A piece copied in this half slab
#pragma unroll
      for (int j = 0; j < (kMma > 0 ? kMma : 1); ++j) {
        if (j < kMma) Mma<T>::run(fb1[j & 3], fa1[j >> 2], acc[j >> 2][j & 3]);
        if (SUMS && (j & ~1) == kSumFrom) colsum[j & 1] = add_fragment<T>(fb1[j & 3], colsum[j & 1]);
        if (j < kSlots) {
#pragma unroll
          for (int i = j * kItems / kSlots; i < (j + 1) * kItems / kSlots; ++i) {
            if (i < kC) {
              if (i == 0) { if constexpr (GATHER) rows_of(s + 3, 0, ix); else copy_a(s + 3, 0, 0u); }
              else copy_b(s + 3, i - 1);
            }
            else read_frag(s + 1, 0, i - kC, fa0, fb0);
          }
          if (GATHER && kC > 0 && j == kSlots - 1) copy_a(s + 3, 0, row_bytes(ix));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  if (n_slabs >= kSmallPipelined) {
    typedef std::integral_constant<int, 0> S0;
    typedef std::integral_constant<int, 1> S1;
    typedef std::integral_constant<int, 2> S2;
    typedef WStepCfg<true, true, true, false, 6> Steady;
    slab_step(0, WStepCfg<false, true, true, false, 6>(), S0());
    int s = 1;
    for (; s + 5 < n_slabs; s += 3) {  // steady state, three slabs per round: stages 1, 2, 0
      slab_step(s, Steady(), S1());
      slab_step(s + 1, Steady(), S2());
      slab_step(s + 2, Steady(), S0());
    }
    for (; s + 3 < n_slabs; ++s) slab_step_rt(s, Steady());  // at most two
    // the last three slabs (s = n_slabs - 3): no new copies; the last slab's missing rows are zeroed
    slab_step_rt(s, WStepCfg<true, false, true, false, 6>());
    slab_step_rt(s + 1, WStepCfg<false, false, true, true, 0>());
    slab_step_rt(s + 2, WStepCfg<false, false, false, false, -1>());
  } else {
    for (int s = 0; s < n_slabs; ++s) {
      if (kFrags > 0) read_frags(s, 1, fa1, fb1);
#pragma unroll
      for (int j = 0; j < kMma; ++j) Mma<T>::run(fb0[j & 3], fa0[j >> 2], acc[j >> 2][j & 3]);
      if constexpr (SUMS != 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) colsum[i] = add_fragment<T>(fb0[kSumFrom + i], colsum[i]);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (s + 1 < n_slabs && (s + 2) * kBK > rows) zero_tail(s + 1);
      __syncthreads();
      if (s + kSmallStages < n_slabs) copy_slab(s + kSmallStages);
      if (s + 1 < n_slabs) read_frags(s + 1, 0, fa0, fb0);
#pragma unroll
      for (int j = 0; j < kMma; ++j) Mma<T>::run(fb1[j & 3], fa1[j >> 2], acc[j >> 2][j & 3]);
      if constexpr (SUMS != 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) colsum[i] = add_fragment<T>(fb1[kSumFrom + i], colsum[i]);
      }
    }
  }

  if constexpr (SUMS != 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) store_column_sum<T>(args, expert, n0 + wn * 128 + (kSumFrom + i) * 32 + rl, colsum[i], g);
  }
  // epilogue: stage the tile in LDS, store whole row segments
  constexpr int stride = kBN * 2 + 16;
  // (operands exchanged in the MFMAs, as in the forward kernel) acc[mi][ni][v]: tile row (mi*2+wm)*32 + lane%32,
  // tile column wn*128 + ni*32 + 8*(v/4) + 4*(lane/32) + v%4
  __syncthreads();
  {
    char *lp = lds + (wm * 32 + rl) * stride + (wn * 128 + 4 * g) * 2;
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
#pragma unroll
      for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16 &a = acc[mi][ni];
          u32x2 v = {pack2<T>(a[4 * q], a[4 * q + 1]), pack2<T>(a[4 * q + 2], a[4 * q + 3])};
          *(u32x2 *)(lp + mi * 64 * stride + (ni * 32 + 8 * q) * 2) = v;
        }
  }
  __syncthreads();
  store_tile<T, kBN>(args, lds, stride, tid, expert, m0, n0, rows_m, true);
}

// An expert's output tiles are taken in bands of this many row tiles, each band column by column.  An XCD has 64 tiles in
// flight, and they write their gradients as they finish: in a band those are 4 row tiles of 16 neighbouring columns, whole
// 8 KB stretches of a gradient's rows, and 4 + 16 operand tiles shared in the L2.  Column by column over the whole expert
// they were 16 to 23 row tiles of 3 or 4 columns, and the writes (1.1 GB a step) went out as 2 KB pieces one row apart.
// Forward + backward, whole columns / bands of 2 / 3 / 4 / 6 / rows of all columns, us: 1536 x 8 tokens on 64 experts,
// 2048 x 2048: 2022 / 1940 / 1937 / 1953 / 1948 / 1941; 1000 x 4 on 32, 2880 x 2880: 1452 / 1389 / 1388 / 1383 / 1386 / 1400;
// 4096 x 4 on 32, 2880 x 2880: 3319 / 3294 / 3303 / 3286 / 3281 / 3307.  Experts with few row tiles (1024 x 1024) don't care.
constexpr int kWgradBand = 4;

template <typename T, bool GATHER>
__global__ __launch_bounds__(kThreads, 2) void wgrad_small_kernel(const WgradArgs args) {
  const int tid = threadIdx.x, wave = tid >> 6, wm = wave >> 1;
  const int per_expert = args.n_m_tiles * args.n_n_tiles;
  const int total = args.E * per_expert;
  const int total8 = (total + kXcds - 1) / kXcds * kXcds;
  const int b = blockIdx.x;
  if (b >= total8) return;
  const int L = (b % kXcds) * (total8 / kXcds) + b / kXcds;
  if (L >= total) return;
  const int expert = L / per_expert, r = L - expert * per_expert;
  const int band = fast_div(r, args.band_div), in_band = r - band * kWgradBand * args.n_n_tiles;
  const int band_rows = min(kWgradBand, args.n_m_tiles - band * kWgradBand);
  const int col_tile = in_band / band_rows;
  const int n0 = col_tile * kBN, m0 = (band * kWgradBand + in_band - col_tile * band_rows) * kSmallBM;
  const int rows_m = min(kSmallBM, args.Md - m0);
  // (the same for every lane; said explicitly, so that the operand addresses built from them stay in scalar registers)
  int rows = min(__builtin_amdgcn_readfirstlane(args.counts[expert]), args.capacity);
  if (rows < 0) rows = 0;
  const long long first = __builtin_amdgcn_readfirstlane(args.offsets[expert]);
  const int n_blocks32 = (rows_m + 31) >> 5;
  const int n_mi = (n_blocks32 - wm + 1) >> 1;
#define YAMOE_WGRAD(NMI_, SUMS_) run_wgrad_tile_small<T, NMI_, GATHER, SUMS_>(args, tid, expert, m0, n0, rows_m, first, rows)
  if (args.bias_grad != nullptr && m0 == 0) {  // (a wave row without rows of the gradient multiplies a block all the same)
    if (wm == 0) { if (n_mi == 2) YAMOE_WGRAD(2, 1); else YAMOE_WGRAD(1, 1); }
    else { if (n_mi == 2) YAMOE_WGRAD(2, 2); else YAMOE_WGRAD(1, 2); }
    return;
  }
  if (n_mi == 2) YAMOE_WGRAD(2, 0);
  else if (n_mi == 1) YAMOE_WGRAD(1, 0);
  else YAMOE_WGRAD(0, 0);
#undef YAMOE_WGRAD
}

// ---- short contractions ------------------------------------------------------------------------------------------
// Up to kShortRows rows per expert a launch is bound by the store of the gradient (5.5 TB/s reached) and by what
// stands between two stores of a CU: a tile's start, its first slab's trip from memory and the staging, which a contraction of
// one to three slabs does not cover.  So four small workgroups share a CU instead of two: 128 x 128 tiles, 64 accumulators and at
// most 128 registers per lane, 35 KB of LDS (a ring of two slabs, into which the tile is staged afterwards), no hand-made order:
// the other three waves of a SIMD work while one waits.  Both weight gradients of a step, large tiles / these, us: 64 experts,
// 2048 x 2048, 16 rows 294 / 273, 32: 332 / 293, 64: 418 / 360, 80: 479 / 390, 112: 478 / 458, 128: 508 / 503, 192: 585 / 602; 32 of
// 2880 x 2880, 64 rows 379 / 325, 112: 461 / 445, 128: 494 / 481, 192: 573 / 583; 16 of 2048, 64 rows 112 / 91, 112: 117 / 109, 128:
// 118 / 122.  Beyond, the small tiles' operand traffic decides: a slab costs 29 us instead of 24 (64 experts, 2048 x 2048), 23 of
// them for its copies from L2, 33 % more bytes.
// Those are evenly routed experts.  A skewed routing has most of its rows in a few experts with far more, so the average alone is
// a sound line only up to kShortRowsAnyRouting; beyond, the capacity has to keep every expert at kShortMostRows or below.  Whole
// forwards and backwards under Zipf (1.2) routing without a capacity, large tiles / these, 64 experts of 2048 x 2048, 24 rows on
// average: 1043 / 1030, 40: 1185 / 1193, 72: 1477 / 1569, 112: 1824 / 1933; 32 of 2880 x 2880, 24 rows 1057 / 1021, 40: 1192 / 1204,
// 72: 1403 / 1486; with 1.25 times the average as the capacity, 64 of 2048 x 2048, 72 rows 1081 / 1018, 104: 1225 / 1175, 32 of
// 2880 x 2880 1100 / 1019 and 1179 / 1152.  (Both kernels in turn, each for the experts that suit it, lose to either one: a second
// launch's tail; 72 rows, Zipf, 1663 and 1592 us.)
constexpr int kShortRows = 112, kShortRowsAnyRouting = 32, kShortMostRows = 128;
constexpr int kShortBM = 128, kShortBN = 128, kShortStages = 2;
constexpr int kShortOperand = kBK * kShortBM * 2;      // 8 KB: 32 k rows of 256 bytes
constexpr int kShortStage = 2 * kShortOperand;
constexpr int kShortStride = kShortBN * 2 + 16;        // bytes of a row of the staged tile
constexpr int kShortLds = kShortBM * kShortStride > kShortStages * kShortStage ? kShortBM * kShortStride : kShortStages * kShortStage;

template <typename T, bool GATHER>
__global__ __launch_bounds__(kThreads, 4) void wgrad_short_kernel(const WgradArgs args) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int per_expert = args.n_m_tiles * args.n_n_tiles;
  const int total = args.E * per_expert;
  const int total8 = (total + kXcds - 1) / kXcds * kXcds;
  const int b = blockIdx.x;
  const int L = (b % kXcds) * (total8 / kXcds) + b / kXcds;
  if (L >= total) return;
  const int expert = L / per_expert, r = L - expert * per_expert;
  const int band = fast_div(r, args.band_div), in_band = r - band * kWgradBand * args.n_n_tiles;
  const int band_rows = min(kWgradBand, args.n_m_tiles - band * kWgradBand);
  const int col_tile = in_band / band_rows;
  const int n0 = col_tile * kShortBN, m0 = (band * kWgradBand + in_band - col_tile * band_rows) * kShortBM;
  const int rows_m = min(kShortBM, args.Md - m0);
  int rows = min(__builtin_amdgcn_readfirstlane(args.counts[expert]), args.capacity);
  if (rows < 0) rows = 0;
  const long long first = __builtin_amdgcn_readfirstlane(args.offsets[expert]);
  const bool sums = args.bias_grad != nullptr && m0 == 0 && wm == 0;

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
  const int n_slabs = (rows + kBK - 1) / kBK;
  const long long lda_bytes = (long long)args.Md * (long long)sizeof(T), ldb_bytes = (long long)args.Nd * (long long)sizeof(T);

  // copy i (0..1) of either operand: k rows 4*(2*wave + i) + (lane >> 4) of the slab, 256 bytes each; LDS position lane & 15
  // holds piece pos ^ ((k & 3) << 2)
  uint32_t a_off[2], b_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = 4 * (2 * wave + i) + (lane >> 4);
    const int piece = (lane & 15) ^ ((k & 3) << 2);
    const int ca = m0 + piece * 8 < args.Md ? piece * 8 : 0, cb = n0 + piece * 8 < args.Nd ? piece * 8 : 0;
    a_off[i] = (uint32_t)((GATHER ? 0ll : k * lda_bytes) + (long long)ca * (long long)sizeof(T));
    b_off[i] = (uint32_t)(k * ldb_bytes + (long long)cb * (long long)sizeof(T));
  }
  const char *a_base = (const char *)((const T *)args.A + (GATHER ? 0ll : first * args.Md) + m0);
  const char *b_base = (const char *)((const T *)args.B + first * args.Nd + n0);
  typedef const __attribute__((address_space(4))) int *ConstInts;
  ConstInts a_rows = GATHER ? (ConstInts)(uintptr_t)(args.a_rows + first) : (ConstInts)0;
  int ix[2][4];
  auto rows_of = [&](int slab) {
    if constexpr (GATHER) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) ix[i][j] = a_rows[slab * kBK + 4 * (2 * wave + i) + j];
    }
  };
  auto row_bytes = [&](int i) -> uint32_t {
    if constexpr (!GATHER) return 0u;
    int r0 = ix[i][0], r1 = ix[i][1], r2 = ix[i][2], r3 = ix[i][3];
    asm volatile("" : "+s"(r0), "+s"(r1), "+s"(r2), "+s"(r3));
    const bool odd = (lane & 16) != 0, high = (lane & 32) != 0;
    const int lo = odd ? r1 : r0, hi = odd ? r3 : r2;
    const uint32_t rr = min((uint32_t)(high ? hi : lo), (uint32_t)args.a_rows_max);
    return (uint32_t)fast_div((int)rr, args.a_div) * (uint32_t)lda_bytes;
  };
  auto copy_slab = [&](int slab) {
    const uint32_t st = lds0 + (uint32_t)(slab & 1) * kShortStage + (uint32_t)(8 * wave) * 256u;
    const char *ab = a_base + (GATHER ? 0ll : (long long)slab * kBK * lda_bytes), *bb = b_base + (long long)slab * kBK * ldb_bytes;
#pragma unroll
    for (int i = 0; i < 2; ++i) copy16_to_lds(bb, b_off[i], st + kShortOperand + (uint32_t)(4 * i) * 256u);
#pragma unroll
    for (int i = 0; i < 2; ++i) copy16_to_lds(ab, a_off[i] + row_bytes(i), st + (uint32_t)(4 * i) * 256u);
  };
  auto zero_tail = [&](int slab) {
    char *st = lds + (slab & 1) * kShortStage + 8 * wave * 256 + lane * 16;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (slab * kBK + 4 * (2 * wave + i) + (lane >> 4) >= rows) {
        *(u32x4 *)(st + 4 * i * 256) = (u32x4){0, 0, 0, 0};
        *(u32x4 *)(st + kShortOperand + 4 * i * 256) = (u32x4){0, 0, 0, 0};
      }
  };

  const int g = lane >> 5, rl = lane & 31, j4 = (lane & 15) >> 2, q4 = lane & 3;
  int a_rd[2], b_rd[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int ca = (x * 2 + wm) * 32 + 16 * ((lane >> 4) & 1) + 4 * q4, cb = wn * 64 + x * 32 + 16 * ((lane >> 4) & 1) + 4 * q4;
    a_rd[x] = (g * 8 + j4) * 256 + (((ca >> 3) ^ (j4 << 2)) << 4) + (ca & 7) * 2;
    b_rd[x] = kShortOperand + (g * 8 + j4) * 256 + (((cb >> 3) ^ (j4 << 2)) << 4) + (cb & 7) * 2;
  }
  f32x16 acc[2][2];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0.0f;
  float colsum[2] = {0.0f, 0.0f};

  if (n_slabs > 0) {
    rows_of(0);
    copy_slab(0);
    if (n_slabs > 1) {
      rows_of(1);
      copy_slab(1);
      if (n_slabs > 2) rows_of(2);
    }
  }
  for (int s = 0; s < n_slabs; ++s) {
    if (s + 1 < n_slabs) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if ((s + 1) * kBK > rows) zero_tail(s);
    __syncthreads();
    const char *st = lds + (s & 1) * kShortStage;
    u32x4 fa[2][2], fb[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        u32x2 lo = lds_read_tr16(st + b_rd[x] + ks * 4096), hi = lds_read_tr16(st + b_rd[x] + ks * 4096 + 1024);
        fb[ks][x] = (u32x4){lo[0], lo[1], hi[0], hi[1]};
        lo = lds_read_tr16(st + a_rd[x] + ks * 4096), hi = lds_read_tr16(st + a_rd[x] + ks * 4096 + 1024);
        fa[ks][x] = (u32x4){lo[0], lo[1], hi[0], hi[1]};
      }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) Mma<T>::run(fb[ks][ni], fa[ks][mi], acc[mi][ni]);
    if (sums) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int x = 0; x < 2; ++x) colsum[x] = add_fragment<T>(fb[ks][x], colsum[x]);
    }
    __syncthreads();
    if (s + 2 < n_slabs) {
      copy_slab(s + 2);
      if (s + 3 < n_slabs) rows_of(s + 3);
    }
  }
  if (sums) {
#pragma unroll
    for (int x = 0; x < 2; ++x) store_column_sum<T>(args, expert, n0 + wn * 64 + x * 32 + rl, colsum[x], g);
  }
  // (after the last barrier nobody reads the ring)
  {
    char *lp = lds + (wm * 32 + rl) * kShortStride + (wn * 64 + 4 * g) * 2;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16 &a = acc[mi][ni];
          u32x2 v = {pack2<T>(a[4 * q], a[4 * q + 1]), pack2<T>(a[4 * q + 2], a[4 * q + 3])};
          *(u32x2 *)(lp + mi * 64 * kShortStride + (ni * 32 + 8 * q) * 2) = v;
        }
  }
  __syncthreads();
  // Where a gradient's rows are not whole cache lines, two tiles write a line, and a streaming store does not leave it in L2 for
  // the second: 32 experts, 2880 x 2000, 16 rows: 119 us and 65 with plain stores (32 rows 117 / 70, 64: 121 / 87, 128: 130 / 113).
  store_tile<T, kShortBN>(args, lds, kShortStride, tid, expert, m0, n0, rows_m, (args.Nd * (int)sizeof(T)) % 128 == 0);
}

}  // namespace async

// dW[E, Md, Nd] = per expert L^T R over its kept rows.  Both operand buffers must stay readable for 32 rows past
// their last row (the copies of a partial last slab run over; what they fetch is zeroed before use).
bool wgrad_async_supported(int Md, int Nd) { return Md % 8 == 0 && Nd % 8 == 0; }

namespace async {
template <typename T, bool GATHER> static int launch_wgrad(const WgradArgs &args, bool is_short, hipStream_t stream) {
  WgradArgs a = args;
  a.n_m_tiles = ceil_div(a.Md, kSmallBM);
  a.n_n_tiles = ceil_div(a.Nd, is_short ? kShortBN : kBN);
  a.band_div = make_fast_div(kWgradBand * a.n_n_tiles);
  long long total = (long long)a.E * a.n_m_tiles * a.n_n_tiles;
  if (total <= 0) return 0;
  total = (total + kXcds - 1) / kXcds * kXcds;
  if (is_short) {
    hipLaunchKernelGGL((wgrad_short_kernel<T, GATHER>), dim3((unsigned)total), dim3(kThreads), kShortLds, stream, a);
    return check_launch("wgrad_short_kernel");
  }
  auto kernel = wgrad_small_kernel<T, GATHER>;
  static DeviceFlags attr_done;  // one per kernel instantiation
  if (int rc = ensure_dynamic_lds((const void *)kernel, kSmallLds, attr_done, "wgrad_small_kernel")) return rc;
  hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(kThreads), kSmallLds, stream, a);
  return check_launch("wgrad_small_kernel");
}
}  // namespace async

// n_rows: the rows of all experts.  With l_rows the left operand is not in expert order: sorted row p is row l_rows[p] / l_div
// of L (rows of a [n_rows / l_div, Md] tensor gathered by token, which must span less than 4 GiB); l_rows holds n_rows values
// below n_rows and must stay readable for 32 values more, and L needs no readable rows past its end.
// d_bias, optional: [E, Nd], the column sums of every expert's rows of R.
template <typename T>
int gemm_async_wgrad(const void *L, const int *l_rows, int l_div, int n_rows, const void *R, void *dW, void *d_bias,
                     const int *counts, const int *offsets, int capacity, int E, int Md, int Nd, hipStream_t stream) {
  async::WgradArgs a = {};
  a.A = L; a.B = R; a.C = dW; a.counts = counts; a.offsets = offsets; a.capacity = capacity; a.bias_grad = d_bias;
  a.a_rows = l_rows; a.a_div = make_fast_div(l_rows != nullptr ? l_div : 1); a.a_rows_max = n_rows > 0 ? n_rows - 1 : 0;
  a.E = E; a.Md = Md; a.Nd = Nd;
  const int average = min(n_rows / E, capacity), most = min(n_rows, capacity);
  const bool is_short = average <= async::kShortRowsAnyRouting || (average <= async::kShortRows && most <= async::kShortMostRows);
  if (l_rows != nullptr) return async::launch_wgrad<T, true>(a, is_short, stream);
  return async::launch_wgrad<T, false>(a, is_short, stream);
}

#define YAMOE_INSTANTIATE_WGRAD(T)                                                                                   \
  template int gemm_async_wgrad<T>(const void *, const int *, int, int, const void *, void *, void *, const int *,     \
                                   const int *, int, int, int, int, hipStream_t);
YAMOE_INSTANTIATE_WGRAD(bf16_t)
YAMOE_INSTANTIATE_WGRAD(f16_t)

}  // namespace yamoe
