// Grouped expert GEMMs for fp32 data on gfx950: the forward's two products, the two input gradients and the weight
// gradients (the README workload of drbh/yamoe, README.md:67-112, and training in fp32; replaces batch_mm,
// csrc/batch_mm.cu:7-31, the bias / clamped-SwiGLU chain, csrc/moe.cpp:161-187, and the products of
// csrc/experts_backward.cu:198, 279-282, 309-311).
//
// The fp32 matrix instruction (v_mfma_f32_32x32x2_f32, 64 clocks for 4096 flop) is sixteen times slower per
// contraction step than the 16-bit ones, so a tile's operands are cheap next to its arithmetic and the design goes
// the other way from the 16-bit kernels: small tiles, many of them, two workgroups per CU.
//
//  * 128 x 128 output tile, 4 wavefronts 2 x 2, each four 32 x 32 accumulator blocks (64 registers).  An expert's rows are
//    cut here into full tiles and a remainder, whatever the row tiles of the schedule are: with halves of its equal row
//    tiles (160 rows: 128 + 32) a tenth of the matrix work of the README workload went into blocks without rows.
//    The 32-row blocks of a tile alternate between the two wave rows, so that a remainder keeps both busy; of an odd number the
//    last one is shared, half of the k-steps each (the sums meet in LDS, 16 KB each way), and a tile takes as long as its blocks
//    rather than as the wave row with one more of them.  Whole forwards, us, before / so, nothing else changed: 140 x 2 tokens on 16
//    experts of 2880 x 2880 491 / 361, 300 x 2 505 / 505, 700 x 2 897 / 865, 1547 x 2 1580 / 1447; 450 x 4 on 32, 1024 wide,
//    185 / 168; 4096 x 2 on 8 of 2880 x 2880, nearly all of it whole tiles, 3288 / 3288 to 3299;
//    forward + backward of 1500 x 2 on 16, 1024 wide, 800 / 787.
//  * Operands go global -> LDS with asynchronous 16-byte copies (no staging registers), two stages of 32 KB, one
//    workgroup barrier per slab of 32 (4096 clocks of MFMA issue on each SIMD): while a workgroup waits at its barrier or
//    runs its epilogue, the other workgroup on the CU keeps the matrix pipe busy.
//  * The workgroups are resident, two per CU, and go through the tiles that have rows; the next tile is looked up and its
//    first slab requested before the epilogue of the one before.
//  README workload, gate_up and down product: 2328 + 1342 us with a workgroup per half row tile, 2100 + 1160 now, 130 and 117
//  TFLOP/s of the 154 that a register-only loop of the instruction reaches on random data; of the difference, 5 % is LDS
//  reads and barriers (a loop of these alone runs at 148), the rest the turn from tile to tile (20 us for the two tiles of a
//  CU, most of it the stores) and the last, partly filled round.  Over 143 layers (4 to 64 experts, 1 to 4096 tokens, widths of
//  512 to 2880) and 140 plain products, time against a workgroup per half row tile: forward 0.66, backward 0.52, products 0.50 in
//  the mean; at worst 1.04, where an expert's rows are whole tiles and the tiles whole rounds for that form as well (64 experts x
//  1024 rows, 2880 x 720: 2040 and 2111 us; 8 experts, 3000 x 2 rows, 1024 wide, forward: 395 and 405).
//  * An operand that is [row][k] in memory (activations, [n][k] weights of the input gradients) keeps that layout in LDS
//    (128-byte rows, 16-byte pieces XOR-swizzled with the row number on the global side of the copy); a lane's 16-byte
//    read holds four contraction steps.
//  * An operand that is [k][column] (the forward's weights, both operands of a weight gradient) keeps that layout too and
//    needs no transpose: a lane's operand for one instruction is ONE value, B[k][n of the lane], so an 8-byte read of
//    row k gives a lane columns 2l and 2l+1, i.e. the operands of the wave's "even" and "odd" accumulator blocks.  The
//    interleaved (gate, up) columns of the clamped SwiGLU therefore meet in one lane, and outputs leave as 8-byte stores,
//    256 contiguous bytes per half wave.
//  * The contraction may end inside a slab: the last slab's copies re-read valid data past its end, and the waves
//    overwrite what they copied of both operands there with zeros before the barrier (an infinity read twice would make a
//    NaN with a zero).
//
// Requirements: leading dimensions and, for row products, the contraction length multiples of 4 elements.
#include <type_traits>

#include "common.h"

namespace yamoe {

namespace f32 {

constexpr int kBM = 128, kBN = 128, kBK = 32;
constexpr int kThreads = 256;
constexpr int kAStage = kBM * kBK * 4;  // 16 KB: 128 rows x 128 bytes, or 32 k rows x 512 bytes
constexpr int kBStage = kBK * kBN * 4;
constexpr int kStage = kAStage + kBStage;
constexpr int kStages = 2;
constexpr int kLds = kStages * kStage;  // 64 KB: two workgroups per CU

constexpr int kWorkgroups = 2 * 256;    // two on each of the 256 CUs, each going through its share of the tiles

static_assert(kRowTile == 2 * kBM, "an expert has at most twice as many tiles here as row tiles in the schedule");

enum { EPI_STORE = 0, EPI_GLU = 1 };
// which products: rows x [k][n] weights (forward), rows x [n][k] weights (input gradients), [k][m]^T x [k][n] over an
// expert's rows (weight gradients)
enum { ROWS_KN = 0, ROWS_NK = 1, WGRAD = 2 };

typedef float f32x2 __attribute__((ext_vector_type(2)));

struct Args {
  const float *A;      // [rows, lda], k-contiguous; WGRAD: [N, Md], rows in expert order
  const float *B;      // [E, Kd, Nd]; ROWS_NK: [E, Nd, Kd]; WGRAD: [N, Nd]
  const float *bias;   // [E, Nd] or null
  float *C;            // EPI_STORE: [rows, ldc]; EPI_GLU: act [rows, Nd/2]; WGRAD: [E, Md, Nd]
  float *C2;           // EPI_GLU: optional pre-activations [rows, Nd]
  const int *a_rows;   // optional gather of A rows: source row = a_rows[p] / a_div
  const int *sched;    // (row products)
  const int *counts, *offsets;  // (WGRAD) kept rows of an expert: the first min(counts, capacity) from offsets on
  int a_div, Kd, Nd, lda, ldb, ldc, n_col_tiles;
  int capacity, E, Md, n_m_tiles;
  long long b_expert_stride;
};

// One output tile: what it is (the same for every lane) and where this lane's copies come from
struct Tile {
  int expert, row0, rows_valid, n0, k_len;  // rows of the tile: sorted rows, or (WGRAD) rows of the gradient
  const char *a_base, *b_base;
  uint32_t a_off[4], b_off[4];
};

template <int EPI, int MODE, bool GATHER>
__global__ __launch_bounds__(kThreads, 2) void gemm_f32_kernel(const Args args) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr bool A_ROWS = MODE != WGRAD, B_ROWS = MODE == ROWS_NK;  // operands that are [row][k]
  constexpr int kStores = MODE == ROWS_NK ? 64 : 32;  // stores of a whole tile per wave (a wait can count 63 at most)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int rl = lane & 31, g = lane >> 5;

  // ---- copies.  A [row][k] operand: copy i (0..3) fetches rows 32*i + 8*wave + (lane >> 3), 16 bytes of each; LDS position
  // lane & 7 of the row holds piece pos ^ ((row >> 1) & 7).  A [k][column] operand: copy i fetches k rows
  // 8*wave + 2*i + (lane >> 5), piece lane & 31 (no swizzle: a half wave reads 256 contiguous bytes of one k row).
  // Rows and columns past the end re-read valid ones; never stored.
  // (a gathering instantiation without a row list reads its rows in order: see gemm_async_tile.h)
  const bool gathers = GATHER && args.a_rows != nullptr;
  const int piece = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);  // (the same for all four copies)
  const long long a_slab_bytes = A_ROWS ? kBK * 4 : (long long)kBK * args.lda * 4;
  const long long b_slab_bytes = B_ROWS ? kBK * 4 : (long long)kBK * args.ldb * 4;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);

  // ---- the tiles: tile L of the launch.  Row products run expert-major, then column tile, then the expert's 128-row
  // tiles; weight gradients expert-major, then column by column of the expert's output tiles.
  const int total = (MODE == WGRAD ? args.E * args.n_m_tiles : args.sched[kSchedHalfTiles]) * args.n_col_tiles;
  // Workgroups go through the tiles in rounds of kWorkgroups.  Where the last round has tiles for at most half of the CUs,
  // they are dealt out in halves of 64 rows (both wave rows stay busy): item i of the launch is tile i up to there.  (The
  // down product of the README workload has 3.05 rounds: 2 % of the whole forward.)
  constexpr bool SPLITS = MODE != WGRAD;
  const int whole_rounds = total / kWorkgroups * kWorkgroups;
  const bool splits = SPLITS && 4 * (total - whole_rounds) <= kWorkgroups;
  const int items = splits ? 2 * total - whole_rounds : total;
  auto set_tile = [&](int item, Tile &t) {
    const bool half = splits && item >= whole_rounds;
    const int L = half ? whole_rounds + ((item - whole_rounds) >> 1) : item;
    long long k_first = 0;
    if constexpr (MODE == WGRAD) {
      const int per_expert = args.n_m_tiles * args.n_col_tiles;
      t.expert = L / per_expert;
      const int local = L - t.expert * per_expert, col_tile = local / args.n_m_tiles;
      t.row0 = (local - col_tile * args.n_m_tiles) * kBM;
      t.rows_valid = min(kBM, args.Md - t.row0);
      t.n0 = col_tile * kBN;
      t.k_len = max(min(__builtin_amdgcn_readfirstlane(args.counts[t.expert]), args.capacity), 0);
      k_first = __builtin_amdgcn_readfirstlane(args.offsets[t.expert]);
    } else {
      // the last row tile of the schedule whose expert starts at or before tile L
      const int *tiles = args.sched + kSchedHeader;
      const int n_tiles = args.sched[0];
      int found = -1;
      for (int base = 0; base < n_tiles; base += kWave) {
        const bool before = base + lane < n_tiles && tiles[8 * (base + lane) + 7] * args.n_col_tiles <= L;
        const int n = __popcll(__ballot(before));
        found += n;
        if (n < kWave) break;
      }
      const int *te = tiles + 8 * __builtin_amdgcn_readfirstlane(found);  // the expert's last row tile
      const int *first = tiles + 8 * __builtin_amdgcn_readfirstlane(te[3]);
      const int row_first = __builtin_amdgcn_readfirstlane(first[1]);
      const int rows = __builtin_amdgcn_readfirstlane(te[1] + te[2]) - row_first;
      const int parts = (rows + kBM - 1) / kBM;
      const int local = L - __builtin_amdgcn_readfirstlane(te[7]) * args.n_col_tiles;
      const int col_tile = (int)((uint32_t)local / (uint32_t)parts);
      const int part = local - col_tile * parts;
      t.expert = __builtin_amdgcn_readfirstlane(te[0]);
      t.row0 = row_first + part * kBM;
      t.rows_valid = min(rows - part * kBM, kBM);
      if (half) {
        // (a half without rows is gone through like the others and stores nothing: its first row only has to exist)
        const bool second = ((item - whole_rounds) & 1) != 0;
        t.rows_valid = second ? t.rows_valid - 64 : min(t.rows_valid, 64);
        if (second && t.rows_valid > 0) t.row0 += 64;
      }
      t.n0 = col_tile * kBN;
      t.k_len = args.Kd;
    }
    const int cols_valid = min(kBN, args.Nd - t.n0);
    auto column_off = [&](int i, int valid, int ld) {
      const int k = 8 * wave + 2 * i + (lane >> 5);
      const int col = (lane & 31) * 4;
      return (uint32_t)(((long long)k * ld + (col >= valid ? 0 : col)) * 4);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 32 * i + 8 * wave + (lane >> 3);
      if constexpr (A_ROWS) {
        const int r = max(min(row, t.rows_valid - 1), 0);
        long long src = r;
        if (gathers) src = args.a_rows[t.row0 + r] / args.a_div;
        t.a_off[i] = (uint32_t)((src * args.lda + piece * 4) * 4);
      } else {
        t.a_off[i] = column_off(i, t.rows_valid, args.lda);
      }
      if constexpr (B_ROWS) t.b_off[i] = (uint32_t)(((long long)min(row, cols_valid - 1) * args.ldb + piece * 4) * 4);
      else t.b_off[i] = column_off(i, cols_valid, args.ldb);
    }
    t.a_base = A_ROWS ? (const char *)(args.A + (gathers ? 0ll : (long long)t.row0 * args.lda))
                      : (const char *)(args.A + k_first * args.lda + t.row0);
    t.b_base = MODE == ROWS_KN   ? (const char *)(args.B + (long long)t.expert * args.b_expert_stride + t.n0)
               : MODE == ROWS_NK ? (const char *)(args.B + (long long)t.expert * args.b_expert_stride + (long long)t.n0 * args.ldb)
                                 : (const char *)(args.B + k_first * args.ldb + t.n0);
  };
  auto issue = [&](const Tile &t, int slab, int stage) {
    const uint32_t st = lds0 + (uint32_t)(stage & (kStages - 1)) * kStage;
    const char *ab = t.a_base + (long long)slab * a_slab_bytes;
    const char *bb = t.b_base + (long long)slab * b_slab_bytes;
    const int left = t.k_len - slab * kBK;  // (below 32 in a last slab that the contraction does not fill)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t a_adj = 0, b_adj = 0;
      if (left < kBK) {  // k rows past the end re-read the last one, pieces past it the row's first
        const int past = max(8 * wave + 2 * i + (lane >> 5) - (left - 1), 0);
        a_adj = A_ROWS ? (piece * 4 >= left ? piece * 16u : 0u) : (uint32_t)past * (uint32_t)args.lda * 4u;
        b_adj = B_ROWS ? (piece * 4 >= left ? piece * 16u : 0u) : (uint32_t)past * (uint32_t)args.ldb * 4u;
      }
      copy16_to_lds(ab, t.a_off[i] - a_adj, st + (uint32_t)(A_ROWS ? (32 * i + 8 * wave) * 128 : (8 * wave + 2 * i) * 512));
      copy16_to_lds(bb, t.b_off[i] - b_adj, st + kAStage + (uint32_t)(B_ROWS ? (32 * i + 8 * wave) * 128 : (8 * wave + 2 * i) * 512));
    }
  };
  // clears what this wave copied of the last slab past the end of the contraction
  auto zero_tail = [&](const Tile &t, int slab, int stage) {
    const int left = t.k_len - slab * kBK;
    char *st = lds + (stage & (kStages - 1)) * kStage + lane * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool past = A_ROWS ? piece * 4 >= left : 8 * wave + 2 * i + (lane >> 5) >= left;
      if (past) *(u32x4 *)(st + (A_ROWS ? (32 * i + 8 * wave) * 128 : (8 * wave + 2 * i) * 512)) = (u32x4){0, 0, 0, 0};
      const bool b_past = B_ROWS ? piece * 4 >= left : 8 * wave + 2 * i + (lane >> 5) >= left;
      if (b_past) *(u32x4 *)(st + kAStage + (B_ROWS ? (32 * i + 8 * wave) * 128 : (8 * wave + 2 * i) * 512)) = (u32x4){0, 0, 0, 0};
    }
  };

  // [row][k] operand of block x in k-step ks (8 contraction steps): row (x*2+w)*32 + rl, piece 2*ks + g; the four values of
  // the piece feed four instructions, in which the lanes of half g hold k = 8*ks + 4*g + q.  (Rows 64 apart share
  // (row >> 1) & 7, so block 1 is the same offset 8192 bytes further.)
  int a_rd[4], b_rd[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int p = ((2 * ks + g) ^ ((rl >> 1) & 7)) << 4;
    a_rd[ks] = A_ROWS ? (wm * 32 + rl) * 128 + p : g * 4 * 512 + (wm * 64 + 2 * rl) * 4 + ks * 8 * 512;
    b_rd[ks] = B_ROWS ? (wn * 32 + rl) * 128 + p : g * 4 * 512 + (wn * 64 + 2 * rl) * 4 + ks * 8 * 512;
  }
  // accumulators: acc[a][b][v], instruction row i = 8*(v/4) + 4*g + v%4 and column rl, is
  //   row (a*2+wm)*32 + i of the tile, or (WGRAD, "even" and "odd" rows) wm*64 + 2*i + a
  //   column wn*64 + 2*rl + b, or (ROWS_NK) (b*2+wn)*32 + rl
  f32x16 acc[2][2];

  // A slab is four k-steps of 4 * NA * 2 MFMAs (1024 clocks for NA = 2).  The operands of a k-step are read from LDS while
  // the MFMAs of the one before run, in a fixed order (left to itself the compiler reads each value right before its use).
  // The wait for the next slab and the barrier stand before the last k-step, whose operands are in registers by then: the
  // copies and the first reads of the next slab are issued under its MFMAs.  (Slab 0's copies are on their way already,
  // into stage `stage`; slab s sits in stage + s.  `stores`: behind them, this wave has exactly
  // kStores stores of the previous tile in flight, which nothing waits for here.)
  // NA blocks are this wave's own; with SHARED there is one more, the tile's last, of which either wave row takes half of the
  // k-steps (row products only: see where the halves meet).
  auto contract = [&](const Tile &t, int stage, bool stores, auto na, auto shared) {
    constexpr int NA = decltype(na)::value;
    constexpr bool SHARED = decltype(shared)::value;
    const int n_slabs = (t.k_len + kBK - 1) / kBK;
    float va[2][4][2], vb[2][4][2];  // [set][q][block]
    auto read = [&](int s, int ks, float (&ra)[4][2], float (&rb)[4][2]) {
      if constexpr (NA > 0 || SHARED) {
        const char *sa = lds + ((stage + s) & (kStages - 1)) * kStage;
        const char *sb = sa + kAStage;
        if constexpr (A_ROWS) {
#pragma unroll
          for (int x = 0; x < NA; ++x) {
            const f32x4 v = *(const f32x4 *)(sa + a_rd[ks] + x * 64 * 128);
#pragma unroll
            for (int q = 0; q < 4; ++q) ra[q][x] = v[q];
          }
          if constexpr (SHARED) {
            if (ks >> 1 == wm) {
              const f32x4 v = *(const f32x4 *)(sa + a_rd[ks] + (NA * 64 - wm * 32) * 128);
#pragma unroll
              for (int q = 0; q < 4; ++q) ra[q][NA] = v[q];
            }
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x2 v = *(const f32x2 *)(sa + a_rd[ks] + q * 512);
            ra[q][0] = v[0];
            ra[q][1] = v[1];
          }
        }
        if constexpr (B_ROWS) {
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const f32x4 v = *(const f32x4 *)(sb + b_rd[ks] + x * 64 * 128);
#pragma unroll
            for (int q = 0; q < 4; ++q) rb[q][x] = v[q];
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x2 v = *(const f32x2 *)(sb + b_rd[ks] + q * 512);
            rb[q][0] = v[0];
            rb[q][1] = v[1];
          }
        }
      }
    };
    auto multiply = [&](int ks, const float (&ra)[4][2], const float (&rb)[4][2]) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[q][a], rb[q][b], acc[a][b], 0, 0, 0);
      if constexpr (SHARED) {
        if (ks >> 1 == wm) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[NA][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[q][NA], rb[q][b], acc[NA][b], 0, 0, 0);
        }
      }
    };
    // slab s is there for every wave, and nobody reads the other stage any more (the reads of a wave are complete when it
    // gets here: its next MFMAs need them)
    auto arrive = [&](int s) {
      // (slab 0 was requested ahead of the previous tile's stores, and vector memory operations complete in order)
      if (s == 0 && stores) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kStores < 64 ? kStores : 0) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      if (s == n_slabs - 1 && (t.k_len & (kBK - 1)) != 0) zero_tail(t, s, stage + s);
      __syncthreads();
      if (s + 1 < n_slabs) issue(t, s + 1, stage + s + 1);
    };
    if (n_slabs > 0) {
      arrive(0);
      read(0, 0, va[0], vb[0]);
    }
    for (int s = 0; s < n_slabs; ++s) {
#pragma unroll
      for (int ks = 0; ks < 3; ++ks) {
        __builtin_amdgcn_sched_barrier(0);
        read(s, ks + 1, va[(ks + 1) & 1], vb[(ks + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(ks, va[ks & 1], vb[ks & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (s + 1 < n_slabs) {
        arrive(s + 1);
        read(s + 1, 0, va[0], vb[0]);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(3, va[1], vb[1]);
    }
  };

  // ---- workgroup b takes tiles b, b + gridDim.x, ...  The next tile is looked up and its first slab requested before the
  // epilogue of the current one.
  // The places in a round of a CU's two, workgroups b and b + 256, are b and 511 - b: in the order of the tiles a full tile
  // and an expert's remainder often alternate, and a CU should get one of each (2 % of the step of a layer of 16 experts
  // with 187 rows).
  int L = blockIdx.x < kWorkgroups / 2 ? blockIdx.x : kWorkgroups / 2 + kWorkgroups - 1 - blockIdx.x, stage = 0;
  bool stores = false;
  if (L >= items) return;
  Tile t;
  set_tile(L, t);
  if (t.k_len > 0) issue(t, 0, stage);
  for (;;) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
    // blocks of this wave that hold anything: rows of a row product by 32-row blocks, everything else by the wave's 64
    // (every wave of the workgroup goes through the same copies, waits and barriers, whatever it multiplies)
    const int cols_valid = min(kBN, args.Nd - t.n0);
    const bool active_n = B_ROWS ? wn * 32 < cols_valid : wn * 64 < cols_valid;
    const int blocks = t.rows_valid <= 0 ? 0 : (t.rows_valid + 31) >> 5;
    const int n_a = !active_n || t.rows_valid <= 0 ? 0 : A_ROWS ? (blocks - wm + 1) >> 1 : (wm * 64 < t.rows_valid ? 2 : 0);
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 2> I2;
    if constexpr (A_ROWS) {
      // An odd number of blocks, which the two wave rows would be 1 and 0 or 2 and 1 of: the last one's k-steps are shared, and
      // the halves of its sums meet in the ring stage of the last slab.
      const int busy = active_n ? blocks : 0;
      if (busy == 4) contract(t, stage, stores, I2(), std::false_type());
      else if (busy == 3) contract(t, stage, stores, I1(), std::true_type());
      else if (busy == 2) contract(t, stage, stores, I1(), std::false_type());
      else if (busy == 1) contract(t, stage, stores, I0(), std::true_type());
      else contract(t, stage, stores, I0(), std::false_type());
      if ((blocks & 1) != 0) {
        const int last = stage + (t.k_len + kBK - 1) / kBK - 1;
        float *meet = (float *)(lds + (last & (kStages - 1)) * kStage) + wn * 32 * kWave + lane;
        auto add = [&](auto which) {
          constexpr int A = decltype(which)::value;
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              if (wm == 1) meet[(b * 16 + v) * kWave] = acc[A][b][v];
              else acc[A][b][v] += meet[(b * 16 + v) * kWave];
            }
        };
        __syncthreads();  // nobody reads the slab any more
        if (wm == 1 && busy == 3) add(I1());
        else if (wm == 1 && busy == 1) add(I0());
        __syncthreads();
        if (wm == 0 && busy == 3) add(I1());
        else if (wm == 0 && busy == 1) add(I0());
      }
    } else {
      if (n_a == 2) contract(t, stage, stores, I2(), std::false_type());
      else contract(t, stage, stores, I0(), std::false_type());
    }

    // (the stage after the last slab's has been free since the barrier in front of that slab)
    stage += (t.k_len + kBK - 1) / kBK;
    const int row0 = t.row0, rows_valid = t.rows_valid, expert = t.expert;
    const bool whole = rows_valid == kBM && cols_valid == kBN;
    const int col = t.n0 + (B_ROWS ? wn * 32 + rl : wn * 64 + 2 * rl);  // (GLU: even, the gate column of pair col / 2)
    float b0 = 0.0f, b1 = 0.0f;
    if (MODE == ROWS_KN && n_a > 0 && args.bias != nullptr && col < args.Nd) {
      const float *bp = args.bias + (long long)expert * args.Nd + col;
      b0 = bp[0];
      b1 = bp[1];
    }
    L += kWorkgroups;
    if (L < items) set_tile(L, t);
    // The bias is waited for here, with the look-ups and ahead of the next slab's request.  Left to its uses, the compiler's
    // wait for all vector memory stands in front of every store of a partial tile, one store at a time, and in the
    // contraction loop, whose registers the load may still be on its way to for all the compiler knows: there it waits for
    // the next slab right after requesting it.  (16 experts, 3000 x 2 rows, 512 wide, forward: 137 us that way, 130 now.)
    asm volatile("" : "+v"(b0), "+v"(b1));
    if (L < items && t.k_len > 0) issue(t, 0, stage);

    // epilogue: straight from the accumulators; a half wave covers 256 (128 for act and ROWS_NK) contiguous bytes of a row
    if (n_a > 0) {
      float *C = args.C + (MODE == WGRAD ? (long long)expert * args.Md * args.Nd : 0ll);
      auto store = [&](int a, int v, long long orow) {
        if constexpr (MODE == ROWS_NK) {
          C[orow * args.ldc + col] = acc[a][0][v];
          C[orow * args.ldc + col + 64] = acc[a][1][v];
        } else {
          const float x0 = acc[a][0][v] + b0, x1 = acc[a][1][v] + b1;
          if constexpr (EPI == EPI_STORE) {
            *(f32x2 *)(C + orow * args.ldc + col) = (f32x2){x0, x1};
          } else {
            C[orow * args.ldc + (col >> 1)] = glu_forward(x0, x1);
            if (args.C2 != nullptr) *(f32x2 *)(args.C2 + orow * args.Nd + col) = (f32x2){x0, x1};
          }
        }
      };
      auto row_of = [&](int a, int v) {
        const int i = 8 * (v >> 2) + 4 * g + (v & 3);
        return A_ROWS ? (a * 2 + wm) * 32 + i : wm * 64 + 2 * i + a;
      };
      if (whole) {  // (kStores stores, one or two per register)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int v = 0; v < 16; ++v) store(a, v, row0 + row_of(a, v));
      } else {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int r = row_of(a, v);
            if (a < n_a && r < rows_valid && col < args.Nd) {
              if constexpr (MODE == ROWS_NK) {
                C[(long long)(row0 + r) * args.ldc + col] = acc[a][0][v];
                if (col + 64 < args.Nd) C[(long long)(row0 + r) * args.ldc + col + 64] = acc[a][1][v];
              } else {
                store(a, v, row0 + r);
              }
            }
          }
      }
    }
    stores = whole && kStores < 64 && (EPI != EPI_GLU || args.C2 == nullptr);
    if (L >= items) return;
  }
}

template <int EPI, int MODE, bool GATHER>
static int launch(const Args &args, hipStream_t stream) {
  auto kernel = gemm_f32_kernel<EPI, MODE, GATHER>;
  static DeviceFlags attr_done;  // one per kernel instantiation
  if (int rc = ensure_dynamic_lds((const void *)kernel, kLds, attr_done, "gemm_f32_kernel")) return rc;
  hipLaunchKernelGGL(kernel, dim3(kWorkgroups), dim3(kThreads), kLds, stream, args);
  return check_launch("gemm_f32_kernel");
}

}  // namespace f32

int gemm_f32_gate_up(const void *x, const int *sorted_idx, const void *w, const void *bias, void *act, void *pre,
                     const void *sched, int N, int K, int E, int H, int I, hipStream_t stream) {
  f32::Args a = {};
  a.A = (const float *)x; a.B = (const float *)w; a.bias = (const float *)bias; a.C = (float *)act; a.C2 = (float *)pre;
  a.a_rows = sorted_idx; a.a_div = K; a.sched = (const int *)sched;
  a.Kd = H; a.Nd = 2 * I; a.lda = H; a.ldb = 2 * I; a.ldc = I;
  a.b_expert_stride = (long long)H * 2 * I;
  a.n_col_tiles = ceil_div(2 * I, f32::kBN);
  return f32::launch<f32::EPI_GLU, f32::ROWS_KN, true>(a, stream);
}

int gemm_f32_down(const void *act, const void *w, const void *bias, void *y, const void *sched, int N, int E, int H,
                  int I, hipStream_t stream) {
  f32::Args a = {};
  a.A = (const float *)act; a.B = (const float *)w; a.bias = (const float *)bias; a.C = (float *)y;
  a.sched = (const int *)sched; a.a_div = 1;
  a.Kd = I; a.Nd = H; a.lda = I; a.ldb = H; a.ldc = H;
  a.b_expert_stride = (long long)I * H;
  a.n_col_tiles = ceil_div(H, f32::kBN);
  return f32::launch<f32::EPI_STORE, f32::ROWS_KN, false>(a, stream);
}

// out[p, :] = g[row p, :] . W[e]^T with W[e] stored [Nd, Kd]; with g_rows the source row of p is g_rows[p] / g_div
int gemm_f32_dgrad(const void *g, const int *g_rows, int g_div, const void *w, void *out, const void *sched, int N, int E,
                   int Kd, int Nd, hipStream_t stream) {
  f32::Args a = {};
  a.A = (const float *)g; a.B = (const float *)w; a.C = (float *)out;
  a.sched = (const int *)sched; a.a_rows = g_rows; a.a_div = g_rows != nullptr ? g_div : 1;
  a.Kd = Kd; a.Nd = Nd; a.lda = Kd; a.ldb = Kd; a.ldc = Nd;
  a.b_expert_stride = (long long)Nd * Kd;
  a.n_col_tiles = ceil_div(Nd, f32::kBN);
  if (g_rows != nullptr) return f32::launch<f32::EPI_STORE, f32::ROWS_NK, true>(a, stream);
  return f32::launch<f32::EPI_STORE, f32::ROWS_NK, false>(a, stream);
}

// dW[e] = L[rows of e]^T . R[rows of e], rows in expert order; an expert without rows gets zeros
int gemm_f32_wgrad(const void *L, const void *R, void *dW, const int *counts, const int *offsets, int capacity, int E, int Md,
                   int Nd, hipStream_t stream) {
  f32::Args a = {};
  a.A = (const float *)L; a.B = (const float *)R; a.C = (float *)dW;
  a.counts = counts; a.offsets = offsets; a.capacity = capacity; a.E = E; a.Md = Md;
  a.Nd = Nd; a.lda = Md; a.ldb = Nd; a.ldc = Nd;
  a.n_col_tiles = ceil_div(Nd, f32::kBN);
  a.n_m_tiles = ceil_div(Md, f32::kBM);
  return f32::launch<f32::EPI_STORE, f32::WGRAD, false>(a, stream);
}

}  // namespace yamoe
