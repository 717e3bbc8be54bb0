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
//    The 32-row blocks of a tile alternate between the two wave rows, so that a remainder keeps both busy.
//  * Operands go global -> LDS with asynchronous 16-byte copies (no staging registers), two stages of 32 KB, one
//    workgroup barrier per slab of 32 (16 000 clocks of matrix work): while a workgroup waits at its barrier or
//    runs its epilogue, the other workgroup on the CU keeps the matrix pipe busy.
//  * An operand that is [row][k] in memory (activations, [n][k] weights of the input gradients) keeps that layout in LDS
//    (128-byte rows, 16-byte pieces XOR-swizzled with the row number on the global side of the copy); a lane's 16-byte
//    read holds four contraction steps.
//  * An operand that is [k][column] (the forward's weights, both operands of a weight gradient) keeps that layout too and
//    needs no transpose: a lane's operand for one instruction is ONE value, B[k][n of the lane], so an 8-byte read of
//    row k gives a lane columns 2l and 2l+1, i.e. the operands of the wave's "even" and "odd" accumulator blocks.  The
//    interleaved (gate, up) columns of the clamped SwiGLU therefore meet in one lane, and outputs leave as 8-byte stores,
//    256 contiguous bytes per half wave.
//  * The contraction may end inside a slab: the last slab's copies re-read valid data past its end, and the waves
//    overwrite what they copied of the left operand there with zeros before the barrier.
//
// Requirements: leading dimensions and, for row products, the contraction length multiples of 4 elements.
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

template <int EPI, int MODE, bool GATHER>
__global__ __launch_bounds__(kThreads, 2) void gemm_f32_kernel(const Args args) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr bool A_ROWS = MODE != WGRAD, B_ROWS = MODE == ROWS_NK;  // operands that are [row][k]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int rl = lane & 31, g = lane >> 5;

  // ---- which tile.  Workgroup ids are dealt round-robin over the XCDs, so id b takes logical tile
  // (b % 8) * per_xcd + b / 8.  Row products run expert-major, then column tile, then the expert's tiles of rows, so the
  // tiles in flight on one XCD share weight columns through its L2; weight gradients run column by column of one expert's
  // output tiles.
  int expert, n0, k_len;
  int row0, rows_valid;  // rows of the output tile: sorted rows, or (WGRAD) rows of the gradient
  long long k_first = 0;
  {
    const int n_rows = MODE == WGRAD ? args.E * args.n_m_tiles : 2 * args.sched[0];
    const int total = n_rows * args.n_col_tiles;
    const int total8 = (total + kXcds - 1) / kXcds * kXcds;
    const int b = blockIdx.x;
    if (b >= total8) return;
    const int L = (b % kXcds) * (total8 / kXcds) + b / kXcds;
    if (L >= total) return;
    if constexpr (MODE == WGRAD) {
      const int per_expert = args.n_m_tiles * args.n_col_tiles;
      expert = L / per_expert;
      const int local = L - expert * per_expert, col_tile = local / args.n_m_tiles;
      row0 = (local - col_tile * args.n_m_tiles) * kBM;
      rows_valid = min(kBM, args.Md - row0);
      n0 = col_tile * kBN;
      k_len = max(min(__builtin_amdgcn_readfirstlane(args.counts[expert]), args.capacity), 0);
      k_first = __builtin_amdgcn_readfirstlane(args.offsets[expert]);
    } else {
      const int *tiles = args.sched + kSchedHeader;
      const int t0 = (L / args.n_col_tiles) >> 1;
      const int gfirst = tiles[8 * t0 + 3], gcount = tiles[8 * t0 + 4];
      const int local = L - 2 * gfirst * args.n_col_tiles;
      const int col_tile = local / (2 * gcount);
      const int part = local - col_tile * 2 * gcount;  // the expert's tile of rows
      const int *last = tiles + 8 * (gfirst + gcount - 1);
      expert = tiles[8 * gfirst];
      row0 = tiles[8 * gfirst + 1] + part * kBM;
      rows_valid = min(last[1] + last[2] - row0, kBM);
      n0 = col_tile * kBN;
      k_len = args.Kd;
      if (rows_valid <= 0) return;  // (the expert has fewer tiles of 128 than twice its row tiles)
    }
  }
  const int cols_valid = min(kBN, args.Nd - n0);
  const int n_slabs = (k_len + kBK - 1) / kBK;

  // ---- copies.  A [row][k] operand: copy i (0..3) fetches rows 32*i + 8*wave + (lane >> 3), 16 bytes of each; LDS position
  // lane & 7 of the row holds piece pos ^ ((row >> 1) & 7).  A [k][column] operand: copy i fetches k rows
  // 8*wave + 2*i + (lane >> 5), piece lane & 31 (no swizzle: a half wave reads 256 contiguous bytes of one k row).
  // Rows and columns past the end re-read valid ones; never stored.
  // (a gathering instantiation without a row list reads its rows in order: see gemm_async_tile.h)
  const bool gathers = GATHER && args.a_rows != nullptr;
  const int piece = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);  // (the same for all four copies)
  uint32_t a_off[4], b_off[4];
  auto column_off = [&](int i, int valid, int ld) {
    const int k = 8 * wave + 2 * i + (lane >> 5);
    const int col = (lane & 31) * 4;
    return (uint32_t)(((long long)k * ld + (col >= valid ? 0 : col)) * 4);
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 32 * i + 8 * wave + (lane >> 3);
    if constexpr (A_ROWS) {
      const int r = min(row, rows_valid - 1);
      long long src = r;
      if (gathers) src = args.a_rows[row0 + r] / args.a_div;
      a_off[i] = (uint32_t)((src * args.lda + piece * 4) * 4);
    } else {
      a_off[i] = column_off(i, rows_valid, args.lda);
    }
    if constexpr (B_ROWS) b_off[i] = (uint32_t)(((long long)min(row, cols_valid - 1) * args.ldb + piece * 4) * 4);
    else b_off[i] = column_off(i, cols_valid, args.ldb);
  }
  const char *a_base = A_ROWS ? (const char *)(args.A + (gathers ? 0ll : (long long)row0 * args.lda))
                              : (const char *)(args.A + k_first * args.lda + row0);
  const char *b_base = MODE == ROWS_KN   ? (const char *)(args.B + (long long)expert * args.b_expert_stride + n0)
                       : MODE == ROWS_NK ? (const char *)(args.B + (long long)expert * args.b_expert_stride + (long long)n0 * args.ldb)
                                         : (const char *)(args.B + k_first * args.ldb + n0);
  const long long a_slab_bytes = A_ROWS ? kBK * 4 : (long long)kBK * args.lda * 4;
  const long long b_slab_bytes = B_ROWS ? kBK * 4 : (long long)kBK * args.ldb * 4;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
  auto issue = [&](int slab) {
    const uint32_t st = lds0 + (uint32_t)(slab & (kStages - 1)) * kStage;
    const char *ab = a_base + (long long)slab * a_slab_bytes;
    const char *bb = b_base + (long long)slab * b_slab_bytes;
    const int left = k_len - slab * kBK;  // (below 32 in a last slab that the contraction does not fill)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 8 * wave + 2 * i + (lane >> 5);
      const int past = max(k - (left - 1), 0);  // k rows past the end re-read the last one, pieces past it the row's first
      const uint32_t a_adj = A_ROWS ? (piece * 4 >= left ? piece * 16u : 0u) : (uint32_t)past * (uint32_t)args.lda * 4u;
      const uint32_t b_adj = B_ROWS ? (piece * 4 >= left ? piece * 16u : 0u) : (uint32_t)past * (uint32_t)args.ldb * 4u;
      copy16_to_lds(ab, a_off[i] - a_adj, st + (uint32_t)(A_ROWS ? (32 * i + 8 * wave) * 128 : (8 * wave + 2 * i) * 512));
      copy16_to_lds(bb, b_off[i] - b_adj, st + kAStage + (uint32_t)(B_ROWS ? (32 * i + 8 * wave) * 128 : (8 * wave + 2 * i) * 512));
    }
  };
  // what this wave copied of the last slab's left operand past the end of the contraction
  auto zero_tail = [&](int slab) {
    const int left = k_len - slab * kBK;
    char *st = lds + (slab & (kStages - 1)) * kStage + lane * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool past = A_ROWS ? piece * 4 >= left : 8 * wave + 2 * i + (lane >> 5) >= left;
      if (past) *(u32x4 *)(st + (A_ROWS ? (32 * i + 8 * wave) * 128 : (8 * wave + 2 * i) * 512)) = (u32x4){0, 0, 0, 0};
    }
  };

  // ---- accumulators: acc[a][b][v], instruction row i = 8*(v/4) + 4*g + v%4 and column rl, is
  //   row (a*2+wm)*32 + i of the tile, or (WGRAD, "even" and "odd" rows) wm*64 + 2*i + a
  //   column wn*64 + 2*rl + b, or (ROWS_NK) (b*2+wn)*32 + rl
  f32x16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;

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
  // blocks of this wave that hold anything: rows of a row product by 32-row blocks, everything else by the wave's 64
  const int blocks = (rows_valid + 31) >> 5;
  const bool active_n = B_ROWS ? wn * 32 < cols_valid : wn * 64 < cols_valid;
  const int n_a = !active_n ? 0 : A_ROWS ? (blocks - wm + 1) >> 1 : (wm * 64 < rows_valid ? 2 : 0);

  if (n_slabs > 0) issue(0);
  for (int s = 0; s < n_slabs; ++s) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (s == n_slabs - 1 && (k_len & (kBK - 1)) != 0) zero_tail(s);
    __syncthreads();  // slab s has landed for every wave, and nobody reads the other stage any more
    if (s + 1 < n_slabs) issue(s + 1);
    const char *sa = lds + (s & (kStages - 1)) * kStage;
    const char *sb = sa + kAStage;
    if (n_a > 0) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        f32x4 fa[2], fb[2];
        if constexpr (A_ROWS) {
          fa[0] = *(const f32x4 *)(sa + a_rd[ks]);
          fa[1] = *(const f32x4 *)(sa + a_rd[ks] + 64 * 128);
        }
        if constexpr (B_ROWS) {
          fb[0] = *(const f32x4 *)(sb + b_rd[ks]);
          fb[1] = *(const f32x4 *)(sb + b_rd[ks] + 64 * 128);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float va[2], vb[2];
          if constexpr (A_ROWS) {
            va[0] = fa[0][q]; va[1] = fa[1][q];
          } else {
            const f32x2 t = *(const f32x2 *)(sa + a_rd[ks] + q * 512);
            va[0] = t[0]; va[1] = t[1];
          }
          if constexpr (B_ROWS) {
            vb[0] = fb[0][q]; vb[1] = fb[1][q];
          } else {
            const f32x2 t = *(const f32x2 *)(sb + b_rd[ks] + q * 512);
            vb[0] = t[0]; vb[1] = t[1];
          }
          acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[0], vb[0], acc[0][0], 0, 0, 0);
          acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[0], vb[1], acc[0][1], 0, 0, 0);
          if (n_a > 1) {
            acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[1], vb[0], acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[1], vb[1], acc[1][1], 0, 0, 0);
          }
        }
      }
    }
  }

  // ---- epilogue: straight from the accumulators; a half wave covers 256 (128 for act and ROWS_NK) contiguous bytes of a row
  if (n_a == 0) return;
  const int col = n0 + (B_ROWS ? wn * 32 + rl : wn * 64 + 2 * rl);  // (GLU: even, the gate column of pair col / 2)
  float b0 = 0.0f, b1 = 0.0f;
  if (MODE == ROWS_KN && args.bias != nullptr && col < args.Nd) {
    const float *bp = args.bias + (long long)expert * args.Nd + col;
    b0 = bp[0];
    b1 = bp[1];
  }
  float *C = args.C + (MODE == WGRAD ? (long long)expert * args.Md * args.Nd : 0ll);
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    if (a < n_a) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int i = 8 * (v >> 2) + 4 * g + (v & 3);
        const int r = A_ROWS ? (a * 2 + wm) * 32 + i : wm * 64 + 2 * i + a;
        if (r < rows_valid) {
          const long long orow = row0 + r;
          if constexpr (MODE == ROWS_NK) {
            if (col < args.Nd) C[orow * args.ldc + col] = acc[a][0][v];
            if (col + 64 < args.Nd) C[orow * args.ldc + col + 64] = acc[a][1][v];
          } else if (col < args.Nd) {
            const float x0 = acc[a][0][v] + b0, x1 = acc[a][1][v] + b1;
            if constexpr (EPI == EPI_STORE) {
              *(f32x2 *)(C + orow * args.ldc + col) = (f32x2){x0, x1};
            } else {
              C[orow * args.ldc + (col >> 1)] = glu_forward(x0, x1);
              if (args.C2 != nullptr) *(f32x2 *)(args.C2 + orow * args.Nd + col) = (f32x2){x0, x1};
            }
          }
        }
      }
    }
  }
}

template <int EPI, int MODE, bool GATHER>
static int launch(const Args &args, long long tiles, hipStream_t stream) {
  auto kernel = gemm_f32_kernel<EPI, MODE, GATHER>;
  static DeviceFlags attr_done;  // one per kernel instantiation
  if (int rc = ensure_dynamic_lds((const void *)kernel, kLds, attr_done, "gemm_f32_kernel")) return rc;
  if (tiles <= 0) return 0;
  tiles = (tiles + kXcds - 1) / kXcds * kXcds;
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(kThreads), kLds, stream, args);
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
  return f32::launch<f32::EPI_GLU, f32::ROWS_KN, true>(a, 2ll * sched_max_row_tiles(N, E) * a.n_col_tiles, stream);
}

int gemm_f32_down(const void *act, const void *w, const void *bias, void *y, const void *sched, int N, int E, int H,
                  int I, hipStream_t stream) {
  f32::Args a = {};
  a.A = (const float *)act; a.B = (const float *)w; a.bias = (const float *)bias; a.C = (float *)y;
  a.sched = (const int *)sched; a.a_div = 1;
  a.Kd = I; a.Nd = H; a.lda = I; a.ldb = H; a.ldc = H;
  a.b_expert_stride = (long long)I * H;
  a.n_col_tiles = ceil_div(H, f32::kBN);
  return f32::launch<f32::EPI_STORE, f32::ROWS_KN, false>(a, 2ll * sched_max_row_tiles(N, E) * a.n_col_tiles, stream);
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
  const long long tiles = 2ll * sched_max_row_tiles(N, E) * a.n_col_tiles;
  if (g_rows != nullptr) return f32::launch<f32::EPI_STORE, f32::ROWS_NK, true>(a, tiles, stream);
  return f32::launch<f32::EPI_STORE, f32::ROWS_NK, false>(a, tiles, stream);
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
  return f32::launch<f32::EPI_STORE, f32::WGRAD, false>(a, (long long)E * a.n_m_tiles * a.n_col_tiles, stream);
}

}  // namespace yamoe
