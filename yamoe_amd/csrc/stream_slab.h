// The weight-streaming product of one (expert, 128-column slab): see stream.hip for the design.  A header of its own because
// the tile kernels' launches carry streamed experts as well (gemm_async_tile.h).
#pragma once

#include "common.h"

namespace yamoe {

constexpr int kStreamWaves = 4;        // waves that finish a slab; a workgroup has 4 or 8
constexpr int kStreamThreads = kWave * kStreamWaves;
constexpr int kSlabCols = 128;

typedef float f32x4v __attribute__((ext_vector_type(4)));

// How a wave multiplies the eight 16-byte loads that each of its lanes makes in a step (8 rows of 8 16-bit columns, or 4 rows
// of 4 + 4 fp32 columns): accumulator j of a lane is column column(lane % 16, j) of the slab.
template <typename T> struct StreamStep {
  static constexpr int kRows = 32;  // contraction rows of a step; a lane's are 8 * (lane / 16) + 0 .. 7
  static constexpr int kLaneRows = 8;
  static __device__ inline int column(int c16, int j) { return c16 * 8 + j; }
  // load i of a lane: which of its rows, and which of the slab's columns
  static __device__ inline int load_row(int i) { return i; }
  static __device__ inline int load_column(int c16, int) { return c16 * 8; }
  static __device__ inline f32x4v mma(const u32x4 &a, const u32x4 &b, f32x4v c) {
    if constexpr (std::is_same_v<T, bf16_t>)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  // (a register transpose: a column's eight values become one operand)
  template <int RB> static __device__ inline void multiply(const u32x4 (&bw)[8], const u32x4 (&aw)[RB], f32x4v (&acc)[RB][8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
      u32x4 col;
#pragma unroll
      for (int d = 0; d < 4; ++d) col[d] = __builtin_amdgcn_perm(bw[2 * d + 1][j >> 1], bw[2 * d][j >> 1], sel);
#pragma unroll
      for (int b = 0; b < RB; ++b) acc[b][j] = mma(aw[b], col, acc[b][j]);
    }
  }
};
// fp32: v_mfma_f32_16x16x4_f32 takes one value of either operand per lane, so a load's four values are the operands of four
// instructions, and no transpose is needed: in the instructions of the lane's row i, lane group g holds row 4 g + i.
template <> struct StreamStep<float> {
  static constexpr int kRows = 16;
  static constexpr int kLaneRows = 4;
  static __device__ inline int column(int c16, int j) { return (j >> 2) * 64 + c16 * 4 + (j & 3); }
  static __device__ inline int load_row(int i) { return i & 3; }
  static __device__ inline int load_column(int c16, int i) { return (i >> 2) * 64 + c16 * 4; }
  template <int RB> static __device__ inline void multiply(const u32x4 (&bw)[8], const u32x4 (&aw)[RB], f32x4v (&acc)[RB][8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < RB; ++b)
          acc[b][(i >> 2) * 4 + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(aw[b][i & 3]), __uint_as_float(bw[i][j]),
                                                                        acc[b][(i >> 2) * 4 + j], 0, 0, 0);
  }
};

struct StreamArgs {
  const void *A;       // activations [rows, lda], k-contiguous
  const void *B;       // weights [E, Kd, Nd]
  const void *bias;    // [E, Nd] or null
  void *C;             // GLU: act [rows, Nd/2]; else [rows, Nd]
  void *C2;            // GLU: optional pre-activations [rows, Nd]
  const int *a_rows;   // optional gather: source row = a_rows[p] / a_div
  const int *sched;
  FastDiv a_div, slab_div;  // divisions by the gather divisor and by n_slabs
  int Kd, Nd, lda, ldc, n_slabs, N, E;
  // The contraction of a slab may be shared by several workgroups (stream_parts in stream.hip), which leave their sums in
  // `partial` ([list entry][slab][part][part_floats], null: never shared) and count themselves in arrivals[list entry * n_slabs +
  // slab] (zero before and after the launch); the one that finds all others there adds the parts up, in their order, and
  // finishes the slab.
  int part_floats;
  bool yields;   // where there are tiles, their launches carry the list
  bool cut_lines;  // a weight row is not a whole number of cache lines
  float *partial;
  int *arrivals;
};
// A part: 16 rows, or 32 where an entry of the list can have more, of a slab's columns
inline int stream_part_floats(int N) { return (N <= 16 ? 16 : kStreamMaxRows) * kSlabCols; }

// One (expert, slab) of RB blocks of 16 rows (RB = 1: up to 16 rows, RB = 2: 17 to 32): the weights are fetched once
// and every column operand built from them goes through RB MFMAs.  item, part, parts: see StreamArgs.
template <typename T, bool GLU, bool GATHER, int WAVES, int DEPTH, int RB>
__device__ inline void stream_slab(const StreamArgs &args, float *red, const int expert, const int first, const int rows,
                                   const int slab, const int item = 0, const int part = 0, const int parts = 1) {
  typedef StreamStep<T> Step;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const int slab0 = slab * kSlabCols;
  const T *Bp = (const T *)args.B + (long long)expert * args.Kd * args.Nd + slab0;

  // A operand of block b: row 16 b + c16 of the expert (zero beyond `rows`), the lane's consecutive k
  bool a_ok[RB];
  const T *Ap[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    a_ok[b] = 16 * b + c16 < rows;
    long long a_src = first + (a_ok[b] ? 16 * b + c16 : 0);
    // (a gathering instantiation without a row list reads its rows in order, like the tile kernels)
    if (GATHER && args.a_rows != nullptr) a_src = fast_div(args.a_rows[a_src], args.a_div);
    Ap[b] = (const T *)args.A + a_src * args.lda + g * Step::kLaneRows;
  }

  f32x4v acc[RB][8];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[b][j] = (f32x4v){0.f, 0.f, 0.f, 0.f};

  const int all_steps = (args.Kd + Step::kRows - 1) / Step::kRows;
  int first_step = 0, n_steps = all_steps;
  if (parts > 1) {
    first_step = (int)((long long)all_steps * part / parts);
    n_steps = (int)((long long)all_steps * (part + 1) / parts);
  }
  u32x4 bw[DEPTH][8], aw[DEPTH][RB];

  auto fetch = [&](int step, u32x4 (&bw)[8], u32x4 (&aw)[RB]) {
    const int k0 = step * Step::kRows, ka = k0 + g * Step::kLaneRows;
    const bool k_ok = ka < args.Kd;  // (the contraction is whole 16-byte chunks: a lane's rows are all there, or none)
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      aw[b] = (u32x4){0, 0, 0, 0};
      if (a_ok[b] && k_ok) aw[b] = *(const u32x4 *)(Ap[b] + k0);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int col = Step::load_column(c16, i);
      u32x4 v = {0, 0, 0, 0};
      if (slab0 + col < args.Nd && k_ok)
        v = __builtin_nontemporal_load((const u32x4 *)(Bp + (long long)(ka + Step::load_row(i)) * args.Nd + col));
      bw[i] = v;
    }
  };

  // steps wave, wave + WAVES, ... ; DEPTH in flight (the loop is unrolled by DEPTH, so the buffers are fixed registers)
  int step = first_step + wave;
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (step + d * WAVES < n_steps) fetch(step + d * WAVES, bw[d], aw[d]);
  for (bool more = step < n_steps; more;) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (more) {
        if (step + (DEPTH - 1) * WAVES < n_steps)
          fetch(step + (DEPTH - 1) * WAVES, bw[(d + DEPTH - 1) % DEPTH], aw[(d + DEPTH - 1) % DEPTH]);
        Step::template multiply<RB>(bw[d], aw[d], acc);
        step += WAVES;
        more = step < n_steps;
      }
    }
  }

  // ---- reduce the partial sums of the waves, one block of 16 rows after the other -------------------------------
  const bool finishes = WAVES == kStreamWaves || wave < kStreamWaves;
  const int col = slab0 + Step::column(c16, 2 * (wave % kStreamWaves));  // wave w finishes accumulators 2w and 2w+1: one (gate, up) pair per lane
  const bool col_ok = finishes && col < args.Nd;
  float b0 = 0.f, b1 = 0.f;
  if (col_ok && args.bias != nullptr) {
    const T *bp = (const T *)args.bias + (long long)expert * args.Nd + col;
    b0 = ElemTraits<T>::to_f32(bp[0]);
    b1 = ElemTraits<T>::to_f32(bp[1]);
  }
  float sum[RB][2][4];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    // eight waves: the last four hand their sums to the first four
    if constexpr (WAVES > kStreamWaves) {
      if (!finishes) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) red[(((wave - kStreamWaves) * 8 + j) * 4 + v) * kWave + lane] = acc[b][j][v];
      }
      __syncthreads();
      if (finishes) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[b][j][v] += red[((wave * 8 + j) * 4 + v) * kWave + lane];
      }
      __syncthreads();
    }
    if (finishes) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[((wave * 8 + j) * 4 + v) * kWave + lane] = acc[b][j][v];
    }
    __syncthreads();
    if (finishes) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float t = 0.f;
#pragma unroll
          for (int w = 0; w < kStreamWaves; ++w) t += red[((w * 8 + 2 * wave + jj) * 4 + v) * kWave + lane];
          sum[b][jj][v] = t;
        }
    }
    if (b + 1 < RB || parts > 1) __syncthreads();  // the next block (or the count below) reuses the buffer
  }

  if (parts > 1) {
    // Device-scope accesses, written through and read past the L2 of the XCD: the parts of a slab may run on different ones.
    float *mine = args.partial + ((long long)item * parts + part) * args.part_floats + tid;
    auto at = [](int b, int jj, int v) { return ((b * 2 + jj) * 4 + v) * kStreamThreads; };
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (col_ok && 16 * b + g * 4 + v < rows) {
          __hip_atomic_store(mine + at(b, 0, v), sum[b][0][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(mine + at(b, 1, v), sum[b][1][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part has arrived; after the barrier, everybody's
    __syncthreads();
    if (tid == 0) {
      const int before = __hip_atomic_fetch_add(args.arrivals + item, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *(int *)red = before;
      if (before == parts - 1) __hip_atomic_store(args.arrivals + item, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (*(int *)red != parts - 1 || !finishes) return;
    asm volatile("" ::: "memory");
    const float *all = args.partial + (long long)item * parts * args.part_floats + tid;
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v) sum[b][0][v] = sum[b][1][v] = 0.f;
    constexpr int kAtOnce = 4;  // parts requested together: one trip to memory for each so many
    for (int p0 = 0; p0 < parts; p0 += kAtOnce) {
      float t[kAtOnce][RB][2][4];
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i)
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            t[i][b][0][v] = t[i][b][1][v] = 0.f;
            if (p0 + i < parts && 16 * b + v < rows) {  // (the same for every lane; what lies past the rows is not used)
              const float *from = all + (long long)(p0 + i) * args.part_floats;
              t[i][b][0][v] = __hip_atomic_load(from + at(b, 0, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              t[i][b][1][v] = __hip_atomic_load(from + at(b, 1, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
          }
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i)
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int v = 0; v < 4; ++v) { sum[b][0][v] += t[i][b][0][v]; sum[b][1][v] += t[i][b][1][v]; }
    }
  }

  if (!col_ok) return;
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 16 * b + g * 4 + v;
      if (r >= rows) continue;
      const long long orow = first + r;
      const float x0 = sum[b][0][v] + b0, x1 = sum[b][1][v] + b1;
      if (GLU) {
        ((T *)args.C)[orow * args.ldc + (col >> 1)] = ElemTraits<T>::from_f32(glu_forward(x0, x1));
        if (args.C2 != nullptr) {
          T *P = (T *)args.C2 + orow * args.Nd + col;
          P[0] = pre_activation_store<T>(x0, false);
          P[1] = pre_activation_store<T>(x1, true);
        }
      } else {
        T *O = (T *)args.C + orow * args.ldc + col;
        O[0] = ElemTraits<T>::from_f32(x0);
        O[1] = ElemTraits<T>::from_f32(x1);
      }
    }
}

}  // namespace yamoe
