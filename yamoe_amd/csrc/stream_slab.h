// The weight-streaming product of one (expert, 128-column slab): see stream.hip for the design.  A header of its own because
// the tile kernels' launches carry streamed experts as well (gemm_async_tile.h).
#pragma once

#include "common.h"

namespace yamoe {

constexpr int kStreamWaves = 4;        // waves that finish a slab; a workgroup has 4 or 8
constexpr int kSlabCols = 128;

typedef float f32x4v __attribute__((ext_vector_type(4)));

template <typename T> struct Mma16;
template <> struct Mma16<bf16_t> {
  __device__ static inline f32x4v run(const u32x4 &a, const u32x4 &b, f32x4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  }
};
template <> struct Mma16<f16_t> {
  __device__ static inline f32x4v run(const u32x4 &a, const u32x4 &b, f32x4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
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
  FastDiv a_div;
  int Kd, Nd, lda, ldc, n_slabs, N, E;
};

// One (expert, slab) of RB blocks of 16 rows (RB = 1: up to 16 rows, RB = 2: 17 to 32): the weights are fetched once
// and every column operand built from them goes through RB MFMAs.
template <typename T, bool GLU, bool GATHER, int WAVES, int DEPTH, int RB>
__device__ inline void stream_slab(const StreamArgs &args, float *red, const int expert, const int first, const int rows,
                                   const int slab) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const int col0 = slab * kSlabCols + c16 * 8;  // first of this lane's 8 output columns
  const bool col_ok = col0 < args.Nd;
  const T *Bp = (const T *)args.B + (long long)expert * args.Kd * args.Nd + col0;

  // A operand of block b: row 16 b + c16 of the expert (zero beyond `rows`), 8 consecutive k starting at 8 g
  bool a_ok[RB];
  const T *Ap[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    a_ok[b] = 16 * b + c16 < rows;
    long long a_src = first + (a_ok[b] ? 16 * b + c16 : 0);
    // (a gathering instantiation without a row list reads its rows in order, like the tile kernels)
    if (GATHER && args.a_rows != nullptr) a_src = fast_div(args.a_rows[a_src], args.a_div);
    Ap[b] = (const T *)args.A + a_src * args.lda + g * 8;
  }

  f32x4v acc[RB][8];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[b][j] = (f32x4v){0.f, 0.f, 0.f, 0.f};

  const int n_steps = (args.Kd + 31) / 32;
  u32x4 bw[DEPTH][8], aw[DEPTH][RB];

  auto fetch = [&](int step, u32x4 (&bw)[8], u32x4 (&aw)[RB]) {
    int k0 = step * 32;
    int ka = k0 + g * 8;
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      aw[b] = (u32x4){0, 0, 0, 0};
      if (a_ok[b] && ka < args.Kd) aw[b] = *(const u32x4 *)(Ap[b] + k0);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      int k = ka + i;
      u32x4 v = {0, 0, 0, 0};
      if (col_ok && k < args.Kd) v = __builtin_nontemporal_load((const u32x4 *)(Bp + (long long)k * args.Nd));
      bw[i] = v;
    }
  };
  auto consume = [&](const u32x4 (&bw)[8], const u32x4 (&aw)[RB]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
      u32x4 col;
#pragma unroll
      for (int d = 0; d < 4; ++d) col[d] = __builtin_amdgcn_perm(bw[2 * d + 1][j >> 1], bw[2 * d][j >> 1], sel);
#pragma unroll
      for (int b = 0; b < RB; ++b) acc[b][j] = Mma16<T>::run(aw[b], col, acc[b][j]);
    }
  };

  // steps wave, wave + WAVES, ... ; DEPTH in flight (the loop is unrolled by DEPTH, so the buffers are fixed registers)
  int step = wave;
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (step + d * WAVES < n_steps) fetch(step + d * WAVES, bw[d], aw[d]);
  for (bool more = step < n_steps; more;) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (more) {
        if (step + (DEPTH - 1) * WAVES < n_steps) fetch(step + (DEPTH - 1) * WAVES, bw[(d + DEPTH - 1) % DEPTH], aw[(d + DEPTH - 1) % DEPTH]);
        consume(bw[d], aw[d]);
        step += WAVES;
        more = step < n_steps;
      }
    }
  }

  // ---- reduce the partial sums and finish, one block of 16 rows after the other -------------------------------
  const int col = col0 + 2 * wave;  // wave w (of the first four) finishes accumulator columns j = 2w, 2w+1: one (gate, up) pair per lane
  float b0 = 0.f, b1 = 0.f;
  if (wave < kStreamWaves && col_ok && args.bias != nullptr) {
    const T *bp = (const T *)args.bias + (long long)expert * args.Nd + col;
    b0 = ElemTraits<T>::to_f32(bp[0]);
    b1 = ElemTraits<T>::to_f32(bp[1]);
  }
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    // more than four waves: waves 4r .. 4r+3 hand their sums to waves 0 .. 3, one group after the other (a fixed order)
    for (int r = 1; r < WAVES / kStreamWaves; ++r) {
      if (wave / kStreamWaves == r) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) red[(((wave - kStreamWaves * r) * 8 + j) * 4 + v) * kWave + lane] = acc[b][j][v];
      }
      __syncthreads();
      if (wave < kStreamWaves) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[b][j][v] += red[((wave * 8 + j) * 4 + v) * kWave + lane];
      }
      __syncthreads();
    }
    if (wave < kStreamWaves) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[((wave * 8 + j) * 4 + v) * kWave + lane] = acc[b][j][v];
    }
    __syncthreads();
    if (wave < kStreamWaves && col_ok) {
      float sum[2][4];
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float t = 0.f;
#pragma unroll
          for (int w = 0; w < kStreamWaves; ++w) t += red[((w * 8 + 2 * wave + jj) * 4 + v) * kWave + lane];
          sum[jj][v] = t;
        }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        int r = 16 * b + g * 4 + v;
        if (r >= rows) continue;
        long long orow = first + r;
        float x0 = sum[0][v] + b0, x1 = sum[1][v] + b1;
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
    if (b + 1 < RB) __syncthreads();  // the next block reuses the buffer
  }
}

}  // namespace yamoe
