// The step before the expert layer: router linear -> top-k -> softmax over the selected logits -> dense scores
// (torch-ext/yamoe/layers.py:128-152, torch-ext/yamoe/vendored/gpt_oss_mlp.py:128-142), in one kernel, and the
// gradient of that step.
//
// A workgroup takes 32 tokens.  logits[32, E] = x[32, H] * W[E, H]^T: both operands are k-contiguous in memory,
// which is exactly the register layout of the 32x32x16 MFMA operands (lane l holds 8 consecutive k of row l % 32,
// starting at 8 * (l / 32)), so a fragment is one 16-byte read.  (fp32: a lane's
// 16 bytes are 4 consecutive k starting at 4 * (l / 32), fed to four v_mfma_f32_32x32x2_f32, whose two lane halves are
// the two k of an instruction: any pairing of k values is fine as long as both operands use the same.)  Four waves
// split the contraction of a block of 32 experts, their partial tiles meet in LDS, the bias is added and the logits are
// rounded to the activation dtype as the reference's linear does.  Then the lanes of a token pick the top-k together (ties: lowest
// expert id first) and the softmax of the k picked values is computed in fp32, rounded once, and written into the dense
// [T, E] score row (zero elsewhere).
#include <type_traits>

#include "common.h"

namespace yamoe {

constexpr int kRouterTokens = 32;
constexpr int kRouterThreads = 256;
constexpr int kRouterMaxE = 256;
constexpr int kRouterMaxK = 16;
constexpr int kRouterCus = 256;

template <typename T> struct RouterMma;
template <> struct RouterMma<bf16_t> {
  __device__ static inline void run(const u32x4 &a, const u32x4 &b, f32x16 &c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct RouterMma<f16_t> {
  __device__ static inline void run(const u32x4 &a, const u32x4 &b, f32x16 &c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct RouterMma<float> {
  __device__ static inline void run(const u32x4 &a, const u32x4 &b, f32x16 &c) {
    const f32x4 af = __builtin_bit_cast(f32x4, a), bf = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int q = 0; q < 4; ++q) c = __builtin_amdgcn_mfma_f32_32x32x2f32(af[q], bf[q], c, 0, 0, 0);
  }
};

// NB = number of 32-expert column blocks (E <= 32 * NB), WB = how many of them a wave computes.  A workgroup has
// 4 * NB / WB waves: in every chunk of the contraction (128 bytes of a row, four steps) wave w takes step w % 4 of the
// blocks starting at (w / 4) * WB, so every logit is summed in the same order whatever NB is.
//
// What bounds it is getting the operands in: a workgroup reads its 32 token rows and all E weight rows, 32 * (1 + NB) * 128
// bytes per chunk against a handful of MFMAs.  The chunks come in by asynchronous copies of whole 128-byte pieces, eight
// rows per instruction, into a ring of S stages of G chunks each (S - 1 stages on their way while one is used).  Fragments
// fetched straight from global memory touch 32 cache lines per instruction for 32 bytes of each, which the L1's tag rate
// holds at 30 us for one token and 58 us for 8192 on a [128, 2880] router (17.7 and 20.1 us this way).
//
// With few experts that tag rate is no limit (lanes of the same row share their lines), and what counts is the wave's own
// chain from stage to stage: wait, barrier, copies, LDS read, MFMA, about 500 clocks however little a stage holds.  Hence
// G: up to 64 experts a stage is several chunks.  [E, 2880] bf16, top-2, us by fragments from global memory / stages of one
// chunk / now: 1 token, 8 experts 9.8 / 13.9 / 8.3, 32 experts 13.3 / 13.8 / 8.6; fp32, 2048 tokens, 8 experts 26.6 / 33.7 / 21.9.
// The form of up to 32 experts with most in flight fills a CU's LDS; where there are more workgroups than CUs, small rings of which
// five share a CU are the better ones (32768 tokens, 8 experts, 1024 wide bf16: 25.3 / 14.2; 2048 tokens: 6.0 / 7.2).  Up
// to 64 experts two share a CU (40 experts, 32768 tokens, 1024 wide fp32: 58.8 by fragments, 64.6 with one per CU, 52.8 now).
//
// The pick is made by the lanes of the token together: L = 8 * NB / WB lanes hold 32 * NB / L consecutive logits each in
// registers, and every round is a maximum over the lane's own values followed by log2(L) exchanges.  (One thread per
// token walking its row in LDS, the picks in scratch memory, took 90 of the kernel's 103 us at 1536 tokens of 2048 values,
// 64 experts, top-8, which takes 13.3 us now.)
template <int NB, int G_, int S_> struct RouterRing {
  static constexpr int G = G_, S = S_;
  static constexpr int kRows = kRouterTokens + 32 * NB;
  static constexpr int kChunk = kRows * 128;
  static constexpr int kStage = G * kChunk, kBytes = S * kStage;
  static constexpr int kLd = 32 * NB + 1;                  // padded row of the logits tile, which takes the ring's place
  static_assert(kRouterTokens * kLd * 4 <= kBytes && kBytes <= 160 * 1024, "the logits tile fits the ring, the ring a CU");
};

// a logit as an unsigned number in the same order (equal floats give equal numbers: -0 becomes +0 first); every NaN is the
// largest, whatever its sign, as in torch.topk; 0 is below all
__device__ inline uint32_t router_order(float v) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v + 0.0f);
  return v != v ? 0xffffffffu : (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ inline float router_unorder(uint32_t o) {
  return __builtin_bit_cast(float, (o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

template <typename T, int NB, int WB, class R>
__global__ __launch_bounds__(kRouterThreads *NB / WB) void router_topk_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                                     const T *__restrict__ bias, int Tn, int H, int E, int K,
                                                                     long long *__restrict__ indices, T *__restrict__ scores,
                                                                     T *__restrict__ topk_weights, T *__restrict__ logits_out) {
  constexpr int kThreads = kRouterThreads * NB / WB, kWaves = kThreads / kWave;
  constexpr int kLd = R::kLd, S = R::S, G = R::G;
  extern __shared__ __attribute__((aligned(16))) char ring[];
  float *tile = (float *)ring;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kq = wave & 3, nb0 = (wave >> 2) * WB;
  const int rl = lane & 31, g = lane >> 5;
  const int t0 = blockIdx.x * kRouterTokens;

  f32x16 acc[WB];
#pragma unroll
  for (int nb = 0; nb < WB; ++nb)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[nb][v] = 0.0f;

  // Copies: copy q of a chunk brings rows 8 q + lane / 8 of it (32 token rows, then the weight rows), 16 bytes per
  // lane; position lane % 8 of row r holds piece pos ^ ((r >> 1) & 7), so that 32 lanes reading one piece of 32 rows touch
  // every bank.  Wave w issues copies w, w + kWaves, ...  Rows past the end re-read the last valid one, pieces and
  // chunks past the end of a row its first; their products are never used.
  constexpr int kCopies = R::kRows / 8, kPerWave = (kCopies + kWaves - 1) / kWaves;
  constexpr int kFewer = kPerWave * kWaves - kCopies;  // the last kFewer waves issue one copy less
  const bool fewer = wave >= kWaves - kFewer;
  const int row_bytes = H * (int)sizeof(T);
  const char *src[kPerWave];
#pragma unroll
  for (int i = 0; i < kPerWave; ++i) {
    const int row = 8 * (wave + i * kWaves) + (lane >> 3);
    src[i] = row < kRouterTokens ? (const char *)x + (long long)min(t0 + row, Tn - 1) * row_bytes
                                 : (const char *)w + (long long)min(row - kRouterTokens, E - 1) * row_bytes;
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)ring);
  auto issue = [&](int group, int stage) {
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int i = 0; i < kPerWave; ++i) {
        if (i == kPerWave - 1 && fewer) break;
        const int row = 8 * (wave + i * kWaves) + (lane >> 3);
        int at = (group * G + j) * 128 + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
        if (at >= row_bytes) at = 0;
        copy16_to_lds(src[i] + at, lds0 + (uint32_t)(stage * R::kStage + j * R::kChunk + 8 * (wave + i * kWaves) * 128));
      }
  };
  // every copy but those of the youngest `groups` has landed
  auto wait_but = [&](auto groups) {
    constexpr int C = decltype(groups)::value * G;
    if (kFewer > 0 && fewer) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C * (kPerWave - 1)) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C * kPerWave) : "memory");
  };
  const int n_steps = row_bytes / 32, n_groups = (n_steps + 4 * G - 1) / (4 * G);
  const int rd = rl * 128 + (((2 * kq + g) ^ ((rl >> 1) & 7)) << 4);
  auto use = [&](int group, int stage) {
    const char *st = ring + stage * R::kStage + rd;
    u32x4 fa[G], fb[G][WB];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      fa[j] = *(const u32x4 *)(st + j * R::kChunk);
#pragma unroll
      for (int nb = 0; nb < WB; ++nb) fb[j][nb] = *(const u32x4 *)(st + j * R::kChunk + (1 + nb0 + nb) * 4096);
    }
#pragma unroll
    for (int j = 0; j < G; ++j)
      if (4 * (group * G + j) + kq < n_steps) {
#pragma unroll
        for (int nb = 0; nb < WB; ++nb) RouterMma<T>::run(fa[j], fb[j][nb], acc[nb]);
      }
  };
#pragma unroll
  for (int c = 0; c < S - 1; ++c)
    if (c < n_groups) issue(c, c);
  int c = 0, stage = 0;
  for (; c + S - 1 < n_groups; ++c) {
    wait_but(std::integral_constant<int, S - 2>());
    __syncthreads();  // group c is there for every wave, and nobody reads the stage of group c - 1 any more
    const int free_stage = stage == 0 ? S - 1 : stage - 1;
    issue(c + S - 1, free_stage);
    use(c, stage);
    stage = stage == S - 1 ? 0 : stage + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (; c < n_groups; ++c) {
    use(c, stage);
    stage = stage == S - 1 ? 0 : stage + 1;
  }
  __syncthreads();  // the ring is dead: the logits tile takes its place
  // acc[nb][v]: token 8 * (v / 4) + 4 * g + v % 4, expert (nb0 + nb) * 32 + rl; the four waves of a block add up in LDS,
  // one after another
  for (int turn = 0; turn < 4; ++turn) {
    if (kq == turn) {
#pragma unroll
      for (int nb = 0; nb < WB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          float *at = tile + (8 * (v >> 2) + 4 * g + (v & 3)) * kLd + (nb0 + nb) * 32 + rl;
          *at = turn == 0 ? acc[nb][v] : *at + acc[nb][v];
        }
    }
    __syncthreads();
  }

  // The L lanes of token r take its logits M * sub .. M * sub + M - 1: bias, rounding to the activation dtype (the value
  // the reference's top-k sees), and the sortable form; experts past the end are 0, below every logit.
  constexpr int L = kThreads / kRouterTokens, M = 32 * NB / L;
  const int r = tid / L, sub = tid % L;
  const long long t = t0 + r;
  uint32_t key[M];
  float prob[M];
#pragma unroll
  for (int j = 0; j < M; ++j) {
    const int e = sub * M + j;
    key[j] = 0u;
    prob[j] = 0.0f;
    if (e < E) {
      const T q = ElemTraits<T>::from_f32(tile[r * kLd + e] + (bias != nullptr ? ElemTraits<T>::to_f32(bias[e]) : 0.0f));
      key[j] = router_order(ElemTraits<T>::to_f32(q));
      if (logits_out != nullptr && t < Tn) logits_out[t * E + e] = q;
    }
  }
  float first = 0.0f, sum = 0.0f;
  float mine[kRouterMaxK / 8] = {};  // lane `sub` keeps the weights of picks sub and (8 lanes per token) sub + 8
  for (int k = 0; k < K; ++k) {
    uint32_t best = 0u;
    int at = 0;
#pragma unroll
    for (int j = 0; j < M; ++j)
      if (key[j] > best) { best = key[j]; at = sub * M + j; }
#pragma unroll
    for (int d = 1; d < L; d <<= 1) {
      const uint32_t other = (uint32_t)__shfl_xor((int)best, d);
      const int other_at = __shfl_xor(at, d);
      // ties: the lower expert id (the lower lane holds the lower ids)
      if (other > best || (other == best && other_at < at)) { best = other; at = other_at; }
    }
    const float v = router_unorder(best);
    if (k == 0) first = v;
    const float p = expf(v - first);
    sum += p;
#pragma unroll
    for (int j = 0; j < M; ++j)
      if (at == sub * M + j) { key[j] = 0u; prob[j] = p; }
#pragma unroll
    for (int i = 0; i < kRouterMaxK / 8; ++i)
      if (k == sub + i * L) mine[i] = p;
    if (sub == 0 && t < Tn) indices[t * K + k] = at;
  }
  if (t >= Tn) return;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    const int e = sub * M + j;
    // (a key of 0 is a pick; the others divide nothing, as the sum may not be finite)
    if (e < E) scores[t * E + e] = ElemTraits<T>::from_f32(key[j] != 0u ? 0.0f : prob[j] / sum);
  }
  if (topk_weights != nullptr) {
#pragma unroll
    for (int i = 0; i < kRouterMaxK / 8; ++i)
      if (sub + i * L < K) topk_weights[t * K + sub + i * L] = ElemTraits<T>::from_f32(mine[i] / sum);
  }
}

template <typename T, int NB, int WB, int G, int S>
static int launch_router(const void *x, const void *w, const void *bias, int Tn, int H, int E, int K, long long *indices,
                         void *scores, void *topk_weights, void *logits, hipStream_t stream) {
  typedef RouterRing<NB, G, S> R;
  auto kernel = router_topk_kernel<T, NB, WB, R>;
  static DeviceFlags attr_done;  // one per kernel instantiation
  if (int rc = ensure_dynamic_lds((const void *)kernel, R::kBytes, attr_done, "router_topk_kernel")) return rc;
  hipLaunchKernelGGL(kernel, dim3(ceil_div(Tn, kRouterTokens)), dim3(kRouterThreads * NB / WB), R::kBytes, stream,
                     (const T *)x, (const T *)w, (const T *)bias, Tn, H, E, K, indices, (T *)scores, (T *)topk_weights,
                     (T *)logits);
  return check_launch("router_topk_kernel");
}

template <typename T>
static int router_dispatch(const void *x, const void *w, const void *bias, int Tn, int H, int E, int K, long long *indices,
                           void *scores, void *topk_weights, void *logits, hipStream_t stream) {
  const int nb = ceil_div(E, 32);
  if (nb <= 1) {  // 128 KB of LDS while a CU has one workgroup at most, 32 KB where several should share it
    if (Tn <= kRouterTokens * kRouterCus) return launch_router<T, 1, 1, 8, 2>(x, w, bias, Tn, H, E, K, indices, scores, topk_weights, logits, stream);
    return launch_router<T, 1, 1, 2, 2>(x, w, bias, Tn, H, E, K, indices, scores, topk_weights, logits, stream);
  }
  if (nb <= 2) return launch_router<T, 2, 1, 2, 3>(x, w, bias, Tn, H, E, K, indices, scores, topk_weights, logits, stream);  // 72 KB
  if (nb <= 4) return launch_router<T, 4, 1, 1, 6>(x, w, bias, Tn, H, E, K, indices, scores, topk_weights, logits, stream);  // 120 KB
  return launch_router<T, 8, 2, 1, 4>(x, w, bias, Tn, H, E, K, indices, scores, topk_weights, logits, stream);  // 144 KB
}

// ---- gradient of the step, first part: from the gradient of the dense scores to the gradient of the logits --------
// With p_k the softmax weights of the token's K picks (the scores the forward stored) and
// g_k = d_scores[t, pick_k]:  d_logits[t, pick_k] = p_k * (g_k - sum_j p_j g_j), zero for every other expert: what
// autograd gives through scatter, softmax over the K picked logits and top-k (torch-ext/yamoe/layers.py:136-149).
// 16 lanes per token: lane k holds pick k (of 16 at a time), every lane adds the picks up in their order and writes every
// 16th expert, so that the row is stored once.  It is bound by the three dependent fetches of a token; with one thread per
// token, which also walked its row storing zeros, 1536 tokens of 64 experts, top-8, took 13.9 us (5.3 now).
constexpr int kPickLanes = 16;
template <typename T>
__global__ __launch_bounds__(256) void router_backward_logits_kernel(const T *__restrict__ d_scores,
                                                                     const long long *__restrict__ indices,
                                                                     const T *__restrict__ scores, int Tn, int E, int K,
                                                                     T *__restrict__ d_logits) {
  const int l = threadIdx.x & (kPickLanes - 1);
  const long long t = (long long)blockIdx.x * (256 / kPickLanes) + threadIdx.x / kPickLanes;
  if (t >= Tn) return;  // (all lanes of a token together)
  int pick = -1;
  float p = 0.0f, g = 0.0f;  // (an index outside the experts adds nothing and is written nowhere)
  auto fetch = [&](int k0) {
    const int k = k0 + l;
    const long long e = k < K ? indices[t * K + k] : -1;
    const bool ok = e >= 0 && e < E;
    pick = ok ? (int)e : -1;
    p = ok ? ElemTraits<T>::to_f32(scores[t * E + e]) : 0.0f;
    g = ok ? ElemTraits<T>::to_f32(d_scores[t * E + e]) : 0.0f;
  };
  float inner = 0.0f;
  for (int k0 = 0; k0 < K; k0 += kPickLanes) {
    fetch(k0);
    for (int j = 0; j < min(kPickLanes, K - k0); ++j) inner += __shfl(p, j, kPickLanes) * __shfl(g, j, kPickLanes);
  }
  for (int e0 = 0; e0 < E; e0 += kPickLanes) {
    float v = 0.0f;
    for (int k0 = 0; k0 < K; k0 += kPickLanes) {
      if (K > kPickLanes) fetch(k0);
      for (int j = 0; j < min(kPickLanes, K - k0); ++j) {
        const float pj = __shfl(p, j, kPickLanes), gj = __shfl(g, j, kPickLanes);
        if (__shfl(pick, j, kPickLanes) == e0 + l) v = pj * (gj - inner);
      }
    }
    if (e0 + l < E) d_logits[t * E + e0 + l] = ElemTraits<T>::from_f32(v);
  }
}

template <typename T>
int launch_router_backward_logits(const void *d_scores, const long long *indices, const void *scores, int Tn, int E, int K,
                                  void *d_logits, hipStream_t stream) {
  hipLaunchKernelGGL(router_backward_logits_kernel<T>, dim3(ceil_div(Tn, 256 / kPickLanes)), dim3(256), 0, stream,
                     (const T *)d_scores, indices, (const T *)scores, Tn, E, K, (T *)d_logits);
  return check_launch("router_backward_logits_kernel");
}
template int launch_router_backward_logits<float>(const void *, const long long *, const void *, int, int, int, void *, hipStream_t);
template int launch_router_backward_logits<bf16_t>(const void *, const long long *, const void *, int, int, int, void *, hipStream_t);
template int launch_router_backward_logits<f16_t>(const void *, const long long *, const void *, int, int, int, void *, hipStream_t);

// ---- second part, 16-bit data: d_weight[E, H] = d_logits^T . hidden and d_bias = column sums of d_logits ----------
// A product with a small result and a long contraction (the tokens), so it is bound by the latency of walking the tokens
// and the walk is what is split: a workgroup owns 64 experts x 32 columns, its 16 waves take every 16th slab of 32 tokens,
// each through a staging area of its own (no workgroup barrier before the end, the next slab's rows on their way while one
// is multiplied), and their fp32 partial tiles meet in LDS in the order of the waves.  Partial sums that stay inside the
// workgroup need neither workspace nor a second launch, and 32 columns give 64 to 90 workgroups at widths of 2048 to 2880.
// Both operands are [token][.] in memory and in LDS and are read with the LDS transpose read (see common.h); the
// bias gradient is summed from the same operand registers by the workgroups of the first columns.  1536 tokens, 64 experts,
// H = 2048: 8.7 us; on eight 256 x 256 tiles that each walked all tokens 59 us, and 19 to 42 us more in a launch for the bias.
constexpr int kRwWaves = 16, kRwThreads = kRwWaves * kWave, kRwSlab = 32, kRwExperts = 64, kRwCols = 32;
constexpr int kRwDRow = kRwExperts * 2 + 16, kRwXRow = kRwCols * 2 + 16;     // bytes of a staged row (padded)
constexpr int kRwStage = kRwSlab * (kRwDRow + kRwXRow);                      // staging bytes of a wave
constexpr int kRwPart = kRwExperts * kRwCols * (int)sizeof(float);           // partial tile of a wave (over the staging)
constexpr int kRwBias = kRwWaves * kRwPart;                                  // partial bias sums, behind both
constexpr int kRwLds = kRwBias + kRwWaves * kRwExperts * (int)sizeof(float);
static_assert(kRwStage <= kRwPart, "the staging areas end where the bias sums start");

// four k rows `row_bytes` apart, twice: the eight consecutive k of this lane's row of a 32 x 32 x 16 operand
__device__ inline u32x4 rw_operand(const char *p, int row_bytes) {
  const u32x2 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 4 * row_bytes);
  return (u32x4){lo[0], lo[1], hi[0], hi[1]};
}

template <typename T>
__global__ __launch_bounds__(kRwThreads) void router_weight_grad_kernel(const T *__restrict__ d_logits,
                                                                        const T *__restrict__ hidden, int Tn, int H, int E,
                                                                        T *__restrict__ d_weight, T *__restrict__ d_bias) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * kRwCols, e0 = blockIdx.y * kRwExperts;
  const int n_slabs = (Tn + kRwSlab - 1) / kRwSlab;
  const bool sums_bias = d_bias != nullptr && blockIdx.x == 0;
  char *const ds = lds + wave * kRwStage, *const xs = ds + kRwSlab * kRwDRow;

  // this lane's pieces of a slab: d_logits rows (lane >> 3) + 8 i, 16 bytes at lane & 7; hidden rows (lane >> 2) + 16 i, at
  // lane & 3.  Tokens, experts and columns past the end are zeros.
  const int dp = lane & 7, xp = lane & 3;
  const bool d_in = e0 + dp * 8 < E, x_in = n0 + xp * 8 < H;
  u32x4 draw[4], xraw[2];
  auto fetch = [&](int slab) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const long long t = (long long)slab * kRwSlab + (lane >> 3) + 8 * i;
      draw[i] = (u32x4){0, 0, 0, 0};
      if (d_in && t < Tn) draw[i] = *(const u32x4 *)(d_logits + t * E + e0 + dp * 8);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const long long t = (long long)slab * kRwSlab + (lane >> 2) + 16 * i;
      xraw[i] = (u32x4){0, 0, 0, 0};
      if (x_in && t < Tn) xraw[i] = *(const u32x4 *)(hidden + t * H + n0 + xp * 8);
    }
  };

  f32x16 acc[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[b][v] = 0.0f;
  float bias[2] = {0.0f, 0.0f};
  const int g = lane >> 5, rl = lane & 31, j4 = (lane & 15) >> 2, q4 = lane & 3;
  const int col = (16 * ((lane >> 4) & 1) + 4 * q4) * 2;
  if (wave < n_slabs) fetch(wave);
  for (int s = wave; s < n_slabs; s += kRwWaves) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *(u32x4 *)(ds + ((lane >> 3) + 8 * i) * kRwDRow + dp * 16) = draw[i];
#pragma unroll
    for (int i = 0; i < 2; ++i) *(u32x4 *)(xs + ((lane >> 2) + 16 * i) * kRwXRow + xp * 16) = xraw[i];
    if (s + kRwWaves < n_slabs) fetch(s + kRwWaves);
    // (one wave's LDS operations are carried out in order: nothing to wait for between its stores and its reads)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const u32x4 fx = rw_operand(xs + (ks * 16 + g * 8 + j4) * kRwXRow + col, kRwXRow);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const u32x4 fd = rw_operand(ds + (ks * 16 + g * 8 + j4) * kRwDRow + b * 64 + col, kRwDRow);
        RouterMma<T>::run(fd, fx, acc[b]);
        if (sums_bias) {
          const T *h = (const T *)&fd;
#pragma unroll
          for (int j = 0; j < 8; ++j) bias[b] += ElemTraits<T>::to_f32(h[j]);
        }
      }
    }
    asm volatile("" ::: "memory");
  }

  __syncthreads();  // (the partial tiles lie over the staging areas)
  // acc[b][v]: expert b*32 + 8*(v/4) + 4*g + v%4, column rl
  float *const part = (float *)(lds + wave * kRwPart), *const bias_part = (float *)(lds + kRwBias);
  if (wave < n_slabs) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) part[(b * 32 + 8 * (v >> 2) + 4 * g + (v & 3)) * kRwCols + rl] = acc[b][v];
    if (sums_bias) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const float sum = bias[b] + __shfl_xor(bias[b], 32);
        if (g == 0) bias_part[wave * kRwExperts + b * 32 + rl] = sum;
      }
    }
  }
  __syncthreads();
  const int n_parts = min(n_slabs, kRwWaves);
  {
    typedef T T2 __attribute__((ext_vector_type(2)));
    const int o = 2 * tid, e = e0 + o / kRwCols, c = n0 + (o & (kRwCols - 1));
    float s0 = 0.0f, s1 = 0.0f;
    for (int w = 0; w < n_parts; ++w) {
      s0 += ((const float *)(lds + w * kRwPart))[o];
      s1 += ((const float *)(lds + w * kRwPart))[o + 1];
    }
    if (e < E && c < H) *(T2 *)(d_weight + (long long)e * H + c) = (T2){ElemTraits<T>::from_f32(s0), ElemTraits<T>::from_f32(s1)};
  }
  if (sums_bias && tid < kRwExperts && e0 + tid < E) {
    float sum = 0.0f;
    for (int w = 0; w < n_parts; ++w) sum += bias_part[w * kRwExperts + tid];
    d_bias[e0 + tid] = ElemTraits<T>::from_f32(sum);
  }
}
static_assert(2 * kRwThreads == kRwExperts * kRwCols, "two outputs per thread");

// d_weight [E, H] and, if wanted, d_bias [E]; E and H multiples of 8
template <typename T>
int launch_router_weight_grad(const void *d_logits, const void *hidden, int Tn, int H, int E, void *d_weight, void *d_bias,
                              hipStream_t stream) {
  static DeviceFlags attr_done;  // one per kernel instantiation
  if (int rc = ensure_dynamic_lds((const void *)router_weight_grad_kernel<T>, kRwLds, attr_done, "router_weight_grad_kernel")) return rc;
  hipLaunchKernelGGL(router_weight_grad_kernel<T>, dim3(ceil_div(H, kRwCols), ceil_div(E, kRwExperts)), dim3(kRwThreads), kRwLds,
                     stream, (const T *)d_logits, (const T *)hidden, Tn, H, E, (T *)d_weight, (T *)d_bias);
  return check_launch("router_weight_grad_kernel");
}
template int launch_router_weight_grad<bf16_t>(const void *, const void *, int, int, int, void *, void *, hipStream_t);
template int launch_router_weight_grad<f16_t>(const void *, const void *, int, int, int, void *, void *, hipStream_t);

}  // namespace yamoe

using namespace yamoe;

extern "C" int yamoe_router_topk(const void *hidden, const void *weight, const void *bias, int32_t T_, int32_t H, int32_t E,
                                 int32_t K, int32_t dtype, int64_t *router_indices, void *router_scores, void *topk_weights,
                                 void *logits, void *stream) {
  const int step = dtype == YAMOE_F32 ? 8 : 16;
  if (T_ < 0 || H <= 0 || H % step != 0 || E <= 0 || E > kRouterMaxE || K <= 0 || K > kRouterMaxK || K > E) {
    set_error("yamoe_router_topk: need H %% %d == 0, 1 <= E <= %d, 1 <= top_k <= min(E, %d) (got H=%d E=%d top_k=%d)",
              step, kRouterMaxE, kRouterMaxK, H, E, K);
    return YAMOE_E_ARG;
  }
  if (T_ == 0) return 0;
  if (!hidden || !weight || !router_indices || !router_scores) {
    set_error("yamoe_router_topk: null pointer");
    return YAMOE_E_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case YAMOE_BF16:
      return router_dispatch<bf16_t>(hidden, weight, bias, T_, H, E, K, (long long *)router_indices, router_scores,
                                     topk_weights, logits, s);
    case YAMOE_F16:
      return router_dispatch<f16_t>(hidden, weight, bias, T_, H, E, K, (long long *)router_indices, router_scores,
                                    topk_weights, logits, s);
    case YAMOE_F32:
      return router_dispatch<float>(hidden, weight, bias, T_, H, E, K, (long long *)router_indices, router_scores,
                                    topk_weights, logits, s);
    default:
      set_error("yamoe_router_topk: unknown dtype %d", dtype);
      return YAMOE_E_DTYPE;
  }
}
