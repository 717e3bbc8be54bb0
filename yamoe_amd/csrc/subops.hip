// The public helper ops of drbh/yamoe (torch-ext/torch_binding.cpp:9-56) on the reference's own data
// layouts: `sort`, `bincount_cumsum`, `gather`, `scatter`, `index_select_out`.  (`batch_mm` is served by
// the grouped GEMM kernels, see cabi.hip.)  The fused forward does not use these: it keeps
// expert-contiguous buffers without padding.  They exist so that code written against the reference's
// helper ops keeps working, with the padded [E, C, H] buffers and inclusive `bins` it expects.
#include <type_traits>

#include "common.h"

namespace yamoe {

// ---- sort: stable LSD radix sort of integer keys with an iota payload (csrc/sort.cu:17-91) --------------
// 8-bit digits; one pass = per-wave segment histograms, a scan to per-(digit, segment) cursors, and an
// in-order placement with wavefront-ballot ranking, exactly the scheme of route.hip with 256 buckets.
constexpr int kSortThreads = 1024;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortSeg = 1024;  // elements per wave segment
constexpr int kRadix = 256;
constexpr int kScatterWaves = 16 * 256;    // waves that keep HBM busy in the scatter
// Slots that one workgroup indexes in one launch; beyond, a clearing launch and a grid.  Whole scatter, 1024 wide, bf16, us, one
// workgroup / grid, where launches queue up (or are replayed) and where each waits for the host: 4096 slots of 32 experts 9.2 / 7.9
// and 10.1 / 12.8, 5120 10.6 / 8.4 and 11.3 / 13.1, 6144 11.8 / 8.8 and 12.3 / 13.2; 4096 of 128 9.7 / 8.1 and 10.5 / 13.0, 5120
// 11.2 / 8.5 and 11.8 / 12.7, 6144 12.7 / 9.1 and 13.1 / 12.8; with the bins in global memory (2000 experts) 2048 9.0 / 8.0 and 9.7 /
// 12.6, 3072 11.8 / 8.7 and 12.2 / 12.9.  The search for a slot's expert takes longer the more there are, so the lines, where one
// caller's loss comes up to the other's gain, do too.
constexpr int kScatterLdsBins = 1024;  // up to this many experts the search for a position's expert runs in LDS
static int scatter_one_block(int E) { return E <= 32 ? 5120 : E <= kScatterLdsBins ? 4096 : 2048; }

template <typename K>
__device__ inline unsigned digit_of(K key, int shift, int bits, bool flip_sign) {
  typedef typename std::make_unsigned<K>::type U;
  U u = (U)key;
  if (flip_sign) u ^= (U)((U)1 << (sizeof(K) * 8 - 1));
  return (unsigned)((u >> shift) & (U)((1u << bits) - 1u));
}

template <typename K>
__global__ __launch_bounds__(kSortThreads) void sort_hist_kernel(const K *keys, int n, int shift, int bits,
                                                                 bool flip_sign, int *seg_counts) {
  __shared__ int hist[kSortWaves * kRadix];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < kSortWaves * kRadix; i += kSortThreads) hist[i] = 0;
  __syncthreads();
  long long seg = (long long)blockIdx.x * kSortWaves + wave;
  long long b = seg * kSortSeg, e = b + kSortSeg;
  if (e > n) e = n;
  for (long long i = b + lane; i < e; i += kWave) atomicAdd(&hist[wave * kRadix + digit_of(keys[i], shift, bits, flip_sign)], 1);
  __syncthreads();
  for (int i = tid; i < kSortWaves * kRadix; i += kSortThreads)
    seg_counts[(size_t)blockIdx.x * kSortWaves * kRadix + i] = hist[i];
}

// one block of 256 threads: thread d owns digit d
__global__ __launch_bounds__(kRadix) void sort_scan_kernel(int *seg_counts, int n_seg) {
  __shared__ int total[kRadix];
  const int d = threadIdx.x;
  int s = 0;
  for (int g = 0; g < n_seg; ++g) s += seg_counts[(size_t)g * kRadix + d];
  total[d] = s;
  __syncthreads();
  int base = 0;
  for (int j = 0; j < d; ++j) base += total[j];
  for (int g = 0; g < n_seg; ++g) {
    int c = seg_counts[(size_t)g * kRadix + d];
    seg_counts[(size_t)g * kRadix + d] = base;
    base += c;
  }
}

// Places keys b .. e-1, one wave, in order: `cursor` (LDS, of this wave alone) holds where each digit's next key goes.
template <typename K>
__device__ inline void sort_place_segment(const K *keys, const K *vals, bool iota_vals, long long b, long long e, int lane, int shift,
                                          int bits, bool flip_sign, int *cursor, K *keys_out, K *vals_out) {
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  // the next step's key and payload are fetched one step ahead (10 000 int32 keys of 8 bits: 14.5 us without, 13.9 with; int16:
  // 14.6 and 16.1, so those are fetched where they are used)
  constexpr bool AHEAD = sizeof(K) > 2;
  if (b >= e) return;
  K next_key = (K)0, next_val = (K)0;
  auto fetch = [&](long long i) {
    i = i < e ? i : e - 1;
    next_key = keys[i];
    next_val = iota_vals ? (K)i : vals[i];
  };
  if (AHEAD) fetch(b + lane);
  for (long long base = b; base < e; base += kWave) {
    long long i = base + lane;
    bool active = i < e;
    K key, val;
    if constexpr (AHEAD) {
      key = active ? next_key : (K)0;
      val = active ? next_val : (K)0;
      if (base + kWave < e) fetch(i + kWave);
    } else {
      key = active ? keys[i] : (K)0;
      val = active ? (iota_vals ? (K)i : vals[i]) : (K)0;
    }
    unsigned dg = digit_of(key, shift, bits, flip_sign);
    uint64_t peers = __ballot(active);
    for (int bit = 0; bit < bits; ++bit) {
      bool s = (dg >> bit) & 1;
      uint64_t m = __ballot(active && s);
      peers &= s ? m : ~m;
    }
    int rank = __popcll(peers & lt_mask);
    int start = 0;
    if (active) start = cursor[dg];
    __builtin_amdgcn_wave_barrier();
    if (active) {
      keys_out[start + rank] = key;
      vals_out[start + rank] = val;
      if (rank == 0) cursor[dg] = start + __popcll(peers);
    }
    // the cursor is private to this wave and LDS operations of one wave complete in order: the next step's
    // read sees this step's write without a fence or a volatile access (both would also wait for the global
    // stores above); lanes address the cursor by key, so the compiler cannot carry its values across steps
    __builtin_amdgcn_wave_barrier();
  }
}

template <typename K>
__global__ __launch_bounds__(kSortThreads) void sort_place_kernel(const K *keys, const K *vals, bool iota_vals, int n,
                                                                  int shift, int bits, bool flip_sign,
                                                                  const int *seg_cursors, K *keys_out, K *vals_out) {
  __shared__ int cursor_all[kSortWaves * kRadix];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < kSortWaves * kRadix; i += kSortThreads)
    cursor_all[i] = seg_cursors[(size_t)blockIdx.x * kSortWaves * kRadix + i];
  __syncthreads();
  int *cursor = cursor_all + wave * kRadix;
  long long seg = (long long)blockIdx.x * kSortWaves + wave;
  long long b = seg * kSortSeg, e = b + kSortSeg;
  if (e > n) e = n;
  sort_place_segment(keys, vals, iota_vals, b, e, lane, shift, bits, flip_sign, cursor, keys_out, vals_out);
}

// One pass over at most kSortWaves * kSortSeg keys, by one workgroup: each wave takes an equal contiguous segment, counts
// its digits in LDS, the counts become cursors, and the wave places its keys.  Three launches in one; each launch of the
// chain costs 4 us or more, whatever it does (4096 int32 keys of 4 bits: 25.0 us in three, 6.8 us in one).
template <typename K>
__global__ __launch_bounds__(kSortThreads) void sort_block_kernel(const K *keys, const K *vals, bool iota_vals, int n, int shift,
                                                                  int bits, bool flip_sign, K *keys_out, K *vals_out) {
  __shared__ int hist[kSortWaves * kRadix];
  __shared__ int group_total[kRadix / kWave];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < kSortWaves * kRadix; i += kSortThreads) hist[i] = 0;
  __syncthreads();
  const int seg = ceil_div(ceil_div(n, kSortWaves), kWave) * kWave;
  const int b = min(wave * seg, n), e = min(b + seg, n);
  int *cursor = hist + wave * kRadix;
  for (int i0 = b; i0 < e; i0 += 4 * kWave) {  // four loads on their way (positions past the end: the last key, not counted)
    std::conditional_t<sizeof(K) == 2, int, K> k[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u == 0 || i0 + u * kWave < e) k[u] = keys[min(i0 + u * kWave + lane, n - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + u * kWave + lane < e) atomicAdd(&cursor[digit_of((K)k[u], shift, bits, flip_sign)], 1);
  }
  __syncthreads();
  // thread d: keys of digit d in the waves before each one, then in all smaller digits
  int total = 0, before = 0;
  if (tid < kRadix) {
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      const int c = hist[w * kRadix + tid];
      hist[w * kRadix + tid] = total;
      total += c;
    }
    int sum;
    before = wave_exclusive_scan(total, sum);
    if (lane == 0) group_total[wave] = sum;
  }
  __syncthreads();
  if (tid < kRadix) {
    for (int g = 0; g < wave; ++g) before += group_total[g];
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) hist[w * kRadix + tid] += before;
  }
  __syncthreads();
  sort_place_segment(keys, vals, iota_vals, b, e, lane, shift, bits, flip_sign, cursor, keys_out, vals_out);
}

template <typename K>
__global__ void sort_copy_iota_kernel(const K *keys, K *keys_out, K *vals_out, int n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    keys_out[i] = keys[i];
    vals_out[i] = (K)i;
  }
}

template <typename K>
static int sort_impl(const void *x, int n, int end_bit, void *x_out, void *iota_out, void *ws, hipStream_t stream) {
  const int width = (int)sizeof(K) * 8;
  if (end_bit > width) end_bit = width;
  if (end_bit <= 0) {
    hipLaunchKernelGGL(sort_copy_iota_kernel<K>, dim3(ceil_div(n, 256)), dim3(256), 0, stream, (const K *)x, (K *)x_out,
                       (K *)iota_out, n);
    return check_launch("sort_copy_iota_kernel");
  }
  const int passes = ceil_div(end_bit, 8);
  const int n_blocks = ceil_div(ceil_div(n, kSortSeg), kSortWaves);
  const int n_seg = n_blocks * kSortWaves;
  K *tmp_k = (K *)ws;
  K *tmp_v = tmp_k + align_up((size_t)n, 64);
  int *seg_counts = (int *)(tmp_v + align_up((size_t)n, 64));
  // ping-pong so that the last pass writes x_out / iota_out
  const K *src_k = (const K *)x;
  const K *src_v = nullptr;
  for (int p = 0; p < passes; ++p) {
    bool to_out = ((passes - 1 - p) % 2) == 0;
    K *dst_k = to_out ? (K *)x_out : tmp_k, *dst_v = to_out ? (K *)iota_out : tmp_v;
    int shift = 8 * p, bits = end_bit - shift < 8 ? end_bit - shift : 8;
    bool flip = (end_bit == width) && (p == passes - 1);
    if (n_blocks == 1) {
      hipLaunchKernelGGL(sort_block_kernel<K>, dim3(1), dim3(kSortThreads), 0, stream, src_k, src_v, p == 0, n, shift, bits, flip,
                         dst_k, dst_v);
      if (int rc = check_launch("sort_block_kernel")) return rc;
      src_k = dst_k;
      src_v = dst_v;
      continue;
    }
    hipLaunchKernelGGL(sort_hist_kernel<K>, dim3(n_blocks), dim3(kSortThreads), 0, stream, src_k, n, shift, bits, flip,
                       seg_counts);
    hipLaunchKernelGGL(sort_scan_kernel, dim3(1), dim3(kRadix), 0, stream, seg_counts, n_seg);
    hipLaunchKernelGGL(sort_place_kernel<K>, dim3(n_blocks), dim3(kSortThreads), 0, stream, src_k, src_v, p == 0, n, shift,
                       bits, flip, seg_counts, dst_k, dst_v);
    int rc = check_launch("sort pass");
    if (rc) return rc;
    src_k = dst_k;
    src_v = dst_v;
  }
  return 0;
}

// ---- bincount + inclusive cumsum (csrc/bincount_cumsum.cu:7-97) ---------------------------------------
// One workgroup: LDS histogram of the whole input, then a scan.  out[0..minlength) = inclusive prefix
// sums, out[minlength..out_len) = 0 (the reference zeroes the whole buffer first).  4096 sorted values in 16 bins: 2.8 us; 5.7 with
// a barrier pair per doubling step of the scan, one load at a time and an addition per value.
constexpr int kBincountMaxBins = 8192;
__global__ __launch_bounds__(1024) void bincount_cumsum_kernel(const int *in, int n, int *out, int out_len, int minlength) {
  __shared__ int hist[kBincountMaxBins];
  __shared__ int wave_total[1024 / kWave];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  for (int i = tid; i < minlength; i += blockDim.x) hist[i] = 0;
  __syncthreads();
  const unsigned count = n;  // (positions are unsigned: the last step's end passes 2^31 - 1 for an n just below it)
  for (unsigned i0 = 0; i0 < count; i0 += 4 * blockDim.x) {  // four loads on their way
    int bin[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned i = i0 + u * blockDim.x + tid;
      bin[u] = i < count ? in[i] : -1;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      // sorted input: the 64 values of a wave are usually the same one, which would be 64 additions in a row to one address
      if (u > 0 && i0 + u * blockDim.x >= count) break;
      const int first = __builtin_amdgcn_readfirstlane(bin[u]);
      const bool one = __all(bin[u] == first);
      if (bin[u] >= 0 && bin[u] < minlength && (!one || lane == 0)) atomicAdd(&hist[bin[u]], one ? kWave : 1);
    }
  }
  __syncthreads();
  // inclusive prefix sums, 1024 bins at a time: within the wave, then over the waves
  if (minlength <= kWave) {  // (one wave has them all)
    if (wave == 0) {
      const int sum = wave_inclusive_scan(lane < minlength ? hist[lane] : 0);
      if (lane < minlength) out[lane] = sum;
    }
  }
  int carry = 0;
  for (int base = minlength <= kWave ? minlength : 0; base < minlength; base += blockDim.x) {
    const int i = base + tid;
    const int sum = wave_inclusive_scan(i < minlength ? hist[i] : 0);
    if (lane == kWave - 1) wave_total[wave] = sum;
    __syncthreads();
    int before = carry;
#pragma unroll
    for (int w = 0; w < 1024 / kWave; ++w) {
      const int t = wave_total[w];
      before += w < wave ? t : 0;
      carry += t;
    }
    if (i < minlength) out[i] = before + sum;
    __syncthreads();
  }
  for (unsigned i = minlength + tid; i < (unsigned)out_len; i += blockDim.x) out[i] = 0;
}

// ---- padded gather (csrc/gather.cu:6-109): out[e,i,:] = x[idx[start_e+i] / top_k,:] or 0 -----------------
template <typename T>
__global__ __launch_bounds__(256) void padded_gather_kernel(const T *x, const int *idx, const int *bins, T *out, int Tn,
                                                            int H, int E, int C, int top_k) {
  const int lane = threadIdx.x & 63;
  const long long n_rows = (long long)E * C;
  for (long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); row < n_rows; row += (long long)gridDim.x * 4) {
    int e = (int)(row / C), i = (int)(row - (long long)e * C);
    int start = e == 0 ? 0 : bins[e - 1], n = bins[e] - start;
    bool valid = i < n;
    int tok = 0;
    if (valid) {
      tok = idx[start + i] / top_k;
      if (tok < 0 || tok >= Tn) valid = false;
    }
    T *dst = out + row * H;
    const T *src = x + (long long)tok * H;
    constexpr int V = ElemTraits<T>::kVec;
    if (H % V == 0) {
      for (int c = lane; c < H / V; c += 64) {
        u32x4 v = {0, 0, 0, 0};
        if (valid) v = ((const u32x4 *)src)[c];
        ((u32x4 *)dst)[c] = v;
      }
    } else {
      for (int c = lane; c < H; c += 64) dst[c] = valid ? src[c] : ElemTraits<T>::from_f32(0.0f);
    }
  }
}

// ---- padded scatter (csrc/scatter.cu:66-147): y[tok,:] += src[e,i,:] * w[start_e+i] -----------------------
// Done without atomics: pass 1 records, for every flat slot, which padded row (if any) feeds it; in pass 2 one to four
// waves own an output row and add that token's rows in slot order.
// slots[flat] = {padded row, sorted position} of every flat slot, {-1, -1} for slots without a row.  With few slots one
// workgroup clears and fills them in one launch; `clear` is false where scatter_clear_kernel has run before.
__global__ __launch_bounds__(1024) void scatter_index_kernel(const int *idx, const int *bins_in, int2 *slots, int S, int E, int C,
                                                             bool clear) {
  __shared__ int lds_bins[kScatterLdsBins];
  const bool in_lds = E <= kScatterLdsBins;
  if (in_lds)
    for (int e = threadIdx.x; e < E; e += blockDim.x) lds_bins[e] = bins_in[e];
  if (in_lds && !clear) __syncthreads();
  const int *bins = in_lds ? lds_bins : bins_in;
  if (clear) {  // (a grid of one workgroup)
    for (int p = threadIdx.x; p < S; p += blockDim.x) slots[p] = make_int2(-1, -1);
    __syncthreads();
  }
  const long long step = (long long)gridDim.x * blockDim.x;
  for (long long at = (long long)blockIdx.x * blockDim.x + threadIdx.x; at < S; at += step) {
    const int p = (int)at;
    // expert of sorted position p: first e with bins[e] > p
    int lo = 0, hi = E;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (bins[mid] > p) hi = mid; else lo = mid + 1;
    }
    if (lo >= E) continue;
    int start = lo == 0 ? 0 : bins[lo - 1];
    int i = p - start;
    int flat = idx[p];
    if (i < C && flat >= 0 && flat < S) slots[flat] = make_int2(lo * C + i, p);
  }
}
// KS > 0: 16-byte chunks, all rows of a token (at most KS slots, the same for all lanes of the wave) requested together;
// 0: any number of slots, any width or alignment.  Both add the rows to y in slot order.  HBM-bound; one element per lane
// with the row number looked up and divided for each took 37.6 us for 2048 tokens x 2 x 1024 fp16, this takes 5.5.  (With the
// index launch, 4096 tokens x 3, 5, 6 x 1024 bf16: 59.4 -> 22.4, 97.4 -> 15.4, 114.6 -> 16.8.)
template <typename T, int KS>
__global__ __launch_bounds__(256) void padded_scatter_kernel(const T *__restrict__ src, const int2 *__restrict__ slots,
                                                             const T *__restrict__ weights, T *__restrict__ y, int Tn, int H,
                                                             int top_k, int split) {
  typedef typename ElemTraits<T>::acc_t acc_t;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int part = wave % split;
  for (int t = wave / split; t < Tn; t += gridDim.x * 4 / split) {
    if constexpr (KS > 0) {
      constexpr int V = ElemTraits<T>::kVec;
      int row[KS];
      acc_t w[KS];
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const int2 at = k < top_k ? slots[t * top_k + k] : make_int2(-1, -1);
        row[k] = at.x;
        w[k] = at.x >= 0 && weights != nullptr ? ElemTraits<T>::to_acc(weights[at.y]) : (acc_t)1;
      }
      u32x4 *dst = (u32x4 *)(y + (long long)t * H);
      for (int c = part * kWave + lane; c < H / V; c += kWave * split) {
        u32x4 raw[KS], o = dst[c];
#pragma unroll
        for (int k = 0; k < KS; ++k) raw[k] = ((const u32x4 *)(src + (long long)max(row[k], 0) * H))[c];
        T *ov = (T *)&o;
        acc_t acc[V];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] = ElemTraits<T>::to_acc(ov[j]);
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          if (row[k] < 0) continue;
          const T *v = (const T *)&raw[k];
#pragma unroll
          for (int j = 0; j < V; ++j) acc[j] += w[k] * ElemTraits<T>::to_acc(v[j]);
        }
#pragma unroll
        for (int j = 0; j < V; ++j) ov[j] = ElemTraits<T>::from_acc(acc[j]);
        dst[c] = o;
      }
    } else {
      for (int c = part * kWave + lane; c < H; c += kWave * split) {
        acc_t acc = ElemTraits<T>::to_acc(y[(long long)t * H + c]);
        for (int k = 0; k < top_k; ++k) {
          const int2 at = slots[t * top_k + k];
          if (at.x < 0) continue;
          acc_t w = weights != nullptr ? ElemTraits<T>::to_acc(weights[at.y]) : (acc_t)1;
          acc += w * ElemTraits<T>::to_acc(src[(long long)at.x * H + c]);
        }
        y[(long long)t * H + c] = ElemTraits<T>::from_acc(acc);
      }
    }
  }
}
template <typename T>
static void launch_padded_scatter(const void *src, const int2 *slots, const void *weights, void *y, int Tn, int H, int top_k,
                                  hipStream_t stream) {
  const int split = Tn >= kScatterWaves ? 1 : 2 * Tn >= kScatterWaves ? 2 : 4;
  const int blocks = min(ceil_div(Tn, 4 / split), 65536);
  const bool chunks = H % ElemTraits<T>::kVec == 0 && ((uintptr_t)src | (uintptr_t)y) % 16 == 0 && top_k <= 8;
#define YAMOE_SCATTER(KS)                                                                                             \
  hipLaunchKernelGGL((padded_scatter_kernel<T, KS>), dim3(blocks), dim3(256), 0, stream, (const T *)src, slots,       \
                     (const T *)weights, (T *)y, Tn, H, top_k, split)
  if (!chunks) YAMOE_SCATTER(0);
  else if (top_k > 4) YAMOE_SCATTER(8);
  else if (top_k > 2) YAMOE_SCATTER(4);
  else YAMOE_SCATTER(2);
#undef YAMOE_SCATTER
}
__global__ void scatter_clear_kernel(int2 *slots, int S) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < S) slots[i] = make_int2(-1, -1);
}

// ---- index_select_out (csrc/index_select.cu:7-51): out[i] = in[idx[i]] ------------------------------------
template <typename T>
__global__ void index_select_kernel(const T *in, const int *idx, T *out, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[idx[i]];
}

// counts[e] = rows, offsets[e] = e * rows: the regular [E, C, *] layout as a ragged one (for callers of the C ABI)
__global__ void regular_groups_kernel(int *counts, int *offsets, int E, int rows) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < E) counts[e] = rows;
  if (e <= E) offsets[e] = e * rows;
}

}  // namespace yamoe

using namespace yamoe;

extern "C" size_t yamoe_sort_workspace_bytes(int32_t n, int32_t elem_bytes) {
  size_t nn = align_up((size_t)(n > 0 ? n : 1), 64);
  int n_blocks = ceil_div(ceil_div(n > 0 ? n : 1, kSortSeg), kSortWaves);
  return align_up(2 * nn * (size_t)elem_bytes + (size_t)n_blocks * kSortWaves * kRadix * sizeof(int), 256);
}

extern "C" int yamoe_sort(const void *x, int32_t elem_bytes, int32_t n, int32_t end_bit, void *x_out, void *iota_out,
                          void *workspace, size_t workspace_bytes, void *stream) {
  if (n < 0 || (elem_bytes != 2 && elem_bytes != 4 && elem_bytes != 8)) {
    set_error("yamoe_sort: keys must be int16, int32 or int64 and n >= 0");
    return YAMOE_E_ARG;
  }
  if (n == 0) return 0;
  if (!x || !x_out || !iota_out || !workspace) { set_error("yamoe_sort: null pointer"); return YAMOE_E_ARG; }
  if (workspace_bytes < yamoe_sort_workspace_bytes(n, elem_bytes)) {
    set_error("yamoe_sort: workspace too small");
    return YAMOE_E_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  if (elem_bytes == 2) return sort_impl<short>(x, n, end_bit, x_out, iota_out, workspace, st);
  if (elem_bytes == 4) return sort_impl<int>(x, n, end_bit, x_out, iota_out, workspace, st);
  return sort_impl<long long>(x, n, end_bit, x_out, iota_out, workspace, st);
}

extern "C" int yamoe_bincount_cumsum(const int32_t *input, int32_t n, int32_t *output, int32_t output_len,
                                     int32_t minlength, void *stream) {
  if (n < 0 || minlength < 0 || output_len < minlength || minlength > kBincountMaxBins || (n > 0 && !input) ||
      (output_len > 0 && !output)) {
    set_error("yamoe_bincount_cumsum: need 0 <= minlength <= min(output_len, %d)", kBincountMaxBins);
    return YAMOE_E_ARG;
  }
  if (output_len == 0) return 0;
  hipLaunchKernelGGL(bincount_cumsum_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, input, n, output, output_len,
                     minlength);
  return check_launch("bincount_cumsum_kernel");
}

#define YAMOE_DISPATCH(dtype, CALL)                                       \
  switch (dtype) {                                                        \
    case YAMOE_F32: { typedef float T; CALL; break; }                     \
    case YAMOE_BF16: { typedef bf16_t T; CALL; break; }                   \
    case YAMOE_F16: { typedef f16_t T; CALL; break; }                     \
    case YAMOE_F64: { typedef double T; CALL; break; }                    \
    default: set_error("unknown dtype %d", dtype); return YAMOE_E_DTYPE;  \
  }

extern "C" int yamoe_padded_gather(const void *x, const int32_t *indices, const int32_t *bins, void *output, int32_t T_,
                                   int32_t H, int32_t E, int32_t C, int32_t top_k, int32_t dtype, void *stream) {
  if (T_ < 0 || H <= 0 || E <= 0 || C < 0 || top_k <= 0) { set_error("yamoe_padded_gather: bad size"); return YAMOE_E_ARG; }
  if ((long long)E * C == 0) return 0;
  if (!x || !indices || !bins || !output) { set_error("yamoe_padded_gather: null pointer"); return YAMOE_E_ARG; }
  long long rows = (long long)E * C;
  int blocks = (int)((rows + 3) / 4 < 65536 ? (rows + 3) / 4 : 65536);
  YAMOE_DISPATCH(dtype, hipLaunchKernelGGL(padded_gather_kernel<T>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                                           (const T *)x, indices, bins, (T *)output, T_, H, E, C, top_k));
  return check_launch("padded_gather_kernel");
}

extern "C" size_t yamoe_padded_scatter_workspace_bytes(int32_t S) { return align_up((size_t)(S > 0 ? S : 1) * 8, 256); }

extern "C" int yamoe_padded_scatter(const void *src, const int32_t *indices, const int32_t *bins, const void *weights,
                                    void *y, int32_t T_, int32_t H, int32_t E, int32_t C, int32_t top_k, int32_t dtype,
                                    void *workspace, size_t workspace_bytes, void *stream) {
  if (T_ < 0 || H <= 0 || E <= 0 || C < 0 || top_k <= 0) { set_error("yamoe_padded_scatter: bad size"); return YAMOE_E_ARG; }
  const int S = T_ * top_k;
  if (S == 0 || C == 0) return 0;  // (a capacity of zero keeps no row: y stays as it is, and src may be an empty tensor)
  if (!src || !indices || !bins || !y || !workspace || workspace_bytes < yamoe_padded_scatter_workspace_bytes(S)) {
    set_error("yamoe_padded_scatter: null pointer or workspace too small");
    return YAMOE_E_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  int2 *slots = (int2 *)workspace;
  const bool one = S <= scatter_one_block(E);
  if (!one) hipLaunchKernelGGL(scatter_clear_kernel, dim3(ceil_div(S, 256)), dim3(256), 0, st, slots, S);
  hipLaunchKernelGGL(scatter_index_kernel, dim3(one ? 1 : ceil_div(S, 256)), dim3(one ? 1024 : 256), 0, st, indices, bins, slots,
                     S, E, C, one);
  YAMOE_DISPATCH(dtype, launch_padded_scatter<T>(src, slots, weights, y, T_, H, top_k, st));
  return check_launch("padded_scatter_kernel");
}

extern "C" int yamoe_index_select(const void *input, const int32_t *idx, void *out, int64_t n, int32_t dtype,
                                  void *stream) {
  if (n < 0) { set_error("yamoe_index_select: n < 0"); return YAMOE_E_ARG; }
  if (n == 0) return 0;
  if (!input || !idx || !out) { set_error("yamoe_index_select: null pointer"); return YAMOE_E_ARG; }
  unsigned blocks = (unsigned)((n + 255) / 256);
  YAMOE_DISPATCH(dtype, hipLaunchKernelGGL(index_select_kernel<T>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                                           (const T *)input, idx, (T *)out, (long long)n));
  return check_launch("index_select_kernel");
}

extern "C" int yamoe_regular_groups(int32_t *counts, int32_t *offsets, int32_t E, int32_t rows, void *stream) {
  if (E <= 0 || rows < 0 || !counts || !offsets) { set_error("yamoe_regular_groups: bad argument"); return YAMOE_E_ARG; }
  hipLaunchKernelGGL(regular_groups_kernel, dim3(ceil_div(E + 1, 256)), dim3(256), 0, (hipStream_t)stream, counts, offsets,
                     E, rows);
  return check_launch("regular_groups_kernel");
}
