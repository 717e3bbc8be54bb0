// Routing for the expert layer: a stable counting sort of the N = T*K (token, slot) assignments by
// expert id, the per-expert counts and exclusive offsets, the inverse permutation, and the work
// lists the expert GEMM kernels walk.
//
// Replaces cub::DeviceRadixSort::SortPairs (csrc/sort.cu:17-91) and bincount_cumsum_kernel
// (csrc/bincount_cumsum.cu:7-56).  The keys have ceil(log2 E) meaningful bits, so one counting pass
// is enough: the input is cut into contiguous segments, one per wavefront; each wave histograms
// its segment, a scan turns (expert-major, segment-minor) counts into write cursors, and each wave
// then walks its segment in order and places every element at cursor[expert] + (number of equal
// keys in lower lanes of the same 64-element step), found with wavefront ballots.  Walking in order
// and ranking by lane keeps equal keys in input order, i.e. the sort is stable.
#include "common.h"

namespace yamoe {

constexpr int kRouteThreads = 1024;
constexpr int kRouteWaves = kRouteThreads / kWave;
constexpr int kRouteMaxBuckets = 769;    // E + 1 must not exceed this (keeps dynamic LDS under 64 KB)
constexpr int kSingleBlockMaxN = 32768;  // the single-workgroup kernel's limit (its keys sit in LDS as 16-bit values)
// Up to this many assignments the single-workgroup kernel is used.  A whole forward of 64-wide experts, which is mostly this, us,
// two or three launches / one: 4096 assignments on 8 experts 22.3 / 22.9, on 32 22.4 / 22.3, on 128 27.2 / 26.3, on 512 40.5 / 32.3; 6144
// on 8 23.3 / 25.6, on 128 26.4 / 26.8, on 256 37.6 / 37.5, on 512 48.1 / 40.7.  The line lies where it is right for few experts;
// from 64 on it could lie higher (5000 on 64: 24.5 / 23.7; 12 288 on 512: 65.2 / 64.6).
constexpr int kSingleBlockN = 4096;

template <bool I64>
__device__ inline int load_key(const void *idx, int i, int E) {
  long long v = I64 ? ((const long long *)idx)[i] : (long long)((const int *)idx)[i];
  // ids outside [0,E) go to bucket E, after every valid expert
  return (v < 0 || v >= E) ? E : (int)v;
}
template <bool I64>
__device__ inline int load_raw(const void *idx, int i) {
  return I64 ? (int)((const long long *)idx)[i] : ((const int *)idx)[i];
}

// Lanes of this wave whose key equals mine (only among lanes with `active`).
__device__ inline uint64_t match_key(int key, bool active, int key_bits) {
  uint64_t peers = __ballot(active);
  for (int b = 0; b < key_bits; ++b) {
    bool bit = (key >> b) & 1;
    uint64_t m = __ballot(active && bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}

__device__ inline int bits_for(int buckets) {
  int b = 0;
  while ((1 << b) < buckets) ++b;
  return b;
}

// Histogram of one wave's segment [seg_begin, seg_end) into `hist_lds` (zeroed by the caller), four loads on their way.
template <bool I64>
__device__ inline void wave_histogram(const void *idx, int seg_begin, int seg_end, int E,
                                      int *hist_lds) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int base = seg_begin; base < seg_end; base += 4 * kWave) {
    int key[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) key[u] = load_key<I64>(idx, min(base + u * kWave + lane, seg_end - 1), E);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (base + u * kWave + lane < seg_end) atomicAdd(&hist_lds[key[u]], 1);
  }
}

// The first kAhead steps of a wave's segment (a whole segment of 256 keys), requested before the table that their placement
// has to wait for: 12 288 keys on 64 experts 10.1 -> 8.8 us, 65 536 on 128 (the first half of each segment) 22 -> 20.3.
constexpr int kAhead = 4;
struct KeysAhead {
  int raw[kAhead];
  bool bad[kAhead];
};
template <bool I64> __device__ inline void load_ahead(const void *idx, int seg_begin, int seg_end, int E, KeysAhead &k) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int u = 0; u < kAhead; ++u) {
    const int i = min(seg_begin + u * kWave + lane, seg_end - 1);
    k.raw[u] = 0;
    k.bad[u] = false;
    if (seg_begin < seg_end) {  // (an empty segment may lie behind the last key)
      k.raw[u] = load_raw<I64>(idx, i);
      k.bad[u] = load_key<I64>(idx, i, E) == E;
    }
  }
}

// Walk one segment in order and place its elements.  `cursor` (LDS, private to this wave) holds
// the next free sorted position per bucket.
template <bool I64>
__device__ inline void wave_place(const void *idx, int seg_begin, int seg_end, int E, int capacity,
                                  int *cursor, const int *offsets_lds,
                                  int *sorted_expert, int *sorted_idx, int *inv_pos, const KeysAhead &ahead) {
  const int lane = threadIdx.x & (kWave - 1);
  const int key_bits = bits_for(E + 1);
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  auto place = [&](int base, int raw, bool bad) {
    const int i = base + lane;
    const bool active = i < seg_end;
    int key = bad ? E : raw;
    if (!active) key = 0;
    uint64_t peers = match_key(key, active, key_bits);
    int rank = __popcll(peers & lt_mask);
    int start = 0;
    if (active) start = cursor[key];
    __builtin_amdgcn_wave_barrier();
    if (active) {
      int pos = start + rank;
      sorted_expert[pos] = raw;
      sorted_idx[pos] = i;
      bool kept = key < E && (pos - offsets_lds[key]) < capacity;
      inv_pos[i] = kept ? pos : -1;
      if (rank == 0) cursor[key] = start + __popcll(peers);
    }
    // the cursor is private to this wave and LDS operations of one wave complete in order: the next step's
    // read sees this step's write without a fence or a volatile access (both would also wait for the global
    // stores above); lanes address the cursor by key, so the compiler cannot carry its values across steps
    __builtin_amdgcn_wave_barrier();
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u)
    if (seg_begin + u * kWave < seg_end) place(seg_begin + u * kWave, ahead.raw[u], ahead.bad[u]);
  // the raw id of the next step is fetched one step ahead so that its latency hides behind this step
  int base = seg_begin + kAhead * kWave;
  int raw_next = (base + lane < seg_end) ? load_raw<I64>(idx, base + lane) : 0;
  bool bad_next = (base + lane < seg_end) ? (load_key<I64>(idx, base + lane, E) == E) : false;
  for (; base < seg_end; base += kWave) {
    const int raw = raw_next, in = base + lane + kWave;
    const bool bad = bad_next;
    if (in < seg_end) {
      raw_next = load_raw<I64>(idx, in);
      bad_next = load_key<I64>(idx, in, E) == E;
    }
    place(base, raw, bad);
  }
}

// The routing of a small batch is one chain of wave scans (common.h), barriers and divisions.  Kernel times, us, with six trips
// through the LDS crossbar a scan, the bucket scan by the whole workgroup and 64-bit divisions / with DPP moves, by one wave
// and without: 4 keys on 128 experts 8.0 / 4.6, 4096 on 16 12.9 / 9.5, 4004 on 128 15.8 / 10.9; work lists of one expert's rows
// alone 8.4 / 5.0.
// Exclusive scan over buckets of `total` into `offsets` (both LDS), by the first wave of the workgroup; offsets[buckets] = N.
// The caller puts a barrier on both sides.
__device__ inline void first_wave_exclusive_scan(const int *total, int *offsets, int buckets) {
  if (threadIdx.x >= kWave) return;
  const int lane = threadIdx.x;
  int carry = 0;
  for (int base = 0; base < buckets; base += kWave) {
    int sum;
    const int before = wave_exclusive_scan(base + lane < buckets ? total[base + lane] : 0, sum);
    if (base + lane < buckets) offsets[base + lane] = carry + before;
    carry += sum;
  }
  if (lane == 0) offsets[buckets] = carry;
}

// ---- work lists ------------------------------------------------------------------------------
// Which experts stream: see build_schedule_wave.  cols: the column tiles of the gate_up product where an expert's last rows may
// stream, else 0; with kStreamEither, the 128-wide column tiles of both products.
struct StreamRule { int max_rows, cols; };
// Where an expert has a few rows more than whole tiles, cutting all of them into equal tiles takes one tile more, which costs
// little in a launch of many rounds and a whole round where it is the first tile of one.  There those rows go to the
// streaming list, if that saves the gate_up product a round (a round of it takes at least as long as one of the down product in
// layers and slices of them, whose I is at most H): its launch then carries them on CUs that have no tile.  2003 tokens x
// 4 on 32 experts, 2880 x 720, 258 gate_up tiles on 256 CUs: 128 + 72 us, and 89 + 64 with 12 experts' last rows streamed.
// They read the expert's weights once more, behind the tiles on CUs that are not idle, so there may be at most four slabs of them (two
// per column tile) for five CUs, those that the tiles leave idle in their last round counted twice.  Whole forwards, us, tiled /
// streamed: 2032 x 4 on 32, 2880 x 720, 192 slabs, 64 CUs idle 226 / 187, 264 slabs, 52 idle 205 / 210; 2007 x 4 on 32, 2880 x 1440, 264,
// 116 idle 312 / 285, about 2150 x 4, 504, 80 idle 328 / 359; about 2000 x 4 on 32 of 1024 x 1024, none idle, 160: 102 / 96, 208: 102 /
// 102, 224: 99 / 106; about 2000 x 8 on 64 of 2048 x 1024, none idle, 80: 324 / 303, 288: 304 / 335.
// A round is little of a launch beyond four of them, and beyond three where an expert has more than six times the average rows:
// 115 drawn calls that the rest of the rule takes, streamed over tiled, 0.90 in the mean for 2 rounds (0.78 to 1.045), 0.92 for 3 (0.81 to
// 1.02), 0.96 for 4 (0.87 to 1.026), but 1.00 (0.946 to 1.044) for 4 with such an expert.
constexpr int kRemainderRounds = 4;

// One wave; lane l takes experts l, l+64, ...  Experts with 1..stream_max_rows kept rows go to the
// streaming list, larger ones are cut into row tiles of kRowTile rows.  Both lists stay in expert
// order: positions come from wave prefix sums.
__device__ inline void build_schedule_wave(const int *counts, const int *offsets, int N, int E, int capacity,
                                           StreamRule streams, int *sched, const int lane) {
  int *row_tiles = sched + kSchedHeader;
  int *small = row_tiles + 8 * sched_max_row_tiles(N, E);
  int n_tiles = 0, n_small = 0, n_active = 0, n_kept = 0, n_half = 0;
  // Experts of 17 to 32 rows stream only when every expert streams: next to experts that need the tile kernels anyway
  // they are better off as tiles (two half-filled launches one after the other are slower than one: 0.35 against
  // 0.31 ms for 32 experts of about 32 rows, where 0.27 against 0.31 ms is gained when all of them have at most 32).
  int stream_max_rows = streams.max_rows;
  bool everything = stream_max_rows == kStreamEverything;  // (the host checked sched_may_stream_everything)
  if (stream_max_rows == kStreamEither) {
    int as_streams = 0, as_tiles = 0;
    for (int base = 0; base < E; base += kWave) {
      const int kept = base + lane < E ? max(min(counts[base + lane], capacity), 0) : 0;
      as_streams += wave_sum(f32_stream_cost(kept));
      as_tiles += wave_sum(f32_tile_cost(kept));
    }
    everything = as_streams <= max(as_tiles, kF32FewTiles / streams.cols);
    stream_max_rows = 0;
  }
  if (everything) {  // (only then do workgroups share slabs: see stream.hip)
    stream_max_rows = kStreamMaxRows;
    int *arrivals = small + 4 * sched_max_small(N, E);
    for (int i = lane; i < kSchedArrivals; i += kWave) arrivals[i] = 0;
  }
  if (!everything && stream_max_rows > kStreamMixedRows) {
    bool beyond = false;
    for (int base = lane; base < E; base += kWave) beyond |= min(counts[base], capacity) > stream_max_rows;
    if (__any(beyond)) stream_max_rows = kStreamMixedRows;
  }
  // an expert's tiled rows: all of them, or (`remainders`) whole tiles' worth
  auto tiled_rows = [&](int kept, bool remainders) {
    if (kept <= stream_max_rows || everything) return 0;
    const int past = kept % kRowTile;
    return remainders && kept > kRowTile && past <= kStreamMaxRows ? kept - past : kept;
  };
  bool remainders = false;
  if (streams.max_rows != kStreamEither && streams.cols > 0 && !everything) {
    int all = 0, fewer = 0;
    bool skewed = false;
    for (int base = 0; base < E; base += kWave) {
      const int kept = base + lane < E ? max(min(counts[base + lane], capacity), 0) : 0;
      all += wave_sum(ceil_div(tiled_rows(kept, false), kRowTile));
      fewer += wave_sum(ceil_div(tiled_rows(kept, true), kRowTile));
      skewed |= __any((long long)kept * E > 6ll * N);
    }
    const int rounds = ceil_div(all * streams.cols, kXcds * kXcdCus);
    const int left = ceil_div(fewer * streams.cols, kXcds * kXcdCus), idle = left * kXcds * kXcdCus - fewer * streams.cols;
    remainders = rounds <= kRemainderRounds - skewed && left < rounds &&
                 (all - fewer) * 2 * streams.cols * 5 <= (kXcds * kXcdCus + idle) * 4;
  }
  for (int base = 0; base < E; base += kWave) {
    int e = base + lane;
    int kept = e < E ? min(counts[e], capacity) : 0;
    if (kept < 0) kept = 0;
    int first = e < E ? offsets[e] : 0;
    // entries on the streaming list: one, or with `everything` one per chunk of kStreamMaxRows rows
    const int tiled = tiled_rows(kept, remainders);
    int is_small = everything ? ceil_div(kept, kStreamMaxRows) : kept > tiled;
    int tiles = ceil_div(tiled, kRowTile);
    int tot_small, tot_tiles, tot_half;
    int pos_small = wave_exclusive_scan(is_small, tot_small);
    int pos_tiles = wave_exclusive_scan(tiles, tot_tiles);
    const int halves = ceil_div(tiled, kRowTile / 2);
    const int pos_half = n_half + wave_exclusive_scan(halves, tot_half);
    const int tot_active = __popcll(__ballot(kept > 0)), tot_kept = wave_sum(kept);
    for (int c = 0; c < is_small; ++c) {
      int *s = small + 4 * (n_small + pos_small + c);
      s[0] = e; s[1] = first + tiled + c * kStreamMaxRows; s[2] = min(kStreamMaxRows, kept - tiled - c * kStreamMaxRows); s[3] = 0;
    }
    int gfirst = n_tiles + pos_tiles;
    // An expert's rows are cut into equal tiles (a multiple of 32 rows, the MFMA block), not into full
    // tiles plus a remainder: tiles of one expert then advance through the contraction at the same pace
    // and the weight slabs one of them fetches are still in L2 when the others ask for them.
    int per_tile = tiles > 0 ? min(kRowTile, (ceil_div(tiled, tiles) + 31) & ~31) : 0;
    FastDiv by_tiles = {1u, 0u};  // the GEMM kernels divide by the group size (a 64-bit division: only where there is a group)
    if (tiles > 1) by_tiles = make_fast_div(tiles);
    for (int t = 0; t < tiles; ++t) {
      int *w = row_tiles + 8 * (gfirst + t);
      w[0] = e; w[1] = first + t * per_tile; w[2] = min(per_tile, tiled - t * per_tile); w[3] = gfirst; w[4] = tiles;
      w[5] = (int)by_tiles.mul; w[6] = (int)by_tiles.shift; w[7] = pos_half;
    }
    n_small += tot_small; n_tiles += tot_tiles; n_active += tot_active; n_kept += tot_kept; n_half += tot_half;
  }
  // Second pass: cut the tile list into 8 shares of equal cost.  Groups (experts with row tiles) are weighed
  // by the sum of their tiles' weights; cut x falls into the group that contains x/8 of the total.
  auto group = [&](int e, int &tiles) {
    const int tiled = tiled_rows(e < E ? max(min(counts[e], capacity), 0) : 0, remainders);
    tiles = ceil_div(tiled, kRowTile);
    const int per_tile = tiles > 0 ? min(kRowTile, (ceil_div(tiled, tiles) + 31) & ~31) : 0;
    return sched_group_weight(tiles, per_tile, tiled);
  };
  int w_total = 0, tiles;
  if (n_tiles > 0)
    for (int base = 0; base < E; base += kWave) w_total += wave_sum(group(base + lane, tiles));
  // lane x < 8 gets cut x: its group's first row tile and tiles, how far into the group's 8-fold weight it falls
  int cut_first = 0, cut_tiles = 0;
  long long cut_num = 0, cut_w = 1;
  if (w_total > 0) {
    int w_before = 0, t_before = 0;
    for (int base = 0; base < E; base += kWave) {
      int tot_w, tot_t;
      const int w = group(base + lane, tiles);
      const int w_pre = w_before + wave_exclusive_scan(w, tot_w), t_pre = t_before + wave_exclusive_scan(tiles, tot_t);
      for (int x = 0; x < kXcds; ++x) {
        const long long t = (long long)x * w_total;  // compare x * W / 8 with the group's weight interval, times 8
        const uint64_t hit = __ballot(tiles > 0 && t >= 8ll * w_pre && t < 8ll * (w_pre + w));
        if (hit == 0) continue;
        const int from = __ffsll((unsigned long long)hit) - 1;
        const int first = __builtin_amdgcn_readlane(t_pre, from), count = __builtin_amdgcn_readlane(tiles, from);
        const int pre = __builtin_amdgcn_readlane(w_pre, from), weight = __builtin_amdgcn_readlane(w, from);
        if (lane == x) { cut_first = first; cut_tiles = count; cut_num = t - 8ll * pre; cut_w = 8ll * weight; }
      }
      w_before += tot_w; t_before += tot_t;
    }
  }
  if (lane < kXcds) {
    // floor(2^16 * num / w) in double precision: below 2^51 over below 2^35, so a quotient that is no whole number is further
    // from the next one (2^-35) than it is rounded (2^-37)
    int *c = sched + kSchedCuts + 4 * lane;
    c[0] = cut_first; c[1] = (int)((double)(cut_num << 16) / (double)cut_w); c[2] = w_total > 0 ? n_tiles : 0; c[3] = cut_tiles;
  }
  if (lane == 0) {
    sched[0] = n_tiles; sched[1] = n_small; sched[2] = n_active; sched[3] = n_kept;
    sched[4] = w_total; sched[kSchedHalfTiles] = n_half; sched[6] = 0; sched[7] = 0;
    int *c = sched + kSchedCuts + 4 * kXcds;  // the end of the list
    c[0] = n_tiles; c[1] = 0; c[2] = 0; c[3] = 0;
    for (int i = kSchedCuts + 4 * (kXcds + 1); i < kSchedHeader; ++i) sched[i] = 0;
  }
}

__global__ __launch_bounds__(kWave) void build_schedule_kernel(const int *counts, const int *offsets, int N, int E,
                                                               int capacity, StreamRule streams, int *sched) {
  build_schedule_wave(counts, offsets, N, E, capacity, streams, sched, threadIdx.x);
}

// counts[e] = rows, offsets[e] = e * rows and their work lists in one launch (a lane reads back only what it wrote itself)
__global__ __launch_bounds__(kWave) void regular_schedule_kernel(int *counts, int *offsets, int E, int rows, StreamRule streams,
                                                                 int *sched) {
  for (int e = threadIdx.x; e < E; e += kWave) { counts[e] = rows; offsets[e] = e * rows; }
  if (threadIdx.x == 0) offsets[E] = E * rows;
  build_schedule_wave(counts, offsets, E * rows, E, rows, streams, sched, threadIdx.x);
}

// ---- single-block form: everything in one launch -------------------------------------------------
// Dynamic LDS: hist[kRouteWaves][buckets] + total[buckets] + offsets[buckets+1] + the N keys as 16-bit
// values.  The kernel runs once per forward on a cold instruction cache, so its loops stay rolled (straight-line
// code would run at instruction-fetch speed); the keys are read from memory once and kept in LDS for the
// placement pass.
__host__ __device__ inline size_t route_single_lds_bytes(int N, int buckets) {
  size_t ints = (size_t)kRouteWaves * buckets + buckets + buckets + 1;
  return align_up(ints * sizeof(int), 16) + align_up((size_t)(N > 0 ? N : 1) * sizeof(unsigned short), 16);
}

template <bool I64>
__global__ __launch_bounds__(kRouteThreads) void route_single_kernel(
    const void *idx, int N, int E, int capacity, int *sorted_expert, int *sorted_idx, int *counts,
    int *offsets_out, int *inv_pos, int *sched, StreamRule streams) {
  extern __shared__ int lds[];
  const int buckets = E + 1;
  int *hist = lds;                          // [kRouteWaves][buckets]
  int *total = hist + kRouteWaves * buckets;  // [buckets]
  int *offs = total + buckets;              // [buckets + 1]
  unsigned short *keys = (unsigned short *)((char *)lds + align_up(((size_t)kRouteWaves * buckets + 2 * buckets + 1) * sizeof(int), 16));
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid & (kWave - 1);

  for (int i = tid; i < kRouteWaves * buckets; i += blockDim.x) hist[i] = 0;
  __syncthreads();

  int seg = ceil_div(ceil_div(N, kRouteWaves), kWave) * kWave;
  int seg_begin = min(wave * seg, N), seg_end = min(seg_begin + seg, N);
  {
    // four loads in flight per lane; positions past the end are clamped, their keys dropped
    int *h = hist + wave * buckets;
    for (int base = seg_begin; base < seg_end; base += 4 * kWave) {
      int k[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) k[u] = load_key<I64>(idx, min(base + u * kWave + lane, N - 1), E);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int i = base + u * kWave + lane;
        if (i < seg_end) {
          keys[i] = (unsigned short)k[u];
          atomicAdd(&h[k[u]], 1);
        }
      }
    }
  }
  __syncthreads();

  // hist[w][b] <- keys of bucket b in the segments before w; the cursor of a wave is that plus the bucket's offset
  for (int b = tid; b < buckets; b += blockDim.x) {
    int run = 0;
    for (int w = 0; w < kRouteWaves; ++w) {
      const int c = hist[w * buckets + b];
      hist[w * buckets + b] = run;
      run += c;
    }
    total[b] = run;
  }
  __syncthreads();
  first_wave_exclusive_scan(total, offs, buckets);
  __syncthreads();
  for (int b = tid; b < buckets; b += blockDim.x) {
    if (b < E) {
      counts[b] = total[b];
      offsets_out[b] = offs[b];
    } else {
      offsets_out[E] = offs[E];
    }
  }

  // placement, in input order: position = cursor[key] + number of equal keys in lower lanes of the step
  {
    int *cursor = hist + wave * buckets;
    const int key_bits = bits_for(E + 1);
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int base = seg_begin; base < seg_end; base += kWave) {
      const int i = base + lane;
      const bool active = i < seg_end;
      const int k = active ? (int)keys[i] : 0;
      uint64_t peers = match_key(k, active, key_bits);
      int rank = __popcll(peers & lt_mask);
      int start = 0;
      if (active) start = cursor[k];
      const int first = active ? offs[k] : 0;
      __builtin_amdgcn_wave_barrier();
      if (active) {
        const int in_bucket = start + rank, pos = first + in_bucket;
        // a valid id is its own key; the rare invalid one is fetched again for the sorted_expert output
        sorted_expert[pos] = k < E ? k : load_raw<I64>(idx, i);
        sorted_idx[pos] = i;
        inv_pos[i] = k < E && in_bucket < capacity ? pos : -1;
        if (rank == 0) cursor[k] = start + __popcll(peers);
      }
      // the cursor is private to this wave and LDS operations of one wave complete in order: the next step's
      // read sees this step's write without a fence or a volatile access (both would also wait for the global
      // stores above); lanes address the cursor by key, so the compiler cannot carry its values across steps
      __builtin_amdgcn_wave_barrier();
    }
  }
  // the work lists of the GEMM kernels, from the counts and offsets still in LDS (the last wave, after its share
  // of the placement): saves the launch of build_schedule_kernel
  if (sched != nullptr && wave == kRouteWaves - 1) build_schedule_wave(total, offs, N, E, capacity, streams, sched, lane);
}

// ---- three-kernel form for large N -----------------------------------------------------------
// seg_counts is [n_seg][buckets] in global memory; one wave per segment of `seg` elements.
template <bool I64>
__global__ __launch_bounds__(kRouteThreads) void route_hist_kernel(const void *idx, int N, int E,
                                                                   int seg, int *seg_counts) {
  extern __shared__ int lds[];
  const int buckets = E + 1;
  const int tid = threadIdx.x, wave = tid / kWave;
  int *hist = lds + wave * buckets;
  for (int i = tid; i < kRouteWaves * buckets; i += blockDim.x) lds[i] = 0;
  __syncthreads();
  int s = blockIdx.x * kRouteWaves + wave;
  int seg_begin = min((long long)s * seg, (long long)N), seg_end = min(seg_begin + seg, N);
  wave_histogram<I64>(idx, seg_begin, seg_end, E, hist);
  __syncthreads();
  for (int i = tid; i < kRouteWaves * buckets; i += blockDim.x)
    seg_counts[(size_t)blockIdx.x * kRouteWaves * buckets + i] = lds[i];
}

// One block: totals, offsets, then per-segment cursors written back over seg_counts: the form for tables too large for LDS
// (many experts and many assignments at once); smaller ones take route_place_scan_kernel.  A lane holds a bucket and a
// wave walks its stretch of the segments for 64 of them, kScanAhead rows of the table on their way: whole cache lines, where a
// wave that walks one bucket's column, 64 segments a step, fetches a line for every word it reads.  Us for 32 768 keys on 700
// experts, 65 536 on 512, 200 000 on 700, by columns / like this: 133 / 22, 94 / 21, 118 / 19.
constexpr int kScanAhead = 8;
__host__ __device__ inline size_t route_scan_lds_ints(int buckets) { return 2 * (size_t)buckets + 1 + kRouteThreads; }
__global__ __launch_bounds__(kRouteThreads) void route_scan_kernel(int *seg_counts, int n_seg, int E, int *counts,
                                                                   int *offsets_out) {
  extern __shared__ int lds[];
  const int buckets = E + 1;
  int *total = lds;
  int *offs = total + buckets;
  int *part = offs + buckets + 1;  // [stretch][64 * groups of buckets]
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int groups = ceil_div(buckets, kWave), stretches = kRouteWaves / groups, width = groups * kWave;
  const int stretch = wave / groups, b = (wave - stretch * groups) * kWave + lane;
  const int len = ceil_div(n_seg, stretches);
  // (waves left over get an empty stretch; a lane beyond the last bucket reads the last one and writes nothing)
  const int first = stretch < stretches ? min(stretch * len, n_seg) : n_seg, end = stretch < stretches ? min(first + len, n_seg) : n_seg;
  int *column = seg_counts + min(b, buckets - 1);
  int sum = 0;
  for (int g0 = first; g0 < end; g0 += kScanAhead) {
    int c[kScanAhead];
#pragma unroll
    for (int u = 0; u < kScanAhead; ++u) c[u] = column[(size_t)min(g0 + u, end - 1) * buckets];
#pragma unroll
    for (int u = 0; u < kScanAhead; ++u) sum += g0 + u < end ? c[u] : 0;
  }
  if (stretch < stretches) part[stretch * width + b] = sum;
  __syncthreads();
  for (int i = tid; i < buckets; i += blockDim.x) {
    int run = 0;
    for (int w = 0; w < stretches; ++w) run += part[w * width + i];
    total[i] = run;
  }
  __syncthreads();
  first_wave_exclusive_scan(total, offs, buckets);
  __syncthreads();
  int run = b < buckets ? offs[b] : 0;
  for (int w = 0; w < min(stretch, stretches); ++w) run += part[w * width + b];
  for (int g0 = first; g0 < end; g0 += kScanAhead) {
    int c[kScanAhead];
#pragma unroll
    for (int u = 0; u < kScanAhead; ++u) c[u] = column[(size_t)min(g0 + u, end - 1) * buckets];
#pragma unroll
    for (int u = 0; u < kScanAhead; ++u) {
      if (g0 + u < end && b < buckets) column[(size_t)(g0 + u) * buckets] = run;
      run += c[u];
    }
  }
  for (int b = tid; b < buckets; b += blockDim.x) {
    if (b < E) {
      counts[b] = total[b];
      offsets_out[b] = offs[b];
    } else {
      offsets_out[E] = offs[E];
    }
  }
}

// With sched the grid has one workgroup more than there are blocks of segments: its first wave writes the work lists
// of the GEMM kernels from the counts and offsets, next to the placement instead of in a launch of its own.
template <bool I64>
__global__ __launch_bounds__(kRouteThreads) void route_place_kernel(
    const void *idx, int N, int E, int capacity, int seg, const int *seg_cursors,
    const int *offsets_in, int *sorted_expert, int *sorted_idx, int *inv_pos, int n_blocks, const int *counts,
    StreamRule streams, int *sched) {
  extern __shared__ int lds[];
  const int buckets = E + 1;
  const int tid = threadIdx.x, wave = tid / kWave;
  if ((int)blockIdx.x >= n_blocks) {  // (uniform for the workgroup: nobody of it reaches the barrier below)
    if (sched != nullptr && wave == 0)
      build_schedule_wave(counts, offsets_in, N, E, capacity, streams, sched, tid);
    return;
  }
  int *cursor = lds + wave * buckets;
  int *offs = lds + kRouteWaves * buckets;
  int s = blockIdx.x * kRouteWaves + wave;
  int seg_begin = min((long long)s * seg, (long long)N), seg_end = min(seg_begin + seg, N);
  KeysAhead ahead;
  load_ahead<I64>(idx, seg_begin, seg_end, E, ahead);
  for (int i = tid; i < kRouteWaves * buckets; i += blockDim.x)
    lds[i] = seg_cursors[(size_t)blockIdx.x * kRouteWaves * buckets + i];
  for (int b = tid; b <= E; b += blockDim.x) offs[b] = offsets_in[b];
  __syncthreads();
  wave_place<I64>(idx, seg_begin, seg_end, E, capacity, cursor, offs, sorted_expert, sorted_idx,
                  inv_pos, ahead);
}

// ---- two-kernel form: every workgroup of the placement scans the table for itself -----------------------------
// The segments x buckets table of route_hist_kernel is small (65 536 keys in segments of 512 and 128 experts: 66 KB),
// so instead of one workgroup scanning it in a launch of its own, every workgroup of the placement reads all of it
// into LDS and derives what it needs: the bucket totals and offsets, and the cursors of its own 16 segments (a wave
// per bucket column, wave prefix sums over the segments).  Workgroup 0 also writes counts and offsets; with sched
// one workgroup more than there are blocks of segments writes the work lists.
__host__ __device__ inline size_t route_place_scan_lds_ints(int n_seg, int buckets) {
  return (size_t)buckets + (buckets + 1) + (size_t)kRouteWaves * buckets + (size_t)n_seg * buckets;
}
constexpr size_t kPlaceScanMaxLdsInts = 40000;  // 160 000 bytes

template <bool I64>
__global__ __launch_bounds__(kRouteThreads) void route_place_scan_kernel(
    const void *idx, int N, int E, int capacity, int seg, const int *seg_counts, int n_seg, int *sorted_expert,
    int *sorted_idx, int *inv_pos, int *counts, int *offsets_out, int n_blocks, StreamRule streams, int *sched) {
  extern __shared__ int lds[];
  const int buckets = E + 1;
  int *total = lds;                              // [buckets]
  int *offs = total + buckets;                   // [buckets + 1]
  int *cursors = offs + buckets + 1;             // [kRouteWaves][buckets]
  int *table = cursors + kRouteWaves * buckets;  // [n_seg][buckets]
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int cells = n_seg * buckets;
  const int sgm = blockIdx.x * kRouteWaves + wave;
  const int seg_begin = (int)min((long long)sgm * seg, (long long)N), seg_end = min(seg_begin + seg, N);
  KeysAhead ahead;  // (the extra workgroup's segments are empty)
  load_ahead<I64>(idx, seg_begin, seg_end, E, ahead);
  for (int i = tid; i < cells; i += blockDim.x) table[i] = seg_counts[i];
  __syncthreads();
  const int my_first = blockIdx.x * kRouteWaves;  // this workgroup's segments: my_first + 0..15 (none for the extra one)
  for (int b = wave; b < buckets; b += kRouteWaves) {
    int run = 0;
    for (int g0 = 0; g0 < n_seg; g0 += kWave) {
      const int g = g0 + lane;
      const int c = g < n_seg ? table[g * buckets + b] : 0;
      int step_total;
      const int before = wave_exclusive_scan(c, step_total);
      if (g < n_seg && g >= my_first && g < my_first + kRouteWaves) cursors[(g - my_first) * buckets + b] = run + before;
      run += step_total;
    }
    if (lane == 0) total[b] = run;
  }
  __syncthreads();
  first_wave_exclusive_scan(total, offs, buckets);
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int b = tid; b < buckets; b += blockDim.x) {
      if (b < E) {
        counts[b] = total[b];
        offsets_out[b] = offs[b];
      } else {
        offsets_out[E] = offs[E];
      }
    }
  }
  if ((int)blockIdx.x >= n_blocks) {  // (uniform for the workgroup: nobody of it reaches the barrier below)
    if (sched != nullptr && wave == 0) build_schedule_wave(total, offs, N, E, capacity, streams, sched, lane);
    return;
  }
  for (int i = tid; i < kRouteWaves * buckets; i += blockDim.x) cursors[i] += offs[i % buckets];
  __syncthreads();
  wave_place<I64>(idx, seg_begin, seg_end, E, capacity, cursors + wave * buckets, offs, sorted_expert, sorted_idx, inv_pos, ahead);
}

}  // namespace yamoe

using namespace yamoe;

// Keys per wave in the forms with more than one launch: short segments spread the counting and the placement over
// more workgroups, long ones keep the segments x buckets table small.  Whole routing without work lists, us, with segments of 128 /
// 256 / 512 / 1024 / 2048 keys: 16 384 keys on 32 experts 9.2 / 9.5 / 13.8 / 22.6 / 33.5, 32 768 on 128 22.6 / 18.2 / 20.8 / 31.3 / 53.8,
// 65 536 on 128 28.1 / 24.3 / 23.9 / 32.2 / 55.0, 131 072 on 256 68.4 / 43.0 / 35.3 / 45.9 / 64.8.  Beyond that only a large table
// wants 2048 (1 048 576 on 256: 248 / 138 / 94 / 91 with 256 and up); 262 144 on 32 experts take 44.0, and 22.9 / 20.9 / 27.1
// with 256 / 512 / 1024.
static int route_segment(int N) { return N <= 32768 ? 256 : N <= 131072 ? 512 : 2048; }
static_assert(kSingleBlockN <= kSingleBlockMaxN, "the single-workgroup kernel keeps its keys in LDS");

extern "C" size_t yamoe_route_workspace_bytes(int32_t N, int32_t E) {
  if (N <= kSingleBlockN) return 256;
  int seg = route_segment(N);
  int n_seg = ceil_div(ceil_div(N, seg), kRouteWaves) * kRouteWaves;
  return align_up((size_t)n_seg * (E + 1) * sizeof(int), 256);
}

// yamoe_route, optionally with the work lists of yamoe_build_schedule (schedule != nullptr): one launch for N up to
// kSingleBlockN, two above (histograms, then scan + placement), three where the histogram table does not fit LDS;
// with more than one launch the lists come from an extra workgroup of the placement kernel.
int yamoe::route_and_schedule(const void *router_indices, int32_t idx_i64, int32_t N, int32_t E, int32_t capacity,
                              int32_t *sorted_expert, int32_t *sorted_idx, int32_t *counts, int32_t *offsets,
                              int32_t *inv_pos, void *workspace, size_t workspace_bytes, int32_t stream_max_rows, int32_t cols,
                              void *schedule, size_t schedule_bytes, void *stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (schedule != nullptr && schedule_bytes < yamoe_schedule_bytes(N, E)) {
    set_error("yamoe_build_schedule: schedule region too small");
    return YAMOE_E_WORKSPACE;
  }
  if (stream_max_rows == kStreamEverything && !sched_may_stream_everything(N, E, 4)) stream_max_rows = kStreamMaxRows;
  if (stream_max_rows < 0 && stream_max_rows != kStreamEverything && stream_max_rows != kStreamEither) stream_max_rows = 0;
  if (stream_max_rows > kStreamMaxRows) stream_max_rows = kStreamMaxRows;
  if (N < 0 || E <= 0 || E + 1 > kRouteMaxBuckets) {
    set_error("yamoe_route: need N >= 0 and 1 <= E < %d (got N=%d E=%d)", kRouteMaxBuckets, N, E);
    return YAMOE_E_ARG;
  }
  if (!counts || !offsets || (N > 0 && (!router_indices || !sorted_expert || !sorted_idx || !inv_pos))) {
    set_error("yamoe_route: null pointer");
    return YAMOE_E_ARG;
  }
  if (capacity < 0) capacity = 0;
  const StreamRule streams = {stream_max_rows, cols};
  const int buckets = E + 1;
  if (N <= kSingleBlockN) {
    size_t lds = route_single_lds_bytes(N, buckets);
    static DeviceFlags attr_i64, attr_i32;
    const int max_lds = (int)route_single_lds_bytes(kSingleBlockMaxN, kRouteMaxBuckets);
    int rc = idx_i64 ? ensure_dynamic_lds((const void *)route_single_kernel<true>, max_lds, attr_i64, "route_single_kernel")
                     : ensure_dynamic_lds((const void *)route_single_kernel<false>, max_lds, attr_i32, "route_single_kernel");
    if (rc != 0) return rc;
    if (idx_i64)
      hipLaunchKernelGGL(route_single_kernel<true>, dim3(1), dim3(kRouteThreads), lds, stream,
                         router_indices, N, E, capacity, sorted_expert, sorted_idx, counts, offsets, inv_pos, (int *)schedule,
                         streams);
    else
      hipLaunchKernelGGL(route_single_kernel<false>, dim3(1), dim3(kRouteThreads), lds, stream,
                         router_indices, N, E, capacity, sorted_expert, sorted_idx, counts, offsets, inv_pos, (int *)schedule,
                         streams);
    return check_launch("route_single_kernel");
  }
  if (workspace_bytes < yamoe_route_workspace_bytes(N, E) || !workspace) {
    set_error("yamoe_route: workspace too small (%zu < %zu)", workspace_bytes, yamoe_route_workspace_bytes(N, E));
    return YAMOE_E_WORKSPACE;
  }
  const int seg = route_segment(N);
  const int n_blocks = ceil_div(ceil_div(N, seg), kRouteWaves);
  const int n_seg = n_blocks * kRouteWaves;
  int *seg_counts = (int *)workspace;
  size_t lds_a = (size_t)kRouteWaves * buckets * sizeof(int);
  size_t lds_b = route_scan_lds_ints(buckets) * sizeof(int);
  size_t lds_c = ((size_t)kRouteWaves * buckets + buckets) * sizeof(int);
  if (idx_i64)
    hipLaunchKernelGGL(route_hist_kernel<true>, dim3(n_blocks), dim3(kRouteThreads), lds_a, stream,
                       router_indices, N, E, seg, seg_counts);
  else
    hipLaunchKernelGGL(route_hist_kernel<false>, dim3(n_blocks), dim3(kRouteThreads), lds_a, stream,
                       router_indices, N, E, seg, seg_counts);
  int rc = check_launch("route_hist_kernel");
  if (rc) return rc;
  if (route_place_scan_lds_ints(n_seg, buckets) <= kPlaceScanMaxLdsInts) {
    // two launches: the placement's workgroups scan the table themselves
    static DeviceFlags attr_ps64, attr_ps32;
    const int max_lds = (int)(kPlaceScanMaxLdsInts * sizeof(int));
    rc = idx_i64 ? ensure_dynamic_lds((const void *)route_place_scan_kernel<true>, max_lds, attr_ps64, "route_place_scan_kernel")
                 : ensure_dynamic_lds((const void *)route_place_scan_kernel<false>, max_lds, attr_ps32, "route_place_scan_kernel");
    if (rc) return rc;
    const size_t lds_ps = route_place_scan_lds_ints(n_seg, buckets) * sizeof(int);
    const dim3 grid(n_blocks + (schedule != nullptr ? 1 : 0));
    if (idx_i64)
      hipLaunchKernelGGL(route_place_scan_kernel<true>, grid, dim3(kRouteThreads), lds_ps, stream, router_indices, N, E,
                         capacity, seg, seg_counts, n_seg, sorted_expert, sorted_idx, inv_pos, counts, offsets, n_blocks,
                         streams, (int *)schedule);
    else
      hipLaunchKernelGGL(route_place_scan_kernel<false>, grid, dim3(kRouteThreads), lds_ps, stream, router_indices, N, E,
                         capacity, seg, seg_counts, n_seg, sorted_expert, sorted_idx, inv_pos, counts, offsets, n_blocks,
                         streams, (int *)schedule);
    return check_launch("route_place_scan_kernel");
  }
  hipLaunchKernelGGL(route_scan_kernel, dim3(1), dim3(kRouteThreads), lds_b, stream, seg_counts, n_seg, E, counts, offsets);
  rc = check_launch("route_scan_kernel");
  if (rc) return rc;
  if (idx_i64)
    hipLaunchKernelGGL(route_place_kernel<true>, dim3(n_blocks + (schedule != nullptr ? 1 : 0)), dim3(kRouteThreads), lds_c,
                       stream, router_indices, N, E, capacity, seg, seg_counts, offsets, sorted_expert, sorted_idx, inv_pos,
                       n_blocks, counts, streams, (int *)schedule);
  else
    hipLaunchKernelGGL(route_place_kernel<false>, dim3(n_blocks + (schedule != nullptr ? 1 : 0)), dim3(kRouteThreads), lds_c,
                       stream, router_indices, N, E, capacity, seg, seg_counts, offsets, sorted_expert, sorted_idx, inv_pos,
                       n_blocks, counts, streams, (int *)schedule);
  return check_launch("route_place_kernel");
}

extern "C" int yamoe_route(const void *router_indices, int32_t idx_i64, int32_t N, int32_t E,
                           int32_t capacity, int32_t *sorted_expert, int32_t *sorted_idx,
                           int32_t *counts, int32_t *offsets, int32_t *inv_pos, void *workspace,
                           size_t workspace_bytes, void *stream_) {
  return route_and_schedule(router_indices, idx_i64, N, E, capacity, sorted_expert, sorted_idx, counts, offsets, inv_pos,
                            workspace, workspace_bytes, 0, 0, nullptr, 0, stream_);
}

int yamoe::regular_schedule(int *counts, int *offsets, int E, int rows, int stream_max_rows, void *schedule,
                            size_t schedule_bytes, hipStream_t stream) {
  if (schedule_bytes < yamoe_schedule_bytes(E * rows, E)) {
    set_error("regular_schedule: schedule region too small");
    return YAMOE_E_WORKSPACE;
  }
  hipLaunchKernelGGL(regular_schedule_kernel, dim3(1), dim3(kWave), 0, stream, counts, offsets, E, rows, StreamRule{stream_max_rows, 0},
                     (int *)schedule);
  return check_launch("regular_schedule_kernel");
}

extern "C" size_t yamoe_schedule_bytes(int32_t N, int32_t E) {
  size_t words = kSchedHeader + 8 * (size_t)sched_max_row_tiles(N, E) + 4 * (size_t)sched_max_small(N, E) + kSchedArrivals;
  return align_up(words * sizeof(int), 256);
}

extern "C" int yamoe_build_schedule(const int32_t *counts, const int32_t *offsets, int32_t N, int32_t E,
                                    int32_t capacity, int32_t stream_max_rows, void *schedule,
                                    size_t schedule_bytes, void *stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!counts || !offsets || !schedule || N < 0 || E <= 0) {
    set_error("yamoe_build_schedule: bad argument");
    return YAMOE_E_ARG;
  }
  if (schedule_bytes < yamoe_schedule_bytes(N, E)) {
    set_error("yamoe_build_schedule: schedule region too small");
    return YAMOE_E_WORKSPACE;
  }
  if (capacity < 0) capacity = 0;
  if (stream_max_rows == kStreamEverything && !sched_may_stream_everything(N, E, 2)) stream_max_rows = kStreamMaxRows;
  if (stream_max_rows < 0 && stream_max_rows != kStreamEverything) stream_max_rows = 0;
  if (stream_max_rows > kStreamMaxRows) stream_max_rows = kStreamMaxRows;
  hipLaunchKernelGGL(build_schedule_kernel, dim3(1), dim3(kWave), 0, stream, counts, offsets, N, E, capacity,
                     StreamRule{stream_max_rows, 0}, (int *)schedule);
  return check_launch("build_schedule_kernel");
}
