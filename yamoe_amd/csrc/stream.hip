// Weight-streaming path for experts with at most 32 kept rows (the decode regime).
//
// Such an expert does 2*rows flops per weight element, far below the machine balance, so the job
// is to pull each expert's weights through the chip once at HBM rate.  A workgroup owns one
// (expert, 128-column slab) of a [K, N] weight matrix.  Its 4 wavefronts take the 32-row k-steps
// of the slab round-robin; in a step every lane fetches an 8(k) x 8(column) block as eight 16-byte
// loads (a wave reads 32 rows x 256 contiguous bytes), transposes it in registers and feeds it to
// eight v_mfma_f32_16x16x32 instructions whose 16-row A operand is the expert's (zero-padded)
// activations (an expert with 17 to 32 rows has two such operands and runs every column operand through both).  No LDS is
// touched until the final cross-wave reduction.  Two steps of loads are kept in flight per wave, at least 8 waves per CU.
//
// A launch of a few experts (a handful of tokens) has too few workgroups to keep HBM busy that way: one token of a 2880-wide
// layer on two experts is 90 slabs in the gate_up product and 46 in the down product, on 256 CUs, and a CU alone moves 43 GB/s.
// There the contraction of a slab is shared by several workgroups (stream_parts), which costs about 2 us: the parts go
// through memory, and whoever comes last adds them up.  What counts is how evenly the workgroups fill the CUs, which is known
// on the device: us for 1 / 2 / 3 / 4 / 6 / 8 parts, 46 slabs of 90 steps 20.1 / 14.3 / 11.6 / 10.6 / 11.9 / 11.0, 92: 21.1 / 15.6 / 17.8 /
// 15.9 / 16.7 / 15.6, 161: 22.6 / 25.3 / 21.6 / 23.4 / 25.7 / 25.4, 180: 23.4 / 25.4 / 26.1 / 24.7 / 26.7 / 27.5, 64 of 32 steps: 11.7 /
// 10.2 / 8.5 / 8.0 / 9.0 / 9.4, 144 of 32: 12.5 / 14.4 / 12.2 / 13.7 / 15.9 / -, 112 of 16: 7.0 / 8.0 / 7.7 / 7.9 / 8.5 / 11.1 (workgroups
// of four waves, weights from memory): many parts of a short contraction cost more than they spread.  Where no list of the call
// can have more than a slab per CU, a workgroup takes eight waves with three steps in flight each, as much as a CU holds,
// folded into the first four before the same finish: one token on four experts 44.9 us, with four waves 47.5 (four tokens x 4 on
// 32 experts, 1024 wide: 28.6 and 30.5).
//
// An XCD's workgroups take neighbouring slabs, eight at a time.  Where a weight row is not a whole number of cache lines, a
// slab's piece of it shares a line with the next slab's, and both come from memory unless they meet in one L2: 64 experts, 2048 x
// 1544, 16 tokens x 8, whole layer 206 us with neighbours on different XCDs, 200 / 196 / 194 / 193 in groups of 2 / 4 / 8 / 16.  Whole
// lines gain up to 2 % (64 tokens of the 128-expert layer 812 / 806 / 806 / 796 / 797), and more where experts have rows that their
// slabs share (16 experts of 1024 x 1024, whole layer one by one / in groups: 12 rows each 38.1 / 36.3 us, 5 rows 35.0 / 34.0).  But
// groups of eight put 32 slabs of a short list on one XCD and 24 on another where 28 each would do, so with up to kXcdGroupRows
// rows per expert and kXcdGroupFrom workgroups whole lines are dealt out one by one: 168 such products of one row per expert
// 1.013 in groups (0.89 to 1.22; 224 slabs of 64 steps 24.8 / 23.4 us, 225 of 90 30.0 / 27.4), cut lines 0.94.  One stretch for each XCD
// gains no more, and with a skewed routing the experts of many rows meet on one (24 x 8 on 64, 2880 wide, Zipf: 251 us dealt out one by
// one, 263 in stretches, 250 in groups of eight).
//
// fp32 takes the same path with v_mfma_f32_16x16x4_f32.  One token on two experts of 2880 x 2880: 229 us on the tile kernel, 53
// so; 32 x 2 on 16 of them 489 / 267; 128 x 2 492 / 418; 16 x 4 on 32, 1024 wide, 123 / 74.
//
// These are the launches of calls in which every expert streams, and of calls whose tile launches are long.  Where those
// are short and there are tiles, streamed experts ride in them (stream_items in gemm_async_tile.h): the slab code is the
// same, two steps in flight beside 128 x 128 tiles and three beside 256 x 256 ones (two for 17 to 32 rows).
//
// The lane that holds accumulator column c of MFMA j owns output column 8c + j, so the 8
// accumulators of a lane are 8 consecutive output columns: the interleaved (gate, up) pairs of the
// clamped SwiGLU (csrc/moe.cpp:164-180) meet in one lane.
#include "stream_slab.h"

namespace yamoe {

constexpr int kStreamManyWaves = 8, kStreamMaxParts = 8, kStreamMostShared = 1024;
constexpr int kXcdGroup = 8, kXcdGroupFrom = 1024, kXcdGroupRows = 4;
constexpr int kChipCus = kXcds * kXcdCus;

// How many workgroups of `waves` waves share the contraction of a slab, for `slabs` of them of `steps` steps each: what takes the
// fewest steps on the CU that gets most of them, where every wave of a workgroup takes as long as the one with most steps, a
// workgroup's start and finish cost about as much as 16 steps, the parts' way through memory as 6, and each part one more.  (Fitted
// to 154 lists of 16 to 1440 slabs of 16 to 90 steps: 0.6 % over the best number of parts on average, 10 % in the worst of them.  With
// ten steps for the sharing and none for a workgroup's start it was 1.9 and 25 %: 9 x 4 tokens on 64 experts, 1024 wide, Zipf (2)
// routing, 144 slabs in seven parts, whole layer 29.8 us, 27.0 so, 26.7 unshared with eight waves; 5 x 4 on 128, Zipf, 30.9 / 28.0.)
__host__ __device__ inline int stream_parts(int slabs, int steps, int waves) {
  auto steps_of = [&](int parts) { return ceil_div(ceil_div(steps, parts), waves) * waves + 16; };
  int best = 1, cost = ceil_div(slabs, kChipCus) * steps_of(1);
  if (slabs > kSchedArrivals) return 1;
  const int most = waves == kStreamManyWaves ? kChipCus : kStreamMostShared;
#pragma unroll
  for (int p = 2; p <= kStreamMaxParts; ++p) {  // (unrolled: divisions by constants; seven parts: never better than six or eight)
    if (slabs * p > most || steps < 4 * p) break;
    const int c = ceil_div(slabs * p, kChipCus) * steps_of(p) + 6 + p;
    if (p != 7 && c < cost) { best = p; cost = c; }
  }
  return best;
}
// Whether a launch takes eight waves per workgroup, one of which fills a CU (a list holds one entry per expert here, or
// per assignment where these are fewer, unless an expert has more than a chunk of rows).
static bool stream_many_waves(int N, int E, int n_slabs) { return (long long)(N < E ? N : E) * n_slabs <= kChipCus; }

template <typename T, bool GLU, bool GATHER, int WAVES>
__global__ __launch_bounds__(kWave * WAVES, WAVES == kStreamWaves ? 2 : 1) void stream_gemm_kernel(const StreamArgs args) {
  __shared__ float red[kStreamWaves * 8 * 4 * kWave];  // [wave][j][v][lane]
  const ScheduleView sv = schedule_view(args.sched, args.N, args.E);
  if (args.yields && sv.hdr[0] > 0) return;
  const int slabs = sv.hdr[1] * args.n_slabs;
  const int parts = args.partial != nullptr ? stream_parts(slabs, ceil_div(args.Kd, StreamStep<T>::kRows), WAVES) : 1;
  const int total = slabs * parts;
  int b = blockIdx.x;
  // workgroup b runs on XCD b % 8: groups of neighbours there, dealt to the XCDs in turn (hdr[3]: the rows of all experts)
  if (args.cut_lines || total > kXcdGroupFrom || sv.hdr[3] > kXcdGroupRows * sv.hdr[1]) {
    const int place = b / kXcds, group = place / kXcdGroup;
    b = (group * kXcds + b % kXcds) * kXcdGroup + place % kXcdGroup;
  }
  if (b >= total) return;
  const int item = parts == 1 ? b : b / parts, part = b - item * parts;
  const int s = fast_div(item, args.slab_div), slab = item - s * args.n_slabs;
  const int expert = sv.small[4 * s], first = sv.small[4 * s + 1], rows = sv.small[4 * s + 2];
  constexpr int DEPTH = WAVES == kStreamWaves ? 2 : 3;
  if (rows > 16) stream_slab<T, GLU, GATHER, WAVES, 2, 2>(args, red, expert, first, rows, slab, item, part, parts);
  else stream_slab<T, GLU, GATHER, WAVES, DEPTH, 1>(args, red, expert, first, rows, slab, item, part, parts);
}

// The most workgroups that a launch may need, whatever is on its list, and (`shared`) the most of them that leave parts.
static int stream_max_entries(int N, int E, int elem_bytes) {
  return (N < E ? N : E) + (sched_may_stream_everything(N, E, elem_bytes) ? N / kStreamMaxRows : 0) + 1;
}
static long long stream_max_blocks(int N, int E, int Kd, int Nd, int elem_bytes, long long *shared) {
  const int step_rows = elem_bytes == 4 ? StreamStep<float>::kRows : StreamStep<bf16_t>::kRows;
  const int entries = stream_max_entries(N, E, elem_bytes), n_slabs = ceil_div(Nd, kSlabCols), steps = ceil_div(Kd, step_rows);
  const int waves = stream_many_waves(N, E, n_slabs) ? kStreamManyWaves : kStreamWaves;
  long long most = (long long)entries * n_slabs;
  *shared = 0;
  for (int n = 1; n <= entries && (long long)n * n_slabs <= kSchedArrivals; ++n) {
    const int parts = stream_parts(n * n_slabs, steps, waves);
    const long long blocks = (long long)n * n_slabs * parts;
    if (parts > 1 && blocks > *shared) *shared = blocks;
  }
  return most > *shared ? most : *shared;
}
// Bytes of the parts of a product, 0 where its slabs are certain not to be shared.
size_t stream_partial_bytes(int N, int E, int Kd, int Nd, int elem_bytes) {
  long long shared;
  stream_max_blocks(N, E, Kd, Nd, elem_bytes, &shared);
  return (size_t)shared * stream_part_floats(N) * sizeof(float);
}

template <typename T, bool GLU, bool GATHER>
static int launch_stream(StreamArgs a, float *partial, hipStream_t stream) {
  a.n_slabs = ceil_div(a.Nd, kSlabCols);
  a.slab_div = make_fast_div(a.n_slabs);
  a.cut_lines = a.Nd * (int)sizeof(T) % 128 != 0;
  a.partial = partial;
  a.part_floats = stream_part_floats(a.N);
  a.arrivals = const_cast<int *>(schedule_view(a.sched, a.N, a.E).arrivals);
  long long shared, blocks = stream_max_blocks(a.N, a.E, a.Kd, a.Nd, (int)sizeof(T), &shared);
  if (partial == nullptr) blocks = (long long)stream_max_entries(a.N, a.E, (int)sizeof(T)) * a.n_slabs;
  if (blocks <= 0) return 0;
  blocks = (blocks + kXcds * kXcdGroup - 1) / (kXcds * kXcdGroup) * (kXcds * kXcdGroup);
  if (stream_many_waves(a.N, a.E, a.n_slabs))
    hipLaunchKernelGGL((stream_gemm_kernel<T, GLU, GATHER, kStreamManyWaves>), dim3((unsigned)blocks), dim3(kWave * kStreamManyWaves), 0, stream, a);
  else
    hipLaunchKernelGGL((stream_gemm_kernel<T, GLU, GATHER, kStreamWaves>), dim3((unsigned)blocks), dim3(kStreamThreads), 0, stream, a);
  return check_launch("stream_gemm_kernel");
}

// partial: room for stream_partial_bytes of this product, or null (the slabs are not shared then)
template <typename T>
int stream_gate_up(const void *x, const int *sorted_idx, const void *w, const void *bias, void *act, void *pre,
                   const void *sched, int N, int K, int E, int H, int I, float *partial, bool yields, hipStream_t stream) {
  StreamArgs a = {};
  a.yields = yields;
  a.A = x; a.B = w; a.bias = bias; a.C = act; a.C2 = pre; a.a_rows = sorted_idx; a.a_div = make_fast_div(K);
  a.sched = (const int *)sched; a.Kd = H; a.Nd = 2 * I; a.lda = H; a.ldc = I; a.N = N; a.E = E;
  return launch_stream<T, true, true>(a, partial, stream);
}

template <typename T>
int stream_down(const void *act, const void *w, const void *bias, void *y, const void *sched, int N, int E, int H,
                int I, float *partial, bool yields, hipStream_t stream) {
  StreamArgs a = {};
  a.yields = yields;
  a.A = act; a.B = w; a.bias = bias; a.C = y; a.a_div = make_fast_div(1); a.sched = (const int *)sched;
  a.Kd = I; a.Nd = H; a.lda = I; a.ldc = H; a.N = N; a.E = E;
  return launch_stream<T, false, false>(a, partial, stream);
}

#define YAMOE_INSTANTIATE_STREAM(T)                                                                                  \
  template int stream_gate_up<T>(const void *, const int *, const void *, const void *, void *, void *, const void *, \
                                 int, int, int, int, int, float *, bool, hipStream_t);                                     \
  template int stream_down<T>(const void *, const void *, const void *, void *, const void *, int, int, int, int, \
                              float *, bool, hipStream_t);
YAMOE_INSTANTIATE_STREAM(float)
YAMOE_INSTANTIATE_STREAM(bf16_t)
YAMOE_INSTANTIATE_STREAM(f16_t)

}  // namespace yamoe
