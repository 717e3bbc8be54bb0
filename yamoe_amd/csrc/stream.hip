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
// A launch that can hold only a few experts (a handful of tokens: at most kStreamFewBlocks workgroups) has too few
// workgroups to keep HBM busy that way: 4 experts x 23 slabs with two steps of 8 KB in flight per wave are 6 MB on
// the way, where 8 TB/s x 2 us of latency want 16 MB.  Such a launch takes 8 waves per workgroup with three steps in
// flight each instead (16 waves with two steps each measured 3 % slower), folded into the first four before the same
// finish.  One token of a 2880-wide layer on four experts is 180 workgroups in the gate_up product and 92 in the down
// product, on 256 CUs: 22 us for 132 MB of weights and 19 us for 66 MB.
//
// These are the launches of calls in which every expert streams, and of calls whose tile launches are long.  Where those
// are short and there are tiles, streamed experts ride in them (stream_items in gemm_async_tile.h): the slab code is the
// same, with four waves whatever the number of experts, two steps in flight beside 128 x 128 tiles and three beside
// 256 x 256 ones (two for 17 to 32 rows).
//
// The lane that holds accumulator column c of MFMA j owns output column 8c + j, so the 8
// accumulators of a lane are 8 consecutive output columns: the interleaved (gate, up) pairs of the
// clamped SwiGLU (csrc/moe.cpp:164-180) meet in one lane.
#include "stream_slab.h"

namespace yamoe {

constexpr int kStreamManyWaves = 8;
constexpr int kStreamFewBlocks = 1024;  // launches with fewer (expert, slab) workgroups than this take 8 waves each
template <typename T, bool GLU, bool GATHER, int WAVES, int DEPTH>
__global__ __launch_bounds__(64 * WAVES, WAVES == kStreamWaves ? 2 : 1) void stream_gemm_kernel(const StreamArgs args) {
  __shared__ float red[kStreamWaves * 8 * 4 * kWave];  // [wave][j][v][lane]
  const ScheduleView sv = schedule_view(args.sched, args.N, args.E);
  const int n_small = sv.hdr[1];
  const int s = blockIdx.x / args.n_slabs;
  if (s >= n_small) return;
  const int slab = blockIdx.x - s * args.n_slabs;
  const int expert = sv.small[4 * s], first = sv.small[4 * s + 1], rows = sv.small[4 * s + 2];
  if (rows > 16) stream_slab<T, GLU, GATHER, WAVES, DEPTH, 2>(args, red, expert, first, rows, slab);
  else stream_slab<T, GLU, GATHER, WAVES, DEPTH, 1>(args, red, expert, first, rows, slab);
}

template <typename T, bool GLU, bool GATHER>
static int launch_stream(const StreamArgs &a, hipStream_t stream) {
  long long blocks = (long long)sched_max_small(a.N, a.E) * a.n_slabs;
  if (blocks <= 0) return 0;
  if (blocks < kStreamFewBlocks) {
    hipLaunchKernelGGL((stream_gemm_kernel<T, GLU, GATHER, kStreamManyWaves, 3>), dim3((unsigned)blocks),
                       dim3(64 * kStreamManyWaves), 0, stream, a);
  } else {
    hipLaunchKernelGGL((stream_gemm_kernel<T, GLU, GATHER, kStreamWaves, 2>), dim3((unsigned)blocks), dim3(64 * kStreamWaves),
                       0, stream, a);
  }
  return check_launch("stream_gemm_kernel");
}

template <typename T>
int stream_gate_up(const void *x, const int *sorted_idx, const void *w, const void *bias, void *act, void *pre,
                   const void *sched, int N, int K, int E, int H, int I, hipStream_t stream) {
  StreamArgs a = {};
  a.A = x; a.B = w; a.bias = bias; a.C = act; a.C2 = pre; a.a_rows = sorted_idx; a.a_div = make_fast_div(K);
  a.sched = (const int *)sched; a.Kd = H; a.Nd = 2 * I; a.lda = H; a.ldc = I;
  a.n_slabs = ceil_div(2 * I, kSlabCols); a.N = N; a.E = E;
  return launch_stream<T, true, true>(a, stream);
}

template <typename T>
int stream_down(const void *act, const void *w, const void *bias, void *y, const void *sched, int N, int E, int H,
                int I, hipStream_t stream) {
  StreamArgs a = {};
  a.A = act; a.B = w; a.bias = bias; a.C = y; a.a_div = make_fast_div(1); a.sched = (const int *)sched;
  a.Kd = I; a.Nd = H; a.lda = I; a.ldc = H;
  a.n_slabs = ceil_div(H, kSlabCols); a.N = N; a.E = E;
  return launch_stream<T, false, false>(a, stream);
}

#define YAMOE_INSTANTIATE_STREAM(T)                                                                                  \
  template int stream_gate_up<T>(const void *, const int *, const void *, const void *, void *, void *, const void *, \
                                 int, int, int, int, int, hipStream_t);                                              \
  template int stream_down<T>(const void *, const void *, const void *, void *, const void *, int, int, int, int,    \
                              hipStream_t);
YAMOE_INSTANTIATE_STREAM(bf16_t)
YAMOE_INSTANTIATE_STREAM(f16_t)

}  // namespace yamoe
