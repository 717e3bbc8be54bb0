// Grouped expert GEMMs for 16-bit data on gfx950: the products over the rows of the schedule's tiles (the forward's two
// and the two input gradients).  This file holds the instantiations for 256 x 256 tiles and contractions of whole slab
// pairs; gemm_async_ragged.hip (other contractions) and gemm_async_small.hip (128 x 128 tiles) include it, so that the
// three compile side by side.
#include "gemm_async_tile.h"

namespace yamoe {

static_assert(async::Tile<256, 256>::BM == kRowTile && async::Tile<256, 256>::BN == kColTile,
              "tiles of the schedule must match the GEMM tile");

#if defined(YAMOE_TILE_STAMPS) && !defined(YAMOE_INSTANTIATE_ROWS)
// Where the next launches of gemm_async_kernel leave their per-tile clock stamps (device memory, 8 words per tile, room
// for `tiles` tiles; nullptr switches them off).  Exported by the diagnostic build only.
extern "C" void yamoe_debug_tile_stamps(void *buffer, int32_t tiles) {
  async::g_tile_stamps = (unsigned long long *)buffer;
  async::g_tile_stamps_cap = buffer ? tiles : 0;
}
#endif

// the streaming list of the schedule goes with the tiles
static void add_streams(async::Args &a, int N, int E, int carries) {
  a.n_stream_slabs = ceil_div(a.Nd, kSlabCols);
  const long long items = (long long)(N < E ? N : E) * a.n_stream_slabs;
  a.stream_wgs = items < kXcds * kXcdCus ? ceil_div((int)items, kXcds) : kXcdCus;
  a.small = schedule_view(a.sched, N, E).small;
  a.carries_alone = carries == CARRY_ALWAYS;
}

template <typename T, int TILE, bool RAGGED>
int gemm_async_gate_up(const void *x, const int *sorted_idx, const void *w, const void *bias, void *act, void *pre,
                       const void *sched, int N, int K, int E, int H, int I, int small_rows, int carries, hipStream_t stream) {
  async::Args a = {};
  a.A = x; a.B = w; a.bias = bias; a.C = act; a.C2 = pre;
  a.a_rows = sorted_idx; a.a_div = make_fast_div(K); a.sched = (const int *)sched;
  a.Kd = H; a.Nd = 2 * I; a.lda = H; a.ldb = 2 * I; a.ldc = I;
  a.b_expert_stride = (long long)H * 2 * I;
  a.n_col_tiles = ceil_div(2 * I, TILE);
  a.n_col_div = make_fast_div(a.n_col_tiles);
  a.band_div = make_fast_div(async::kBandRows * a.n_col_tiles);
  const int row_tiles = sched_grid_row_tiles(N, E, small_rows);
  using S = async::Tile<TILE, TILE>;
  if (carries == CARRY_NOT) return async::launch<T, S, async::EPI_GLU, true, false, RAGGED, async::FORM_LIST>(a, row_tiles, stream);
  add_streams(a, N, E, carries);
  return async::launch<T, S, async::EPI_GLU, true, false, RAGGED, async::FORM_CARRIER>(a, row_tiles, stream);
}

template <typename T, int TILE, bool RAGGED>
int gemm_async_down(const void *act, const void *w, const void *bias, void *y, const void *sched, int N, int E, int H,
                    int I, int small_rows, int carries, int regular_rows, hipStream_t stream) {
  async::Args a = {};
  a.A = act; a.B = w; a.bias = bias; a.C = y; a.sched = (const int *)sched;
  a.Kd = I; a.Nd = H; a.lda = I; a.ldb = H; a.ldc = H;
  a.b_expert_stride = (long long)I * H;
  a.n_col_tiles = ceil_div(H, TILE);
  a.n_col_div = make_fast_div(a.n_col_tiles);
  a.band_div = make_fast_div(async::kBandRows * a.n_col_tiles);
  using S = async::Tile<TILE, TILE>;
  if (regular_rows > 0) {  // cut like the schedule's: equal tiles, multiples of 32 rows
    a.reg_rows = regular_rows;
    a.reg_tiles = ceil_div(regular_rows, kRowTile);
    a.reg_per_tile = (ceil_div(regular_rows, a.reg_tiles) + 31) & ~31;
    a.reg_units = E * a.n_col_tiles;
    a.reg_div = make_fast_div(a.reg_tiles * a.n_col_tiles);
    a.reg_tile_div = make_fast_div(a.reg_tiles);
    return async::launch<T, S, async::EPI_STORE, false, false, RAGGED, async::FORM_REGULAR>(a, E * a.reg_tiles, stream);
  }
  const int row_tiles = sched_grid_row_tiles(N, E, small_rows);
  if (carries == CARRY_NOT) return async::launch<T, S, async::EPI_STORE, false, false, RAGGED, async::FORM_LIST>(a, row_tiles, stream);
  add_streams(a, N, E, carries);
  return async::launch<T, S, async::EPI_STORE, false, false, RAGGED, async::FORM_CARRIER>(a, row_tiles, stream);
}

// C[rows, Nd] = A[rows, Kd] * W[e]^T with W[e] stored [Nd, Kd]: the input gradients of both projections
// (csrc/experts_backward.cu:279-282, 309-311), without materialising a transposed weight.
// With g_rows the source row of sorted row p is g_rows[p] / g_div (rows of a [T, Kd] tensor gathered by token).
template <typename T, int TILE, bool RAGGED>
int gemm_async_dgrad(const void *g, const int *g_rows, int g_div, const void *w, void *out, const void *sched, int N,
                     int E, int Kd, int Nd, const void *dot_with, float *dot_part, hipStream_t stream) {
  async::Args a = {};
  a.A = g; a.B = w; a.bias = nullptr; a.C = out; a.sched = (const int *)sched;
  a.dot_with = dot_with; a.dot_part = dot_part;
  a.a_rows = g_rows; a.a_div = make_fast_div(g_rows != nullptr ? g_div : 1);
  a.Kd = Kd; a.Nd = Nd; a.lda = Kd; a.ldb = Kd; a.ldc = Nd;
  a.b_expert_stride = (long long)Nd * Kd;
  a.n_col_tiles = ceil_div(Nd, TILE);
  a.n_col_div = make_fast_div(a.n_col_tiles);
  a.band_div = make_fast_div(async::kBandRows * a.n_col_tiles);
  using S = async::Tile<TILE, TILE>;
  if (g_rows != nullptr)
    return async::launch<T, S, async::EPI_STORE, true, true, RAGGED, async::FORM_LIST>(a, sched_max_row_tiles(N, E), stream);
  return async::launch<T, S, async::EPI_STORE, false, true, RAGGED, async::FORM_LIST>(a, sched_max_row_tiles(N, E), stream);
}

#define YAMOE_INSTANTIATE_ASYNC(T, TILE, RAGGED)                                                                        \
  template int gemm_async_gate_up<T, TILE, RAGGED>(const void *, const int *, const void *, const void *, void *,       \
                                                   void *, const void *, int, int, int, int, int, int, int, hipStream_t);     \
  template int gemm_async_down<T, TILE, RAGGED>(const void *, const void *, const void *, void *, const void *, int,    \
                                                int, int, int, int, int, int, hipStream_t);                                   \
  template int gemm_async_dgrad<T, TILE, RAGGED>(const void *, const int *, int, const void *, void *, const void *,    \
                                                 int, int, int, int, const void *, float *, hipStream_t);
#ifndef YAMOE_INSTANTIATE_ROWS
#define YAMOE_INSTANTIATE_ROWS            \
  YAMOE_INSTANTIATE_ASYNC(bf16_t, 256, false) \
  YAMOE_INSTANTIATE_ASYNC(f16_t, 256, false)
#endif
YAMOE_INSTANTIATE_ROWS

}  // namespace yamoe
