// The pipelined tiled product with the gated epilogue (gate/up + activation): the kernel of gemm_pipe.h in the shapes that
// gemm_pipe.hip's cost model picks.
#include "gemm_pipe.h"

namespace sprout {

// out[T, I] = silu(x . w[:I]^T) * (x . w[I:]^T): a block's weight rows are half gate rows, half the matching up rows.
int gemm_bf16_pipe_silu(hipStream_t s, const void* x, const void* w, void* out, int T, int I, int K, int act, float limit,
                        const float* row_gate, long long row_gate_stride) {
  const uint16_t *xp = (const uint16_t*)x, *wp = (const uint16_t*)w;
  RopeArgs epi = {};
  epi.act = act;
  epi.limit = limit;
  epi.row_gate = row_gate;
  epi.row_gate_stride = row_gate_stride;
  int shape, splits;
  pipe_choice(T, 2 * I, K, false, &shape, &splits, true);
  if (shape == 0) return launch_pipe_mode<4, 2, 2, 4, 2, kSilu, float>(s, 1, xp, wp, nullptr, out, T, I, K, K, epi);
  if (shape == 1) return launch_pipe_mode<2, 2, 4, 2, 3, kSilu, float>(s, 1, xp, wp, nullptr, out, T, I, K, K, epi);
  if (shape == 4) return launch_pipe_mode<1, 2, 2, 4, 3, kSilu, float>(s, 1, xp, wp, nullptr, out, T, I, K, K, epi);
  if (shape == 5) return launch_pipe_mode<1, 2, 2, 2, 3, kSilu, float>(s, 1, xp, wp, nullptr, out, T, I, K, K, epi);
  if (shape == 6) return launch_pipe_mode<6, 2, 2, 4, 2, kSilu, float>(s, 1, xp, wp, nullptr, out, T, I, K, K, epi);
  if (shape == 7) return launch_pipe_mode<1, 2, 2, 1, 4, kSilu, float>(s, 1, xp, wp, nullptr, out, T, I, K, K, epi);
  return launch_pipe_mode<1, 2, 4, 2, 4, kSilu, float>(s, 1, xp, wp, nullptr, out, T, I, K, K, epi);
}

// Rows and columns of every block shape, by its index in gemm_pipe.hip's list.
static const int kShapeRows[] = {256, 256, 128, 64, 64, 64, 384, 64, 256};
static const int kShapeCols[] = {256, 128, 128, 64, 256, 128, 256, 64, 160};
static const int kShapeWaves[] = {8, 8, 8, 4, 8, 4, 8, 2, 4};

}  // namespace sprout

// What the pipelined product would do with T x N x K: kind 0 store, 1 accumulate, 2 gated (N = 2 I rows of w).
// plan = {block rows, block columns, splits of K, waves of a block}.  Returns 1 where the pipelined kernel
// does not take the product, else 0.  Runs nothing: for tests and tools.
extern "C" int sp_pipe_plan(int kind, int T, int N, int K, int* plan) {
  using namespace sprout;
  if (T < 1 || N < 1 || K < 1 || kind < 0 || kind > 2 || !plan || !gemm_pipe_takes(T, N, K)) return 1;
  int shape, splits = 1;
  pipe_choice(T, N, K, kind == 1, &shape, &splits, kind == 2);
  if (shape < 0 || shape >= int(sizeof(kShapeRows) / sizeof(kShapeRows[0]))) return 1;
  plan[0] = kShapeRows[shape];
  plan[1] = kShapeCols[shape];
  plan[2] = splits;
  plan[3] = kShapeWaves[shape];
  return 0;
}

// The tile of every block of a launch over tiles_t token tiles and tiles_n weight tiles, as the kernel numbers them:
// tile_of[2 b] = token tile and tile_of[2 b + 1] = weight tile of block b, both -1 for a block with nothing to do.
// Returns the number of blocks (8 for each place on an XCD), or -1; writes at most `room` blocks.  Runs nothing.
extern "C" int sp_pipe_tiles(int tiles_t, int tiles_n, int* tile_of, int room) {
  using namespace sprout;
  if (tiles_t < 1 || tiles_n < 1 || !tile_of) return -1;
  const PipeTiles tiles = pipe_tiles(tiles_t, tiles_n);
  const int blocks = 8 * (tiles.own + tiles.run);
  for (int b = 0; b < blocks && b < room; ++b)
    if (!pipe_tile_of(tiles, b, &tile_of[2 * b], &tile_of[2 * b + 1])) tile_of[2 * b] = tile_of[2 * b + 1] = -1;
  return blocks;
}
