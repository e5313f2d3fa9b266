// The four-wave tiled product that adds to its output, and the choice between the block shapes.  The kernel is in gemm_quad.h;
// the stores and the gated and rotating epilogues are instantiated in gemm_quad_store.hip and gemm_quad_epilogues.hip, so that
// the parts compile side by side.
#include "gemm_quad.h"

namespace sprout {

// 17 to 64 tokens, where the weights are read from memory once and the other kernels do that as well.  Both were timed at ten numbers of
// tokens from 17 to 64 on 325 matrices (a launch of a captured graph, weights from memory).  Time here over time there, on either side of
// each line: mean, and the least and the most of the side that is taken.
//   gated, up to 16,384 rows: below 64 M weights 0.76 (0.58 .. 0.96), above 0.99; more rows: K up to 1,536 0.96 (0.87 .. 1.04; beyond
//     24,576 rows and 40 tokens 0.99), K above 1.07;
//   added, 33 tokens and more: 4 to 64 M weights 0.85 (0.67 .. 1.08; the first 4 M of them 0.84), 2 to 4 M 0.94, more than 64 M 0.95 with
//     1.15 among them; up to 32 tokens: from 6 M weights on, where the other kernel is the eight-wave one, 0.87 (0.67 .. 1.06; to 12 M
//     0.83), 3 to 6 M 1.02;
//   stored, 33 tokens and more: from 2 M weights on 0.70 (0.39 .. 0.94; to 4 M 0.76), less 1.00; up to 32 tokens: 8,192 rows and more,
//     or 6,144 with K up to 4,096, from 8 M weights on 0.78 (0.53 .. 1.04), others 1.02 with 1.16 among them; heads of 32,768 rows and more:
//     K up to 2,048 0.91 (0.82 .. 0.99), 2,560 to 3,584 1.02 with 1.19 among them.
static bool quad_pays_for_few(int kind, int T, int N, int K) {
  const size_t weights = size_t(N) * K, million = 1000000;
  if (kind == kQuadGated) return N <= 16384 ? weights < 64 * million : K <= 1536 && (N <= 24576 || T <= 40);
  if (kind == kQuadAccumulate) return weights >= (T > 32 ? 4 * million : size_t(6) << 20) && weights < 64 * million;
  if (kind != kQuadStore) return false;
  if (N >= 32768) return K <= 2048;
  return T > 32 ? weights >= 2 * million : weights >= 8 * million && (N >= 8192 || (N >= 6144 && K <= 4096));
}

bool gemm_quad_takes(int kind, int T, int N, int K, int hd) {
  if (T <= 16 || !gemm_pipe_takes(T, N, K)) return false;
  if (T <= 64 && !quad_pays_for_few(kind, T, N, K)) return false;
  if (kind == kQuadGated) return N % 16 == 0;
  if (kind == kQuadRotating) return hd % 64 == 0 && N % hd == 0;
  return N % 8 == 0;
}

// What was measured of the block shapes, fitted over 56 products (weights of 896 to 37,888 rows and K of 896 to 18,944, 80 to 2,048
// tokens) with every shape and split: microseconds a step of 64 along K on a full chip, and, where two blocks share a CU, of one that
// has a CU to itself.
struct QuadShape { int wm, wn, buffers, per_cu; };
#define SPROUT_QUAD_ROW(I, WM, WN, NA) {WM, WN, NA, quad_shares_cu<WM, WN, NA> ? 2 : 1},
static const QuadShape kQuadShapes[] = {SPROUT_QUAD_SHAPES(SPROUT_QUAD_ROW)};
static const QuadShape kQuadOddShapes[] = {SPROUT_QUAD_ODD_SHAPES(SPROUT_QUAD_ROW)};
#undef SPROUT_QUAD_ROW
static const float kStepUs[] = {0.36f, 0.77f, 0.35f, 0.85f, 0.48f, 0.68f, 0.80f, 0.66f, 0.86f, 0.77f, 0.81f, 0.96f, 0.93f, 1.06f, 1.06f, 1.19f, 1.33f};
static const float kAloneUs[] = {0.24f, 0.45f, 0.35f, 0.50f, 0.48f, 0.68f, 0.80f, 0.66f, 0.86f, 0.77f, 0.81f, 0.96f, 0.93f, 1.06f, 1.06f, 1.19f, 1.33f};
static const float kOddStepUs[] = {0.98f, 1.14f, 1.22f, 1.40f};

// The estimate: rounds of blocks on the XCD that holds the most (blocks are numbered as pipe_tiles says), a block being its steps
// (longer by 7 % each beyond 20 where two blocks share a CU) and its two ends; a last round that does not fill the chip runs
// somewhat faster, fewer blocks share the caches.  Memory: the weights once at 5.4 TB/s and, at 9 TB/s together (8 with two buffers of x), the tokens once an
// XCD, or, where there are less than 8 weight tiles and an XCD has a run of their blocks, once a weight tile; it adds to the blocks'
// time where both are alike (fourth powers).  A split's float atomics cost 1.9 us a million, the sums read and written without a split
// 1.4.  Over 1,100 products (65 to 8,192 tokens, 512 to 6,144 weight rows, K of 896 to 18,944) the choice takes 1.3 % longer than the best
// of all shapes and splits (mean; 25 % at worst), 10 % less than the eight-wave kernel, and more than 3 % longer than that one on 18 (10 %
// at worst).  (With the tokens read once an XCD whatever the weight tiles: 4,096 tokens by 512 rows of 8,192 in one part on 128 x 64, 80 us,
// where 128 x 128 in two takes 48 and the eight-wave kernel 50.)
//
// Parts that are stored side by side and joined by the norm that reads them: their blocks are an equal run an XCD (quad_part_of), whose
// operands are what the XCD reads, once each where the caches serve it; 0.7 us a million sums stored, and 5 TB/s for the norm to read all
// parts and to write their sum.  Over 80 products (70 to 2,048 tokens, eight matrices of 896 to 5,120 rows) the choice takes 3 % longer than
// the best of all shapes and parts, 10 % at worst.
static float least_time(int kind, int T, int N, int K, const QuadShape* shapes, const float* step_us, const float* alone_us, int n_shapes, int* shape,
                        int* splits) {
  const int steps = K / 64;
  const bool parts = kind == kQuadParts, cuts_k = parts || (kind == kQuadAccumulate && gemm_cuts_k(T, N, K));
  float best = 1e30f;
  for (int c = 0; c < n_shapes; ++c) {
    const QuadShape& p = shapes[c];
    if (kind == kQuadRotating && p.wn != 2 && p.wn % 4 != 0) continue;     // a lane holds both of a pair
    const int bm = 32 * p.wm, bn = 32 * p.wn, slots = 32 * p.per_cu;
    const PipeTiles tiles = pipe_tiles((T + bm - 1) / bm, (N + bn - 1) / bn);
    const float caches = p.buffers == 2 ? 8e6f : 9e6f;
    float memory = float(N) * float(K) * 2.f / 5.4e6f + float(tiles.full ? 8 : tiles.left) * 2.f * float(T) * float(K) / caches;
    for (int sp : {1, 2, 3, 4, 6, 8, 12, 16}) {
      if (sp > 1 && (!cuts_k || steps / sp < 4)) break;
      if (sp == 1 && parts) continue;
      const int k_steps = (steps + sp - 1) / sp;
      if ((steps + k_steps - 1) / k_steps != sp) continue;
      int blocks = (tiles.full * tiles.tiles_t + tiles.run) * sp;
      if (parts) {
        const int tiles_n = (N + bn - 1) / bn;
        blocks = (tiles.tiles_t * tiles_n * sp + 7) / 8;
        // what an XCD's run holds of one part: all token tiles and some weight tiles, or some token tiles of one weight tile
        const float of_parts = fmaxf(1.f, float(sp) / 8.f), run = float(blocks) / of_parts;
        const float rows = fminf(float(N), fminf(float(tiles_n), ceilf(run / tiles.tiles_t)) * bn), tokens = fminf(float(T), run * bm);
        const float fetched = 16.f * of_parts * (rows + tokens) * float(K) / float(sp);
        memory = float(N) * float(K) * 2.f / 5.4e6f + (fetched - float(N) * float(K) * 2.f) / caches;
      }
      const float memory2 = memory * memory;
      const int full = blocks / slots, rest = blocks % slots;
      const float ends = 0.14f * float(p.wm * p.wn) + 0.95f;
      const float block = k_steps * step_us[c] * (p.per_cu == 2 && k_steps > 20 ? 1.07f : 1.f) + ends, alone = k_steps * alone_us[c] + ends;
      float t = full * block;
      if (rest > 32) t += fmaxf(alone, block * (0.81f + 0.19f * float(rest - 32) / 32.f));
      else if (rest) t += alone * (0.79f + 0.21f * float(rest) / 32.f);
      t = sqrtf(sqrtf(t * t * t * t + memory2 * memory2));
      if (parts) t += (0.7e-6f * sp + 0.8e-6f * (sp + 1)) * float(T) * float(N);
      else if (sp > 1) t += 1.9e-6f * float(T) * float(N) * sp;
      else if (kind == kQuadAccumulate) t += 1.4e-6f * float(T) * float(N);
      if (t < best) { best = t; *shape = c; *splits = sp; }
    }
  }
  return best;
}

float quad_choice(int kind, int T, int N, int K, int* shape, int* splits) {
  *shape = 3;
  *splits = 1;
  return least_time(kind, T, N, K, kQuadShapes, kStepUs, kAloneUs, int(sizeof(kQuadShapes) / sizeof(kQuadShapes[0])), shape, splits);
}

// Where the estimate says 2 % less: of 57 gated products (65 to 2,048 tokens at 0.5B, 7B and 32B sizes), each timed on every shape, the 17 that
// this takes are 0.81 to 0.99 of the time (0.93 on average) and none is longer; without the margin one is, by 2.6 %.
bool quad_takes_odd(int T, int N, int K, int* shape) {
  int even, splits;
  return least_time(kQuadGated, T, N, K, kQuadOddShapes, kOddStepUs, kOddStepUs, int(sizeof(kQuadOddShapes) / sizeof(kQuadOddShapes[0])), shape, &splits) <
         0.98f * quad_choice(kQuadGated, T, N, K, &even, &splits);
}

// Parts of K in which the accumulating product is better stored for the norm behind it to join, 0 where it is better added: more than 64
// tokens, at most 128 MiB of sums.
int quad_parts(int T, int N, int K) {
  int shape, parts, splits;
  if (T <= 64 || !gemm_quad_takes(kQuadAccumulate, T, N, K) || K / 64 < 8) return 0;
  const float stored = quad_choice(kQuadParts, T, N, K, &shape, &parts), added = quad_choice(kQuadAccumulate, T, N, K, &shape, &splits);
  return stored < added && size_t(parts) * T * N <= (size_t(32) << 20) ? parts : 0;
}

int gemm_bf16_quad_store(hipStream_t s, const void* x, const void* w, int bias_dtype, const void* bias, bool f32, void* out, int T, int N, int K,
                         const RopeArgs& epilogue);

int gemm_bf16_quad(hipStream_t s, const void* x, const void* w, int bias_dtype, const void* bias, int mode, void* out, int T, int N, int K) {
  if (mode == kAccumulate) return quad_run<kAccumulate>(s, kQuadAccumulate, x, w, bias, bias_dtype, out, T, N, K);
  return gemm_bf16_quad_store(s, x, w, bias_dtype, bias, mode == kStoreF32, out, T, N, K, RopeArgs{});
}

}  // namespace sprout

// What the four-wave product would do with T x N x K on blocks of an even number of tile columns a wave: kind 0 store, 1 accumulate, 2 gated (N = 2 I
// rows of w; sp_quad_odd_plan says where others take its place), 3 rotating (head size hd), 4 parts side by side.  plan = {block rows, block columns, splits of K, buffers of x}.  Returns 1 where it does not take the product, else 0.  Runs
// nothing: for tests and tools.
extern "C" int sp_quad_plan(int kind, int T, int N, int K, int hd, int* plan) {
  using namespace sprout;
  if (T < 1 || N < 1 || K < 1 || kind < 0 || kind > 4 || !plan || (kind == kQuadRotating && hd < 1) || !gemm_quad_takes(kind, T, N, K, hd)) return 1;
  int shape, splits;
  quad_choice(kind, T, N, K, &shape, &splits);
  plan[0] = 32 * kQuadShapes[shape].wm;
  plan[1] = 32 * kQuadShapes[shape].wn;
  plan[2] = splits;
  plan[3] = kQuadShapes[shape].buffers;
  return 0;
}

// Whether a gated product that the four-wave kernel takes (T tokens, N = 2 I rows of w) runs on blocks of an odd number of tile columns a wave: plan =
// {block rows, block columns, buffers of x}.  Returns 1 where it does not, else 0.  Runs nothing: for tests.
extern "C" int sp_quad_odd_plan(int T, int N, int K, int* plan) {
  using namespace sprout;
  int shape;
  if (T < 1 || N < 1 || K < 1 || !plan || !gemm_quad_takes(kQuadGated, T, N, K, 0) || !quad_takes_odd(T, N, K, &shape)) return 1;
  plan[0] = 32 * kQuadOddShapes[shape].wm;
  plan[1] = 32 * kQuadOddShapes[shape].wn;
  plan[2] = kQuadOddShapes[shape].buffers;
  return 0;
}

// The tiles of a product in `parts` parts side by side, block by block: tile_of[3 b] = (token tile, weight tile, part) of block b of
// tiles_t * tiles_n * parts.  Runs nothing: for tests.
extern "C" int sp_quad_part_tiles(int tiles_t, int tiles_n, int parts, int* tile_of) {
  if (tiles_t < 1 || tiles_n < 1 || parts < 1 || !tile_of) return 1;
  const int blocks = tiles_t * tiles_n * parts;
  for (int b = 0; b < blocks; ++b) sprout::quad_part_of(tiles_t, tiles_n, b, blocks, &tile_of[3 * b], &tile_of[3 * b + 1], &tile_of[3 * b + 2]);
  return 0;
}
