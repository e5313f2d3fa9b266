// bfloat16 attention with softmax weights: the instantiations, the sizes the kernels take, and the one-query kernel with the
// output projection folded in.
#include "attention_mfma.h"

namespace sprout {

bool gemm_adds_parts(int T, int N, int K);      // gemm_bf16.hip
constexpr int kProjectColumns = 512;      // most columns of w_o that a set of heads has where attention and projection share a block

bool attention_mfma_supports(int hd, int page_size, int nq, int nkv) {
  const int dt = hd / 16;
  const bool hd_ok = hd % 16 == 0 && (dt <= 6 || dt == 8 || dt == 10 || dt == 12 || dt == 16);
  return hd_ok && page_size % 4 == 0;
}
bool attention_mfma_decode_supports(int nq, int nkv) { return true; }
int attention_mfma_tile_q(int hd) { return 32; }

// Blocks per tile and set of heads along the keys: the number of parts with the least estimated time in microseconds.  A step with few
// queries over a long context (a portion of a long prompt) has few tiles, each with a long walk.  `stage`: a block's 128 keys while
// `places` blocks run at once (a CU holds one block of eight waves; of four waves as many as share it without taking longer); `ends`: its
// queries, its waves' merge, its stores.  One-query blocks that share the launch (`beside`) take hd / 16 us for their 256 keys, in
// the places which the last round of prompt blocks leaves free and in rounds behind it.  Every part costs the
// merge what it writes and reads again, 0.8 us a million bytes.  max_tile_ctx is the longest walk, mean_tile_walk what tiles walk on average.
// A part holds two stages at least, of wide heads one (8 heads of 256, 128 queries behind 512: five parts 22.5 us, two 34.7).
// Fitted to 1,555 steps (fifteen shapes of heads; 48 to 960 queries behind 0 to 30,720 keys, alone, beside one to 45 answers and beside short
// prompts) timed with one to 24 parts: the choice takes 2.3 % longer than the best of them on average, 25 % or more at 10.  A rule by the number
// of blocks alone (as many parts as give every CU a block, half as many beside answers) took 5 to 9 % longer on walks of up to 2,500
// keys and 56 % on longer ones at 28 heads of 128 in 4 groups: 257 queries behind 30,720 beside eight answers one part 608 us, three
// 219; 512 of them one 605, two 333; 640 alone one 604, three 425; 40 heads in 8 groups, 257 queries behind 30,720 one 586, eight 376.
int attention_prefill_parts(int n_tiles, int nq, int nkv, int hd, int page_size, int max_tile_ctx, int mean_tile_walk, long long beside) {
  if (!staged_prefill(page_size) || n_tiles < 1) return 1;
  const StagedShape shape = staged_shape(nq, nkv, hd, n_tiles);
  const int G = nq / nkv, blocks = n_tiles * nkv * ((G + shape.hpb - 1) / shape.hpb), stages = (max_tile_ctx + kStageKeys - 1) / kStageKeys;
  if (blocks >= 2048 / (shape.wpt * shape.hpb) || stages <= 4) return 1;
  const bool small = shape.wpt * shape.hpb == 4 && hd <= 128;      // blocks of four waves of which a CU holds several
  const int places = !small ? 256 : hd <= 32 ? 1024 : hd <= 64 ? 768 : 512;
  const float ends = small ? 2.f : 6.f;
  const float stage = hd > 192 ? 6.f : hd > 128 ? 4.8f : small ? (hd <= 32 ? 0.8f : hd <= 64 ? 1.1f : 2.5f)
                    : shape.hpb == 4 ? 2.3f : hd <= 64 ? 1.45f : 1.95f;
  const float walked = fminf(1.f, float(max(1, mean_tile_walk)) / float(max_tile_ctx));
  const float unit = float(hd) / 16.f, units = float(beside) / (float(shape.wpt * shape.hpb) / 4.f);
  const float merged = 0.8e-6f * float(n_tiles) * 32.f * float(nq) * float(hd + 2) * 4.f;
  const int most = min(hd > 128 ? stages : stages / 2, kMaxPrefillSplits);
  int best = 1;
  float least = 1e30f;
  for (int parts = 1; parts <= most; ++parts) {
    const float longest = ends + float((stages + parts - 1) / parts) * stage, mean = ends + float((stages + parts - 1) / parts) * stage * walked;
    const int full = blocks * parts / places, rest = blocks * parts % places;
    const float behind = rest ? fmaxf(0.f, units - float(places - rest) * floorf(mean / unit)) : units;
    float us = fmaxf(longest, float(full + (rest > 0)) * mean + ceilf(behind / float(places)) * unit);
    if (parts > 1) us += merged * float(parts);
    if (us < least) least = us, best = parts;
  }
  return best;
}

size_t attention_prefill_workspace_floats(int n_tiles, int nq, int nkv, int hd, int page_size, int max_tile_ctx, int mean_tile_walk, int n_decode,
                                          int max_decode_ctx, long long one_query_keys) {
  const long long beside = chunks_beside(hd, nq, nkv, n_tiles, n_decode, max_decode_ctx, one_query_keys);
  const size_t splits = max(attention_prefill_parts(n_tiles, nq, nkv, hd, page_size, max_tile_ctx, mean_tile_walk, beside),
                            attention_rows_plan(n_tiles, nq, nkv, hd, page_size, max_tile_ctx, mean_tile_walk, beside).parts);
  return splits <= 1 ? 0 : size_t(n_tiles) * 32 * nq * splits * (hd + 2);
}

// (In whole 16 bytes: a prompt's parts, written and read as float4, lie behind it in a mixed step's workspace.)
size_t attention_decode_workspace_floats(int n_decode, int nq, int hd, int max_ctx) {
  const size_t splits = (max_ctx + kDecodeChunk - 1) / kDecodeChunk;
  return splits <= 1 ? 0 : (size_t(n_decode) * nq * splits * (hd + 2) + 3) / 4 * 4;
}

int attention_mfma_wide(hipStream_t s, const void* q, int q_stride, const void* k_pool, const void* v_pool,
                        const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* q_len,
                        const int32_t* ctx_len, const int32_t* tiles, int n_tiles, const int32_t* decode_seqs, int n_decode,
                        int max_decode_ctx, int max_tile_ctx, int mean_tile_walk, long long one_query_keys, float* workspace, void* out, int nq, int nkv,
                        int hd, int page_size, int num_pages, ScoreStage st, float scale);

int attention_mfma(hipStream_t s, const void* q, int q_stride, const void* k_pool, const void* v_pool,
                   const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* q_len,
                   const int32_t* ctx_len, const int32_t* tiles, int n_tiles, const int32_t* decode_seqs, int n_decode,
                   int max_decode_ctx, int max_tile_ctx, int mean_tile_walk, long long one_query_keys, float* workspace, void* out, int nq, int nkv,
                   int hd, int page_size, int num_pages, ScoreStage st, float scale) {
#define SP_MFMA(DT)                                                                                              \
  case DT:                                                                                                       \
    return launch_mfma<DT, false>(s, q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, q_len, ctx_len,    \
                           tiles, n_tiles, decode_seqs, n_decode, max_decode_ctx, max_tile_ctx, mean_tile_walk, one_query_keys, \
                           workspace, out, nq, nkv, page_size, num_pages, st, scale)
  switch (hd / 16) {
    SP_MFMA(1); SP_MFMA(2); SP_MFMA(3); SP_MFMA(4); SP_MFMA(5); SP_MFMA(6); SP_MFMA(8);
    default:
      return attention_mfma_wide(s, q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, q_len, ctx_len, tiles, n_tiles,
                                 decode_seqs, n_decode, max_decode_ctx, max_tile_ctx, mean_tile_walk, one_query_keys, workspace, out, nq, nkv, hd,
                                 page_size, num_pages, st, scale);
  }
#undef SP_MFMA
}

// Attention of one-query sequences whose keys one block walks (64 a wave: up to 256 on four waves, 512 on eight), with the output projection behind it
// in the same launch:
//   residual[row(di), n] += sum over the heads of a set and d of attention[di, head, d] * w_o[n, head * HD + d]
// grid (blocks of 64 rows of w_o, sets of heads, sequences).  A short context's attention is a few trips to memory and as long again in the launch
// of the product behind it; here every block of rows walks its set's keys again (a set of 256 keys of 64 numbers is 64 KB out of the caches) and
// its rows of w_o are in registers by the time the keys are weighed.  Each wave takes 16 rows and, with eight waves, half of the columns.
// What bounds it is the chain: page numbers, keys, the waves' merge in LDS, sixteen matrix instructions, the adds.  One sequence of 79 keys, 14 heads
// of 64 in 2 groups, a width of 896: 1.4 us a layer less than attention and product in launches of their own (5.1 and 3.2 us).
template <int DT, int NW, bool POW2>
__global__ __launch_bounds__(64 * NW) void attention_project_kernel(
    const uint16_t* __restrict__ q, int q_stride, const uint16_t* __restrict__ k_pool, const uint16_t* __restrict__ v_pool,
    const int32_t* __restrict__ block_tables, int max_blocks, const int32_t* __restrict__ q_start, const int32_t* __restrict__ ctx_len,
    const int32_t* __restrict__ decode_seqs, const uint16_t* __restrict__ w_o, float* __restrict__ residual, int hidden, int nq, int nkv,
    int kv_stored, int page_size, int num_pages, ScoreStage st, float scale2) {
  constexpr int HD = 16 * DT, HC = (DT + 1) / 2, KEYS = 64 * NW, SHARES = NW / 4, CHUNKS = kProjectColumns / 32 / SHARES;
  __shared__ float s_o[NW][16][HD + 1];
  __shared__ float s_m[NW][16], s_l[NW][16];
  __shared__ int32_t s_table[KEYS / 4 + 4];
  __shared__ __attribute__((aligned(16))) uint16_t xs[kProjectColumns];
  __shared__ float sums[SHARES][64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lj = lane >> 4;
  const int g = blockIdx.y, di = blockIdx.z, seq = decode_seqs ? decode_seqs[di] : di, n_begin = blockIdx.x * 64;
  const int G = nq / nkv, columns = G * HD;
  const int pages = (KEYS - 1) / page_size + 1;
  if (tid < pages) s_table[tid] = block_tables[size_t(seq) * max_blocks + min(tid, max_blocks - 1)];
  const int q_row = decode_seqs ? q_start[seq] : seq;
  const int pos = ctx_len[seq] - 1, k_lo = first_visible(pos, st.window, st.chunk);

  PagedKV kv;
  kv.page_size = page_size;
  kv.num_pages = num_pages;
  kv.page_stride = size_t(kv_stored) * page_size * HD;
  kv.k = k_pool + size_t(g / (nkv / kv_stored)) * page_size * HD;
  kv.v = v_pool + size_t(g / (nkv / kv_stored)) * page_size * HD;
  kv.table = s_table;
  kv.page_shift = POW2 ? 31 - __builtin_clz(page_size) : 0;
  bf16x8 qop[1][HC];
  int qpos[1] = {lr < G ? pos : -1}, qlo[1] = {k_lo};
  const StepRule rule = step_rule(st, scale2);
  load_q_operand<DT>(qop[0], lr < G ? q + size_t(q_row) * q_stride + (g * G + lr) * HD : nullptr);
  __syncthreads();   // the page numbers are in LDS
  const int w0 = wave * 64;
  KVStep<DT> steps[2];
  bool live[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    live[i] = w0 + 32 * i <= pos && w0 + 32 * i + 32 > k_lo;
    if (live[i]) load_step<DT, POW2>(steps[i], kv, w0 + 32 * i, k_lo, pos);
  }
  // this wave's rows of w_o, asked for behind the keys: they are multiplied last
  const int share = wave >> 2, tile = n_begin + 16 * (wave & 3);
  uint4 wa[CHUNKS];
  {
    const uint16_t* wrow = w_o + size_t(min(tile + lr, hidden - 1)) * (size_t(nq) * HD) + g * columns;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int d = 32 * (c * SHARES + share) + 8 * lj;
      wa[c] = d < columns ? ldg128(wrow + d) : make_uint4(0, 0, 0, 0);
    }
  }
  floatx4 o[1][DT];
  float m[1], lsum[1];
  start_row<false>(m[0], lsum[0]);
  if (st.sinks && wave == 0 && lr < G) {      // a term of the denominator without a key: in one lane of a row's four
    m[0] = st.sinks[g * G + lr] * kLog2e;
    lsum[0] = lj == 0 ? 1.f : 0.f;
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[0][dt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (live[i]) attend_step<DT, 1, false>(steps[i], qop, o, m, lsum, w0 + 32 * i, k_lo, qpos, qlo, rule, scale2, 0.f, pos);
  float l = lsum[0];
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (lj == 0) { s_m[wave][lr] = m[0]; s_l[wave][lr] = l; }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) s_o[wave][lr][16 * dt + 4 * lj + r] = o[0][dt][r];
  __syncthreads();
  for (int i = tid; i < kProjectColumns; i += 64 * NW) {
    const int qh = i / HD, d = i % HD;
    float value = 0.f;
    if (i < columns) {
      float mx = -INFINITY, num = 0.f, den = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) mx = fmaxf(mx, s_m[w][qh]);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float f = exp2f(s_m[w][qh] - mx);
        num += f * s_o[w][qh][d];
        den += f * s_l[w][qh];
      }
      value = den > 0.f ? num / den : 0.f;
    }
    xs[i] = f32_to_bf16_bits(value);      // as where the attention output passes through memory
  }
  __syncthreads();
  floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c)      // every column of the result is this sequence's
    acc[c & 1] = mfma16(as_bf16x8(wa[c]), as_bf16x8(*reinterpret_cast<const uint4*>(&xs[32 * (c * SHARES + share) + 8 * lj])), acc[c & 1]);
  if (lr == 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) sums[share][16 * (wave & 3) + 4 * lj + r] = acc[0][r] + acc[1][r];
  __syncthreads();
  if (tid < 64 && n_begin + tid < hidden) {
    float sum = sums[0][tid];
    if (SHARES == 2) sum += sums[SHARES - 1][tid];
    unsafeAtomicAdd(residual + size_t(q_row) * hidden + n_begin + tid, sum);
  }
}

// Decode steps whose chunks' merge is folded into the output projection.  Worth it where the merged partial
// results, which every block of a head and a tile of 16 sequences reads again, stay small beside the rows of w_o
// (measured at 14 heads of 64, a width of 896, contexts of 4,096, tokens a second with the fold against merge and
// projection kernels of their own: 8 sequences 8,250 against 7,930, 24 sequences 21,870 against 21,260, 32
// sequences 27,400 against 26,660, 64 sequences 39,840 against 40,350).
static bool merge_projects(int n_decode, int max_decode_ctx, int hidden) {
  const int n_splits = (max_decode_ctx + kDecodeChunk - 1) / kDecodeChunk;
  return n_decode <= 32 && n_splits > 1 && min(n_decode, 16) * n_splits <= 256 &&
         hidden <= 2048;   // (wider: 28 heads of 128 at 3,584 +1%, 40 heads at 5,120 -0.5% with four tiles a wave)
}

// Whether the kernel above takes a step, on how many waves (0: no).  Where its blocks are at most the CUs.  us a step of 24 layers at 14 heads of 64
// in 2 groups and a width of 896, with attention and product (or the merge that projects) in launches of their own and so:
//   contexts of 79: one sequence 683 and 648, 4 706 and 662, 8 (224 blocks) 726 and 680, 16 (448) 771 and 768;
//   of 250: one 702 and 667, 8 750 and 721, 16 797 and 835; of 400 on eight waves: one 704 and 692, 4 728 and 705, 8 752 and 730.
// Over 24 other layouts (1 to 16 heads a set, 1 to 16 groups, heads of 32 to 64, widths of 128 to 8,192, 1 to 64 sequences) a layer's share takes 0.65 to 1.0 of
// the time at contexts of up to 256.  On eight waves 0.75 to 0.98 at contexts of 300, at 500 0.84 to 1.02 and, where the model is narrow, so that the product's
// launch is short, and most CUs walk 500 keys of 64 numbers each, to 1.18 (8 heads in 8 groups, 512 wide, 4 sequences 8.4 and 9.1; in one group, 32
// sequences 9.2 and 10.9; with 160 blocks and fewer 0.84 to 0.99, but for 8 heads in one group and 3 to 6 sequences 1.03 to 1.09, 0.92 to 0.98 at 300).
// Its sets add into the residual in whatever order they end, so where there are several it takes a step only if the launches of its own would add parts
// in no fixed order either (the merge that projects, a product with K cut): a step that comes out the same bit for bit every time stays so.  (4 heads of 64
// in 2 groups, a width of 256, contexts of 60: 6.4 us a layer and not 4.9; 14 in 2, 8,192 wide: 10.2 and not 7.5.)
static int project_waves(int hd, int nq, int nkv, int n_decode, int max_decode_ctx, int hidden) {
  const int sets = decode_sets(nq, nkv);
  const long long blocks = (long long)((hidden + 63) / 64) * sets * n_decode;
  if (hd > 64 || nq / sets * hd > kProjectColumns || max_decode_ctx > 512 || blocks > 256) return 0;
  if (max_decode_ctx > 256 && hidden < 768 && blocks * hd > 160 * 64) return 0;
  if (sets > 1 && !merge_projects(n_decode, max_decode_ctx, hidden) && !gemm_adds_parts(n_decode, hidden, nq * hd)) return 0;
  return max_decode_ctx <= 256 ? 4 : 8;
}

bool attention_decode_project_takes(int hd, int page_size, int nq, int nkv, int n_decode, int max_decode_ctx, int hidden) {
  if (hd > 128 || !attention_mfma_supports(hd, page_size, nq, nkv) || !attention_mfma_decode_supports(nq, nkv)) return false;
  if (n_decode < 1 || max_decode_ctx < 1 || hidden < 16) return false;
  return project_waves(hd, nq, nkv, n_decode, max_decode_ctx, hidden) || merge_projects(n_decode, max_decode_ctx, hidden);
}

// Tiles of 16 rows of w_o a wave takes in the folded kernel: one up to 16 sequences; with more, every tile of 16
// sequences is a block of its own and merges the head's chunks again, so a block takes as many rows as still
// leaves about 200 blocks (24 and 32 sequences, 14 heads, a width of 896: two tiles a wave 21,870 and 27,400
// tokens a second, one 21,600 and 27,100, four 21,400 and 26,990).
static int project_tiles_per_wave(int n_decode, int nq, int hidden) {
  if (n_decode <= 16) return 1;
  const int seq_tiles = (n_decode + 15) / 16;
  for (int tpw = 4; tpw > 1; tpw /= 2)
    if (nq * ((hidden + 64 * tpw - 1) / (64 * tpw)) * seq_tiles >= 192) return tpw;
  return 1;
}

template <int DT>
static int launch_decode_project(hipStream_t s, const void* q, int q_stride, const void* k_pool, const void* v_pool,
                                 const int32_t* block_tables, int max_blocks, const int32_t* q_start,
                                 const int32_t* ctx_len, const int32_t* decode_seqs, int n_decode, int max_decode_ctx,
                                 float* workspace, const void* w_o, float* residual, int hidden, int nq, int nkv,
                                 int page_size, int num_pages, ScoreStage st, float scale) {
  constexpr int HD = 16 * DT;
  if constexpr (DT <= 4) {
    if (const int waves = project_waves(HD, nq, nkv, n_decode, max_decode_ctx, hidden)) {
      const int sets = decode_sets(nq, nkv);
      const dim3 grid((hidden + 63) / 64, sets, n_decode);
#define SP_PROJECT(NW, POW2)                                                                                                            \
  attention_project_kernel<DT, NW, POW2><<<grid, 64 * NW, 0, s>>>((const uint16_t*)q, q_stride, (const uint16_t*)k_pool,               \
                                                                 (const uint16_t*)v_pool, block_tables, max_blocks, q_start, ctx_len,  \
                                                                 decode_seqs, (const uint16_t*)w_o, residual, hidden, nq, sets, nkv,   \
                                                                 page_size, num_pages, st, scale * kLog2e)
      const bool pow2 = (page_size & (page_size - 1)) == 0;
      if (waves == 4) { if (pow2) SP_PROJECT(4, true); else SP_PROJECT(4, false); }
      else { if (pow2) SP_PROJECT(8, true); else SP_PROJECT(8, false); }
#undef SP_PROJECT
      return check_launch("sp_attention_decode_project (one block a context)");
    }
  }
  const int n_splits = (max_decode_ctx + kDecodeChunk - 1) / kDecodeChunk;
  float* part_o = workspace;
  float* part_ml = workspace + size_t(n_decode) * nq * n_splits * HD;
  if ((page_size & (page_size - 1)) == 0)
    attention_decode_kernel<DT, true, false><<<dim3(n_splits, decode_sets(nq, nkv), n_decode), 256, 0, s>>>(
        (const uint16_t*)q, q_stride, (const uint16_t*)k_pool, (const uint16_t*)v_pool, block_tables, max_blocks,
        chunk_mask(n_splits), q_start, ctx_len, decode_seqs, nullptr, part_o, part_ml, n_splits, nq, decode_sets(nq, nkv), nkv,
        page_size, num_pages, st, scale * kLog2e);
  else
    attention_decode_kernel<DT, false, false><<<dim3(n_splits, decode_sets(nq, nkv), n_decode), 256, 0, s>>>(
        (const uint16_t*)q, q_stride, (const uint16_t*)k_pool, (const uint16_t*)v_pool, block_tables, max_blocks,
        chunk_mask(n_splits), q_start, ctx_len, decode_seqs, nullptr, part_o, part_ml, n_splits, nq, decode_sets(nq, nkv), nkv,
        page_size, num_pages, st, scale * kLog2e);
  if (check_launch("sp_attention_decode_project (decode)")) return 1;
  const int tpw = project_tiles_per_wave(n_decode, nq, hidden);
  const dim3 grid(nq, (hidden + 64 * tpw - 1) / (64 * tpw), (n_decode + 15) / 16);
#define SP_PROJECT(TPW)                                                                                         \
  attention_merge_project_kernel<DT, 1, TPW><<<grid, 256, 0, s>>>(part_o, part_ml, q_start, decode_seqs,        \
                                                                   (const uint16_t*)w_o, residual, n_decode,     \
                                                                   n_splits, nq, hidden)
  if (tpw == 1) SP_PROJECT(1);
  else if (tpw == 2) SP_PROJECT(2);
  else SP_PROJECT(4);
#undef SP_PROJECT
  return check_launch("sp_attention_decode_project (merge and projection)");
}

int attention_mfma_decode_project(hipStream_t s, const void* q, int q_stride, const void* k_pool, const void* v_pool,
                                  const int32_t* block_tables, int max_blocks, const int32_t* q_start,
                                  const int32_t* ctx_len, const int32_t* decode_seqs, int n_decode, int max_decode_ctx,
                                  float* workspace, const void* w_o, float* residual, int hidden, int nq, int nkv,
                                  int hd, int page_size, int num_pages, ScoreStage st, float scale) {
#define SP_MFMA(DT)                                                                                              \
  case DT:                                                                                                       \
    return launch_decode_project<DT>(s, q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, ctx_len, \
                                     decode_seqs, n_decode, max_decode_ctx, workspace, w_o, residual, hidden,    \
                                     nq, nkv, page_size, num_pages, st, scale)
  switch (hd / 16) {
    SP_MFMA(1); SP_MFMA(2); SP_MFMA(3); SP_MFMA(4); SP_MFMA(5); SP_MFMA(6); SP_MFMA(8);
  }
#undef SP_MFMA
  set_error("sp_attention_decode_project: no matrix-core kernel for head size %d", hd);
  return 1;
}

}  // namespace sprout

// On how many waves a block takes attention and output projection of a step of one-query sequences, 0 where they are launches of their own (or the
// merge of the chunks projects).  Runs nothing: for tests.
extern "C" int sp_attention_project_waves(int hd, int nq, int nkv, int n_decode, int max_decode_ctx, int hidden) {
  using namespace sprout;
  if (hd < 16 || hd % 16 || nkv < 1 || nq < nkv || nq % nkv || n_decode < 1 || max_decode_ctx < 1 || hidden < 16) return 0;
  return project_waves(hd, nq, nkv, n_decode, max_decode_ctx, hidden);
}

// Whether a step's prompts and one-query sequences may share a launch (sp_attention takes it where no other kernel takes the prompts): 1 or
// 0.  Runs nothing: for tests.
extern "C" int sp_attention_mixed_pays(int hd, int nq, int nkv, int n_tiles, int n_decode, int max_decode_ctx, long long one_query_keys) {
  using namespace sprout;
  if (hd < 16 || hd > 128 || nkv < 1 || nq < nkv || nq % nkv || n_tiles < 1 || n_decode < 1 || max_decode_ctx < 1) return 0;
  return chunks_beside(hd, nq, nkv, n_tiles, n_decode, max_decode_ctx, one_query_keys) > 0;
}
