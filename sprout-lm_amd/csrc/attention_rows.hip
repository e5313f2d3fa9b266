// bfloat16 attention of prompts for head sizes of 64: more rows a wave than the kernels of attention_mfma.h.
//
// A wave of those kernels holds 32 queries of one head; every 32 keys it reads 8 KB from LDS for 256 cycles of matrix
// instructions, which is all that LDS gives four SIMDs, and four lanes share a row's statistics.  Here the queries of a set of up to
// eight heads of a key/value head are one run of rows, query by query and head by head, of which a block takes 256 and a wave 64, as
// two tiles of 32 rows on 32x32x16 MFMA: a key or value operand read from LDS serves both, a row's statistics lie in two lanes, and
// no slot is empty whatever the number of heads (with two heads a wave, seven heads left an eighth of the chip idle).  Two stages
// of 128 keys travel straight into LDS (global_load_lds, asked for a whole stage ahead, one barrier a stage).  Two blocks run on a CU.
//
// Per 32 keys a wave issues 16 matrix instructions (512 cycles) and 116 vector ones (620 cycles: a multiply-add, an exponential at 8
// cycles, a sum and half a conversion a score).  Two waves on a SIMD overlap the two kinds badly by themselves (947 cycles for the
// work of one, where the same instructions dealt out among each other take 810, from one wave too), so each half of a step weighs one
// tile's scores while the matrix cores sum the other tile's values and multiply its next keys (rows_half).  Whether a row has outgrown its
// running maximum is seen from the sum of the weights that were taken against it: no maximum of the scores is formed (30 instructions
// less a step) until that happens.
// A step takes 1,070 cycles, at 1.75 GHz with random numbers and at 2.24 GHz with zeros: the clock is power's, the cycles are not.  810 of them are the
// instructions; what the other 260 wait for has not been found (once in four steps there is a barrier, for which the loads of a stage have to have landed).
// An even share of all stages for every block instead of parts of each walk (one run of stages, cut anywhere) took as long: where CUs have one block
// instead of two the others run faster.
// 14 heads of 64 in 2 groups, 2,048 queries over 32,768 keys, merge included: 309 -> 279 us on one machine (233 GFLOP, 840 TFLOP/s), 283 -> 263 on another; on
// that one 640 over 8,192 59 -> 48, 250 over 31,250 78 -> 55; 32 heads in 8 groups, 2,048 over 10,240 407 -> 176 (those took the kernels of attention_mfma.h).
// (Stages of 64 keys in a ring of three with operands read where they are used: 366 us where 128 took 298; s_setprio around the matrix
// instructions changed nothing.)
//
//   S^T[key, row]  = K[key, :] . Q[row, :]           A = 32 keys of K, B = Q (32 rows in registers)
//   O^T[dim, row] += V^T[dim, key] . P^T[key, row]    A = V^T (the value pool is stored [dim][key]), B = P
// The result layout of S^T (lane row, keys 8 a + 4 h + b of a run of 16 in lane half h) becomes the operand layout of P^T (keys
// 8 h + 4 a + b) when the key rows of the stage lie in LDS with bits 2 and 3 of their number swapped.
#include "attention_mfma.h"
#include "gemm_pipe.h"

namespace sprout {

namespace {

// A stage: two runs of 64 keys, each 8 KB of key rows (64 keys of 128 bytes), then 8 KB of value rows (64 dimensions of 128 bytes).
constexpr int kRowsBlock = 256, kRowsKeys = 128, kRowsStageBytes = 2 * 2 * 64 * 128, kRowsTable = 2048;
// The longest list of tiles whose blocks an entry (a byte) and a group of 64 (four) fit where the stages lie afterwards.
constexpr int kRowsEntries = 64 * (2 * kRowsStageBytes / (64 + 4));
static_assert(kRowsEntries + kRowsEntries / 64 * 4 <= 2 * kRowsStageBytes && kRowsEntries % 64 == 0, "both lie in the stages' place");

// 64 lanes x 16 bytes, each from an address of its own, into LDS at lds_address + 16 lane.
__device__ __forceinline__ void lanes_to_lds(const void* address, uint32_t lds_address) {
  asm volatile(
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off"
      :
      : "v"(address), "s"(lds_address)
      : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void rows_wait_then_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(N) : "memory");
}

// The other half of a row's keys lies in lane ^ 32.
__device__ __forceinline__ float max_over_halves(float x) {
  const unsigned u = __float_as_uint(x);
  const auto f = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return vmax(__uint_as_float(f[0]), __uint_as_float(f[1]));
}

// What a wave holds: two tiles of 32 rows with their queries, sums and statistics, the scores and weights on their way, and the
// operands of the 32 keys and the 32 values that are multiplied next.
struct RowState {
  bf16x8 q[2][4];
  floatx16 o[2][2], s[2];
  float m[2], l[2];
  uint4 p[2][2], k[4], v[2][2];
};

// Weights of the scores of tile X against its running maximum, and their sum over this lane's 16 keys.
template <int X>
__device__ __forceinline__ float rows_weights(RowState& st, float scale2) {
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    float e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      e[j] = __builtin_amdgcn_exp2f(fmaf(st.s[X][8 * c + j], scale2, -st.m[X]));
      sum += e[j];
    }
    st.p[X][c] = make_uint4(pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3]), pack_bf16x2(e[4], e[5]), pack_bf16x2(e[6], e[7]));
  }
  return sum;
}

// The weighted sums of tile Y with the weights and the values in registers.
template <int Y>
__device__ __forceinline__ void rows_sums(RowState& st) {
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) st.o[Y][dt] = mfma32(as_bf16x8(st.v[c][dt]), as_bf16x8(st.p[Y][c]), st.o[Y][dt]);
}

// The scores of tile Y with the keys in registers.
template <int Y>
__device__ __forceinline__ void rows_scores(RowState& st) {
#pragma unroll
  for (int r = 0; r < 16; ++r) st.s[Y][r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) st.s[Y] = mfma32(as_bf16x8(st.k[ks]), st.q[Y][ks], st.s[Y]);
}

// Keys behind a row's position are taken out.  key of register r: first + 16 (r / 8) + r % 8.
template <int X>
__device__ __forceinline__ void rows_mask(RowState& st, int first, int pos) {
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (first + 16 * (r / 8) + r % 8 > pos) st.s[X][r] = -INFINITY;
}

// Sums of 16 weights up to this say that none of them is above 2^kRescaleStep (or no number).
constexpr float kRowsSumStep = 256.f;
static_assert(kRescaleStep == 8.0f, "the two belong together");

// After the weights of tile X were taken against maxima that some row may have outgrown: all rows' maxima are brought up to date, and
// the weights taken again.  The largest weight of a row is then 1, which bfloat16 holds: where few keys have most of the weight, the rounding of theirs is
// seen in the result.  Error against 64 bits over that of the kernels before this one (seven steps, 14 to 32 heads), scores of a deviation of 1.7 / 3 / 4: 1.000 /
// 0.98 to 1.02 / 0.94 to 1.03.  (With the test at 16 times 2^kRescaleStep, so that maxima stay behind by up to 2^12, 1.001 / 1.02 to 1.08 / 1.04 to 1.08; at a
// quarter of this 0.995 to 0.999 / 0.92 to 0.99 / 0.90 to 0.99, prompts of 0.5B sizes 0.6 % longer.)
template <int X>
__device__ __forceinline__ float rows_rescale(RowState& st, float scale2) {
  float top = st.s[X][0] * scale2;
#pragma unroll
  for (int r = 1; r < 16; ++r) top = vmax(top, st.s[X][r] * scale2);
  top = max_over_halves(top);
  const float mx = vmax(top, st.m[X]);
  const float alpha = __builtin_amdgcn_exp2f(st.m[X] - mx);
  st.m[X] = mx;
  st.l[X] *= alpha;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) st.o[X][dt][r] *= alpha;
  return rows_weights<X>(st, scale2);
}

// Half a step: the weights of tile X, and among them, dealt out one by one, the eight matrix instructions of the other tile: its weighted
// sums with the values in registers, then (behind `between`) its next scores with the keys in registers.  An exponential's result is used
// in the group behind it, so that no instruction waits for the one before.  Returns the sum of this lane's weights.
template <int X, typename BETWEEN>
__device__ __forceinline__ float rows_half(RowState& st, float scale2, const BETWEEN& between) {
  constexpr int Y = 1 - X;
  float e[16], arg[2];
  float sum[2] = {0.f, 0.f};
  uint32_t packed[8];
#pragma unroll
  for (int u = 0; u < 2; ++u) arg[u] = fmaf(st.s[X][u], scale2, -st.m[X]);
  floatx16 next;
#pragma unroll
  for (int r = 0; r < 16; ++r) next[r] = 0.f;
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    if (n < 4) st.o[Y][n & 1] = mfma32(as_bf16x8(st.v[n >> 1][n & 1]), as_bf16x8(st.p[Y][n >> 1]), st.o[Y][n & 1]);
    else next = mfma32(as_bf16x8(st.k[n - 4]), st.q[Y][n - 4], next);
#pragma unroll
    for (int u = 0; u < 2; ++u) e[2 * n + u] = __builtin_amdgcn_exp2f(arg[u]);
    if (n < 7) {
#pragma unroll
      for (int u = 0; u < 2; ++u) arg[u] = fmaf(st.s[X][2 * n + 2 + u], scale2, -st.m[X]);
    }
    if (n > 0) {
      packed[n - 1] = pack_bf16x2(e[2 * n - 2], e[2 * n - 1]);
#pragma unroll
      for (int u = 0; u < 2; ++u) sum[u] += e[2 * n - 2 + u];
    }
    // what this group has made exists here: the compiler keeps the groups apart and in order
    if (n < 4) asm volatile("" : "+v"(st.o[Y][n & 1]));
    else asm volatile("" : "+v"(next));
    asm volatile("" : "+v"(e[2 * n]), "+v"(e[2 * n + 1]), "+v"(arg[0]), "+v"(arg[1]), "+v"(sum[0]), "+v"(sum[1]));
    if (n > 0) asm volatile("" : "+v"(packed[n - 1]));
    if (n == 3) between();
    __builtin_amdgcn_sched_barrier(0);
  }
  packed[7] = pack_bf16x2(e[14], e[15]);
#pragma unroll
  for (int u = 0; u < 2; ++u) sum[u] += e[14 + u];
  st.s[Y] = next;
#pragma unroll
  for (int c = 0; c < 2; ++c) st.p[X][c] = make_uint4(packed[4 * c], packed[4 * c + 1], packed[4 * c + 2], packed[4 * c + 3]);
  return sum[0] + sum[1];
}

// Each wave's sums and statistics of the block's 64 rows to LDS, once no wave reads its stages any more: four numbers of row r from dimension
// 4 n .. of wave w at ((w * 64 + r) * 16 + (n ^ r % 16)) * 16, so that rows lie on different banks.
__device__ __forceinline__ void join_waves(const RowState& st, unsigned char* ring, float2* ml, int wave, int lane) {
  const int li = lane & 31, lk = lane >> 5;
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int r = 32 * rt + li;
    float l = st.l[rt];
    l += __shfl_xor(l, 32, 64);
    if (lk == 0) ml[64 * wave + r] = make_float2(st.m[rt], l);
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        *reinterpret_cast<float4*>(ring + ((64 * wave + r) * 16 + ((8 * dt + 2 * a + lk) ^ (r & 15))) * 16) =
            make_float4(st.o[rt][dt][4 * a], st.o[rt][dt][4 * a + 1], st.o[rt][dt][4 * a + 2], st.o[rt][dt][4 * a + 3]);
  }
  __syncthreads();
}
// Row r's dimensions 16 n .. over all waves, and what they are to be multiplied with.
__device__ __forceinline__ void joined_row(const unsigned char* ring, const float2* ml, int r, int n, float (&sum)[16], float& inv) {
  float2 of[4];
  float mx = kNoKeyYet, den = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) of[w] = ml[64 * w + r], mx = fmaxf(mx, of[w].x);
#pragma unroll
  for (int e = 0; e < 16; ++e) sum[e] = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float f = __builtin_amdgcn_exp2f(of[w].x - mx);
    den += f * of[w].y;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const float4 v = *reinterpret_cast<const float4*>(ring + ((64 * w + r) * 16 + ((4 * n + p) ^ (r & 15))) * 16);
      sum[4 * p] += f * v.x, sum[4 * p + 1] += f * v.y, sum[4 * p + 2] += f * v.z, sum[4 * p + 3] += f * v.w;
    }
  }
  inv = row_factor<false>(den);
}

// The shape of a launch.  An entry of the tile list stands for rows 256 n .. of its sequence and set, n counted by its place in the
// sequence, which has at least as many tiles of 32 queries as blocks of rows: a set holds up to eight heads.  Entries beyond the last rows
// have nothing to do.  (The list holds every tile of its sequences, each once.)
struct RowsShape {
  int heads, sets, n_tiles, parts;      // heads of a set, sets of all key/value heads, entries of the tile list, parts of a walk
  bool direct;                          // a block takes the entry of its own number, rows or not
  const int32_t *tiles, *q_start, *q_len, *ctx_len;
};

// NARROW: either pool is below 4 GB, so that a page's place is 32 bits of bytes.
// SHARED: the four waves of a block share 64 rows and the keys of a stage, 32 each, and their sums are joined in LDS.  A prompt has four times
// the blocks, none of which walks its keys alone, so short walks fill the chip without parts that another launch joins.  What bounds it
// is the longest walk's chain: 0.85 us a stage (loads of the stage after the next asked for in the middle of one, one barrier), 16 stages for
// 2,048 tokens, and 7 before and behind it.  14 heads of 64 in 2 groups, 2,048 tokens 29.7 -> 22.9 us, 47 to 611 tokens five times 14.5 -> 12.0, 1,800
// queries over 2,900 keys 49.6 -> 30.5; 32 heads in 8 groups, 1,024 tokens 19.6 -> 15.9.  (Keys and values waited for apart, with a step and
// a half for their way and two barriers a stage: 27.5 us for the first.)
template <bool NARROW, bool SHARED>
__global__ __launch_bounds__(256, 2) void attention_rows_kernel(
    const uint16_t* __restrict__ q, int q_stride, const uint16_t* __restrict__ k_pool, const uint16_t* __restrict__ v_pool,
    const int32_t* __restrict__ block_tables, int max_blocks, RowsShape shape, uint16_t* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, int nq, int nkv, int page_shift, int num_pages, float scale2) {
  constexpr int HD = 64, BLOCK_ROWS = SHARED ? 64 : kRowsBlock, SUBS = kRowsBlock / BLOCK_ROWS;      // blocks of an entry
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];      // two stages, then the pages' places
  uint32_t* s_table = reinterpret_cast<uint32_t*>(ring + 2 * kRowsStageBytes);
  auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 31, lk = lane >> 5;
  // Which rows, set and part.  Blocks go round the 8 XCDs and in each its 4 groups of CUs in turn, so the blocks with something to do are the first
  // of the launch, whichever entries they belong to (24 heads in 2 groups, 250 queries behind 31,000: two of eight entries are without rows, and as
  // blocks of their own left two XCDs idle: 98 us, so 75).  Entries are listed in order of position; the last ones walk the most keys, so
  // they start first; all sets and parts of an entry one after another, so that an XCD keeps to few of them where they come in eights.  Two blocks
  // run on a CU, the second 256 blocks behind the first: those behind take the entries the other way round, so that a CU has a long walk and a short
  // one (1,024 queries over 4,096 keys beside eight prompts of 128, 14 heads in 2 groups: 51 -> 40 us).
  // What the list says of up to 256 entries, four a lane, is asked for together, and kept: one by one they would be trips to memory of their own.
  // A longer list is read by the four waves, 1,024 entries in a trip, into LDS (`ring`, where no stage is yet): the blocks of each entry, and their sums
  // over 64.  (With trips for 64 entries one behind the other, and all of them twice, a list of 512 entries took a block 24 us, those without rows too:
  // 8 heads in 8 groups on shared rows, 256 prompts of 33 tokens 125 us and now 40, 32 of 1,024 272 and 119; 14 in 2, 256 of 64 37 and 32.)
  // Sets of eight heads have no entries without rows: a block of a long list takes the entry of its own number (`direct`; 16 heads in 2 groups, 100
  // prompts of 100 tokens 30 us and so 26.  With seven heads 256 prompts of 33, half of whose entries are without, 17 and so 25).
  struct Entry { int seq, nth, qlen, ctx, qs; };
  auto entry_of = [&](int e) __attribute__((always_inline)) {
    Entry entry = {0, 0, 0, 0, 0};
    if (e < shape.n_tiles) {
      const int at = shape.tiles[2 * e];
      entry = {at, shape.tiles[2 * e + 1] / 32, shape.q_len[at], shape.ctx_len[at], shape.q_start[at]};
    }
    return entry;
  };
  auto blocks_of = [&](int nth, int qlen) { return min(max((qlen * shape.heads - kRowsBlock * nth + BLOCK_ROWS - 1) / BLOCK_ROWS, 0), SUBS); };
  // over the wave: the sum of numbers 0 .. SUBS, and of those in the lanes before this one
  auto sums = [&](int n, int& before) __attribute__((always_inline)) {
    int all = 0;
    before = 0;
#pragma unroll
    for (int bit = 0; 1 << bit <= SUBS; ++bit) {
      const unsigned long long with = __builtin_amdgcn_ballot_w64(n >> bit & 1);
      all += __builtin_popcountll(with) << bit;
      before += int(__builtin_amdgcn_mbcnt_hi(uint32_t(with >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(with), 0))) << bit;
    }
    return all;
  };
  constexpr int KEPT = 4;
  const bool listed_once = shape.n_tiles <= 64 * KEPT, direct = !SHARED && shape.direct;
  const int groups = (shape.n_tiles + 63) / 64;
  int* s_groups = reinterpret_cast<int*>(ring + kRowsEntries);
  Entry kept[KEPT];
  int here[KEPT], before[KEPT], all[KEPT], n_units = 0;
  if (direct) {
    n_units = shape.n_tiles;
  } else if (groups == 1) {      // most steps: by itself, so that they run past what follows
    kept[0] = entry_of(lane);
    here[0] = blocks_of(kept[0].nth, kept[0].qlen);
    n_units = sums(here[0], before[0]);
  } else if (listed_once) {
    int at[KEPT];
#pragma unroll
    for (int j = 0; j < KEPT; ++j) {
      const int e = 64 * j + lane;
      at[j] = 0, kept[j] = {0, 0, 0, 0, 0};
      if (e < shape.n_tiles) at[j] = shape.tiles[2 * e], kept[j].nth = shape.tiles[2 * e + 1] / 32;
    }
#pragma unroll
    for (int j = 0; j < KEPT; ++j)
      if (64 * j + lane < shape.n_tiles) kept[j] = {at[j], kept[j].nth, shape.q_len[at[j]], shape.ctx_len[at[j]], shape.q_start[at[j]]};
#pragma unroll
    for (int j = 0; j < KEPT; ++j) {
      here[j] = blocks_of(kept[j].nth, kept[j].qlen);
      all[j] = sums(here[j], before[j]);
      n_units += all[j];
    }
  } else {
    for (int group0 = wave; group0 < groups; group0 += 16) {
      int at[4], nth[4], qlen[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = 64 * (group0 + 4 * j) + lane, in = min(e, shape.n_tiles - 1);
        at[j] = shape.tiles[2 * in], nth[j] = e == in ? shape.tiles[2 * in + 1] / 32 : 1 << 20;      // (beyond any sequence: without rows)
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) qlen[j] = shape.q_len[at[j]];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (group0 + 4 * j >= groups) break;
        const int n = blocks_of(nth[j], qlen[j]), of_group = sums(n, before[0]);
        ring[64 * (group0 + 4 * j) + lane] = uint8_t(n);
        if (lane == 0) s_groups[group0 + 4 * j] = of_group;
      }
    }
    __syncthreads();
    for (int group = lane; group < groups; group += 64) n_units += s_groups[group];
#pragma unroll
    for (int step = 1; step < 64; step *= 2) n_units += __shfl_xor(n_units, step, 64);
    n_units = uniform(n_units);
  }
  const int sets_parts = shape.sets * shape.parts, n_blocks = n_units * sets_parts;
  int id = blockIdx.x;
  if (id >= n_blocks) return;
  if (const int first = id & ~255, eights = min(256, n_blocks - first) / 8; id & 256 && id - first < 8 * eights)
    id = first + 8 * (eights - 1 - (id - first) / 8) + id % 8;
  const int set = id % sets_parts % shape.sets, part = SHARED ? 0 : id % sets_parts / shape.sets;
  int left = n_units - 1 - id / sets_parts, group = 0, tile = left, sub = 0;      // number `left` of the blocks of all entries
  Entry entry;
  if (direct) {
    entry = entry_of(tile);
    if (blocks_of(entry.nth, entry.qlen) == 0) return;
  } else {
    if (groups > 1 && listed_once) {
#pragma unroll
      for (int j = 0; j + 1 < KEPT; ++j)
        if (group == j && left >= all[j]) {
          left -= all[j];
          group = j + 1, kept[0] = kept[j + 1], here[0] = here[j + 1], before[0] = before[j + 1];
        }
    } else if (groups > 1) {
      for (int first = 0;; first += 64) {
        const int sum = first + lane < groups ? s_groups[first + lane] : 0;
        int upto = sum;
#pragma unroll
        for (int step = 1; step < 64; step *= 2) {
          const int below = __shfl_up(upto, step, 64);
          upto += lane >= step ? below : 0;
        }
        const int of_all = __builtin_amdgcn_readlane(upto, 63);
        if (left < of_all) {
          const int from = __builtin_ctzll(__builtin_amdgcn_ballot_w64(left < upto));
          group = first + from;
          left -= __builtin_amdgcn_readlane(upto - sum, from);
          break;
        }
        left -= of_all;
      }
      here[0] = ring[64 * group + lane];
      sums(here[0], before[0]);
    }
    const int from = __builtin_ctzll(__builtin_amdgcn_ballot_w64(before[0] <= left && left < before[0] + here[0]));
    tile = 64 * group + from;
    sub = left - __builtin_amdgcn_readlane(before[0], from);
    if (listed_once) {
      auto its = [&](int v) { return __builtin_amdgcn_readlane(v, from); };
      entry = {its(kept[0].seq), its(kept[0].nth), its(kept[0].qlen), its(kept[0].ctx), its(kept[0].qs)};
    } else {
      entry = entry_of(tile);
    }
  }
  const int seq = uniform(entry.seq), nth = uniform(entry.nth), qlen = uniform(entry.qlen), ctx = uniform(entry.ctx), qs = uniform(entry.qs);
  const int G = nq / nkv, heads = shape.heads, sets_of_group = shape.sets / nkv;
  const int g = set / sets_of_group, first_head = set % sets_of_group * heads;      // the last set of a group may have heads to spare
  // row r of the sequence: query r / heads, head first_head + r % heads
  const int rows = qlen * heads, row0 = kRowsBlock * nth + BLOCK_ROWS * sub;
  const int pos0 = ctx - qlen, k_last = pos0 + (min(row0 + BLOCK_ROWS, rows) - 1) / heads;
  int lo = 0, hi = k_last;
  if (!SHARED && shape.parts > 1) share_of_walk(lo, hi, kRowsKeys, part, shape.parts);
  const int stages = hi >= lo ? (hi - lo) / kRowsKeys + 1 : 0;

  typedef __attribute__((address_space(3))) unsigned char* lds_address_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_address_t)ring;
  const int page_mask = (1 << page_shift) - 1;
  // a page's place in either pool, in units of 512 numbers (it holds 8 tokens of 64 at least), which 32 bits reach 4 TB with, or in bytes
  const uint32_t page_units = (uint32_t(nkv) << page_shift >> 3) << (NARROW ? 10 : 0);
  auto place_of = [&](int page) __attribute__((always_inline)) { return uint32_t(min(max(page, 0), num_pages - 1)) * page_units; };
  // What this lane fetches of a run of 64 keys: of row r = 8 (4 j + wave) + lane / 8 the piece (lane % 8) ^ swz(r); key rows hold the key
  // with bits 2 and 3 of their number swapped, value rows are dimensions.  A run begins at a multiple of 64, so a key's page and
  // its place there are the run's and the lane's own, added: kplace and vplace, and page kpage (vpage) from the run's first.
  int kkey[2], vkey[2], kcol[2], vrow[2], kpage[2], vpage[2];
  uint32_t kplace[2], vplace[2];      // numbers
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * (4 * j + wave) + (lane >> 3), piece = (lane & 7) ^ swz(r);
    kkey[j] = (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1);
    kcol[j] = 8 * piece;
    vkey[j] = 8 * piece;
    vrow[j] = r;
    kpage[j] = kkey[j] >> page_shift;
    vpage[j] = vkey[j] >> page_shift;
    kplace[j] = (kkey[j] & page_mask) * HD + kcol[j];
    vplace[j] = (vrow[j] << page_shift) + (vkey[j] & page_mask);
  }
  uint32_t kaddr[4];      // row li (or li + 32, where piece bits are the other way round), pieces 2 ks + lk
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) kaddr[ks] = li * 128 + (((2 * ks + lk) ^ swz(li)) << 4);

  const int32_t* table = block_tables + size_t(seq) * max_blocks;
  const int first_page = lo >> page_shift, n_pages = stages ? (hi >> page_shift) - first_page + 1 : 0;
  const bool table_in_lds = n_pages <= kRowsTable;
  if (table_in_lds)
    for (int i = threadIdx.x; i < n_pages; i += 256) s_table[i] = place_of(table[first_page + i]);
  __syncthreads();

  const uint16_t* kbase = k_pool + (size_t(g) << page_shift) * HD;
  const uint16_t* vbase = v_pool + (size_t(g) << page_shift) * HD;
  // A stage's fetch in two parts: where this lane's eight pieces of 16 bytes lie (from LDS, asked for together: the compiler moves no
  // LDS read over the loads below, and each would be waited for by itself), and the loads.
  struct Pieces { uint32_t place[2][4]; };
  auto places_from = [&](int s, auto in_lds) __attribute__((always_inline)) {
    auto place = [&](int page) __attribute__((always_inline)) {
      if constexpr (decltype(in_lds)::value) return s_table[page - first_page];
      else return place_of(table[page]);
    };
    Pieces at;
#pragma unroll
    for (int run = 0; run < 2; ++run) {
      const int key0 = lo + s * kRowsKeys + 64 * run;
      if (key0 + 63 <= hi) {
        const int page0 = key0 >> page_shift;
#pragma unroll
        for (int j = 0; j < 2; ++j) at.place[run][j] = place(page0 + kpage[j]), at.place[run][2 + j] = place(page0 + vpage[j]);
      } else {      // keys behind the walk's end repeat the last one: masked by position
#pragma unroll
        for (int j = 0; j < 2; ++j)
          at.place[run][j] = place(min(key0 + kkey[j], hi) >> page_shift), at.place[run][2 + j] = place(min(key0 + vkey[j], hi & ~7) >> page_shift);
      }
    }
    return at;
  };
  auto places = [&](int s) __attribute__((always_inline)) {
    return table_in_lds ? places_from(s, std::true_type{}) : places_from(s, std::false_type{});
  };
  auto fetch = [&](int s, int buf, const Pieces& at) __attribute__((always_inline)) {
    // 64 pieces of 16 bytes: number `within` of the page at `place`, from `base` on
    auto piece = [&](const uint16_t* base, uint32_t place, uint32_t within, uint32_t dst) __attribute__((always_inline)) {
      if constexpr (NARROW) load_to_lds(base, place + 2 * within, dst);
      else lanes_to_lds(base + ((size_t(place) << 9) + within), dst);
    };
#pragma unroll
    for (int run = 0; run < 2; ++run) {
      const int key0 = lo + s * kRowsKeys + 64 * run;
      const uint32_t dst = lds0 + buf * kRowsStageBytes + run * 16384 + wave * 1024;
      if (key0 + 63 <= hi) {
        const int in_page = key0 & page_mask;
#pragma unroll
        for (int j = 0; j < 2; ++j) piece(kbase + in_page * HD, at.place[run][j], kplace[j], dst + j * 4096);
#pragma unroll
        for (int j = 0; j < 2; ++j) piece(vbase + in_page, at.place[run][2 + j], vplace[j], dst + 8192 + j * 4096);
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) piece(kbase, at.place[run][j], (min(key0 + kkey[j], hi) & page_mask) * HD + kcol[j], dst + j * 4096);
#pragma unroll
        for (int j = 0; j < 2; ++j) piece(vbase, at.place[run][2 + j], (vrow[j] << page_shift) + (min(key0 + vkey[j], hi & ~7) & page_mask), dst + 8192 + j * 4096);
      }
    }
  };

  // this wave's rows; one without any walks along for its share of the fetches
  const int wave_row = SHARED ? row0 : row0 + 64 * wave;
  const bool has_rows = SHARED || wave_row < rows;
  if (stages > 0) fetch(0, 0, places(0));
  if (SHARED && stages > 1) fetch(1, 1, places(1));
  int pos[2], query[2], head[2];
  RowState st;
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int r = wave_row + 32 * rt + li, row = min(r, rows - 1);
    query[rt] = row / heads;
    const int h = first_head + row - query[rt] * heads;
    head[rt] = h < G && r < rows ? g * G + h : -1;
    pos[rt] = head[rt] >= 0 ? min(pos0 + query[rt], hi) : -1;
    const uint16_t* from_q = q + size_t(qs + query[rt]) * q_stride + (g * G + min(h, G - 1)) * HD + 8 * lk;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) st.q[rt][ks] = as_bf16x8(ldg128(from_q + 16 * ks));
    st.m[rt] = kNoKeyYet;
    st.l[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
#pragma unroll
      for (int r16 = 0; r16 < 16; ++r16) st.o[rt][dt][r16] = 0.f;
      st.p[rt][dt] = st.v[rt][dt] = make_uint4(0, 0, 0, 0);
    }
  }
  // the last key of the part that every row of the wave sees
  const int last_seen = min(has_rows ? pos0 + wave_row / heads : ctx, hi);
  const int steps = stages ? (hi - lo) / 32 + 1 : 0;      // of 32 keys, four a stage
  if constexpr (SHARED) {
    if (stages > 1) rows_wait_then_barrier<8>();      // the first stage has landed
    else rows_wait_then_barrier<0>();
  } else {
    rows_wait_then_barrier<0>();
    if (stages > 1) fetch(1, 1, places(1));
  }
  // The keys of step `i` of the stage in buffer `buf`; its values.  Where waves share a stage, this wave's step of it.
  uint32_t my_keys[4], my_values[2][2];
  if constexpr (SHARED) {
    const uint32_t at = (wave >> 1) * 16384;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) my_keys[ks] = at + (wave & 1) * 4096 + (kaddr[ks] ^ ((wave & 1) * 64));
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) my_values[c][dt] = at + 8192 + dt * 4096 + li * 128 + ((((4 * (wave & 1) + 2 * c + lk) ^ swz(li)) << 4) ^ (dt * 64));
  }
  auto keys = [&](int buf, int i) __attribute__((always_inline)) {
    if constexpr (SHARED) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) st.k[ks] = *reinterpret_cast<const uint4*>(ring + buf * kRowsStageBytes + my_keys[ks]);
      return;
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      st.k[ks] = *reinterpret_cast<const uint4*>(ring + buf * kRowsStageBytes + (i >> 1) * 16384 + (i & 1) * 4096 + (kaddr[ks] ^ ((i & 1) * 64)));
  };
  auto values = [&](int buf, int i) __attribute__((always_inline)) {
    // value row 32 dt + li, keys 32 i + 16 c + 8 lk ..
    if constexpr (SHARED) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) st.v[c][dt] = *reinterpret_cast<const uint4*>(ring + buf * kRowsStageBytes + my_values[c][dt]);
      return;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
        st.v[c][dt] = *reinterpret_cast<const uint4*>(ring + buf * kRowsStageBytes + (i >> 1) * 16384 + 8192 + dt * 4096 + (kaddr[2 * (i & 1) + c] ^ (dt * 64)));
  };
  // In the middle of a stage's last step: every wave has read all of the stage, and every wave's loads of the next one have
  // landed; the one after it is asked for.
  auto turn = [&](int s, int buf) __attribute__((always_inline)) {
    Pieces next;
    const bool more = s + 2 < stages;
    if (more) next = places(s + 2);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
    if (more) fetch(s + 2, buf, next);
  };
  // Rows that have outgrown their maximum are few and far between: the weights are taken first and the test comes behind them.
  auto settle = [&](auto which, float sum) __attribute__((always_inline)) {
    constexpr int X = decltype(which)::value;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(sum <= kRowsSumStep)) != 0, 0)) sum = rows_rescale<X>(st, scale2);
    st.l[X] += sum;
  };
  constexpr std::integral_constant<int, 0> A{};
  constexpr std::integral_constant<int, 1> B{};
  // A step: two halves, in each of which one tile's weights are taken while the matrix cores sum the other's values and multiply
  // its next keys.
  auto step_of = [&](int s, int buf, int i, bool more, auto masked) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked)::value;
    const int first = lo + s * kRowsKeys + 32 * i;
    const bool beyond = MASKED && first + 31 > last_seen;
    if (beyond) rows_mask<0>(st, first + 8 * lk, pos[0]);
    settle(A, rows_half<0>(st, scale2, [&]() __attribute__((always_inline)) { values(buf, i); }));
    __builtin_amdgcn_sched_barrier(0);
    if (i == 3 && more) turn(s, buf);
    if (i < 3) keys(buf, i + 1);
    else if (more) keys(buf ^ 1, 0);
    if (beyond) rows_mask<1>(st, first + 8 * lk, pos[1]);
    settle(B, rows_half<1>(st, scale2, [] {}));
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (SHARED) {
    keys(0, 0);
    rows_scores<0>(st);
    int s = 0, buf = 0;
    // A stage is a step: the one after the next is asked for in its middle, from places that were looked up at its start.
    auto shared_step = [&](auto masked, bool more, bool another) __attribute__((always_inline)) {
      constexpr bool MASKED = decltype(masked)::value;
      const int first = s * kRowsKeys + 32 * wave;
      const bool beyond = MASKED && first + 31 > last_seen;
      const Pieces next = places(min(s + 2, stages - 1));
      if (beyond) rows_mask<0>(st, first + 8 * lk, pos[0]);
      settle(A, rows_half<0>(st, scale2, [&]() __attribute__((always_inline)) { values(buf, 0); }));
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
        if (another) fetch(s + 2, buf, next);
        keys(buf ^ 1, 0);
      }
      if (beyond) rows_mask<1>(st, first + 8 * lk, pos[1]);
      settle(B, rows_half<1>(st, scale2, [] {}));
      __builtin_amdgcn_sched_barrier(0);
    };
    for (; s + 2 < stages && s * kRowsKeys + 32 * wave + 31 <= last_seen; ++s, buf ^= 1) shared_step(std::false_type{}, true, true);
    for (; s < stages; ++s, buf ^= 1) shared_step(std::true_type{}, s + 1 < stages, s + 2 < stages);
    rows_sums<1>(st);
    join_waves(st, ring, reinterpret_cast<float2*>(s_table), wave, lane);
    // four lanes a row, 16 dimensions each
    const int r = threadIdx.x >> 2, row = row0 + r, n = threadIdx.x & 3;
    if (row >= rows) return;
    const int h = first_head + row % heads;
    if (h >= G) return;
    float sum[16], inv;
    joined_row(ring, reinterpret_cast<const float2*>(s_table), r, n, sum, inv);
    uint16_t* dst = out + size_t(qs + row / heads) * (size_t(nq) * HD) + (g * G + h) * HD + 16 * n;
#pragma unroll
    for (int e = 0; e < 16; e += 8)
      *reinterpret_cast<uint4*>(dst + e) = make_uint4(pack_bf16x2(sum[e] * inv, sum[e + 1] * inv), pack_bf16x2(sum[e + 2] * inv, sum[e + 3] * inv),
                                                      pack_bf16x2(sum[e + 4] * inv, sum[e + 5] * inv), pack_bf16x2(sum[e + 6] * inv, sum[e + 7] * inv));
    return;
  }
  if (has_rows && steps > 0) {
    keys(0, 0);
    rows_scores<0>(st);
  }
  int s = 0, buf = 0, step = 0;
  // whole stages that every row sees, with another stage behind them
  for (; s + 1 < stages && lo + s * kRowsKeys + kRowsKeys - 1 <= last_seen; ++s, buf ^= 1, step += 4) {
    if (has_rows) {
#pragma unroll
      for (int i = 0; i < 4; ++i) step_of(s, buf, i, true, std::false_type{});
    } else {
      turn(s, buf);
    }
  }
  for (; step < steps; ++step) {
    const int i = step & 3;
    const bool more = step + 1 < steps;
    if (has_rows) step_of(s, buf, i, more, std::true_type{});
    else if (i == 3 && more) turn(s, buf);
    if (i == 3) { ++s; buf ^= 1; }
  }
  if (!has_rows) return;
  rows_sums<1>(st);
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    float l = st.l[rt];
    l += __shfl_xor(l, 32, 64);
    if (head[rt] < 0) continue;
    if (shape.parts > 1) {
      // where the merge looks for them: by the entry of the list that holds the query.  A sequence's entries follow one another in
      // the lists that the engine makes; in others they are looked for.
      const int want = query[rt] / 32 * 32;
      int entry = tile - nth + query[rt] / 32;
      auto holds = [&](int e) { return e >= 0 && e < shape.n_tiles && shape.tiles[2 * e] == seq && shape.tiles[2 * e + 1] == want; };
      if (!holds(entry))
        for (entry = 0; entry < shape.n_tiles && !holds(entry);) ++entry;
      if (entry >= shape.n_tiles) continue;
      const size_t slot = ((size_t(entry) * 32 + query[rt] - want) * nq + head[rt]) * shape.parts + part;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *reinterpret_cast<float4*>(part_o + slot * HD + 32 * dt + 8 * a + 4 * lk) =
              make_float4(st.o[rt][dt][4 * a], st.o[rt][dt][4 * a + 1], st.o[rt][dt][4 * a + 2], st.o[rt][dt][4 * a + 3]);
      if (lk == 0) *reinterpret_cast<float2*>(part_ml + 2 * slot) = make_float2(st.m[rt], l);
      continue;
    }
    const float inv = row_factor<false>(l);
    uint16_t* dst = out + size_t(qs + query[rt]) * (size_t(nq) * HD) + head[rt] * HD + 4 * lk;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int a = 0; a < 4; ++a)
        *reinterpret_cast<uint2*>(dst + 32 * dt + 8 * a) = make_uint2(pack_bf16x2(st.o[rt][dt][4 * a] * inv, st.o[rt][dt][4 * a + 1] * inv),
                                                                      pack_bf16x2(st.o[rt][dt][4 * a + 2] * inv, st.o[rt][dt][4 * a + 3] * inv));
  }
}

}  // namespace

// The launch for a step, no parts where the kernels of attention_mfma.h are the faster ones.
//
// This kernel costs 12 us before and behind its walks, so it pays where there is much to walk: `work` counts stages over all blocks.  Timed on both
// kernels over 180 steps (nine shapes of heads; 64 to 2,048 queries behind 0 to 30,720 keys, alone and several together), this one's time over that of
// the kernels before it (where blocks without rows still took places, those below the lines):
//   longest walk of 3,000 keys and more, three heads a group and more: work from 1,400 on 0.77 (0.42 to 0.97; 14 heads in 2 groups 0.87, 0.70 to
//     1.00), below 1.18 (0.98 to 1.4); two heads a group, whose blocks of 128 queries reach further past the diagonal: from 3,500 on 0.59 (0.53 to
//     0.67), below 1.1 to 1.4 but for two; one head a group 1.0 to 2.8;
//   shorter walks, whole: from 192 blocks and 400 stages on 0.76 (0.38 to 1.06), fewer 1.0 to 3.3.
// Beside one-query sequences, whose blocks share a launch with the other kernel's and take about 12 us by themselves, from 2,200 stages on.
// Parts: two blocks a CU, each of eight stages at least, walks of less than 3,000 keys whole; where most tiles walk little beside a few long ones, those few
// count.  Over 75 steps these cost 3 % more than the best of 1 to 32.
RowsPlan attention_rows_plan(int n_tiles, int nq, int nkv, int hd, int page_size, int max_tile_ctx, int mean_tile_walk, long long beside) {
  RowsPlan plan = {0, 0, 0, false};
  if (hd != 64 || !staged_prefill(page_size) || n_tiles < 1 || n_tiles > kRowsEntries) return plan;
  const int G = nq / nkv, sets = (G + 7) / 8;
  plan.heads = (G + sets - 1) / sets;
  plan.sets = nkv * sets;
  const long long blocks = (long long)(((long long)n_tiles * plan.heads + 7) / 8) * plan.sets, longest = max(1, max_tile_ctx), mean = min(longest, (long long)max(1, mean_tile_walk));
  const long long work = blocks * max(mean, (long long)kRowsKeys) / kRowsKeys;
  const bool cut = longest >= 3000;
  if (G < (cut ? 2 : 3) || (!cut && blocks < 192) || work < (G == 2 ? 3500 : beside > 0 ? 2200 : cut ? 1400 : 400)) return plan;
  const long long count = 2 * mean < longest ? max(1LL, blocks * mean / longest) : blocks;
  plan.direct = n_tiles > 64 && plan.heads == 8;
  plan.parts = !cut ? 1 : int(max(1LL, min(min(512 / count, (longest + kRowsKeys - 1) / kRowsKeys / 8), (long long)kMaxPrefillSplits)));
  return plan;
}

// The launch for a step, between that one, the one whose waves share a block's rows (SHARED), and none.
//
// Both estimates in us.  Shared rows: 7 before and behind the walks; `chain`, the longest walk, at 0.85 a stage where its block has a CU's memory path
// to itself, 1.2 beside another all along; `chip`, all stages on 512 places and 4.8 a round of blocks; where the places are taken once or
// twice, what two blocks of a CU walk together.  Rows of their own: 12, 1.95 a stage of a part, all stages, and what the merge reads.  (Measured,
// 14 heads in 2 groups: 2,048 tokens twice 34.8 and 43.1, 4,096 at once 52 and 61, 1,024 behind 7,168 60 and 52, 2,048 behind 30,720 314 and
// 258; 32 heads in 8 groups: 2,048 tokens 37 and 43, twice 71 and 51.)
// Beside the kernels of attention_mfma.h (where rows of their own do not pay) the lines are in blocks and stages: over 560 steps (ten shapes of
// heads, one to eight prompts of 24 to 2,048 queries behind 0 to 30,000) those with 224 blocks of 64 rows and more took 0.32 to 1.02 of the time, with
// fewer 0.8 to 1.4 and, from 150 and 1,000 stages on, 0.78 to 1.03; with one head a group and less than 600 stages up to 1.36, and with more than a round of
// blocks whose walks are shorter than two stages on average 1.08 to 1.35 (256 prompts of 64 tokens 1.25, 32 of 512 0.98); one long walk among
// little else is what those cut.  Beside answers, which then have a launch of their own: from 250 blocks and 1,800 stages on 0.61 to 1.0, below to 1.6.
// With this choice the steps take 0.84 of the time of before on average, the worst 1.03.  Over 220 more, among them 130 of nine to 256 prompts at once, 0.68; what
// takes longer are some of a hundred short prompts and more, for which two heads a wave had less to do before and behind its walks (14 heads in 2
// groups, 256 prompts of 64 tokens 24.5 and 32 us, 100 of 100 21.8 and 27; 64 in 8, 64 of 32 14 and 15).  Rows of their own take 4 us more for every further
// round of blocks (78 prompts of 2 to 207 tokens, 64 heads in 8 groups, one walk of 4,037 keys: in three parts 144 us, on shared rows 116).
RowsPlan attention_rows_choice(int n_tiles, int nq, int nkv, int hd, int page_size, int max_tile_ctx, int mean_tile_walk, long long beside) {
  RowsPlan rows = attention_rows_plan(n_tiles, nq, nkv, hd, page_size, max_tile_ctx, mean_tile_walk, beside);
  if (hd != 64 || !staged_prefill(page_size) || n_tiles < 1 || n_tiles > kRowsEntries) return rows;
  const int G = nq / nkv;
  RowsPlan shared = {0, 0, 1, true};
  const int sets_of_group = (G + 7) / 8;
  shared.heads = (G + sets_of_group - 1) / sets_of_group;
  shared.sets = nkv * sets_of_group;
  const float longest = ceilf(float(max(1, max_tile_ctx)) / kRowsKeys), mean = fminf(longest, float(max(1, mean_tile_walk)) / kRowsKeys);      // stages
  const float blocks = 0.5f * float(n_tiles) * float(shared.heads) * float(shared.sets), stages = blocks * (mean + 0.5f);
  const float rounds = floorf(blocks / 512.f), rest = blocks - 512.f * rounds;
  const float of_rest = (rest > 256.f ? 1.22f : rest > 0.f ? 0.85f : 0.f) * (rounds > 0.f ? fmaxf(0.f, 2.f * mean - longest) : mean);
  const float chain = (rounds > 0.f ? 1.2f : 0.85f) * longest, chip = fmaxf(0.65f / 256.f * stages + 4.8f / 512.f * blocks, 1.22f * rounds * mean + of_rest);
  if (rows.parts) {
    const float further = fmaxf(0.f, float(n_tiles) * float(rows.heads) / 8.f * float(rows.sets * rows.parts) / 512.f - 1.f);
    float us = 12.f + fmaxf(1.95f * ceilf(longest / float(rows.parts)), 0.55f / 256.f * stages + 4.f * further);
    if (rows.parts > 1) us += 2.f + 5.3e-5f * float(n_tiles) * 32.f * float(nq) * float(rows.parts);
    return 1.05f * (7.f + fmaxf(chain, chip)) < us ? shared : rows;
  }
  if (beside > 0) return blocks >= 250.f && stages >= 1800.f && chain <= 8.f + 1.4f * chip ? shared : rows;
  if (blocks < 224.f) return blocks >= 150.f && stages >= 1000.f && chain <= 12.f + 1.5f * chip ? shared : rows;
  return (G > 1 || (stages >= 600.f && (blocks <= 512.f || mean >= 2.f))) && chain <= 12.f + (G > 1 ? 3.f : 1.6f) * chip ? shared : rows;
}

int launch_attention_rows(hipStream_t s, const RowsPlan& plan, const uint16_t* q, int q_stride, const uint16_t* k_pool, const uint16_t* v_pool,
                          const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* q_len, const int32_t* ctx_len,
                          const int32_t* tiles, int n_tiles, uint16_t* out, float* part_o, float* part_ml, int nq, int nkv, int page_shift, int num_pages, float scale2) {
  constexpr int lds = 2 * kRowsStageBytes + kRowsTable * 4;
  const bool narrow = (size_t(num_pages) * nkv << page_shift) * 128 < (size_t(1) << 32);
  const bool shared = plan.shared;
  auto kernel = shared ? (narrow ? attention_rows_kernel<true, true> : attention_rows_kernel<false, true>)
                       : (narrow ? attention_rows_kernel<true, false> : attention_rows_kernel<false, false>);
  static bool raised[2][2] = {};
  if (!raised[shared][narrow]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      set_error("sp_attention (prefill): cannot raise the LDS limit: %s", hipGetErrorString(e));
      return 1;
    }
    raised[shared][narrow] = true;
  }
  const RowsShape shape = {plan.heads, plan.sets, n_tiles, plan.parts, plan.direct, tiles, q_start, q_len, ctx_len};
  // blocks of 64 rows of a sequence of t tiles: at most 32 t heads / 64, rounded up, which is t times (heads + 1) / 2 at most
  kernel<<<n_tiles * plan.sets * plan.parts * (shared ? (plan.heads + 1) / 2 : 1), 256, lds, s>>>(q, q_stride, k_pool, v_pool, block_tables, max_blocks, shape, out, part_o, part_ml,
                                                                 nq, nkv, page_shift, num_pages, scale2);
  return check_launch("sp_attention (prefill)");
}

}  // namespace sprout

// A step's prompts on rows of a wave's own, were there no blocks that share them (sp_attention_rows_choice says what runs; the workspace is for the larger of
// both): plan = {heads of a set, sets, parts}.  Returns 1 where the other kernels are the faster ones, else 0.  Runs nothing: for tests.
extern "C" int sp_attention_rows_plan(int hd, int page_size, int nq, int nkv, int n_tiles, int max_tile_ctx, int mean_tile_walk, long long beside,
                                      int* plan) {
  if (nkv < 1 || nq < nkv || nq % nkv || page_size < 1 || n_tiles < 1 || max_tile_ctx < 1 || !plan) return 1;
  const sprout::RowsPlan p = sprout::attention_rows_plan(n_tiles, nq, nkv, hd, page_size, max_tile_ctx, mean_tile_walk > 0 ? mean_tile_walk : max_tile_ctx, beside);
  plan[0] = p.heads;
  plan[1] = p.sets;
  plan[2] = p.parts;
  return p.parts == 0;
}

// ... and what it does with them in the end: plan = {heads of a set, sets, parts, whether a block's waves share its rows}.  Returns 1 where the other
// kernels take them, else 0.  Runs nothing: for tests.
extern "C" int sp_attention_rows_choice(int hd, int page_size, int nq, int nkv, int n_tiles, int max_tile_ctx, int mean_tile_walk, long long beside,
                                        int* plan) {
  if (nkv < 1 || nq < nkv || nq % nkv || page_size < 1 || n_tiles < 1 || max_tile_ctx < 1 || !plan) return 1;
  const sprout::RowsPlan p = sprout::attention_rows_choice(n_tiles, nq, nkv, hd, page_size, max_tile_ctx, mean_tile_walk > 0 ? mean_tile_walk : max_tile_ctx, beside);
  plan[0] = p.heads;
  plan[1] = p.sets;
  plan[2] = p.parts;
  plan[3] = p.shared;
  return p.parts == 0;
}
