// bfloat16 attention of prompts for head sizes of 64: more rows a wave than the kernels of attention_mfma.h.
//
// A wave of those kernels holds 32 queries of one head; every 32 keys it reads 8 KB from LDS for 256 cycles of matrix
// instructions, which is all that LDS gives four SIMDs, and four lanes share a row's statistics.  Here a wave holds 32 queries of
// TWO heads of a key/value head, as two tiles of 32 rows on 32x32x16 MFMA: a key or value operand read from LDS serves both,
// and a row's statistics lie in two lanes.  Four waves (eight heads) share two stages of 128 keys that travel straight into LDS
// (global_load_lds, asked for a whole stage ahead, one barrier a stage); every operand is read a phase before it is used: the
// values before the scores are multiplied, the next keys before they are weighed.  Two blocks run on a CU.
// What bounds it: per 32 keys a wave issues 16 matrix instructions (512 cycles) and 130 vector ones (700 cycles: a multiply-add,
// an exponential at 9 cycles, a sum, half a maximum and half a conversion a score); two waves on a SIMD overlap in part.  A stage's
// loads ask for little beside: a page's place in the pools is in LDS as it is added, and a lane's share of it is its own for the whole walk
// (with every place worked out from its key 130 vector instructions a stage, 8 % more time).  14 heads of 64 in 2 groups, 2,048 queries over
// 32,768 keys: 511 -> 298 us (780 TFLOP/s; 292 on another machine) with four parts of the keys, and 8 for their merge; over 8,192: 137 -> 92 + 8; two prompts of
// 2,048: 80 -> 52.
// (One head's weights between the other's products, in one wave: the matrix cores and the vector unit then overlap within a wave too,
// but the launch takes 5 % longer; four waves a CU with all registers to themselves: 450 us, the vector unit takes 2.7 cycles an
// instruction from two waves and 5 from one.)
// (Stages of 64 keys in a ring of three with operands read where they are used: 366 us; s_setprio around the matrix
// instructions changed nothing.)
//
//   S^T[key, row]  = K[key, :] . Q[row, :]           A = 32 keys of K, B = Q (32 rows in registers)
//   O^T[dim, row] += V^T[dim, key] . P^T[key, row]    A = V^T (the value pool is stored [dim][key]), B = P
// The result layout of S^T (lane row, keys 8 a + 4 h + b of a run of 16 in lane half h) becomes the operand layout of P^T (keys
// 8 h + 4 a + b) when the key rows of the stage lie in LDS with bits 2 and 3 of their number swapped.
#include "attention_mfma.h"

namespace sprout {

namespace {

// A stage: two runs of 64 keys, each 8 KB of key rows (64 keys of 128 bytes), then 8 KB of value rows (64 dimensions of 128 bytes).
constexpr int kRowsKeys = 128, kRowsStageBytes = 2 * 2 * 64 * 128, kRowsTable = 2048;

__device__ __forceinline__ int rows_swz(int row) { return (row ^ (row >> 3)) & 7; }
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

// NRT row tiles (heads) of a wave: its queries, sums and statistics, and the key operands of the 32 keys it multiplies next.
template <int NRT>
struct RowState {
  bf16x8 q[NRT][4];
  floatx16 o[NRT][2];
  float m[NRT], l[NRT];
  uint4 k[4];
};

// Scores of 32 keys from the key operands in registers.
template <int NRT>
__device__ __forceinline__ void rows_scores(const RowState<NRT>& st, floatx16 (&s)[NRT]) {
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[rt][r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) s[rt] = mfma32(as_bf16x8(st.k[ks]), st.q[rt][ks], s[rt]);
}

// Weights and weighted sums of the 32 keys from key0 on with the value operands v[c][dt].
template <int NRT, bool MASKED>
__device__ __forceinline__ void rows_weigh(RowState<NRT>& st, floatx16 (&s)[NRT], const uint4 (&v)[2][2], int key0, int pos, float scale2) {
  if (MASKED) {
    const int first = key0 + 8 * ((threadIdx.x & 63) >> 5);      // key of register r: first + 16 (r / 8) + r % 8
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (first + 16 * (r / 8) + r % 8 > pos) s[rt][r] = -INFINITY;
  }
  // A row's running maximum is brought up to date only where a number of the row exceeds it by more than kRescaleStep, then for
  // all tiles in one go.
  bool grown = false;
  float top[NRT];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) {
    float x = vmax3(s[rt][0], s[rt][1], s[rt][2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) x = vmax3(x, s[rt][r], s[rt][r + 1]);
    top[rt] = vmax(x, s[rt][15]) * scale2;
    grown = grown || top[rt] > st.m[rt] + kRescaleStep;
  }
  if (__builtin_amdgcn_ballot_w64(grown) != 0) {
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      const float t = max_over_halves(top[rt]);
      const float mx = t > st.m[rt] + kRescaleStep ? t : st.m[rt];
      const float alpha = __builtin_amdgcn_exp2f(st.m[rt] - mx);
      st.m[rt] = mx;
      st.l[rt] *= alpha;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) st.o[rt][dt][r] *= alpha;
    }
  }
  uint4 p[NRT][2];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) {
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        e[j] = __builtin_amdgcn_exp2f(fmaf(s[rt][8 * c + j], scale2, -st.m[rt]));
        sum += e[j];
      }
      p[rt][c] = make_uint4(pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3]), pack_bf16x2(e[4], e[5]), pack_bf16x2(e[6], e[7]));
    }
    st.l[rt] += sum;
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) st.o[rt][dt] = mfma32(as_bf16x8(v[c][dt]), as_bf16x8(p[rt][c]), st.o[rt][dt]);
}

__global__ __launch_bounds__(256, 2) void attention_rows_kernel(
    const uint16_t* __restrict__ q, int q_stride, const uint16_t* __restrict__ k_pool, const uint16_t* __restrict__ v_pool,
    const int32_t* __restrict__ block_tables, int max_blocks, const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len,
    const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ tiles, uint16_t* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, int n_splits, int nq, int nkv, int page_shift, int num_pages, float scale2,
    int n_tiles) {
  constexpr int HD = 64;
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];      // two stages, then the page numbers
  int32_t* s_table = reinterpret_cast<int32_t*>(ring + 2 * kRowsStageBytes);
  // Tiles are listed in order of position; the last ones walk the most keys, so they start first.  Two blocks run on a CU, the second
  // 256 blocks behind the first: where the blocks of a part of the keys fill the 256 in whole numbers, those behind take the tiles the
  // other way round, so that a CU has a long walk and a short one (1,024 queries over 4,096 keys beside eight prompts of 128, 14 heads
  // in 2 groups: 51 -> 40 us, the paired walks of attention_mfma.h 46; over 32,768 beside five of 256 276 -> 188).
  const unsigned part = gridDim.x * gridDim.y;
  const bool turned = 256 % part == 0 && (blockIdx.z * part / 256 & 1);
  const int tile = turned ? int(blockIdx.x) : n_tiles - 1 - int(blockIdx.x);
  const int seq = tiles[2 * tile], q_off = tiles[2 * tile + 1];
  const int G = nq / nkv, sets = (G + 7) / 8, g = blockIdx.y / sets, first_head = (blockIdx.y % sets) * 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 31, lk = lane >> 5;
  const int qlen = q_len[seq], ctx = ctx_len[seq], qs = q_start[seq];
  const int nvalid = min(32, qlen - q_off);
  if (nvalid <= 0) return;
  const int pos0 = ctx - qlen + q_off, k_hi = pos0 + nvalid - 1;
  const int split = blockIdx.z;
  int lo = 0, hi = k_hi;
  if (n_splits > 1) share_of_walk(lo, hi, kRowsKeys, split, n_splits);
  const int heads = max(0, min(2, G - first_head - 2 * wave)), head0 = g * G + first_head + 2 * wave;

  const int32_t* table = block_tables + size_t(seq) * max_blocks;
  const int first_page = lo >> page_shift, n_pages = hi >= lo ? (hi >> page_shift) - first_page + 1 : 0;
  const bool table_in_lds = n_pages <= kRowsTable;
  // a page's place in either pool, in units of 512 numbers (it holds 8 tokens of 64 at least): 32 bits reach 4 TB
  const uint32_t page_units = uint32_t(nkv) << page_shift >> 3;
  auto place_of = [&](int page) __attribute__((always_inline)) { return uint32_t(min(max(page, 0), num_pages - 1)) * page_units; };
  if (table_in_lds)
    for (int i = threadIdx.x; i < n_pages; i += 256) s_table[i] = int32_t(place_of(table[first_page + i]));
  __syncthreads();

  const int stages = hi >= lo ? (hi - lo) / kRowsKeys + 1 : 0;
  typedef __attribute__((address_space(3))) unsigned char* lds_address_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_address_t)ring;
  const uint16_t* kbase = k_pool + (size_t(g) << page_shift) * HD;
  const uint16_t* vbase = v_pool + (size_t(g) << page_shift) * HD;
  const int page_mask = (1 << page_shift) - 1;
  // What this lane fetches of a run of 64 keys: of row r = 8 (4 j + wave) + lane / 8 the piece (lane % 8) ^ swz(r); key rows hold the key
  // with bits 2 and 3 of their number swapped, value rows are dimensions.  A run begins at a multiple of 64, so a key's page and
  // its place there are the run's and the lane's own, added: kplace and vplace, and page kpage (vpage) from the run's first.
  int kkey[2], vkey[2], kcol[2], vrow[2], kpage[2], vpage[2];
  const uint16_t *kplace[2], *vplace[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * (4 * j + wave) + (lane >> 3), piece = (lane & 7) ^ rows_swz(r);
    kkey[j] = (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1);
    kcol[j] = 8 * piece;
    vkey[j] = 8 * piece;
    vrow[j] = r;
    kpage[j] = kkey[j] >> page_shift;
    vpage[j] = vkey[j] >> page_shift;
    kplace[j] = kbase + (kkey[j] & page_mask) * HD + kcol[j];
    vplace[j] = vbase + (size_t(vrow[j]) << page_shift) + (vkey[j] & page_mask);
  }
  auto fetch_from = [&](int s, int buf, auto in_lds) __attribute__((always_inline)) {
    auto page_at = [&](int page) __attribute__((always_inline)) {
      if constexpr (decltype(in_lds)::value) return size_t(uint32_t(s_table[page - first_page])) << 9;
      else return size_t(place_of(table[page])) << 9;
    };
#pragma unroll
    for (int run = 0; run < 2; ++run) {
      const int key0 = lo + s * kRowsKeys + 64 * run;
      const uint32_t dst = lds0 + buf * kRowsStageBytes + run * 16384 + wave * 1024;
      if (key0 + 63 <= hi) {
        const int page0 = key0 >> page_shift, in_page = key0 & page_mask;
#pragma unroll
        for (int j = 0; j < 2; ++j) lanes_to_lds(kplace[j] + (page_at(page0 + kpage[j]) + size_t(in_page * HD)), dst + j * 4096);
#pragma unroll
        for (int j = 0; j < 2; ++j) lanes_to_lds(vplace[j] + (page_at(page0 + vpage[j]) + size_t(in_page)), dst + 8192 + j * 4096);
        continue;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int key = min(key0 + kkey[j], hi);      // keys behind the walk's end repeat the last one: masked by position
        lanes_to_lds(kbase + page_at(key >> page_shift) + (key & page_mask) * HD + kcol[j], dst + j * 4096);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int key = min(key0 + vkey[j], hi & ~7);
        lanes_to_lds(vbase + page_at(key >> page_shift) + (size_t(vrow[j]) << page_shift) + (key & page_mask), dst + 8192 + j * 4096);
      }
    }
  };
  auto fetch = [&](int s, int buf) __attribute__((always_inline)) {
    if (table_in_lds) fetch_from(s, buf, std::true_type{});
    else fetch_from(s, buf, std::false_type{});
  };
  uint32_t kaddr[4];      // row li (or li + 32, where piece bits are the other way round), pieces 2 ks + lk
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) kaddr[ks] = li * 128 + (((2 * ks + lk) ^ rows_swz(li)) << 4);

  // A wave without a head walks along for its share of the fetches.
  auto walk = [&](auto nrt) __attribute__((always_inline)) {
    constexpr int NRT = decltype(nrt)::value;
    RowState<NRT == 0 ? 1 : NRT> st;
    const int pos = li < nvalid ? pos0 + li : -1;
    if constexpr (NRT > 0) {
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        const uint16_t* row = q + size_t(qs + q_off + min(li, nvalid - 1)) * q_stride + (head0 + rt) * HD + 8 * lk;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) st.q[rt][ks] = as_bf16x8(ldg128(row + 16 * ks));
        st.m[rt] = kNoKeyYet;
        st.l[rt] = 0.f;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) st.o[rt][dt][r] = 0.f;
      }
    }
    const int steps = hi >= lo ? (hi - lo) / 32 + 1 : 0;      // of 32 keys, four a stage
    if (steps > 0) fetch(0, 0);
    rows_wait_then_barrier<0>();
    if (stages > 1) fetch(1, 1);
    // The keys of step `i` of the stage in buffer `buf`; its values.
    auto keys = [&](int buf, int i) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        st.k[ks] = *reinterpret_cast<const uint4*>(ring + buf * kRowsStageBytes + (i >> 1) * 16384 + (i & 1) * 4096 + (kaddr[ks] ^ ((i & 1) * 64)));
    };
    auto values = [&](uint4 (&v)[2][2], int buf, int i) __attribute__((always_inline)) {
      // value row 32 dt + li, keys 32 i + 16 c + 8 lk ..
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
          v[c][dt] = *reinterpret_cast<const uint4*>(ring + buf * kRowsStageBytes + (i >> 1) * 16384 + 8192 + dt * 4096 + (kaddr[2 * (i & 1) + c] ^ (dt * 64)));
    };
    // Between the scores of a stage's last step and their weights: every wave has read all of the stage, and every wave's loads of
    // the next one have landed; the one after it is asked for, and the next step's keys are read.
    auto turn = [&](int s, int buf) __attribute__((always_inline)) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
      if (s + 2 < stages) fetch(s + 2, buf);
      if constexpr (NRT > 0) keys(buf ^ 1, 0);
    };
    if constexpr (NRT > 0) if (steps > 0) keys(0, 0);
    int s = 0, buf = 0, step = 0;
    // whole stages that every row sees, with another stage behind them
    for (; s + 1 < stages && lo + s * kRowsKeys + kRowsKeys - 1 <= pos0; ++s, buf ^= 1, step += 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (NRT > 0) {
          uint4 v[2][2];
          floatx16 sc[NRT];
          values(v, buf, i);
          rows_scores<NRT>(st, sc);
          if (i < 3) keys(buf, i + 1);
          else turn(s, buf);
          rows_weigh<NRT, false>(st, sc, v, 0, 0, scale2);
        } else if (i == 3) turn(s, buf);
      }
    }
    for (; step < steps; ++step) {
      const int i = step & 3;
      if constexpr (NRT > 0) {
        uint4 v[2][2];
        floatx16 sc[NRT];
        values(v, buf, i);
        rows_scores<NRT>(st, sc);
        if (i < 3) keys(buf, i + 1);
        else if (step + 1 < steps) turn(s, buf);
        rows_weigh<NRT, true>(st, sc, v, lo + 32 * step, min(pos, hi), scale2);
      } else if (i == 3 && step + 1 < steps) turn(s, buf);
      if (i == 3) { ++s; buf ^= 1; }
    }
    if constexpr (NRT > 0) {
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        float l = st.l[rt];
        l += __shfl_xor(l, 32, 64);
        if (li >= nvalid) continue;
        const int head = head0 + rt;
        if (n_splits > 1) {
          const size_t slot = ((size_t(tile) * 32 + li) * nq + head) * n_splits + split;
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
        uint16_t* dst = out + size_t(qs + q_off + li) * (size_t(nq) * HD) + head * HD + 4 * lk;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
          for (int a = 0; a < 4; ++a)
            *reinterpret_cast<uint2*>(dst + 32 * dt + 8 * a) = make_uint2(pack_bf16x2(st.o[rt][dt][4 * a] * inv, st.o[rt][dt][4 * a + 1] * inv),
                                                                          pack_bf16x2(st.o[rt][dt][4 * a + 2] * inv, st.o[rt][dt][4 * a + 3] * inv));
      }
    }
  };
  if (heads == 2) walk(std::integral_constant<int, 2>{});
  else if (heads == 1) walk(std::integral_constant<int, 1>{});
  else walk(std::integral_constant<int, 0>{});
}

}  // namespace

// Blocks along the keys for the kernel above, or 0 where the kernels of attention_mfma.h are the faster ones.  The eight head
// slots of a block have to be mostly taken (3 heads a group, 2,048 queries over 4,096 keys: 74 us against 69), and the blocks
// have to fill the CUs while each still walks 2,048 keys: the merge of parts costs about 10 us, and the paired walks of a
// prompt's first 2,048 tokens take 32 us where this kernel takes 43; from 256 blocks on it wins with whole walks.  Walks count in fractions of
// 2,048 keys: at 70 steps that rounding down left out it takes 0.68 of the other's time (0.42 to 0.88; 48 heads in 6 groups, 768 queries behind 3,000
// 62 us and 123).
int attention_rows_splits(int n_tiles, int nq, int nkv, int hd, int page_size, int max_tile_ctx) {
  if (hd != 64 || !staged_prefill(page_size) || n_tiles < 1) return 0;
  const int G = nq / nkv, sets = (G + 7) / 8;
  if (4 * G < 3 * 8 * sets) return 0;
  const long blocks = long(n_tiles) * nkv * sets;
  if (blocks < 256 && blocks * max_tile_ctx < 256L * 2048) return 0;
  return max(1, min(int(512 / blocks), max_tile_ctx / (blocks >= 256 ? 4096 : 1024)));
}

// Whether this kernel is the slower one all the same: one walk among many short ones bounds the launch where it is longer than three
// times a CU's share of all walks, and a block of this kernel walks alone at 0.0203 us a key where the blocks of attention_mfma.h share
// its keys out over four waves a head, in `there` parts.  Timed on both kernels over 613 steps (eight shapes of heads; 32 to 1,024 queries behind
// 2,048 to 32,000 keys, alone and with two or eight prompts of 64 to 1,024, alone and beside eight answers) the rule's choice takes 1.6 % longer than the faster
// one on average, 55 of them more than 10 %; this kernel always 3.9 %, that one always 55 %.  The worst: 24 heads in 2 groups, 1,024 queries behind
// 32,000 beside eight prompts of 300, 938 us here and 596 there, where the longest walk is not three times the share.
bool attention_rows_bound_by_one_walk(int n_tiles, int nq, int nkv, int splits, int page_size, int max_tile_ctx, int mean_tile_walk, int there) {
  const int G = nq / nkv, sets = (G + 7) / 8;
  const float longest = float(max_tile_ctx) / float(splits);
  if (longest <= 3.f * float(n_tiles) * float(nkv * sets) * float(mean_tile_walk) / 256.f) return false;
  StagedShape shape = staged_shape(nq, nkv, 64, n_tiles);
  staged_paired(n_tiles, nq, nkv, 64, there, max_tile_ctx, mean_tile_walk, &shape);
  const float per_key = shape.hpb == 4 ? 0.0184f : shape.hpb == 2 ? 0.0088f : 0.0085f;
  return 0.0203f * longest + (splits > 1 ? 15.f : 7.f) > per_key * float(max_tile_ctx) / float(there) + 24.f;
}

int launch_attention_rows(hipStream_t s, const uint16_t* q, int q_stride, const uint16_t* k_pool, const uint16_t* v_pool,
                          const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* q_len,
                          const int32_t* ctx_len, const int32_t* tiles, int n_tiles, int splits, uint16_t* out,
                          float* part_o, float* part_ml, int nq, int nkv, int page_shift, int num_pages, float scale2) {
  constexpr int lds = 2 * kRowsStageBytes + kRowsTable * 4;
  static bool raised = false;
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_rows_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      set_error("sp_attention (prefill): cannot raise the LDS limit: %s", hipGetErrorString(e));
      return 1;
    }
    raised = true;
  }
  attention_rows_kernel<<<dim3(n_tiles, nkv * ((nq / nkv + 7) / 8), splits), 256, lds, s>>>(
      q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, q_len, ctx_len, tiles, out, part_o, part_ml, splits,
      nq, nkv, page_shift, num_pages, scale2, n_tiles);
  return check_launch("sp_attention (prefill)");
}

}  // namespace sprout
