// Tiled bfloat16 product for many rows on four waves a block: out[T, N] = x[T, K] . w[N, K]^T with K a multiple of 64.
// The kernel and its launch; included by the files that instantiate its shapes.
//
// What bounds a product of many tokens here is power first: with random numbers the card lowers its clock until the
// matrix cores, the LDS and the caches together stay within their budget.  From registers alone, random operands
// run at 1.80 PFLOP/s through 32x32x16 and at 2.07 through 16x16x32 (2.45 with zeros, either): half as many sums are
// read and written a product.  So the products are 16x16x32, walked back and forth over the wave's tiles, so that one
// of the two operands stays where it is from one instruction to the next (2-3 %), and a wave holds as large a share of
// the block as its registers allow: at 256 x 256 four waves of 128 x 128 read two thirds of what eight of 128 x 64 read
// from LDS.  2,048 tokens by 37,888 rows of 3,584: 410 us, 1.36 PFLOP/s, where eight waves on 32x32x16 with one barrier
// between whole steps take 498-537.
//
// One wave a SIMD (two for the small blocks) hides nothing behind another, so a wave's own instructions are dealt out:
// a step of 64 along K is two halves of 32; while a half is multiplied, the operands of the next one are read from LDS
// into a second set of registers, and the loads of a later step from memory straight into LDS
// (global_load_lds_dwordx4) go out one by one between the products.  Loads in one run keep the matrix cores waiting:
// with 32x32x16 on four waves 547 us against 508 on eight.
//
// x has a ring of NA buffers, w of NA + 1: a step's operands are in registers when its second half begins, so that
// half's barrier both says that the next step has landed and frees this step's buffers.  x of step s + NA is asked for
// in the second half of step s, w of step s + NA already in the first half, into the buffer that step s - 1 has left.
//
// LDS layout, as in gemm_pipe.h: 128 bytes a row, piece p of row r at position p ^ swz(r); a lane of 16x16x32 reads row
// l % 16, piece l / 16 (+ 4 in the second half) of its 16 rows.
#pragma once
#include "gemm_pipe.h"

namespace sprout {

template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

template <int WM, int WN, int NA> constexpr size_t quad_lds = size_t(NA * WM + (NA + 1) * WN) * 4096;
// Two blocks fit a CU: then a wave has 256 registers, else 512, of which the sums take the half that only the matrix
// instructions and moves can reach.
template <int WM, int WN, int NA> constexpr bool quad_shares_cu = quad_lds<WM, WN, NA> <= 80 * 1024;

// Where row `p` of 32 tile rows (two tiles of 16) lies among 32 rows of w: a lane of 16x16x32 ends with rows
// 4 (l / 16) .. + 3 of either tile, which are eight neighbours in this order.
__device__ __forceinline__ int neighbours8(int p) { return 8 * ((p >> 2) & 3) + 4 * (p >> 4) + (p & 3); }

// What a block of the four-wave product does with its sums: lane (li = lane % 16, lq = lane / 16) holds
// out[t = tile row li][4 lq .. + 3 of tile column j] of tile (i, j), in the order of the weight rows that the kernel fetched.
// `turn` is LDS that the block has no more use for, used where K is split over blocks (gridDim.z > 1).
// AGPR: the sums lie in that half of the registers; 16 tokens' worth is moved at a time (`take`), all of them do not fit the other.
template <int WM, int WN, int MODE, bool AGPR>
__device__ __forceinline__ void quad_epilogue(floatx4 (&acc)[WM][WN], float* turn, const void* __restrict__ bias, int bias_dtype,
                                              void* __restrict__ out, int T, int N, int t0, int n0, int wm, int wn, const RopeArgs& rope) {
  const int lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  // `count` numbers of the bias from n on: the loads of all in one run, they wait for memory together
  auto bias_of = [&](int n, auto& v) __attribute__((always_inline)) {
    constexpr int COUNT = sizeof(v) / sizeof(float);
#pragma unroll
    for (int e = 0; e < COUNT; ++e) v[e] = 0.f;
    if (!bias || n >= N) return;
    if (bias_dtype == kBF16) {
#pragma unroll
      for (int e = 0; e < COUNT; ++e) v[e] = to_float(reinterpret_cast<const bf16_t*>(bias)[n + e]);
    } else {
#pragma unroll
      for (int e = 0; e < COUNT; ++e) v[e] = reinterpret_cast<const float*>(bias)[n + e];
    }
  };
  auto take = [&](int i) __attribute__((always_inline)) {
    if constexpr (AGPR) {
#pragma unroll
      for (int j = 0; j < WN; ++j) asm volatile("" : "+a"(acc[i][j]));
    }
  };
  auto pack8 = [](const float (&v)[8]) __attribute__((always_inline)) {
    return make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
  };

  if constexpr (MODE == kRope) {
    // Bias, rounding to bfloat16 (as where the projections pass through memory), rotation of q and k heads; q goes to
    // out [T, nq * hd], k and v into the paged pools.
    // Everything that comes from memory is asked for ahead of its use, the cosines and sines of the next 16 tokens before the
    // results of these are stored: the compiler moves no load over the stores, and each would be a trip to memory of its own
    // (2,048 tokens, 28 + 4 + 4 heads of 128 at K = 3,584: 997 us so, 70 ahead of time; 93 and a rotation kernel of 15 before).
    constexpr int Q = (WN + 2) / 4;                     // a wave's groups of 32 + 32 dimensions (16 + 16 where it has two tile columns)
    constexpr int E = WN == 2 ? 4 : 8;                  // neighbours that a lane holds of either half
    const int hd = rope.hd, half = hd / 2, groups_per_head = half / 32, heads = rope.nq + 2 * rope.nkv;
    int head[Q], d0[Q], slot[WM];
    float add_lo[Q][E], add_hi[Q][E];
#pragma unroll
    for (int i = 0; i < WM; ++i) slot[i] = rope.slot_mapping[min(t0 + (wm * WM + i) * 16 + li, T - 1)];
#pragma unroll
    for (int m = 0; m < Q; ++m) {
      const int group = n0 / 64 + (WN == 2 ? 0 : wn * Q + m);
      head[m] = group / groups_per_head;
      d0[m] = 32 * (group % groups_per_head) + (WN == 2 ? 16 * wn : 0) + E * lq;    // E dimensions of the first half
      bias_of(head[m] * hd + d0[m], add_lo[m]);
      bias_of(head[m] * hd + d0[m] + half, add_hi[m]);
    }
    if (!rope.table) __syncthreads();                   // `turn` below: nobody reads the stages any more
    float turns[2][Q][2 * E];                           // cosines and sines of a lane's dimensions
    auto fetch_turns = [&](int i) __attribute__((always_inline)) {
      const int t = min(t0 + (wm * WM + i) * 16 + li, T - 1);
#pragma unroll
      for (int m = 0; m < Q; ++m) {
        if (rope.table) {
          const float4* row = reinterpret_cast<const float4*>(rope.table + size_t(t) * half + d0[m]);
#pragma unroll
          for (int e = 0; e < E / 2; ++e) {
            const float4 v = row[e];
            turns[i & 1][m][4 * e] = v.x;
            turns[i & 1][m][4 * e + 1] = v.y;
            turns[i & 1][m][4 * e + 2] = v.z;
            turns[i & 1][m][4 * e + 3] = v.w;
          }
        } else {
          // without a table the wave computes those of 16 tokens by 32 dimensions in its own part of the LDS
          float2* mine = reinterpret_cast<float2*>(turn) + (wm * 2 + wn) * 16 * 33;
          const float pos = float(rope.positions[t]);
#pragma unroll 1
          for (int e = 0; e < E; ++e) {
            float sn, cs;
            sincosf(pos * rope.inv_freq[d0[m] + e], &sn, &cs);
            mine[li * 33 + E * lq + e] = make_float2(cs, sn);
          }
          wave_lds_fence();
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const float2 v = mine[li * 33 + E * lq + e];
            turns[i & 1][m][2 * e] = v.x;
            turns[i & 1][m][2 * e + 1] = v.y;
          }
          wave_lds_fence();
        }
      }
    };
    auto put = [&](uint16_t* to, const float (&v)[E]) __attribute__((always_inline)) {
      if constexpr (E == 8) *reinterpret_cast<uint4*>(to) = pack8(v);
      else *reinterpret_cast<uint2*>(to) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    };
    fetch_turns(0);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      take(i);
      if (i + 1 < WM) fetch_turns(i + 1);
      const int t = t0 + (wm * WM + i) * 16 + li;
      if (t >= T) continue;
      const int page = slot[i] >= 0 ? slot[i] / rope.page_size : 0, off = slot[i] >= 0 ? slot[i] % rope.page_size : 0;
#pragma unroll
      for (int m = 0; m < Q; ++m) {
        if (head[m] >= heads) continue;
        float lo[E], hi[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float p = to_float(bf16_t{f32_to_bf16_bits(acc[i][4 * m + e / 4][e % 4] + add_lo[m][e])});
          const float q = to_float(bf16_t{f32_to_bf16_bits(acc[i][4 * m + E / 4 + e / 4][e % 4] + add_hi[m][e])});
          const float cs = turns[i & 1][m][2 * e], sn = turns[i & 1][m][2 * e + 1];
          lo[e] = head[m] < rope.nq + rope.nkv ? p * cs - q * sn : p;
          hi[e] = head[m] < rope.nq + rope.nkv ? q * cs + p * sn : q;
        }
        if (head[m] < rope.nq) {
          uint16_t* q = reinterpret_cast<uint16_t*>(out) + size_t(t) * (size_t(rope.nq) * hd) + head[m] * hd + d0[m];
          put(q, lo);
          put(q + half, hi);
        } else if (slot[i] >= 0) {
          if (head[m] < rope.nq + rope.nkv) {
            uint16_t* k = rope.k_pool + ((size_t(page) * rope.nkv + (head[m] - rope.nq)) * rope.page_size + off) * hd + d0[m];
            put(k, lo);
            put(k + half, hi);
          } else {
            uint16_t* v = rope.v_pool + ((size_t(page) * rope.nkv + (head[m] - rope.nq - rope.nkv)) * hd + d0[m]) * rope.page_size + off;
#pragma unroll
            for (int e = 0; e < E; ++e) {
              v[e * rope.page_size] = f32_to_bf16_bits(lo[e]);
              v[(e + half) * rope.page_size] = f32_to_bf16_bits(hi[e]);
            }
          }
        }
      }
    }
  } else if constexpr (MODE == kSilu) {
    // out[t, n] = silu(gate) * up, both rounded to bfloat16 first, as where they are stored before the gated product; the
    // activation is a compile-time choice of the walk over the tiles (-1: one that gated_value picks)
    auto rows = [&](auto which) __attribute__((always_inline)) {
      constexpr int ACT = decltype(which)::value;
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        const int t = t0 + (wm * WM + i) * 16 + li;
        if (t >= T) continue;
        const float row = rope.row_gate ? 1.0f / (1.0f + expf(-rope.row_gate[size_t(t) * rope.row_gate_stride])) : 1.0f;
        auto value = [&](float gate, float up) __attribute__((always_inline)) {
          const uint32_t both = pack_bf16x2(gate, up);
          const float g = __uint_as_float(both << 16), u = __uint_as_float(both & 0xffff0000u);
          float v;
          if (ACT == kActSilu) v = g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
          else if (ACT == kActGeluTanh) v = g * __builtin_amdgcn_rcpf(1.0f + __expf(gelu_tanh_exponent(g))) * u;
          else v = gated_value(g, u, rope.act, rope.limit);
          return rope.row_gate ? v * row : v;
        };
        uint16_t* dst = reinterpret_cast<uint16_t*>(out) + size_t(t) * N;
        if constexpr (WN % 4 == 0) {
#pragma unroll
          for (int j = 0; j < WN; j += 4) {
            const int n = n0 / 2 + (wn * WN + j) * 8 + 8 * lq;
            if (n >= N) continue;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = value(acc[i][j + e / 4][e % 4], acc[i][j + 2 + e / 4][e % 4]);
            *reinterpret_cast<uint4*>(dst + n) = pack8(v);
          }
        } else if constexpr (WN % 2 == 1) {
          // a lane's four rows of a tile are two gate rows and the matching up rows: it ends with 2 WN neighbours
          struct __attribute__((packed, aligned(4))) Run { uint32_t pair[WN]; };
          const int n = n0 / 2 + wn * 8 * WN + 2 * WN * lq;
          Run run;
#pragma unroll
          for (int j = 0; j < WN; ++j) run.pair[j] = pack_bf16x2(value(acc[i][j][0], acc[i][j][2]), value(acc[i][j][1], acc[i][j][3]));
          if (n + 2 * WN <= N) {
            *reinterpret_cast<Run*>(dst + n) = run;
          } else {
#pragma unroll
            for (int j = 0; j < WN; ++j)
              if (n + 2 * j < N) *reinterpret_cast<uint32_t*>(dst + n + 2 * j) = run.pair[j];
          }
        } else {
          constexpr int G = WN / 2;
#pragma unroll
          for (int j = 0; j < G; ++j) {
            const int n = n0 / 2 + wn * 16 * G + 4 * G * lq + 4 * j;
            if (n >= N) continue;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = value(acc[i][j][r], acc[i][j + G][r]);
            *reinterpret_cast<uint2*>(dst + n) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
          }
        }
      }
    };
    if (rope.act == kActSilu) rows(std::integral_constant<int, kActSilu>{});
    else if (rope.act == kActGeluTanh) rows(std::integral_constant<int, kActGeluTanh>{});
    else rows(std::integral_constant<int, -1>{});
  } else if constexpr (MODE == kStore) {
    float add[WN / 2][8];
#pragma unroll
    for (int j = 0; j < WN; j += 2) bias_of(n0 + (wn * WN + j) * 16 + 8 * lq, add[j / 2]);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      take(i);
      const int t = t0 + (wm * WM + i) * 16 + li;
      if (t >= T) continue;
#pragma unroll
      for (int j = 0; j < WN; j += 2) {
        const int n = n0 + (wn * WN + j) * 16 + 8 * lq;
        if (n >= N) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[i][j + e / 4][e % 4] + add[j / 2][e];
        if (rope.second) {                    // two products in one: see RopeArgs; split and strides in fours
#pragma unroll
          for (int h = 0; h < 8; h += 4) {
            uint16_t* dst;
            if (n + h >= rope.split) {
              dst = rope.second + size_t(t) * rope.second_stride + (n + h - rope.split);
#pragma unroll
              for (int r = 0; r < 4; ++r) v[h + r] = stored_value(v[h + r], rope.act);
            } else {
              dst = reinterpret_cast<uint16_t*>(out) + size_t(t) * rope.out_stride + n + h;
            }
            *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v[h], v[h + 1]), pack_bf16x2(v[h + 2], v[h + 3]));
          }
        } else {
          *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(out) + size_t(t) * N + n) = pack8(v);
        }
      }
    }
  } else if (MODE == kAccumulate && gridDim.z > 1) {
    // K is split over blocks: the partial sums are added with float atomics, turned round in the wave's own part of the
    // LDS first so that an instruction adds runs of a row
    __syncthreads();
    constexpr int COLS = 16 * WN, PITCH = COLS + 4;
    float* mine = turn + (wm * 2 + wn) * 16 * PITCH;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      take(i);
#pragma unroll
      for (int j = 0; j < WN; ++j)
        *reinterpret_cast<float4*>(mine + li * PITCH + j * 16 + 4 * lq) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
      wave_lds_fence();
      const int tbase = t0 + (wm * WM + i) * 16, nbase = n0 + wn * COLS;
#pragma unroll
      for (int e = 0; e < 16 * COLS; e += 64) {
        const int tr = (e + lane) / COLS, col = (e + lane) % COLS;
        if (tbase + tr < T && nbase + col < N) {
          float v = mine[tr * PITCH + col];
          if (bias && blockIdx.z == 0)
            v += bias_dtype == kBF16 ? to_float(reinterpret_cast<const bf16_t*>(bias)[nbase + col]) : reinterpret_cast<const float*>(bias)[nbase + col];
          unsafeAtomicAdd(reinterpret_cast<float*>(out) + size_t(tbase + tr) * N + nbase + col, v);
        }
      }
      wave_lds_fence();
    }
  } else {
    // the sums there are asked for 16 tokens ahead of the stores, which the compiler moves no load over
    const int n = n0 + wn * WN * 16 + 4 * lq;           // + 16 j
    float add[WN][4];
    float4 there[2][WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) bias_of(n + 16 * j, add[j]);
    auto row = [&](int i) __attribute__((always_inline)) {
      return reinterpret_cast<float*>(out) + size_t(min(t0 + (wm * WM + i) * 16 + li, T - 1)) * N + n;
    };
    auto fetch = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < WN; ++j)
        if (MODE == kAccumulate && n + 16 * j < N) there[i & 1][j] = *reinterpret_cast<const float4*>(row(i) + 16 * j);
    };
    fetch(0);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      take(i);
      if (i + 1 < WM) fetch(i + 1);
      if (t0 + (wm * WM + i) * 16 + li >= T) continue;
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        if (n + 16 * j >= N) continue;
        float4 sum = make_float4(acc[i][j][0] + add[j][0], acc[i][j][1] + add[j][1], acc[i][j][2] + add[j][2], acc[i][j][3] + add[j][3]);
        if (MODE == kAccumulate) {
          const float4 old = there[i & 1][j];
          sum = make_float4(old.x + sum.x, old.y + sum.y, old.z + sum.z, old.w + sum.w);
        }
        *reinterpret_cast<float4*>(row(i) + 16 * j) = sum;
      }
    }
  }
}

// Which tile and which part of K block `block` of `blocks` takes where the parts are stored side by side: every XCD has an equal run of
// all of them, numbered part by part and in a part weight tile by weight tile, so that an XCD reads its run's share of K and of the
// weights alone.  (K in two parts, 2,048 tokens, 896 rows of 4,864 on 128 x 128: numbered as the other products are, where an XCD has
// tiles of every part, 28.5 us, so 24.8; 1,238 tokens in four 21.8 and 18.9; 264 tokens, 3,584 rows of 18,944 in six 51.3 and 49.)
__host__ __device__ inline void quad_part_of(int tiles_t, int tiles_n, int block, int blocks, int* tile_t, int* tile_n, int* part) {
  const int xcd = block & 7, each = blocks >> 3, more = blocks & 7;
  const int id = xcd * each + (xcd < more ? xcd : more) + (block >> 3);
  *tile_t = id % tiles_t;
  *tile_n = id / tiles_t % tiles_n;
  *part = id / tiles_t / tiles_n;
}

// A block of 2 x 2 waves, each with WM x WN tiles of 16 x 16: BM = 32 WM tokens by BN = 32 WN weight rows.
// Requires: K and the split multiples of 64, N of 8 (kSilu: N counts gate rows), 16-byte aligned operands, every
// offset of a tile's row within 32 bits (gemm_pipe_takes).
template <int WM, int WN, int NA, int MODE>
__global__ __launch_bounds__(256, (quad_shares_cu<WM, WN, NA> ? 2 : 1)) void gemm_quad_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const void* __restrict__ bias, int bias_dtype,
    void* __restrict__ out, int T, int N, int K, int k_per_split, RopeArgs rope) {
  constexpr int BM = 32 * WM, BN = 32 * WN, ROW = 128;
  constexpr uint32_t ASZ = BM * ROW, BSZ = BN * ROW, B0 = NA * ASZ;
  constexpr int L = WM + WN;                            // a wave's loads of a step
  constexpr bool AGPR = !quad_shares_cu<WM, WN, NA>;
  static_assert((WN % 2 == 0 || MODE == kSilu) && (MODE != kRope || WN == 2 || WN % 4 == 0), "tiles of w are paired");
  static_assert(NA >= 2 && NA <= 4 && (NA - 1) * L <= 63, "vmcnt holds six bits");
  static_assert(quad_lds<WM, WN, NA> <= 160 * 1024, "a CU's LDS");
  extern __shared__ __attribute__((aligned(1024))) unsigned char pipe_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lq = lane >> 4;
  int tile_n, tile_t, part = blockIdx.z;
  if (MODE == kStoreF32 && rope.parts > 0) {
    quad_part_of((T + BM - 1) / BM, (N + BN - 1) / BN, blockIdx.x, gridDim.x, &tile_t, &tile_n, &part);
    out = reinterpret_cast<float*>(out) + size_t(part) * T * N;
  } else {
    const PipeTiles tiles = pipe_tiles((T + BM - 1) / BM, ((MODE == kSilu ? 2 * N : N) + BN - 1) / BN);
    if (!pipe_tile_of(tiles, blockIdx.x, &tile_t, &tile_n)) return;
  }
  const int t0 = tile_t * BM, n0 = tile_n * BN;
  const int k_begin = part * k_per_split, k_end = min(K, k_begin + k_per_split);
  const int steps = (k_end - k_begin) / 64;

  // ---- what this lane fetches: row 8 (4 j + wave) + lane / 8 of each operand tile, for j < WM (WN)
  const unsigned char* xs = reinterpret_cast<const unsigned char*>(x + size_t(t0) * K + k_begin);     // the next step to be asked for
  const unsigned char* ws = reinterpret_cast<const unsigned char*>(w + (MODE == kSilu || MODE == kRope ? size_t(0) : size_t(n0) * K) + k_begin);
  uint32_t xoff[WM], woff[WN];
#pragma unroll
  for (int j = 0; j < WM; ++j) {
    const int r = 8 * (4 * j + wave) + (lane >> 3);
    xoff[j] = uint32_t(min(r, T - 1 - t0)) * uint32_t(K) * 2u + (((lane & 7) ^ swz(r)) << 4);
  }
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int r = 8 * (4 * j + wave) + (lane >> 3);
    int row;
    if (MODE == kSilu) {
      // N counts gate rows; w holds N gate rows, then N up rows.  A lane ends with both of one index.
      int gate, up;
      if (WN % 4 == 0) {            // 32 gate rows, then the 32 up rows
        gate = tile_n * (BN / 2) + (r / 64) * 32 + neighbours8(r & 31);
        up = (r >> 5) & 1;
      } else if (WN % 2 == 1) {     // two gate rows, then their two up rows, four times a tile
        const int own = r % (16 * WN), tile = own / 16;
        gate = tile_n * (BN / 2) + (r / (16 * WN)) * 8 * WN + 2 * WN * ((own >> 2) & 3) + 2 * tile + (own & 1);
        up = (own >> 1) & 1;
      } else {                      // a wave's first half of tiles gate rows, its second half up rows
        constexpr int G = WN / 2;
        const int own = r % (16 * WN), tile = own / 16;
        gate = tile_n * (BN / 2) + (r / (16 * WN)) * 16 * G + 4 * G * ((own >> 2) & 3) + 4 * (tile % G) + (own & 3);
        up = tile / G;
      }
      gate = min(N - 1, gate);
      row = up ? N + gate : gate;
    } else if (MODE == kRope) {
      // 32 dimensions of a head's first half, then their rotation partners half a head further on
      const int half = rope.hd / 2, groups_per_head = half / 32;
      const int group = tile_n * (BN / 64) + r / 64, head = group / groups_per_head, u = group % groups_per_head;
      // with two tile columns a wave has 16 of the 32 dimensions and their partners
      row = WN == 2 ? 16 * (r >> 5) + (r & 15) + ((r >> 4) & 1) * half : neighbours8(r & 31) + ((r >> 5) & 1) * half;
      row = min(N - 1, head * rope.hd + 32 * u + row);
    } else if (MODE == kStore) {
      row = min((r & ~31) + neighbours8(r & 31), N - 1 - n0);
    } else {
      row = min(r, N - 1 - n0);
    }
    woff[j] = uint32_t(row) * uint32_t(K) * 2u + (((lane & 7) ^ swz(r)) << 4);
  }
  typedef __attribute__((address_space(3))) unsigned char* lds_address_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_address_t)pipe_lds;
  const uint32_t xdst = lds0 + wave * 1024, wdst = lds0 + B0 + wave * 1024;
  auto load_x = [&](uint32_t buf, int j) __attribute__((always_inline)) { load_to_lds(xs, xoff[j], xdst + buf + 4096 * j); };
  auto load_w = [&](uint32_t buf, int j) __attribute__((always_inline)) { load_to_lds(ws, woff[j], wdst + buf + 4096 * j); };

  floatx4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  if constexpr (AGPR) {
    // the compiler does not know the products below for matrix instructions: the zeros are written well ahead of them
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) asm volatile("" : "+a"(acc[i][j]));
    asm volatile("s_nop 7" : : : "memory");
  }

#pragma unroll
  for (int p = 0; p < NA; ++p)
    if (p < steps) {
#pragma unroll
      for (int j = 0; j < WN; ++j) load_w(p * BSZ, j);
#pragma unroll
      for (int j = 0; j < WM; ++j) load_x(p * ASZ, j);
      xs += ROW;
      ws += ROW;
    }
  if (steps >= NA) wait_loads_then_barrier<(NA - 1) * L>();
  else wait_loads_then_barrier<0>();

  // ---- what this lane reads: row 16 i + li of its wave's rows, piece lq (+ 4).  swz(16 m + li) = swz(li) ^ 2 (m & 3).
  const int s0 = swz(li);
  const uint32_t xrow0 = (wm * WM * 16 + li) * ROW, wrow0 = B0 + (wn * WN * 16 + li) * ROW;
  uint4 a[2][WM], b[2][WN];
  auto read_x = [&](int h, int i, uint32_t buf) __attribute__((always_inline)) {
    a[h][i] = *reinterpret_cast<const uint4*>(pipe_lds + buf + xrow0 + i * 2048 + ((((h * 4 + lq) ^ s0) << 4) ^ (((wm * WM + i) & 3) << 5)));
  };
  auto read_w = [&](int h, int j, uint32_t buf) __attribute__((always_inline)) {
    b[h][j] = *reinterpret_cast<const uint4*>(pipe_lds + buf + wrow0 + j * 2048 + ((((h * 4 + lq) ^ s0) << 4) ^ (((wn * WN + j) & 3) << 5)));
  };
  auto read = [&](int h, int r, uint32_t xbuf, uint32_t wbuf) __attribute__((always_inline)) {   // in the order of their use
    if (r == 0) read_x(h, 0, xbuf);
    else if (r <= WN) read_w(h, r - 1, wbuf);
    else read_x(h, r - WN, xbuf);
  };

  // One half step: the products of the operands in set H; among them the reads of the next half into the other set
  // (from xbuf and wbuf) and, one at a time, the loads of w (H = 0) or x (H = 1) into the buffer `into`.
  auto half = [&](auto which, auto loads, auto reads, uint32_t xbuf, uint32_t wbuf, uint32_t into) __attribute__((always_inline)) {
    constexpr int H = decltype(which)::value;
    constexpr bool LOADS = decltype(loads)::value, READS = decltype(reads)::value;
    constexpr int NL = H == 0 ? WN : WM, M = WM * WN, EVERY = M / NL;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (READS && m % 2 == 0 && m / 2 < L) read(1 - H, m / 2, xbuf, wbuf);
      if (LOADS && m % EVERY == (EVERY > 1 ? 1 : 0)) {
        if (H == 0) load_w(into, m / EVERY);
        else load_x(into, m / EVERY);
      }
      const int i = m / WN, j = (i & 1) ? WN - 1 - m % WN : m % WN;
      if constexpr (AGPR)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(as_bf16x8(b[H][j])), "v"(as_bf16x8(a[H][i])));
      else
        acc[i][j] = mfma16(as_bf16x8(b[H][j]), as_bf16x8(a[H][i]), acc[i][j]);
      if (m % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    if (READS) {
#pragma unroll
      for (int r = (M + 1) / 2; r < L; ++r) read(1 - H, r, xbuf, wbuf);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // between the halves of a step: the next step has landed (at most `ON_THE_WAY` loads are later ones), and every wave has
  // this step's operands in registers
  auto turn = [&](auto on_the_way) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(decltype(on_the_way)::value) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  constexpr std::true_type yes{};
  constexpr std::false_type no{};

#pragma unroll
  for (int r = 0; r < L; ++r) read(0, r, 0, 0);
  uint32_t xbuf = 0, wbuf = 0;
  auto next_x = [&](uint32_t v) { return v == (NA - 1) * ASZ ? 0u : v + ASZ; };
  auto next_w = [&](uint32_t v) { return v == NA * BSZ ? 0u : v + BSZ; };
  int s = 0;
  for (; s + NA < steps; ++s) {
    const uint32_t xn = next_x(xbuf), wn_ = next_w(wbuf);
    half(first, yes, yes, xbuf, wbuf, wbuf == 0 ? NA * BSZ : wbuf - BSZ);
    // asked for since x of the next step: NA - 2 whole steps and w of one more
    turn(std::integral_constant<int, (NA - 2) * L + WN>{});
    half(second, yes, yes, xn, wn_, xbuf);
    xs += ROW;
    ws += ROW;
    xbuf = xn;
    wbuf = wn_;
  }
  auto tail = [&](auto behind) __attribute__((always_inline)) {       // a step with `behind` more behind it
    constexpr int BEHIND = decltype(behind)::value;
    if (steps - 1 - s == BEHIND) {
      const uint32_t xn = next_x(xbuf), wn_ = next_w(wbuf);
      half(first, no, yes, xbuf, wbuf, 0);
      turn(std::integral_constant<int, (BEHIND - 1) * L>{});
      half(second, no, yes, xn, wn_, 0);
      xbuf = xn;
      wbuf = wn_;
      ++s;
    }
  };
  if constexpr (NA > 3) tail(std::integral_constant<int, 3>{});
  if constexpr (NA > 2) tail(std::integral_constant<int, 2>{});
  tail(std::integral_constant<int, 1>{});
  half(first, no, yes, xbuf, wbuf, 0);
  half(second, no, no, 0, 0, 0);

  if constexpr (AGPR) {
    // the last products' sums are read after enough wait states
    asm volatile("s_nop 15\n\ts_nop 15" : : : "memory");
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) asm volatile("" : "+a"(acc[i][j]));
  }
  quad_epilogue<WM, WN, MODE, AGPR>(acc, reinterpret_cast<float*>(pipe_lds), bias, bias_dtype, out, T, N, t0, n0, wm, wn, rope);
}

template <int WM, int WN, int NA, int MODE>
inline int launch_quad(hipStream_t s, int splits, const uint16_t* x, const uint16_t* w, const void* bias, int bias_dtype, void* out,
                       int T, int N, int K, const RopeArgs& rope = RopeArgs{}) {
  constexpr size_t lds = quad_lds<WM, WN, NA>;
  static bool raised = false;
  if (lds > 48 * 1024 && !raised) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_quad_kernel<WM, WN, NA, MODE>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) {
      set_error("sp_gemm (four waves): cannot raise the LDS limit: %s", hipGetErrorString(e));
      return 1;
    }
    raised = true;
  }
  const int k_per_split = (K / 64 + splits - 1) / splits * 64;
  const PipeTiles tiles = pipe_tiles((T + 32 * WM - 1) / (32 * WM), ((MODE == kSilu ? 2 * N : N) + 32 * WN - 1) / (32 * WN));
  dim3 grid(8 * (tiles.own + tiles.run), 1, (K + k_per_split - 1) / k_per_split);
  if (MODE == kStoreF32 && rope.parts > 0) grid = dim3(((T + 32 * WM - 1) / (32 * WM)) * ((N + 32 * WN - 1) / (32 * WN)) * grid.z, 1, 1);
  gemm_quad_kernel<WM, WN, NA, MODE><<<grid, 256, lds, s>>>(x, w, bias, bias_dtype, out, T, N, K, k_per_split, rope);
  return check_launch("sp_gemm (four waves)");
}


// The block shapes, by the index that quad_choice gives: X(index, WM, WN, NA).
#define SPROUT_QUAD_SHAPES(X) \
  X(0, 2, 2, 4) X(1, 3, 4, 2) X(2, 4, 2, 4) X(3, 4, 4, 2) X(4, 4, 4, 4) X(5, 4, 6, 2) X(6, 5, 6, 2) X(7, 6, 4, 2) X(8, 6, 6, 2) \
  X(9, 8, 4, 3) X(10, 4, 8, 2) X(11, 5, 8, 2) X(12, 10, 4, 2) X(13, 6, 8, 2) X(14, 8, 6, 2) X(15, 9, 6, 2) X(16, 8, 8, 2)

// Blocks of an odd number of tile columns a wave, of gated products alone: X(index, WM, WN, NA).  See gemm_quad_odd.hip.
#define SPROUT_QUAD_ODD_SHAPES(X) X(0, 8, 5, 2) X(1, 10, 5, 2) X(2, 8, 7, 2) X(3, 9, 7, 2)

enum QuadKind { kQuadStore = 0, kQuadAccumulate = 1, kQuadGated = 2, kQuadRotating = 3, kQuadParts = 4 };   // as sp_quad_plan counts them

// Whether the four-wave kernel takes T x N x K (N: all weight rows): more than 64 tokens, from 17 on where it is the faster one; whole
// steps of 64 along K, outputs in whole eights of a row.
bool gemm_quad_takes(int kind, int T, int N, int K, int hd = 0);
// 16-byte stores: an output that is not so aligned stays with gemm_pipe's kernel.
inline bool quad_aligned(const void* x, const void* w, const void* out) {
  return ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
}
// Whether the accumulating product of T x N x K on the other kernels, which take it at other alignments, is cut along K.  Its parts
// are joined with float atomics, whose order differs from run to run and the sums' last bits with it: a product that comes out the
// same in every run there does so on four waves too.
bool gemm_cuts_k(int T, int N, int K);
// Picks the shape and the split of K with the least estimated time, and returns that in microseconds.
float quad_choice(int kind, int T, int N, int K, int* shape, int* splits);
// Whether a gated product of T tokens by N gate and up rows is better on blocks of an odd number of tile columns, and on which.
bool quad_takes_odd(int T, int N, int K, int* shape);

// The product on the shape that quad_choice picks (N as the kernel counts it: gate rows for kSilu).
template <int MODE>
inline int quad_run(hipStream_t s, int kind, const void* x, const void* w, const void* bias, int bias_dtype, void* out, int T, int N, int K,
                    const RopeArgs& epilogue = RopeArgs{}) {
  int shape, splits;
  quad_choice(kind, T, MODE == kSilu ? 2 * N : N, K, &shape, &splits);
  switch (shape) {
#define SPROUT_QUAD_CASE(I, WM, WN, NA) \
    case I: \
      if constexpr (MODE != kRope || WN == 2 || WN % 4 == 0) \
        return launch_quad<WM, WN, NA, MODE>(s, splits, (const uint16_t*)x, (const uint16_t*)w, bias, bias_dtype, out, T, N, K, epilogue); \
      break;
    SPROUT_QUAD_SHAPES(SPROUT_QUAD_CASE)
#undef SPROUT_QUAD_CASE
  }
  set_error("sp_gemm (four waves): no shape for %d tokens, %d rows, K = %d", T, N, K);
  return 1;
}

}  // namespace sprout
