// float32 products of many tokens on the bfloat16 matrix cores: out (float32) = or += a[T, K] . w[N, K]^T, K in 32s.
//
// v_mfma_f32_32x32x2_f32 gives 157 TFLOP/s, the bfloat16 instruction sixteen times that.  A float32 number is the sum of three
// bfloat16 numbers to its last bit (three_parts of mfma.h), and a product is taken as the six products of parts that reach 2^-24 of
// it: a1 b1, a1 b2, a2 b1, a2 b2, a1 b3, a3 b1; what is left out is 2^-26 of it at most, less than the float32 product's own rounding.
// a1 b1 is summed in one float32 accumulator and the other five, 2^-8 of its size, in a second: a result is rounded once for every
// thirty-two numbers of K and once where the two meet, where the float32 instruction rounds once for every number that is not zero
// and at most once for every two.  Relative error of the result against 64 bits, float32 instruction -> this: normal operands,
// K = 896 5.4e-7 -> 1.7e-7, 4,864 1.25e-6 -> 4.3e-7, 27,648 3.0e-6 -> 4.3e-7; weights with 1, 2, 8 and 64 numbers a row that are not
// zero 2.5e-8 -> 2.6e-8, 3.1e-8 -> 2.6e-8, 5.4e-8 -> 2.9e-8, 1.4e-7 -> 5.7e-8; one number 2^100 times the others of its row against a
// weight of zero 5.4e-7 -> 1.7e-7.  Time, whole call (2,048 tokens): 9,728 rows of 896 320 -> 202 us (of it 21 the splits, at 4.6
// TB/s; the product 170, at 1.26 PFLOP/s of bfloat16 products, where 32x32x16 on blocks with one barrier between whole steps took
// 202), 896 rows of 4,864 163 -> 124, 37,888 rows of 3,584 4,095 -> 2,513.
//
// (Pairs of float16 numbers took three products and half the time, but held 23 bits of 24, and numbers below 2^-17 of
// their row's largest less and less of them: one number that stood 2^24 out of its row and met no weight left an error of 2e-5.)
//
// Every row is multiplied by a power of two that brings its largest number into [2^49, 2^50): numbers down to 2^-150 of it keep all
// their bits, whatever the size of the row, and no sum overflows.  Powers of two are exact, and the sums are multiplied back
// by them.  A row with an infinity passes as its bits (upper and lower sixteen in two parts): its results are taken number by
// number behind the others, as the float32 instruction gives them; a row with a NaN gives NaN, whatever it meets (896
// rows of 4,864, 2,048 tokens, whole call: 124 us; with a token that has a NaN 122, with an infinity 567).
//
// The instruction drops the bits below its sum's last place, so that results end a little below the true ones, all to the same
// side, which the averages that attention takes over many tokens' values do not lose as they lose the rest of the error: odd rows
// on either side change their sign, and the results of an odd and an even row change it back.
//
// The rows are split by a kernel of their own before the product (the activations with what stands before the product, the norm
// or the gate, folded in; the weights into a workspace, a chunk of rows at a time, at the speed of memory): two rows together,
// 32 numbers of K a step, a line of 128 bytes a part.  K beyond kMaxK is walked in pieces that add.
#include "gemm_pipe.h"

namespace sprout {

float gemm_f32_time_us(int T, int N, int K);      // of the float32 instruction's kernel (gemm_f32.hip)

namespace {

constexpr int64_t kChunkBytes = int64_t(128) << 20;      // of split weights a launch multiplies
constexpr int kMaxK = 5120;                              // numbers of a row at a time: a chunk of rows then fills the chip
constexpr int kStep = 32, kStepBytes = 3 * 128;          // numbers of K a step, bytes of a step of two rows
constexpr int kNotFinite = 1 << 20;                      // a row's exponent, where the row holds its numbers' bits
constexpr int kHasNan = 1 << 22;                         // ... and where one of them is NaN
constexpr uint32_t kInfinityBits = 0x7f800000u;

enum { kRowsAsTheyAre = 0, kRowsGated = 1, kRowsNormed = 2, kRowsPaired = 3 };

struct SplitSource {
  const float* a;              // [rows][length]; kRowsGated: [rows][2 length], gate then up
  int length, first;           // of a row of the product, and the first of its numbers that is split
  const float* norm_w;         // kRowsNormed: a row is (a * scale) * norm_w, scale = 1 / rms
  float eps;
  int act;                     // kRowsGated
  float limit;
  int row0, half;              // kRowsPaired: the first split row, and the rows of a gate (see paired_row)
};

// A gated product's weights, gate rows then up rows (half of each, in sixteens), are split in pairs of sixteen: split row n of the
// product is this row of them.  The two numbers that meet in an output are then in one lane of the product, in neighbouring tiles.
__device__ __forceinline__ int paired_row(int n, int half) { return (n >> 5) * 16 + (n & 15) + ((n >> 4) & 1) * half; }

__device__ __forceinline__ size_t row_at(int row, int K) { return size_t(row >> 1) * (size_t(K / kStep) * kStepBytes) + (row & 1) * 64; }

// One row a wave (WAVES 1, four rows a block) or a block of four waves: bound by memory, a row's numbers stay in registers
// between its largest and the split (eight pieces of 16 bytes a lane).
template <int WAVES, int KIND>
__global__ __launch_bounds__(256) void split_rows_kernel(SplitSource src, unsigned char* __restrict__ out, int32_t* __restrict__ exponents,
                                                         int rows, int K) {
  constexpr int LANES = 64 * WAVES, PIECES = 8;
  __shared__ float scratch[16];
  __shared__ uint32_t tops[4];
  const int row = WAVES == 1 ? int(blockIdx.x) * 4 + (threadIdx.x >> 6) : int(blockIdx.x);
  const int lane = WAVES == 1 ? threadIdx.x & 63 : threadIdx.x;
  if (row >= rows) return;
  const int n4 = K / 4;
  const float* whole = src.a + size_t(KIND == kRowsPaired ? paired_row(src.row0 + row, src.half) : row) * (KIND == kRowsGated ? 2 * src.length : src.length);
  const float4* a = reinterpret_cast<const float4*>(whole + src.first);
  float4 kept[PIECES];
  if (KIND != kRowsGated) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
      if (lane + p * LANES < n4) kept[p] = a[lane + p * LANES];
  }
  float factor = 1.f;
  if (KIND == kRowsNormed) {
    float squares = 0.f;
    if (K == src.length) {
#pragma unroll
      for (int p = 0; p < PIECES; ++p)
        if (lane + p * LANES < n4) squares += kept[p].x * kept[p].x + kept[p].y * kept[p].y + kept[p].z * kept[p].z + kept[p].w * kept[p].w;
    } else {
      for (int i = lane; i < src.length / 4; i += LANES) {
        const float4 v = reinterpret_cast<const float4*>(whole)[i];
        squares += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
      }
    }
    squares = WAVES == 1 ? wave_sum(squares) : block_sum(squares, scratch);
    factor = 1.0f / sqrtf(squares / float(src.length) + src.eps);
  }
  uint32_t top = 0;      // the bits of the largest magnitude: infinity's are above all numbers', NaN's above infinity's
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const int i = lane + p * LANES;
    if (i >= n4) continue;
    if (KIND == kRowsNormed) {
      const float4 v = kept[p], w = reinterpret_cast<const float4*>(src.norm_w + src.first)[i];
      kept[p] = make_float4(v.x * factor * w.x, v.y * factor * w.y, v.z * factor * w.z, v.w * factor * w.w);
    } else if (KIND == kRowsGated) {
      const float4 g = a[i], u = reinterpret_cast<const float4*>(whole + src.length + src.first)[i];
      kept[p] = make_float4(gated_value(g.x, u.x, src.act, src.limit), gated_value(g.y, u.y, src.act, src.limit),
                            gated_value(g.z, u.z, src.act, src.limit), gated_value(g.w, u.w, src.act, src.limit));
    }
    const float f[4] = {kept[p].x, kept[p].y, kept[p].z, kept[p].w};
#pragma unroll
    for (int c = 0; c < 4; ++c) top = max(top, __float_as_uint(f[c]) & 0x7fffffffu);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) top = max(top, uint32_t(__shfl_xor(int(top), d, 64)));
  if (WAVES > 1) {
    if ((threadIdx.x & 63) == 0) tops[threadIdx.x >> 6] = top;
    __syncthreads();
    top = max(max(tops[0], tops[1]), max(tops[2], tops[3]));
  }
  const bool bits = top >= kInfinityBits;
  int e = 0;
  if (top > 0 && !bits) e = 50 - __builtin_amdgcn_frexp_expf(__uint_as_float(top));      // top = m 2^x, m in [0.5, 1): m 2^50
  if (lane == 0) exponents[row] = top > kInfinityBits ? kHasNan : bits ? kNotFinite : e;
  const uint32_t odd = bits ? 0u : uint32_t(row & 1) << 31;      // odd rows change their sign (see above)
  unsigned char* dst_row = out + row_at(row, K);
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const int i = lane + p * LANES;
    if (i >= n4) continue;
    float f[4] = {kept[p].x, kept[p].y, kept[p].z, kept[p].w};
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = __uint_as_float(__float_as_uint(__builtin_amdgcn_ldexpf(f[c], e)) ^ odd);
    uint2 part[3];
    three_parts(f[0], f[1], part[0].x, part[1].x, part[2].x);
    three_parts(f[2], f[3], part[0].y, part[1].y, part[2].y);
    if (bits) {
      const uint32_t u[4] = {__float_as_uint(kept[p].x), __float_as_uint(kept[p].y), __float_as_uint(kept[p].z), __float_as_uint(kept[p].w)};
      part[0] = make_uint2((u[0] >> 16) | (u[1] & 0xffff0000u), (u[2] >> 16) | (u[3] & 0xffff0000u));
      part[1] = make_uint2((u[0] & 0xffffu) | (u[1] << 16), (u[2] & 0xffffu) | (u[3] << 16));
    }
    unsigned char* dst = dst_row + size_t(i / 8) * kStepBytes + 8 * (i % 8);
#pragma unroll
    for (int c = 0; c < 3; ++c) *reinterpret_cast<uint2*>(dst + 128 * c) = part[c];
  }
}

template <int KIND>
int launch_split(hipStream_t s, const SplitSource& src, unsigned char* out, int32_t* exponents, int rows, int K) {
  if (K <= 2048) split_rows_kernel<1, KIND><<<(rows + 3) / 4, 256, 0, s>>>(src, out, exponents, rows, K);
  else split_rows_kernel<4, KIND><<<rows, 256, 0, s>>>(src, out, exponents, rows, K);
  return check_launch("sp_gemm_f32_split (rows)");
}

// Numbers k .. k + 7 of a split row, as they were (k in eights).
__device__ __forceinline__ void numbers_of(const unsigned char* __restrict__ parts, int row, int k, int K, int exponent, float (&v)[8]) {
  const unsigned char* p = parts + row_at(row, K) + size_t(k / kStep) * kStepBytes + 2 * (k % kStep);
  const uint4 q[3] = {ldg128(p), ldg128(p + 128), ldg128(p + 256)};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    uint32_t part[3];
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      const uint32_t two = e < 2 ? q[h].x : e < 4 ? q[h].y : e < 6 ? q[h].z : q[h].w;
      part[h] = e & 1 ? two >> 16 : two & 0xffffu;
    }
    const float x = __uint_as_float(part[0] << 16) + (__uint_as_float(part[1] << 16) + __uint_as_float(part[2] << 16));
    v[e] = exponent == kNotFinite ? __uint_as_float(part[0] << 16 | part[1]) : __builtin_amdgcn_ldexpf(row & 1 ? -x : x, -exponent);
  }
}

template <int WM, int WN, int STAGES> constexpr int split_lds = STAGES * 32 * (WM + WN) * 192;
template <int WM, int WN, int STAGES> constexpr bool split_shares_cu = split_lds<WM, WN, STAGES> <= 80 * 1024;

// Four waves in two rows of two, each WM x WN tiles of 16 x 16 (see gemm_quad.h: 16x16x32, the instruction that takes the least power
// a product, what else a wave has to do dealt out between its products).  A stage is 32 numbers of K, BM + BN rows of three times 64
// bytes, each part a plane of lines of two rows.  Piece c of 16 bytes of the row r & 1 of line l = r / 2 lies at position
// (4 (r & 1) + c) ^ s(l) of it, s(l) = (l ^ l / 4) & 3: the 16 rows that a quarter of a wave reads together lie on all banks, whether
// the LDS has 32 or 64.  A fetch of 1 KB is eight lines of a plane, which are lines of memory.
//
// A wave walks its 16-row tiles i of x: 6 WN products each, with w's parts of the step in registers and x's read AHEAD tiles before
// their use; at tile WM - AHEAD the reads pass to the next step, so there the wave has read all of this one: the barrier that says that
// the next step has landed also frees this step's stage, and the loads into it follow one by one between the products.
// What bounds it: matrix instructions, 6 WM WN of 16 cycles a stage and SIMD, at the clock that their power leaves; a block of
// 256 x 128 reads 72 KB from L2 for 3,072 cycles.
//
// kSilu: w's rows in pairs of sixteen (paired_row), out [T, N / 2] the gated values of the two products, N in 32s, no bias.
// Half the numbers are stored and read again, and the exponential and the division, which a split behind it hid under its reads, now
// stand beside another block's products (2,048 tokens by 9,728 rows of 896: product 167 -> 169 us, the split of the rows that the
// down product reads 22.7 -> 16.4).
template <int WM, int WN, int STAGES, int MODE>
__global__ __launch_bounds__(256, (split_shares_cu<WM, WN, STAGES> ? 2 : 1)) void split_product_kernel(
    const unsigned char* __restrict__ x, const unsigned char* __restrict__ w, const int32_t* __restrict__ x_exp,
    const int32_t* __restrict__ w_exp, const void* __restrict__ bias, int bias_dtype, float* out, int T, int N, int K, long long out_stride,
    int act, float limit) {
  constexpr int BM = 32 * WM, BN = 32 * WN;
  constexpr int STAGE = (BM + BN) * 192, XBYTES = BM * 192;
  constexpr int LX = 3 * BM / 64, LW = 3 * BN / 64, L = LX + LW;       // load instructions per wave, stage and operand
  static_assert(3 * BM % 64 == 0 && 3 * BN % 64 == 0, "every wave fills whole groups of 8 lines");
  static_assert((STAGES - 2) * L <= 63, "vmcnt holds six bits");
  static_assert(split_lds<WM, WN, STAGES> <= 160 * 1024, "a CU's LDS");
  constexpr bool AGPR = !split_shares_cu<WM, WN, STAGES>;
  constexpr int SETS = WM % 4 == 0 ? 4 : WM % 3 == 0 ? 3 : 2, AHEAD = SETS == 2 ? 1 : 2;
  static_assert(WM % SETS == 0, "a tile's registers are the same in every step");
  extern __shared__ __attribute__((aligned(1024))) unsigned char pipe_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lq = lane >> 4;
  int tile_n, tile_t;
  if (!pipe_tile_of(pipe_tiles((T + BM - 1) / BM, (N + BN - 1) / BN), blockIdx.x, &tile_t, &tile_n)) return;
  const int t0 = tile_t * BM, n0 = tile_n * BN;
  const int steps = K / kStep;
  typedef __attribute__((address_space(3))) unsigned char* lds_address_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_address_t)pipe_lds + wave * 1024;
  const uint32_t pitch = uint32_t(steps) * kStepBytes;      // of a line of two rows
  const unsigned char *xs = x + size_t(t0 / 2) * pitch, *ws = w + size_t(n0 / 2) * pitch;      // the next step to be asked for
  uint32_t off[L];
  // fetch u = 4 j + wave of an operand: eight lines of part u / (rows / 16)
  auto offset_of = [&](int u, int rows, int last_line) {
    const int part = u / (rows / 16), line = (u % (rows / 16)) * 8 + (lane >> 3), piece = (lane & 7) ^ ((line ^ (line >> 2)) & 3);
    return uint32_t(min(line, last_line)) * pitch + part * 128 + piece * 16;
  };
#pragma unroll
  for (int j = 0; j < LX; ++j) off[j] = offset_of(4 * j + wave, BM, (T - 1 - t0) / 2);
#pragma unroll
  for (int j = 0; j < LW; ++j) off[LX + j] = offset_of(4 * j + wave, BN, (N - 1 - n0) / 2);
  auto load = [&](uint32_t stage, int j) __attribute__((always_inline)) {
    if (j < LX) load_to_lds(xs, off[j], lds0 + stage + 4096 * j);
    else load_to_lds(ws, off[j], lds0 + stage + XBYTES + 4096 * (j - LX));
  };

  floatx4 acc[WM][WN], low[WM][WN];      // sums of the first parts' products, and of the others
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = low[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  if constexpr (AGPR) {
    // the compiler does not know the products below for matrix instructions: the zeros are written well ahead of them
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        asm volatile("" : "+a"(acc[i][j]));
        asm volatile("" : "+a"(low[i][j]));
      }
    asm volatile("s_nop 7" : : : "memory");
  }

#pragma unroll
  for (int p = 0; p < STAGES; ++p)
    if (p < steps) {
#pragma unroll
      for (int j = 0; j < L; ++j) load(p * STAGE, j);
      xs += kStepBytes;
      ws += kStepBytes;
    }
  if (steps >= STAGES) wait_loads_then_barrier<(STAGES - 1) * L>();
  else wait_loads_then_barrier<0>();

  // row li of tile i of the wave's, piece lq of a part; s(8 i + l) = s(l) ^ 2 (i & 1)
  const uint32_t position = (li >> 1) * 128 + (((((li & 1) << 2) | lq) ^ (((li >> 1) ^ (li >> 3)) & 3)) << 4);
  const uint32_t xrow = wm * WM * 1024 + position, wrow = XBYTES + wn * WN * 1024 + position;
  bf16x8 a[SETS][3], b[WN][3];
  auto read_x = [&](int i, uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 3; ++h)
      a[i % SETS][h] = as_bf16x8(*reinterpret_cast<const uint4*>(pipe_lds + stage + (xrow ^ (((wm * WM + i) & 1) << 5)) + h * (BM * 64) + i * 1024));
  };
  auto read_w = [&](int j, int h, uint32_t stage) __attribute__((always_inline)) {
    b[j][h] = as_bf16x8(*reinterpret_cast<const uint4*>(pipe_lds + stage + (wrow ^ (((wn * WN + j) & 1) << 5)) + h * (BN * 64) + j * 1024));
  };
  auto mul = [&](floatx4& sum, bf16x8 wp, bf16x8 xp) __attribute__((always_inline)) {
    if constexpr (AGPR) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(sum) : "v"(wp), "v"(xp));
    else sum = mfma16(wp, xp, sum);
  };

  // One step from `stage`; the next step's operands are read from `next`, later loads go into `stage` once it is free.  A tile takes
  // w's parts in their order, three products with the first, two with the second, one with the third: the step's last tile has done
  // with the first two before its end, and they are read for the next step there, the third in the next step's first tile.
  // LOADS: a step is left to be asked for; MORE: a step follows; ON_THE_WAY: loads of later steps than it.
  auto walk = [&](auto loads, auto more, auto on_the_way, uint32_t stage, uint32_t next) __attribute__((always_inline)) {
    constexpr int FREE = WM - AHEAD, PRODUCTS = 6 * WN * AHEAD;      // products from the barrier to the end of the step
    constexpr bool LOADS = decltype(loads)::value, MORE = decltype(more)::value;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      if (i == FREE && MORE) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(decltype(on_the_way)::value) : "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
      if (i + AHEAD < WM) read_x(i + AHEAD, stage);
      else if (MORE) read_x(i + AHEAD - WM, next);
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int jj = 0; jj < WN; ++jj) {
          const int j = (q & 1) ? WN - 1 - jj : jj;
          const int m = (i - FREE) * 6 * WN + q * WN + jj;           // products since the barrier
          if (i == 0 && q == 0) read_w(j, 2, stage);
          if (i == WM - 1 && MORE && q == 3) read_w(jj, 0, next);
          if (i == WM - 1 && MORE && q == 5) read_w(jj, 1, next);
          if (LOADS && m >= 0 && m % 2 == 0 && m / 2 < L) load(stage, m / 2);      // one for every two products from the barrier on
          if (q == 0) mul(low[i][j], b[j][0], a[i % SETS][2]);
          else if (q == 1) mul(acc[i][j], b[j][0], a[i % SETS][0]);
          else if (q == 2) mul(low[i][j], b[j][0], a[i % SETS][1]);
          else if (q == 3) mul(low[i][j], b[j][1], a[i % SETS][1]);
          else if (q == 4) mul(low[i][j], b[j][1], a[i % SETS][0]);
          else mul(low[i][j], b[j][2], a[i % SETS][0]);
          if (m & 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (LOADS) {
#pragma unroll
      for (int j = PRODUCTS / 2; j < L; ++j) load(stage, j);
      xs += kStepBytes;
      ws += kStepBytes;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) read_x(i, 0);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < WN; ++j) read_w(j, h, 0);
  uint32_t stage = 0;
  auto after = [&](uint32_t v) { return v == (STAGES - 1) * STAGE ? 0u : v + STAGE; };
  int s = 0;
  for (; s + STAGES < steps; ++s) {
    const uint32_t next = after(stage);
    walk(yes, yes, std::integral_constant<int, (STAGES - 2) * L>{}, stage, next);
    stage = next;
  }
  auto tail = [&](auto behind) __attribute__((always_inline)) {       // a step with `behind` more behind it
    constexpr int BEHIND = decltype(behind)::value;
    if (steps - 1 - s == BEHIND) {
      const uint32_t next = after(stage);
      walk(no, yes, std::integral_constant<int, (BEHIND - 1) * L>{}, stage, next);
      stage = next;
      ++s;
    }
  };
  if constexpr (STAGES > 3) tail(std::integral_constant<int, 3>{});
  if constexpr (STAGES > 2) tail(std::integral_constant<int, 2>{});
  tail(std::integral_constant<int, 1>{});
  walk(no, no, std::integral_constant<int, 0>{}, stage, 0);
  if constexpr (AGPR) {
    asm volatile("s_nop 15\n\ts_nop 15" : : : "memory");      // the last products' sums are read after enough wait states
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        asm volatile("" : "+a"(acc[i][j]));
        asm volatile("" : "+a"(low[i][j]));
      }
  }

  // lane (li, lq) holds out[t = tile row li][n = 4 lq + r of tile column j].  The sums there are asked for a tile of tokens ahead of the stores.
  const int nbase = n0 + wn * WN * 16 + 4 * lq;
  const bool fours = (out_stride & 3) == 0;
  int ew[WN][4];
  float add[WN][4];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) ew[j][r] = w_exp[min(nbase + 16 * j + r, N - 1)];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = min(nbase + 16 * j + r, N - 1);
      add[j][r] = !bias ? 0.f : bias_dtype == kBF16 ? to_float(reinterpret_cast<const bf16_t*>(bias)[n]) : reinterpret_cast<const float*>(bias)[n];
    }
  int ex[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) ex[i] = x_exp[min(t0 + (wm * WM + i) * 16 + li, T - 1)];
  float4 there[2][WN];
  auto fetch = [&](int i) __attribute__((always_inline)) {
    const float* row = out + size_t(min(t0 + (wm * WM + i) * 16 + li, T - 1)) * out_stride;
#pragma unroll
    for (int j = 0; j < WN; ++j)
      if (MODE == kAccumulate && fours && nbase + 16 * j + 4 <= N) there[i & 1][j] = *reinterpret_cast<const float4*>(row + nbase + 16 * j);
  };
  bool strange = false;
  fetch(0);
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    if constexpr (AGPR) {
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        asm volatile("" : "+a"(acc[i][j]));
        asm volatile("" : "+a"(low[i][j]));
      }
    }
    if (i + 1 < WM) fetch(i + 1);
    const int t = t0 + (wm * WM + i) * 16 + li;
    float* row = out + size_t(min(t, T - 1)) * out_stride;
    auto values = [&](int j, float (&v)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = ex[i] + ew[j][r];
        const float back = __builtin_amdgcn_ldexpf(acc[i][j][r] + low[i][j][r], -e);
        const bool beyond = e >= kNotFinite / 2;      // exponents of finite rows lie between -78 and 199
        v[r] = (beyond ? 0.f : (t ^ (nbase + 16 * j + r)) & 1 ? -back : back) + add[j][r];
        strange |= beyond;
      }
    };
    if constexpr (MODE == kSilu) {
#pragma unroll
      for (int j = 0; j < WN; j += 2) {
        const int n = nbase + 16 * j;      // of the gate rows of a pair, which is whole: N in 32s
        float g[4], u[4];
        values(j, g);
        values(j + 1, u);
        if (t >= T || n >= N) continue;
        auto store = [&](int which) __attribute__((always_inline)) {
          *reinterpret_cast<float4*>(row + (n >> 5) * 16 + (n & 15)) =
              make_float4(gated_value(g[0], u[0], which, limit), gated_value(g[1], u[1], which, limit), gated_value(g[2], u[2], which, limit),
                          gated_value(g[3], u[3], which, limit));
        };
        if (act == kActSilu) store(kActSilu);      // one choice for four numbers
        else store(act);
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int n = nbase + 16 * j;
      float v[4];
      values(j, v);
      if (t >= T || n >= N) continue;
      if (fours && n + 4 <= N) {
        if (MODE == kAccumulate) {
          const float4 old = there[i & 1][j];
          *reinterpret_cast<float4*>(row + n) = make_float4(old.x + v[0], old.y + v[1], old.z + v[2], old.w + v[3]);
        } else {
          *reinterpret_cast<float4*>(row + n) = make_float4(v[0], v[1], v[2], v[3]);
        }
      } else {
        for (int r = 0; r < 4 && n + r < N; ++r) row[n + r] = MODE == kAccumulate ? row[n + r] + v[r] : v[r];
      }
    }
  }
  if (!__syncthreads_or(strange)) return;
  // results of rows that are not finite, number by number
  auto by_number = [&](int t, int n, int et, int en, auto zero) {
    auto sum = zero;
    for (int k = 0; k < K; k += 8) {
      float xv[8], wv[8];
      numbers_of(x, t, k, K, et, xv);
      numbers_of(w, n, k, K, en, wv);
#pragma unroll
      for (int e = 0; e < 8; ++e) sum = __builtin_elementwise_fma(decltype(zero)(xv[e]), decltype(zero)(wv[e]), sum);
    }
    return sum;
  };
  auto value = [&](int t, int n, int et) -> float {
    const int en = w_exp[n];
    if (max(et, en) == kHasNan) return __builtin_nanf("");
    if (max(et, en) == kNotFinite) return by_number(t, n, et, en, 0.f);
    return float(by_number(t, n, et, en, 0.0));      // a finite result that meets one that is not: its sums above are gone
  };
  if constexpr (MODE == kSilu) {
    for (int at = threadIdx.x; at < BM * BN / 2; at += 256) {
      const int t = t0 + at / (BN / 2), c = at % (BN / 2), n = n0 + (c >> 4) * 32 + (c & 15);
      if (t >= T || n >= N) continue;
      const int et = x_exp[t];
      if (max(et, max(w_exp[n], w_exp[n + 16])) < kNotFinite) continue;
      out[size_t(t) * out_stride + n0 / 2 + c] = gated_value(value(t, n, et), value(t, n + 16, et), act, limit);
    }
    return;
  }
  // ... bias, and what was there before, stand in the output; the sums are added to them
  for (int at = threadIdx.x; at < BM * BN; at += 256) {
    const int t = t0 + at / BN, n = n0 + at % BN;
    if (t >= T || n >= N) continue;
    const int et = x_exp[t];
    if (max(et, w_exp[n]) < kNotFinite) continue;
    out[size_t(t) * out_stride + n] += value(t, n, et);
  }
}

// The block shapes: X(index, WM, WN, STAGES), and what was measured of them, fitted over 35 products (256 to 2,048 tokens, 896 to
// 18,944 rows, K of 896 to 4,864) on every shape: microseconds of a step of 32 along K on a full chip, and, where two blocks share a CU,
// of one that has a CU to itself.
#define SPROUT_SPLIT_SHAPES(X) X(0, 8, 4, 2) X(1, 6, 4, 2) X(2, 2, 4, 4) X(3, 4, 2, 2) X(4, 2, 2, 3) X(5, 2, 2, 4) X(6, 6, 2, 3)
struct SplitShape { int wm, wn, per_cu; };
constexpr SplitShape kSplitShapes[] = {
#define SPROUT_SPLIT_ROW(I, WM, WN, STAGES) {WM, WN, split_shares_cu<WM, WN, STAGES> ? 2 : 1},
    SPROUT_SPLIT_SHAPES(SPROUT_SPLIT_ROW)
#undef SPROUT_SPLIT_ROW
};
constexpr float kSplitStepUs[] = {1.95f, 1.48f, 0.61f, 1.10f, 0.66f, 0.37f, 0.85f};
constexpr float kSplitAloneUs[] = {1.95f, 1.48f, 0.61f, 0.69f, 0.38f, 0.37f, 0.85f};

// Rounds of blocks on the XCD that holds the most, as in quad_choice (gemm_quad.hip); the choice takes 1 % longer than the best shape
// over the 35 products (mean; 17 % at worst).
int choose_split_shape(int T, int N, int K, float* time_us) {
  int best = 0;
  const float steps = float(K / kStep);
  for (int i = 0; i < int(sizeof(kSplitShapes) / sizeof(kSplitShapes[0])); ++i) {
    const SplitShape& p = kSplitShapes[i];
    const PipeTiles tiles = pipe_tiles((T + 32 * p.wm - 1) / (32 * p.wm), (N + 32 * p.wn - 1) / (32 * p.wn));
    const int blocks = tiles.full * tiles.tiles_t + tiles.run, slots = 32 * p.per_cu, full = blocks / slots, rest = blocks % slots;
    const float ends = 0.41f * float(p.wm * p.wn) + 0.61f, block = steps * kSplitStepUs[i] + ends, alone = steps * kSplitAloneUs[i] + ends;
    float us = 2.7f + full * block;
    if (rest > 32) us += fmaxf(alone, block * (0.85f + 0.15f * float(rest - 32) / 32.f));
    else if (rest) us += alone * (0.81f + 0.19f * float(rest) / 32.f);
    if (i == 0 || us < *time_us) { best = i; *time_us = us; }
  }
  return best;
}

struct Product {
  const unsigned char *x, *w;
  const int32_t *x_exp, *w_exp;
  const void* bias;      // may be null
  int bias_dtype;
  float* out;
  int T, N, K;
  long long out_stride;
  int act;
  float limit;
};

template <int WM, int WN, int STAGES, int MODE>
int launch_mode(hipStream_t s, const Product& p) {
  constexpr int lds = split_lds<WM, WN, STAGES>;
  static bool raised = false;
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(split_product_kernel<WM, WN, STAGES, MODE>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      set_error("sp_gemm_f32_split: cannot raise the LDS limit: %s", hipGetErrorString(e));
      return 1;
    }
    raised = true;
  }
  const PipeTiles tiles = pipe_tiles((p.T + 32 * WM - 1) / (32 * WM), (p.N + 32 * WN - 1) / (32 * WN));
  split_product_kernel<WM, WN, STAGES, MODE><<<8 * (tiles.own + tiles.run), 256, lds, s>>>(
      p.x, p.w, p.x_exp, p.w_exp, p.bias, p.bias_dtype, p.out, p.T, p.N, p.K, p.out_stride, p.act, p.limit);
  return check_launch("sp_gemm_f32_split");
}

int product(hipStream_t s, const Product& p, int mode) {
  float time_us;
  switch (choose_split_shape(p.T, p.N, p.K, &time_us)) {
#define SPROUT_SPLIT_CASE(I, WM, WN, STAGES) \
    case I: return mode == kSilu ? launch_mode<WM, WN, STAGES, kSilu>(s, p) \
                 : mode == kAccumulate ? launch_mode<WM, WN, STAGES, kAccumulate>(s, p) : launch_mode<WM, WN, STAGES, kStoreF32>(s, p);
    SPROUT_SPLIT_SHAPES(SPROUT_SPLIT_CASE)
#undef SPROUT_SPLIT_CASE
  }
  set_error("sp_gemm_f32_split: no shape for %d tokens, %d rows, K = %d", p.T, p.N, p.K);
  return 1;
}

// ... and of a split of `rows` rows of K numbers, at 4.6 TB/s.
float split_time_us(int rows, int K) { return 4.f + float(rows) * float(K) * 10.f / 4.6e6f; }

int64_t aligned(int64_t bytes) { return (bytes + 255) / 256 * 256; }
int64_t split_bytes(int rows, int K) { return aligned(int64_t((rows + 1) / 2) * (K / kStep) * kStepBytes); }
// Numbers of K of one pass: all, or equal pieces of whole steps.
int piece_of(int K) {
  const int pieces = (K + kMaxK - 1) / kMaxK;
  return ((K / kStep + pieces - 1) / pieces) * kStep;
}
// Rows of w of one launch: all of them; or of those that the chunk holds whole rounds of the largest blocks over the chip.
int chunk_rows(int T, int N, int K) {
  const int64_t rows = kChunkBytes / (int64_t(K) * 6) / 256 * 256;
  if (rows >= N) return N;
  const int token_tiles = (T + 255) / 256, round = token_tiles < 256 ? 256 / token_tiles * 128 : 256;
  return int(rows >= round ? rows / round * round : rows);
}

}  // namespace

}  // namespace sprout

using namespace sprout;

// Bytes of workspace that sp_gemm_f32_split wants for T tokens by N rows of K, or 0 where it does not take the product.
extern "C" int64_t sp_gemm_f32_split_bytes(int T, int N, int K) {
  if (T < 256 || N < 1 || K < 64 || K % kStep) return 0;
  const int piece = piece_of(K);
  return split_bytes(T, piece) + split_bytes(chunk_rows(T, N, piece), piece) + aligned(int64_t(T) * 4) + aligned(int64_t(N) * 4);
}

// Whether sp_gemm_f32_split is taken to be faster than the float32 instruction's kernel: the weights are split once a call, which
// few tokens do not pay for, and small products pay for the launches (float32 instruction's product -> whole calls with the norm or
// the gate, us: 640 tokens by 9,728 rows of 896 101 -> 80, 2,048 320 -> 202; 896 rows of 4,864 at 1,500 tokens 164 -> 115, 2,048 163 -> 124;
// 37,888 of 3,584 at 512 tokens 1,079 -> 1,050, at 1,024 2,120 -> 1,559, at 2,048 4,095 -> 2,513; 3,584 of 18,944 at 512 615 -> 546,
// at 2,048 2,226 -> 1,457; at 2,048 tokens 1,152 of 896 46 -> 44, 896 of 896 36 -> 50, which is not taken).
extern "C" int sp_gemm_f32_split_pays(int T, int N, int K) {
  if (sp_gemm_f32_split_bytes(T, N, K) == 0) return 0;
  const int piece = piece_of(K), chunk = chunk_rows(T, N, piece);
  float us = 0.f;
  for (int k = 0; k < K; k += piece) {
    const int width = min(K - k, piece);
    us += split_time_us(T, width);
    for (int n = 0; n < N; n += chunk) {
      float time_us;
      choose_split_shape(T, min(N - n, chunk), width, &time_us);
      us += split_time_us(min(N - n, chunk), width) + time_us;
    }
  }
  return us < gemm_f32_time_us(T, N, K);
}

// Whether sp_gemm_f32_split takes the product as a gated one (mode 2): gate and up rows in sixteens, K in one piece (the values are
// gated where the sums end).
extern "C" int sp_gemm_f32_split_gates(int T, int N, int K) { return sp_gemm_f32_split_bytes(T, N, K) > 0 && N % 32 == 0 && piece_of(K) == K; }

// out[T, N] = or += rows . w^T + bias, everything float32; rows: `kind` 0: a [T, K]; 1: act(a[:, :K], a[:, K:]) of a [T, 2 K];
// 2: rmsnorm(a) * norm_w.  mode 1 adds into out; mode 2 (not of kind 1, without a bias): out[T, N / 2] = act(rows . first half of w) times
// rows . second half.
extern "C" int sp_gemm_f32_split(void* stream, int kind, const float* a, const float* norm_w, float eps, int activation, float limit,
                                 const float* w, int bias_dtype, const void* bias, int mode, float* out, int T, int N, int K, void* workspace, int64_t workspace_bytes) {
  const int64_t need = sp_gemm_f32_split_bytes(T, N, K);
  SP_REQUIRE(need > 0, "sp_gemm_f32_split: T=%d N=%d K=%d is not taken", T, N, K);
  SP_REQUIRE(kind >= 0 && kind <= 2 && (kind != kRowsNormed || norm_w) && mode >= 0 && mode <= 2, "sp_gemm_f32_split: unknown kind %d or mode %d", kind, mode);
  SP_REQUIRE(activation >= 0 && activation < kGateActs, "sp_gemm_f32_split: no kernel for activation %d", activation);
  SP_REQUIRE(mode != 2 || (kind != kRowsGated && !bias && sp_gemm_f32_split_gates(T, N, K)), "sp_gemm_f32_split: T=%d N=%d K=%d kind %d is not taken as a gated product", T, N, K, kind);
  SP_REQUIRE(!bias || bias_dtype == kF32 || bias_dtype == kBF16, "sp_gemm_f32_split: unsupported bias dtype %d", bias_dtype);
  SP_REQUIRE(a && w && out && workspace && workspace_bytes >= need, "sp_gemm_f32_split: null operand, or a workspace of %lld bytes where %lld are needed",
             (long long)workspace_bytes, (long long)need);
  SP_REQUIRE((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(norm_w) | reinterpret_cast<uintptr_t>(w) |
              reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(workspace)) % 16 == 0,
             "sp_gemm_f32_split: operands must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  const int piece = piece_of(K), chunk = chunk_rows(T, N, piece);
  unsigned char* at = (unsigned char*)workspace;
  unsigned char* xs = at; at += split_bytes(T, piece);
  unsigned char* ws = at; at += split_bytes(chunk, piece);
  int32_t* x_exp = (int32_t*)at; at += aligned(int64_t(T) * 4);
  int32_t* w_exp = (int32_t*)at;
  for (int k = 0; k < K; k += piece) {
    const int width = K - k < piece ? K - k : piece;
    const SplitSource src = {a, K, k, norm_w, eps, activation, limit};
    if (kind == kRowsAsTheyAre ? launch_split<kRowsAsTheyAre>(s, src, xs, x_exp, T, width)
        : kind == kRowsGated   ? launch_split<kRowsGated>(s, src, xs, x_exp, T, width)
                               : launch_split<kRowsNormed>(s, src, xs, x_exp, T, width))
      return 1;
    for (int n = 0; n < N; n += chunk) {
      const int rows = N - n < chunk ? N - n : chunk;
      SplitSource wsrc = {};
      wsrc.a = mode == 2 ? w : w + size_t(n) * K;
      wsrc.length = K;
      wsrc.first = k;
      wsrc.row0 = n;
      wsrc.half = N / 2;
      if (mode == 2 ? launch_split<kRowsPaired>(s, wsrc, ws, w_exp + n, rows, width) : launch_split<kRowsAsTheyAre>(s, wsrc, ws, w_exp + n, rows, width)) return 1;
      const void* rows_bias = !bias || k > 0 ? nullptr : bias_dtype == kBF16 ? (const void*)((const bf16_t*)bias + n) : (const void*)((const float*)bias + n);
      const Product p = {xs, ws, x_exp, w_exp + n, rows_bias, bias_dtype, mode == 2 ? out + n / 2 : out + n, T, rows, width, mode == 2 ? N / 2 : N, activation, limit};
      if (const int rc = product(s, p, mode == 2 ? kSilu : mode == 1 || k > 0 ? kAccumulate : kStoreF32)) return rc;
    }
  }
  return 0;
}
