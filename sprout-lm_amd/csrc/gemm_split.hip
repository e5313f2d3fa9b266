// float32 products of many tokens on the bfloat16 matrix cores: out (float32) = or += a[T, K] . w[N, K]^T, K in 32s.
//
// v_mfma_f32_32x32x2_f32 gives 157 TFLOP/s, the bfloat16 instruction sixteen times that.  A float32 number is the sum of three
// bfloat16 numbers to its last bit (three_parts of mfma.h), and a product is taken as the six products of parts that reach 2^-24 of
// it: a1 b1, a1 b2, a2 b1, a2 b2, a1 b3, a3 b1; what is left out is 2^-26 of it at most, less than the float32 product's own rounding.
// a1 b1 is summed in one float32 accumulator and the other five, 2^-8 of its size, in a second: a result is rounded once for every
// sixteen numbers of K and once where the two meet, where the float32 instruction rounds once for every number that is not zero
// and at most once for every two.  Relative error of the result against 64 bits, float32 instruction -> this: normal operands,
// K = 896 5.4e-7 -> 1.7e-7, 4,864 1.25e-6 -> 4.3e-7, 27,648 3.0e-6 -> 4.3e-7; weights with 1, 2, 8 and 64 numbers a row that are not
// zero 2.5e-8 -> 2.6e-8, 3.1e-8 -> 2.6e-8, 5.4e-8 -> 2.9e-8, 1.4e-7 -> 5.7e-8; one number 2^100 times the others of its row against a
// weight of zero 5.4e-7 -> 1.7e-7.  Time, whole call (2,048 tokens): 9,728 rows of 896 303 -> 235 us (of it 21 the splits, at 4.6
// TB/s; the product 203, at 1.05 PFLOP/s of bfloat16 products), 896 rows of 4,864 182 -> 154, 37,888 rows of 3,584 4,268 -> 2,958.
//
// (Pairs of float16 numbers took three products and half the time, but held 23 bits of 24, and numbers below 2^-17 of
// their row's largest less and less of them: one number that stood 2^24 out of its row and met no weight left an error of 2e-5.)
//
// Every row is multiplied by a power of two that brings its largest number into [2^49, 2^50): numbers down to 2^-150 of it keep all
// their bits, whatever the size of the row, and no sum overflows.  Powers of two are exact, and the sums are multiplied back
// by them.  A row with an infinity passes as its bits (upper and lower sixteen in two parts): its results are taken number by
// number behind the others, as the float32 instruction gives them; a row with a NaN gives NaN, whatever it meets (896
// rows of 4,864, 2,048 tokens, whole call: 159 us; one token with a NaN 1,390 -> 166, 32 of them 2,560 -> 169; with an infinity 1,360).
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

enum { kRowsAsTheyAre = 0, kRowsGated = 1, kRowsNormed = 2 };

struct SplitSource {
  const float* a;              // [rows][length]; kRowsGated: [rows][2 length], gate then up
  int length, first;           // of a row of the product, and the first of its numbers that is split
  const float* norm_w;         // kRowsNormed: a row is (a * scale) * norm_w, scale = 1 / rms
  float eps;
  int act;                     // kRowsGated
  float limit;
};

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
  const float* whole = src.a + size_t(row) * (KIND == kRowsGated ? 2 * src.length : src.length);
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

// Number k of a split row, as it was.
__device__ float number_of(const unsigned char* __restrict__ parts, int row, int k, int K, int exponent) {
  const uint16_t* p = reinterpret_cast<const uint16_t*>(parts + row_at(row, K) + size_t(k / kStep) * kStepBytes) + k % kStep;
  const uint32_t p1 = p[0], p2 = p[64], p3 = p[128];
  if (exponent == kNotFinite) return __uint_as_float(p1 << 16 | p2);
  const float x = __uint_as_float(p1 << 16) + (__uint_as_float(p2 << 16) + __uint_as_float(p3 << 16));
  return __builtin_amdgcn_ldexpf(row & 1 ? -x : x, -exponent);
}

// The pipelined kernel of gemm_pipe.h (its ring, its waits, its numbering of tiles) with three parts an operand: a stage is 32 numbers
// of K, BM + BN rows of three times 64 bytes, each part a plane of lines of two rows.  Piece c of 16 bytes of the row r & 1 of line
// l = r / 2 lies at position (4 (r & 1) + c) ^ s(l) of it, s(l) = (l ^ l / 4) & 3: the 16 rows that a quarter of a wave reads
// together lie on all banks, whether the LDS has 32 or 64, and s is the same 32 rows on.  A fetch of 1 KB is eight lines of a
// plane, which are lines of memory.
// What bounds it: a wave issues 12 WM WN matrix instructions a stage for 6 (WM + WN) KB from LDS; a block of 256 x 128 reads 72 KB
// from L2 for 3,072 cycles of matrix instructions a SIMD, as the bfloat16 product of 384 x 256 reads 80.
template <int WM, int WN, int WAVES_M, int WAVES_N, int STAGES, int MODE, typename TB>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, (WAVES_M * WAVES_N <= 4 ? 2 : 1)) void split_product_kernel(
    const unsigned char* __restrict__ x, const unsigned char* __restrict__ w, const int32_t* __restrict__ x_exp,
    const int32_t* __restrict__ w_exp, const TB* __restrict__ bias, float* out, int T, int N, int K, RopeArgs rope) {
  constexpr int NW = WAVES_M * WAVES_N, BM = 32 * WM * WAVES_M, BN = 32 * WN * WAVES_N;
  constexpr int STAGE = (BM + BN) * 192, XBYTES = BM * 192;
  constexpr int LX = 3 * BM / (16 * NW), LW = 3 * BN / (16 * NW);      // load instructions per wave, stage and operand
  static_assert(3 * BM % (16 * NW) == 0 && 3 * BN % (16 * NW) == 0, "every wave fills whole groups of 8 lines");
  static_assert((STAGES - 2) * (LX + LW) <= 63, "vmcnt holds six bits");
  extern __shared__ __attribute__((aligned(1024))) unsigned char pipe_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int li = lane & 31, lk = lane >> 5;
  int tile_n, tile_t;
  if (!pipe_tile_of(pipe_tiles((T + BM - 1) / BM, (N + BN - 1) / BN), blockIdx.x, &tile_t, &tile_n)) return;
  const int t0 = tile_t * BM, n0 = tile_n * BN;
  const int steps = K / kStep;
  typedef __attribute__((address_space(3))) unsigned char* lds_address_t;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_address_t)pipe_lds;
  const uint32_t pitch = uint32_t(steps) * kStepBytes;      // of a line of two rows
  const unsigned char *xbase = x + size_t(t0 / 2) * pitch, *wbase = w + size_t(n0 / 2) * pitch;
  uint32_t xoff[LX], woff[LW];
  // fetch u = NW j + wave of an operand: eight lines of part u / (rows / 16)
  auto offset_of = [&](int u, int rows, int last_line) {
    const int part = u / (rows / 16), line = (u % (rows / 16)) * 8 + (lane >> 3), piece = (lane & 7) ^ ((line ^ (line >> 2)) & 3);
    return uint32_t(min(line, last_line)) * pitch + part * 128 + piece * 16;
  };
#pragma unroll
  for (int j = 0; j < LX; ++j) xoff[j] = offset_of(NW * j + wave, BM, (T - 1 - t0) / 2);
#pragma unroll
  for (int j = 0; j < LW; ++j) woff[j] = offset_of(NW * j + wave, BN, (N - 1 - n0) / 2);
  auto fetch = [&](int buf, int step) {
    const unsigned char* xs = xbase + size_t(step) * kStepBytes;
    const unsigned char* ws = wbase + size_t(step) * kStepBytes;
    const uint32_t dst = lds0 + buf * STAGE + wave * 1024;
#pragma unroll
    for (int j = 0; j < LX; ++j) load_to_lds(xs, xoff[j], dst + NW * j * 1024);
#pragma unroll
    for (int j = 0; j < LW; ++j) load_to_lds(ws, woff[j], dst + XBYTES + NW * j * 1024);
  };
  // row 32 i + li of the wave's, pieces 2 ks + lk of a part
  const uint32_t position = (li >> 1) * 128 + (((((li & 1) << 2) | lk) ^ (((li >> 1) ^ (li >> 3)) & 3)) << 4);
  const uint32_t xrow = wm * WM * 2048 + position, wrow = XBYTES + wn * WN * 2048 + position;

  floatx16 acc[WM][WN], low[WM][WN];      // sums of the first parts' products, and of the others
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.f;

  auto multiply = [&](int buf) {
    const unsigned char* stage = pipe_lds + buf * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 b[WN][3];
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int h = 0; h < 3; ++h)
          b[j][h] = as_bf16x8(*reinterpret_cast<const uint4*>(stage + (wrow ^ (ks * 32)) + h * (BN * 64) + j * 2048));
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        bf16x8 a[3];
#pragma unroll
        for (int h = 0; h < 3; ++h)
          a[h] = as_bf16x8(*reinterpret_cast<const uint4*>(stage + (xrow ^ (ks * 32)) + h * (BM * 64) + i * 2048));
#pragma unroll
        for (int j = 0; j < WN; ++j) low[i][j] = mfma32(b[j][0], a[2], low[i][j]);
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = mfma32(b[j][0], a[0], acc[i][j]);
#pragma unroll
        for (int j = 0; j < WN; ++j) low[i][j] = mfma32(b[j][2], a[0], low[i][j]);
#pragma unroll
        for (int j = 0; j < WN; ++j) low[i][j] = mfma32(b[j][1], a[1], low[i][j]);
#pragma unroll
        for (int j = 0; j < WN; ++j) low[i][j] = mfma32(b[j][0], a[1], low[i][j]);
#pragma unroll
        for (int j = 0; j < WN; ++j) low[i][j] = mfma32(b[j][1], a[0], low[i][j]);
      }
    }
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < steps) fetch(s, s);
  for (int s0 = 0; s0 < steps; s0 += STAGES) {
#pragma unroll
    for (int u = 0; u < STAGES; ++u) {
      const int s = s0 + u;
      if (s >= steps) break;
      // every wave's loads of step s have landed, and every wave is done with step s - 1
      if (steps - 1 - s >= STAGES - 2) wait_loads_then_barrier<(STAGES - 2) * (LX + LW)>();
      else wait_loads_then_barrier<0>();
      if (s + STAGES - 1 < steps) fetch((u + STAGES - 1) % STAGES, s + STAGES - 1);
      multiply(u);
    }
  }
  bool strange = false;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int t = t0 + (wm * WM + i) * 32 + li, ex = x_exp[min(t, T - 1)];
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + (wn * WN + j) * 32 + 8 * (r / 4) + 4 * lk + r % 4, e = ex + w_exp[min(n, N - 1)];
        const float back = __builtin_amdgcn_ldexpf(acc[i][j][r] + low[i][j][r], -e);
        const bool beyond = e >= kNotFinite / 2;      // exponents of finite rows lie between -78 and 199
        acc[i][j][r] = beyond ? 0.f : (t ^ n) & 1 ? -back : back;
        strange |= beyond;
      }
  }
  tile_epilogue<WM, WN, MODE, TB, WAVES_N, true>(acc, reinterpret_cast<float*>(pipe_lds), bias, out, T, N, t0, n0, rope);
  if (!__syncthreads_or(strange)) return;
  // results of rows that are not finite: bias, and what was there before, stand in the output; the sums are added to them
  for (int at = threadIdx.x; at < BM * BN; at += 64 * NW) {
    const int t = t0 + at / BN, n = n0 + at % BN;
    if (t >= T || n >= N) continue;
    const int ex = x_exp[t], ew = w_exp[n];
    if (max(ex, ew) < kNotFinite) continue;
    const bool nan = max(ex, ew) == kHasNan;
    float sum = nan ? __builtin_nanf("") : 0.f;
    for (int k = 0; k < K && !nan; ++k) sum = fmaf(number_of(x, t, k, K, ex), number_of(w, n, k, K, ew), sum);
    out[size_t(t) * rope.row_stride + n] += sum;
  }
}

// Block shapes, blocks a CU holds, microseconds of a block's start and end, of a step of 32 along K on a CU by itself, and of one
// where the chip is full.
struct SplitShape { int bm, bn, per_cu; float start_us, light_us, full_us; };
constexpr SplitShape kSplitShapes[] = {{256, 128, 1, 8.f, 1.75f, 2.35f}, {128, 64, 2, 3.f, 0.73f, 1.38f}, {64, 64, 2, 3.f, 0.44f, 0.80f}};

int choose_split_shape(int T, int N, int K, float* time_us) {
  int best = 0;
  const float steps = float(K / kStep);
  for (int i = 0; i < int(sizeof(kSplitShapes) / sizeof(kSplitShapes[0])); ++i) {
    const SplitShape& p = kSplitShapes[i];
    const long blocks = long((T + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn), slots = 256 * p.per_cu;
    const long rounds = blocks / slots, rest = blocks % slots;
    float us = float(rounds) * (p.start_us + steps * p.full_us) + 3.f;
    const float shared = p.per_cu == 1 ? float(rest) / float(slots) : rest > 256 ? 1.f : 0.f;
    if (rest) us += p.start_us + steps * (p.light_us + (p.full_us - p.light_us) * shared);
    if (i == 0 || us < *time_us) { best = i; *time_us = us; }
  }
  return best;
}

struct Product {
  const unsigned char *x, *w;
  const int32_t *x_exp, *w_exp;
  const void* bias;      // may be null
  float* out;
  int T, N, K;
  long long out_stride;
};

template <int WM, int WN, int WAVES_M, int WAVES_N, int STAGES, int MODE, typename TB>
int launch_mode(hipStream_t s, const Product& p) {
  constexpr int BM = 32 * WM * WAVES_M, BN = 32 * WN * WAVES_N, lds = STAGES * (BM + BN) * 192;
  static bool raised = false;
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(split_product_kernel<WM, WN, WAVES_M, WAVES_N, STAGES, MODE, TB>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      set_error("sp_gemm_f32_split: cannot raise the LDS limit: %s", hipGetErrorString(e));
      return 1;
    }
    raised = true;
  }
  const PipeTiles tiles = pipe_tiles((p.T + BM - 1) / BM, (p.N + BN - 1) / BN);
  RopeArgs args = {};
  args.row_stride = p.out_stride;
  split_product_kernel<WM, WN, WAVES_M, WAVES_N, STAGES, MODE, TB><<<8 * (tiles.own + tiles.run), 64 * WAVES_M * WAVES_N, lds, s>>>(
      p.x, p.w, p.x_exp, p.w_exp, (const TB*)p.bias, p.out, p.T, p.N, p.K, args);
  return check_launch("sp_gemm_f32_split");
}

template <int WM, int WN, int WAVES_M, int WAVES_N, int STAGES>
int launch_product(hipStream_t s, const Product& p, bool add, int bias_dtype) {
  if (p.bias && bias_dtype == kBF16)
    return add ? launch_mode<WM, WN, WAVES_M, WAVES_N, STAGES, kAccumulate, bf16_t>(s, p)
               : launch_mode<WM, WN, WAVES_M, WAVES_N, STAGES, kStoreF32, bf16_t>(s, p);
  return add ? launch_mode<WM, WN, WAVES_M, WAVES_N, STAGES, kAccumulate, float>(s, p)
             : launch_mode<WM, WN, WAVES_M, WAVES_N, STAGES, kStoreF32, float>(s, p);
}

int product(hipStream_t s, const Product& p, bool add, int bias_dtype) {
  float time_us;
  switch (choose_split_shape(p.T, p.N, p.K, &time_us)) {
    case 0: return launch_product<2, 2, 4, 2, 2>(s, p, add, bias_dtype);
    case 1: return launch_product<2, 1, 2, 2, 2>(s, p, add, bias_dtype);
    default: return launch_product<1, 1, 2, 2, 3>(s, p, add, bias_dtype);
  }
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
// few tokens do not pay for, and small products pay for the launches (whole calls with the norm or the gate before them, float32
// instruction -> this, us: 640 tokens by 9,728 rows of 896 129 -> 92, 2,048 303 -> 235; 896 rows of 4,864 at 1,500 tokens 176 -> 138, 2,048
// 182 -> 154; 37,888 of 3,584 at 512 tokens 1,108 -> 1,216, at 1,024 2,170 -> 1,862, at 2,048 4,268 -> 2,958; 3,584 of 18,944 at 512
// 645 -> 652, at 2,048 2,339 -> 1,654; 896 of 896 at 2,048 34 -> 43).  The two estimates were within a fifth of what was measured
// over 124 products, and took none to the slower side by more than 3 %.
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

// out[T, N] = or += rows . w^T + bias, everything float32; rows: `kind` 0: a [T, K]; 1: act(a[:, :K], a[:, K:]) of a [T, 2 K];
// 2: rmsnorm(a) * norm_w.  mode 1 adds into out.
extern "C" int sp_gemm_f32_split(void* stream, int kind, const float* a, const float* norm_w, float eps, int activation, float limit,
                                 const float* w, int bias_dtype, const void* bias, int mode, float* out, int T, int N, int K, void* workspace, int64_t workspace_bytes) {
  const int64_t need = sp_gemm_f32_split_bytes(T, N, K);
  SP_REQUIRE(need > 0, "sp_gemm_f32_split: T=%d N=%d K=%d is not taken", T, N, K);
  SP_REQUIRE(kind >= 0 && kind <= 2 && (kind != kRowsNormed || norm_w) && (mode == 0 || mode == 1), "sp_gemm_f32_split: unknown kind %d or mode %d", kind, mode);
  SP_REQUIRE(activation >= 0 && activation < kGateActs, "sp_gemm_f32_split: no kernel for activation %d", activation);
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
      wsrc.a = w + size_t(n) * K;
      wsrc.length = K;
      wsrc.first = k;
      if (launch_split<kRowsAsTheyAre>(s, wsrc, ws, w_exp + n, rows, width)) return 1;
      const void* rows_bias = !bias || k > 0 ? nullptr : bias_dtype == kBF16 ? (const void*)((const bf16_t*)bias + n) : (const void*)((const float*)bias + n);
      const Product p = {xs, ws, x_exp, w_exp + n, rows_bias, out + n, T, rows, width, N};
      if (const int rc = product(s, p, mode == 1 || k > 0, bias_dtype)) return rc;
    }
  }
  return 0;
}
