// float32 products of many tokens on the float16 matrix cores: out (float32) = or += a[T, K] . w[N, K]^T, K in 32s.
//
// v_mfma_f32_32x32x2_f32 gives 157 TFLOP/s, the float16 instruction sixteen times that.  A float32 number a is the sum of two
// float16 numbers to its last bit or the one before: upper = rn(a), lower = rn(a - upper) leave at most 2^-23 |a|, on average
// half of that where anything is left at all, and a . w = upper.upper + upper.lower + lower.upper leaves out a product of
// 2^-22 at most: three products at sixteen times the rate.  All three are summed in float32 in one accumulator, sixteen
// numbers of K an instruction instead of two, so that there are fewer roundings of the sums than before and those are what
// the error of a long product is made of: relative error of the result against 64 bits (normal operands, the float32
// instruction -> this): K = 896 5.4e-7 -> 3.4e-7, K = 4,864 1.25e-6 -> 7.8e-7.  Time, whole call (2,048 tokens): 9,728 rows of
// 896 329 -> 132 us (of it 15 the split of the weights at 4.6 TB/s), 896 rows of 4,864 179 -> 97 us, 37,888 rows of 3,584
// 4,150 -> 1,700 us (327 TFLOP/s of float32 products).
//
// float16 has five bits of exponent, so every row is multiplied by a power of two that brings its largest number into
// [2^14, 2^15): numbers down to 2^-17 of the row's largest keep a lower part of full width, and what is lost of smaller ones is
// below 2^-40 of the largest.  Powers of two are exact, and the sums are multiplied back by them.  A row that
// holds an infinity or NaN gives NaN where the float32 instruction gave an infinity or NaN.
//
// The instruction drops the bits below its sum's last place: every result lies a little (2e-8 of the results' size at K = 896,
// 1.1e-7 at 4,864) below the true one, all to the same side, which the averages that attention takes over many tokens' values do
// not lose as they lose the rest of the error.  So odd rows on either side change their sign and the results of an odd and an
// even row change it back: the mean of the error over a row or a column of results goes to 1e-9, for an operation an element.
//
// The rows are split by a kernel of their own before the product (the activations with what stands before the product,
// the norm or the gate, folded in; the weights into a workspace, a chunk of rows at a time, at the speed of memory), into the
// 128-byte slices of 32 numbers (upper, then lower parts) that the pipelined kernel of gemm_pipe.h takes.
#include "gemm_pipe.h"

namespace sprout {

namespace {

constexpr int64_t kChunkBytes = int64_t(256) << 20;      // of split weights a launch multiplies

enum { kRowsAsTheyAre = 0, kRowsGated = 1, kRowsNormed = 2 };

struct SplitSource {
  const float* a;              // [rows][K]; kRowsGated: [rows][2 K], gate then up
  const float* norm_w;         // kRowsNormed: a row is (a * scale) * norm_w, scale = 1 / rms
  float eps;
  int act;                     // kRowsGated
  float limit;
};

__device__ __forceinline__ float max4(float4 v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))); }

// One row a wave (WAVES 1, four rows a block) or a block of four waves: bound by memory, a row's numbers stay in registers
// between its largest and the split where eight pieces of 16 bytes a lane hold it, else they are formed again.
template <int WAVES, int KIND, bool FITS>
__global__ __launch_bounds__(256) void split_rows_kernel(SplitSource src, uint16_t* __restrict__ out, int32_t* __restrict__ exponents,
                                                         int rows, int K) {
  constexpr int LANES = 64 * WAVES, PIECES = 8;
  __shared__ float scratch[16];
  const int row = WAVES == 1 ? int(blockIdx.x) * 4 + (threadIdx.x >> 6) : int(blockIdx.x);
  const int lane = WAVES == 1 ? threadIdx.x & 63 : threadIdx.x;
  if (row >= rows) return;
  const int n4 = K / 4;
  const float4* a = reinterpret_cast<const float4*>(src.a + size_t(row) * (KIND == kRowsGated ? 2 * K : K));
  float factor = 1.f;
  float4 kept[FITS ? PIECES : 1];
  auto raw = [&](int i) { return a[i]; };
  if (FITS && KIND != kRowsGated) {
#pragma unroll
    for (int p = 0; p < (FITS ? PIECES : 0); ++p)
      if (lane + p * LANES < n4) kept[p] = raw(lane + p * LANES);
  }
  if (KIND == kRowsNormed) {
    float squares = 0.f;
    if (FITS) {
#pragma unroll
      for (int p = 0; p < (FITS ? PIECES : 0); ++p)
        if (lane + p * LANES < n4) squares += kept[p].x * kept[p].x + kept[p].y * kept[p].y + kept[p].z * kept[p].z + kept[p].w * kept[p].w;
    } else {
      for (int i = lane; i < n4; i += LANES) { const float4 v = raw(i); squares += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w; }
    }
    squares = WAVES == 1 ? wave_sum(squares) : block_sum(squares, scratch);
    factor = 1.0f / sqrtf(squares / float(K) + src.eps);
  }
  auto value = [&](int i, float4 v) {
    if (KIND == kRowsNormed) {
      const float4 w = reinterpret_cast<const float4*>(src.norm_w)[i];
      return make_float4(v.x * factor * w.x, v.y * factor * w.y, v.z * factor * w.z, v.w * factor * w.w);
    }
    if (KIND == kRowsGated) {
      const float4 g = a[i], u = a[i + n4];
      v = make_float4(gated_value(g.x, u.x, src.act, src.limit), gated_value(g.y, u.y, src.act, src.limit),
                      gated_value(g.z, u.z, src.act, src.limit), gated_value(g.w, u.w, src.act, src.limit));
    }
    return v;
  };
  float top = 0.f;
  bool finite = true;
  auto look = [&](float4 v) {
    const float m = max4(v);
    top = fmaxf(top, m);
    // (a maximum drops a NaN: it is looked for by itself)
    finite = finite && fabsf(v.x) < INFINITY && fabsf(v.y) < INFINITY && fabsf(v.z) < INFINITY && fabsf(v.w) < INFINITY;
  };
  if (FITS) {
#pragma unroll
    for (int p = 0; p < (FITS ? PIECES : 0); ++p)
      if (lane + p * LANES < n4) { kept[p] = value(lane + p * LANES, kept[p]); look(kept[p]); }
  } else {
    for (int i = lane; i < n4; i += LANES) look(value(i, KIND == kRowsGated ? make_float4(0, 0, 0, 0) : raw(i)));
  }
  if (!finite) top = INFINITY;
  top = wave_max(top);
  if (WAVES > 1) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = top;
    __syncthreads();
    top = fmaxf(fmaxf(scratch[0], scratch[1]), fmaxf(scratch[2], scratch[3]));
  }
  int e = 0;
  if (top > 0.f && top < INFINITY) e = 15 - __builtin_amdgcn_frexp_expf(top);      // top = m 2^x, m in [0.5, 1): m 2^15
  if (lane == 0) exponents[row] = e;
  const uint32_t odd = uint32_t(row & 1) << 31;      // odd rows change their sign (see above)
  auto store = [&](int i, float4 v) {
    uint16_t* dst = out + size_t(row) * 2 * K + size_t(i / 8) * 64 + 4 * (i % 8);
    const float f[4] = {v.x, v.y, v.z, v.w};
    uint16_t hi[4], lo[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float x = __uint_as_float(__float_as_uint(__builtin_amdgcn_ldexpf(f[c], e)) ^ odd);
      const _Float16 h = (_Float16)x;
      hi[c] = __builtin_bit_cast(uint16_t, h);
      lo[c] = __builtin_bit_cast(uint16_t, (_Float16)(x - (float)h));
    }
    *reinterpret_cast<uint2*>(dst) = make_uint2(hi[0] | uint32_t(hi[1]) << 16, hi[2] | uint32_t(hi[3]) << 16);
    *reinterpret_cast<uint2*>(dst + 32) = make_uint2(lo[0] | uint32_t(lo[1]) << 16, lo[2] | uint32_t(lo[3]) << 16);
  };
  if (FITS) {
#pragma unroll
    for (int p = 0; p < (FITS ? PIECES : 0); ++p)
      if (lane + p * LANES < n4) store(lane + p * LANES, kept[p]);
  } else {
    for (int i = lane; i < n4; i += LANES) store(i, value(i, KIND == kRowsGated ? make_float4(0, 0, 0, 0) : raw(i)));
  }
}

template <int KIND>
int launch_split(hipStream_t s, const SplitSource& src, uint16_t* out, int32_t* exponents, int rows, int K) {
  if (K <= 2048) split_rows_kernel<1, KIND, true><<<(rows + 3) / 4, 256, 0, s>>>(src, out, exponents, rows, K);
  else if (K <= 8192) split_rows_kernel<4, KIND, true><<<rows, 256, 0, s>>>(src, out, exponents, rows, K);
  else split_rows_kernel<4, KIND, false><<<rows, 256, 0, s>>>(src, out, exponents, rows, K);
  return check_launch("sp_gemm_f32_split (rows)");
}

// Block shapes, blocks a CU holds, and microseconds of a step of 32 along K where few blocks run and where every CU is full,
// measured over 200 to 2,048 tokens at 896 to 9,728 rows and K of 896 and 4,864; a block's start and end take 6 us, 3 us for
// blocks that follow others.  (The model is within 20% of what it was fitted to, and the shape it takes within 10% of the best
// there: 2,048 tokens by 9,728 rows of 896: 384 x 256 113 us, 64 x 128 125, 256 x 128 126, 128 x 128 140, 256 x 256 142;
// 2,048 by 896 rows of 4,864: 64 x 128 73 us, 64 x 64 82, 128 x 128 108; 256 tokens by 896 rows of 4,864: 64 x 64 41, 64 x 128 66.)
struct SplitShape { int bm, bn, per_cu; float light_us, full_us; };
constexpr SplitShape kSplitShapes[] = {{384, 256, 1, 2.5f, 3.8f},   {256, 256, 1, 1.75f, 2.3f}, {256, 128, 1, 1.0f, 1.28f},
                                       {128, 128, 1, 0.68f, 0.79f}, {64, 128, 2, 0.33f, 0.68f}, {64, 64, 2, 0.23f, 0.54f}};

int choose_split_shape(int T, int N, int K) {
  int best = 0;
  float best_us = 0.f;
  const float steps = float(K / 32);
  for (int i = 0; i < int(sizeof(kSplitShapes) / sizeof(kSplitShapes[0])); ++i) {
    const SplitShape& p = kSplitShapes[i];
    const long blocks = long((T + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn), slots = 256 * p.per_cu;
    const long rounds = blocks / slots, rest = blocks % slots;
    float us = float(rounds) * (3.f + steps * p.full_us) + 3.f;
    if (rest) us += 3.f + steps * (p.light_us + (p.full_us - p.light_us) * float(rest) / float(slots));
    if (i == 0 || us < best_us) { best = i; best_us = us; }
  }
  return best;
}

template <int WM, int WN, int WAVES_M, int WAVES_N, int STAGES, typename TB>
int launch_product(hipStream_t s, const split_t* x, const split_t* w, const TB* bias, int mode, float* out, int T, int N, int K,
                   const RopeArgs& args) {
  if (mode == kAccumulate)
    return launch_pipe_mode<WM, WN, WAVES_M, WAVES_N, STAGES, kAccumulate, TB, split_t>(s, 1, x, w, bias, out, T, N, K, K, args);
  return launch_pipe_mode<WM, WN, WAVES_M, WAVES_N, STAGES, kStoreF32, TB, split_t>(s, 1, x, w, bias, out, T, N, K, K, args);
}

template <typename TB>
int product(hipStream_t s, int shape, const split_t* x, const split_t* w, const TB* bias, int mode, float* out, int T, int N, int K,
            const RopeArgs& args) {
  switch (shape) {
    case 0: return launch_product<6, 2, 2, 4, 2, TB>(s, x, w, bias, mode, out, T, N, K, args);
    case 1: return launch_product<4, 2, 2, 4, 2, TB>(s, x, w, bias, mode, out, T, N, K, args);
    case 2: return launch_product<2, 2, 4, 2, 3, TB>(s, x, w, bias, mode, out, T, N, K, args);
    case 3: return launch_product<2, 2, 2, 2, 4, TB>(s, x, w, bias, mode, out, T, N, K, args);
    case 4: return launch_product<1, 2, 2, 2, 3, TB>(s, x, w, bias, mode, out, T, N, K, args);
    default: return launch_product<1, 1, 2, 2, 4, TB>(s, x, w, bias, mode, out, T, N, K, args);
  }
}

int64_t aligned(int64_t bytes) { return (bytes + 255) / 256 * 256; }
// Rows of w of one launch: all of them, or as many whole tiles as the chunk holds.
int chunk_rows(int N, int K) {
  const int64_t rows = kChunkBytes / (int64_t(K) * 4) / 256 * 256;
  return int(rows >= N ? N : rows);
}

}  // namespace

}  // namespace sprout

using namespace sprout;

// Bytes of workspace that sp_gemm_f32_split wants for T tokens by N rows of K, or 0 where it does not take the product or
// the float32 instruction is as fast: the weights are split once a call, which few tokens do not pay for (whole call against the
// float32 instruction: 200 tokens by 1,152 rows of 896 21.5 us against 20.7; 256 by 9,728 of 896 47 against 53, 256 by 896 of
// 4,864 55 against 87; 2,048 by 9,728 of 896 132 against 329).
extern "C" int64_t sp_gemm_f32_split_bytes(int T, int N, int K) {
  if (T < 256 || N < 1 || K < 64 || K % 32 || int64_t(K) * 4 * 384 >= (int64_t(1) << 31) || chunk_rows(N, K) < 1) return 0;
  return aligned(int64_t(T) * K * 4) + aligned(int64_t(chunk_rows(N, K)) * K * 4) + aligned(int64_t(T) * 4) + aligned(int64_t(N) * 4);
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
  const int chunk = chunk_rows(N, K);
  unsigned char* at = (unsigned char*)workspace;
  uint16_t* xs = (uint16_t*)at; at += aligned(int64_t(T) * K * 4);
  uint16_t* ws = (uint16_t*)at; at += aligned(int64_t(chunk) * K * 4);
  int32_t* x_exp = (int32_t*)at; at += aligned(int64_t(T) * 4);
  int32_t* w_exp = (int32_t*)at;
  SplitSource src = {a, norm_w, eps, activation, limit};
  if (kind == kRowsAsTheyAre ? launch_split<kRowsAsTheyAre>(s, src, xs, x_exp, T, K)
      : kind == kRowsGated   ? launch_split<kRowsGated>(s, src, xs, x_exp, T, K)
                             : launch_split<kRowsNormed>(s, src, xs, x_exp, T, K))
    return 1;
  RopeArgs args = {};
  args.row_stride = N;
  args.x_exp = x_exp;
  for (int n = 0; n < N; n += chunk) {
    const int rows = N - n < chunk ? N - n : chunk;
    SplitSource wsrc = {};
    wsrc.a = w + size_t(n) * K;
    if (launch_split<kRowsAsTheyAre>(s, wsrc, ws, w_exp + n, rows, K)) return 1;
    args.w_exp = w_exp + n;
    const int shape = choose_split_shape(T, rows, K);
    const int rc = bias && bias_dtype == kBF16
        ? product<bf16_t>(s, shape, (const split_t*)xs, (const split_t*)ws, (const bf16_t*)bias + n, mode == 1 ? kAccumulate : kStoreF32, out + n, T, rows, K, args)
        : product<float>(s, shape, (const split_t*)xs, (const split_t*)ws, bias ? (const float*)bias + n : nullptr, mode == 1 ? kAccumulate : kStoreF32, out + n, T, rows, K, args);
    if (rc) return rc;
  }
  return 0;
}
