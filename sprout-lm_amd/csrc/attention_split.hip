// float32 attention of prompts for head sizes of 64 on the bfloat16 matrix instruction.
//
// The float32 instruction (attention_f32.hip) multiplies at a sixteenth of the bfloat16 one's rate, and its tiles of 16 read
// every operand from the caches.  A float32 number is the sum of three bfloat16 numbers to its last bit, a = a1 + a2 + a3 with
// a1 = rn(a), a2 = rn(a - a1), a3 = a - a1 - a2 (eight bits each; bfloat16 has float32's exponents, so nothing is scaled), and a
// product is taken as the six products of parts that reach 2^-24 of it (a1 b1, a1 b2, a2 b1, a2 b2, a1 b3, a3 b1), summed in
// float32: sixteen numbers an instruction, so with fewer roundings of the sums than the float32 instruction's chain of two.
// Queries, keys, values and the softmax's weights all pass it like that; scores, statistics and sums are float32.
//
// The instruction drops the bits below its sum's last place, so that its sums end a little below the true ones.  In the scores that
// moves all keys of a query alike, and the softmax drops it.  The sums over the values would carry it to every token alike
// (2.7e-8 of the results' size at 4,095 keys), where a later average over tokens keeps it and loses the rest of the error: the
// weights of odd rows have their sign changed, so that half the rows end above.
//
// What three parts cannot hold: infinities (inf - inf is NaN), numbers that round beyond bfloat16's largest, and the last bits of
// numbers below 2^-110, whose third parts end in bfloat16's subnormal numbers.  The first two end as NaN in the row's sums; values of
// the third kind end as results below kTinyResult; keys of the third kind matter beside queries above kLargeQuery only, and queries
// of the third kind are looked for.  (What stays: a value above 2^100 under a weight below 2^-110.)  A wave that finds one of them at
// the end of its walk walks again by itself, from the pools on the float32 instruction and with every maximum exact, as
// attention_f32.hip's kernel does.  The look at the sums is 50 instructions a wave: no time beyond noise in any size measured (a walk
// of the block again, through LDS, put its check's three barriers behind every block: 3 to 10 % of these launches); the look at the
// queries 83.1 -> 86.8 us for 2,048 tokens under 14 heads (at the walk's start, where the first stage's loads wait for it, 87.5; at
// its end from the queries' first parts 87.9).
//
// A block of four waves takes 32 queries of four heads of a key/value head, a wave a head; stages of 64 keys are loaded into
// registers while the one before is used, split there and written to LDS as three planes each (48 KB), key rows and value
// rows of 128 bytes in the layout of attention_rows.hip, whose tile products these are.  Two blocks run on a CU.  The matrix
// instructions bound it: 48 of them (1,536 cycles) per 32 keys and wave, behind the split of the stage at its start.
// 14 heads of 64 in 2 groups, float32 instruction -> this, merge of the parts included: 2,048 tokens 262 -> 94 us (80 TFLOP/s of
// float32 products), 2,048 behind 2,048 529 -> 192, five prompts of 47 to 611 82 -> 32, 512 tokens 70 -> 21; relative error of
// the result against 64 bits 7.0e-8 -> 4.8e-8, 1.1e-6 -> 5.8e-7, 1.5e-7 -> 9.2e-8, 1.0e-7 -> 6.7e-8.
#include "attention_mfma.h"

namespace sprout {

namespace {

constexpr int kSplitKeys = 64, kPlane = 64 * 128, kSplitTable = 2048;
constexpr float kTinyResult = 0x1p-100f, kLargeQuery = 0x1p60f, kTinyQuery = 0x1p-110f;

__device__ __forceinline__ int split_swz(int row) { return (row ^ (row >> 3)) & 7; }

__device__ __forceinline__ void three_parts8(const float (&f)[8], uint4 (&p)[3]) {
  three_parts(f[0], f[1], p[0].x, p[1].x, p[2].x);
  three_parts(f[2], f[3], p[0].y, p[1].y, p[2].y);
  three_parts(f[4], f[5], p[0].z, p[1].z, p[2].z);
  three_parts(f[6], f[7], p[0].w, p[1].w, p[2].w);
}
// c += a . b of numbers in three parts, the smallest products first.
__device__ __forceinline__ floatx16 mfma_parts(const uint4 (&a)[3], const uint4 (&b)[3], floatx16 c) {
  c = mfma32(as_bf16x8(a[2]), as_bf16x8(b[0]), c);
  c = mfma32(as_bf16x8(a[0]), as_bf16x8(b[2]), c);
  c = mfma32(as_bf16x8(a[1]), as_bf16x8(b[1]), c);
  c = mfma32(as_bf16x8(a[1]), as_bf16x8(b[0]), c);
  c = mfma32(as_bf16x8(a[0]), as_bf16x8(b[1]), c);
  return mfma32(as_bf16x8(a[0]), as_bf16x8(b[0]), c);
}
__device__ __forceinline__ float min3_of_magnitudes(float a, float b, float c) {
  float least;
  asm("v_min3_f32 %0, |%1|, |%2|, |%3|" : "=v"(least) : "v"(a), "v"(b), "v"(c));
  return least;
}
__device__ __forceinline__ float max3_of_magnitudes(float a, float b, float c) {
  float most;
  asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(most) : "v"(a), "v"(b), "v"(c));
  return most;
}
__device__ __forceinline__ float max_over_row(float x) {      // the other half of a row's keys lies in lane ^ 32
  const unsigned u = __float_as_uint(x);
  const auto f = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return vmax(__uint_as_float(f[0]), __uint_as_float(f[1]));
}

__global__ __launch_bounds__(256, 2) void attention_split_kernel(
    const float* __restrict__ q, int q_stride, const float* __restrict__ k_pool, const float* __restrict__ v_pool,
    const int32_t* __restrict__ block_tables, int max_blocks, const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len,
    const int32_t* __restrict__ ctx_len, const int32_t* __restrict__ tiles, float* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, int n_splits, int nq, int nkv, int page_shift, int num_pages, float scale2,
    int n_tiles) {
  constexpr int HD = 64;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];      // three planes of keys, three of values, the page numbers
  int32_t* s_table = reinterpret_cast<int32_t*>(lds + 6 * kPlane);
  const int tile = n_tiles - 1 - int(blockIdx.x);      // the longest walks first
  const int seq = tiles[2 * tile], q_off = tiles[2 * tile + 1];
  const int G = nq / nkv, sets = (G + 3) / 4, g = blockIdx.y / sets, in_group = (blockIdx.y % sets) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 31, lk = lane >> 5;
  const int qlen = q_len[seq], ctx = ctx_len[seq], qs = q_start[seq];
  const int nvalid = min(32, qlen - q_off);
  if (nvalid <= 0) return;
  const int pos0 = ctx - qlen + q_off, k_hi = pos0 + nvalid - 1, split = blockIdx.z;
  int lo = 0, hi = k_hi;
  if (n_splits > 1) share_of_walk(lo, hi, kSplitKeys, split, n_splits);
  const bool live = in_group < G;      // a wave without a head walks along for its share of the stages
  const int head = g * G + min(in_group, G - 1);

  const int32_t* table = block_tables + size_t(seq) * max_blocks;
  const int first_page = lo >> page_shift, n_pages = hi >= lo ? (hi >> page_shift) - first_page + 1 : 0;
  const bool table_in_lds = n_pages <= kSplitTable;
  if (table_in_lds)
    for (int i = threadIdx.x; i < n_pages; i += 256) s_table[i] = table[first_page + i];
  __syncthreads();
  const int page_mask = (1 << page_shift) - 1;
  const float* kbase = k_pool + (size_t(g) << page_shift) * HD;
  const float* vbase = v_pool + (size_t(g) << page_shift) * HD;
  auto page_at = [&](int key) __attribute__((always_inline)) {
    const int page = table_in_lds ? s_table[(key >> page_shift) - first_page] : table[key >> page_shift];
    return size_t(min(max(page, 0), num_pages - 1)) * nkv;
  };

  // What this thread moves of a stage: sixteen dimensions of key fr, and sixteen keys of dimension fr.
  const int fr = threadIdx.x >> 2, fc = threadIdx.x & 3;
  const int krow = (fr & ~12) | ((fr & 4) << 1) | ((fr & 8) >> 1);      // (see attention_rows.hip: bits 2 and 3 swapped)
  float4 kv[4], vv[4];
  auto fetch = [&](int key0) __attribute__((always_inline)) {
    const int key = min(key0 + fr, hi);      // keys behind the walk's end repeat the last one: masked by position
    const float* src = kbase + ((page_at(key) << page_shift) + (key & page_mask)) * HD + 16 * fc;
#pragma unroll
    for (int u = 0; u < 4; ++u) kv[u] = *reinterpret_cast<const float4*>(src + 4 * u);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int kb = min(key0 + 16 * fc + 4 * u, hi & ~3);
      vv[u] = *reinterpret_cast<const float4*>(vbase + ((page_at(kb) * HD + fr) << page_shift) + (kb & page_mask));
    }
  };
  auto to_lds = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      uint4 p[3];
      const float4 a = kv[2 * half], b = kv[2 * half + 1], c = vv[2 * half], d = vv[2 * half + 1];
      three_parts8({a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(lds + i * kPlane + krow * 128 + (((2 * fc + half) ^ split_swz(krow)) << 4)) = p[i];
      three_parts8({c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w}, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(lds + (3 + i) * kPlane + fr * 128 + (((2 * fc + half) ^ split_swz(fr)) << 4)) = p[i];
    }
  };

  const uint32_t odd = uint32_t(li & 1) << 31;      // odd rows' sums are held with the other sign (see above)
  uint4 qp[4][3];
  floatx16 o[2];
  float m = kNoKeyYet, l = 0.f, largest_q = 0.f, least_q = INFINITY;
  {
    const float* row = q + size_t(qs + q_off + min(li, nvalid - 1)) * q_stride + head * HD + 8 * lk;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const float4 a = *reinterpret_cast<const float4*>(row + 16 * ks), b = *reinterpret_cast<const float4*>(row + 16 * ks + 4);
      three_parts8({a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}, qp[ks]);
      largest_q = max3_of_magnitudes(max3_of_magnitudes(largest_q, a.x, a.y), a.z, a.w);
      largest_q = max3_of_magnitudes(max3_of_magnitudes(largest_q, b.x, b.y), b.z, b.w);
      least_q = min3_of_magnitudes(min3_of_magnitudes(least_q, a.x, a.y), a.z, a.w);
      least_q = min3_of_magnitudes(min3_of_magnitudes(least_q, b.x, b.y), b.z, b.w);
    }
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  }
  const int pos = li < nvalid ? min(pos0 + li, hi) : -1;
  uint32_t addr[4];      // row li (piece bits the other way round in row li + 32), pieces 2 ks + lk
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) addr[ks] = li * 128 + (((2 * ks + lk) ^ split_swz(li)) << 4);

  if (hi >= lo) fetch(lo);
  for (int key0 = lo; key0 <= hi; key0 += kSplitKeys) {
    if (key0 > lo) __syncthreads();      // the stage before has been used
    to_lds();
    __syncthreads();
    if (key0 + kSplitKeys <= hi) fetch(key0 + kSplitKeys);
    if (!live) continue;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int first = key0 + 32 * half;
      if (first > hi) break;
      floatx16 s;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        uint4 kp[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) kp[i] = *reinterpret_cast<const uint4*>(lds + i * kPlane + half * 32 * 128 + addr[half ? ks ^ 2 : ks]);
        s = mfma_parts(kp, qp[ks], s);
      }
      if (first + 31 > pos0) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (first + 8 * lk + 16 * (r / 8) + r % 8 > pos) s[r] = -INFINITY;
      }
      float top = vmax3(s[0], s[1], s[2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) top = vmax3(top, s[r], s[r + 1]);
      top = vmax(top, s[15]) * scale2;
      if (__builtin_amdgcn_ballot_w64(top > m + kRescaleStep) != 0) {
        const float t = max_over_row(top);
        const float mx = t > m + kRescaleStep ? t : m;
        const float alpha = __builtin_amdgcn_exp2f(m - mx);
        m = mx;
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      }
      float sum = 0.f;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          e[j] = __builtin_amdgcn_exp2f(fmaf(s[8 * c + j], scale2, -m));
          sum += e[j];
          e[j] = __uint_as_float(__float_as_uint(e[j]) ^ odd);
        }
        uint4 p[3];
        three_parts8(e, p);
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) {
          uint4 vp[3];
#pragma unroll
          for (int i = 0; i < 3; ++i)
            vp[i] = *reinterpret_cast<const uint4*>(lds + (3 + i) * kPlane + dt * 32 * 128 + addr[(2 * half + c) ^ (dt ? 2 : 0)]);
          o[dt] = mfma_parts(vp, p, o[dt]);
        }
      }
      l += sum;
    }
  }
  if (!live) return;
  l += __shfl_xor(l, 32, 64);
  // sums that are not finite, queries at the ends of the range, or (zeros aside) results below kTinyResult
  float total = l, least = INFINITY;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      total += fabsf(o[dt][r]);
      total += fabsf(o[dt][r + 1]);
      least = min3_of_magnitudes(least, o[dt][r], o[dt][r + 1]);
    }
  bool beyond = !(total < INFINITY) || largest_q > kLargeQuery;
  if (least_q < kTinyQuery) {      // zeros, most often
    const float* row = q + size_t(qs + q_off + min(li, nvalid - 1)) * q_stride + head * HD + 8 * lk;
#pragma unroll 1
    for (int d = 0; d < HD; d += 16)
      for (int j = 0; j < 8; ++j) beyond |= (row[d + j] != 0.f) & (fabsf(row[d + j]) < kTinyQuery);
  }
  if (least < kTinyResult * l) {
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) beyond |= (o[dt][r] != 0.f) & (fabsf(o[dt][r]) < kTinyResult * l);
  }
  if (__builtin_amdgcn_ballot_w64(beyond && li < nvalid) != 0) {
    const float* row = q + size_t(qs + q_off + min(li, nvalid - 1)) * q_stride + head * HD + 8 * lk;
    const int in_run = (li & ~12) | ((li & 4) << 1) | ((li & 8) >> 1);      // the key of row li of 32
    m = kNoKeyYet;
    l = 0.f;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
#pragma unroll 1
    for (int first = lo; first <= hi; first += 32) {
      const int key = min(first + in_run, hi);
      const float* krow = kbase + ((page_at(key) << page_shift) + (key & page_mask)) * HD + 8 * lk;
      floatx16 s;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll 1
      for (int d = 0; d < HD; d += 16)
#pragma unroll
        for (int j = 0; j < 8; ++j) s = mfma32_f32(krow[d + j], row[d + j], s);
      float top = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (first + 8 * lk + 16 * (r / 8) + r % 8 > pos) s[r] = -INFINITY;
        top = vmax(top, s[r]);
      }
      const float mx = vmax(m, max_over_row(top * scale2)), alpha = __builtin_amdgcn_exp2f(m - mx);
      m = mx;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (first + 16 * c > hi) break;      // (repeated values would have no weight, but an infinity among them would have a say)
        float e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          e[j] = __builtin_amdgcn_exp2f(fmaf(s[8 * c + j], scale2, -m));
          l += e[j];
          e[j] = __uint_as_float(__float_as_uint(e[j]) ^ odd);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int kb = min(first + 16 * c + 8 * lk + 4 * u, hi & ~3);
#pragma unroll
          for (int dt = 0; dt < 2; ++dt) {
            const float4 v = *reinterpret_cast<const float4*>(vbase + ((page_at(kb) * HD + 32 * dt + li) << page_shift) + (kb & page_mask));
            o[dt] = mfma32_f32(v.x, e[4 * u], o[dt]);
            o[dt] = mfma32_f32(v.y, e[4 * u + 1], o[dt]);
            o[dt] = mfma32_f32(v.z, e[4 * u + 2], o[dt]);
            o[dt] = mfma32_f32(v.w, e[4 * u + 3], o[dt]);
          }
        }
      }
    }
    l += __shfl_xor(l, 32, 64);
  }
  if (li >= nvalid) return;
  float* dst;
  float factor = li & 1 ? -1.f : 1.f;
  if (n_splits > 1) {
    const size_t slot = ((size_t(tile) * 32 + li) * nq + head) * n_splits + split;
    dst = part_o + slot * HD;
    if (lk == 0) *reinterpret_cast<float2*>(part_ml + 2 * slot) = make_float2(m, l);
  } else {
    dst = out + size_t(qs + q_off + li) * (size_t(nq) * HD) + head * HD;
    factor *= row_factor<false>(l);
  }
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int a = 0; a < 4; ++a)
      *reinterpret_cast<float4*>(dst + 32 * dt + 8 * a + 4 * lk) =
          make_float4(o[dt][4 * a] * factor, o[dt][4 * a + 1] * factor, o[dt][4 * a + 2] * factor, o[dt][4 * a + 3] * factor);
}

}  // namespace

// Heads of 64 and pages of a power of two of tokens, of whole pieces of 16 bytes; any number of heads a group, also where three of a
// block's waves then only carry stages (float32 instruction -> this, us, 2,048 tokens: 32 heads in 32 groups 422 -> 403, 16 in 16
// 278 -> 237, 16 in 8 406 -> 133, 12 in 4 281 -> 86, 8 in 1 267 -> 59; 256 tokens: 36 to 39 -> 17 to 18 in all of them; 64 behind
// 8,128: 1,080 -> 37 to 79; eight and 60 one-query sequences beside a prompt 169 -> 35 and 343 -> 158 under 14 heads in 2, 508 -> 480
// under 16 in 16).
bool attention_split_takes(int hd, int page_size) { return hd == 64 && page_size >= 4 && (page_size & (page_size - 1)) == 0; }

// Blocks along the keys: as many as fill the chip's 512 places two and a half times, each with four stages at least.  (14 heads in 2
// groups, 2,048 tokens: one 113 us, two 90, four 91, five 85, eight 90; 256 tokens behind 1,024: one 72, four 29, eight 25; 32 heads in 8
// groups, 2,048 tokens: one 178, two 167, four 168.)
int attention_split_splits(int n_tiles, int nq, int nkv, int max_tile_ctx) {
  const long blocks = long(n_tiles) * nkv * ((nq / nkv + 3) / 4);
  return blocks < 1 ? 1 : max(1, min(min(int(1280 / blocks), max_tile_ctx / (4 * kSplitKeys)), 16));
}

size_t attention_split_workspace_floats(int n_tiles, int nq, int nkv, int hd, int max_tile_ctx) {
  const size_t splits = attention_split_splits(n_tiles, nq, nkv, max_tile_ctx);
  return splits > 1 ? size_t(n_tiles) * 32 * nq * splits * (hd + 2) : 0;
}

int attention_split(hipStream_t s, const float* q, int q_stride, const float* k_pool, const float* v_pool,
                    const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* q_len,
                    const int32_t* ctx_len, const int32_t* tiles, int n_tiles, int max_tile_ctx, float* out, float* workspace, int nq,
                    int nkv, int page_size, int num_pages, float scale) {
  const int splits = attention_split_splits(n_tiles, nq, nkv, max_tile_ctx);
  constexpr int kLds = 6 * kPlane + kSplitTable * 4;
  static bool raised = false;
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_split_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) {
      set_error("sp_attention (float32, parts): cannot raise the LDS limit: %s", hipGetErrorString(e));
      return 1;
    }
    raised = true;
  }
  int page_shift = 0;
  while ((1 << page_shift) < page_size) ++page_shift;
  float* part_ml = splits > 1 ? workspace + size_t(n_tiles) * 32 * nq * splits * 64 : nullptr;
  attention_split_kernel<<<dim3(n_tiles, nkv * ((nq / nkv + 3) / 4), splits), 256, kLds, s>>>(
      q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, q_len, ctx_len, tiles, out, workspace, part_ml, splits,
      nq, nkv, page_shift, num_pages, scale * kLog2e, n_tiles);
  if (check_launch("sp_attention (float32, parts)")) return 1;
  if (splits > 1) {
    const int pairs = n_tiles * 32 * nq;
    attention_prefill_merge_kernel<4, 2, false, float><<<(pairs + 15) / 16, 256, 0, s>>>(workspace, part_ml, q_start, q_len, tiles, out, splits,
                                                                                        nq, ScoreStage{}, pairs);
    return check_launch("sp_attention (float32, parts, merge)");
  }
  return 0;
}

}  // namespace sprout
