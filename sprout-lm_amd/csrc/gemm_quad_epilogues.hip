// The four-wave tiled product with the gated (gate/up and activation) and the rotating (q/k/v, rotation and cache write) epilogue.
#include "gemm_quad.h"

namespace sprout {
int gemm_bf16_quad_odd_silu(int shape, hipStream_t s, const void* x, const void* w, void* out, int T, int I, int K, const RopeArgs& epilogue);

// out[T, I] = silu(x . w[:I]^T) * (x . w[I:]^T): a block's weight rows are half gate rows, half the matching up rows.
int gemm_bf16_quad_silu(hipStream_t s, const void* x, const void* w, void* out, int T, int I, int K, int act, float limit,
                        const float* row_gate, long long row_gate_stride) {
  RopeArgs epilogue = {};
  epilogue.act = act;
  epilogue.limit = limit;
  epilogue.row_gate = row_gate;
  epilogue.row_gate_stride = row_gate_stride;
  int shape;
  if (quad_takes_odd(T, 2 * I, K, &shape)) return gemm_bf16_quad_odd_silu(shape, s, x, w, out, T, I, K, epilogue);
  return quad_run<kSilu>(s, kQuadGated, x, w, nullptr, kF32, out, T, I, K, epilogue);
}

// q, k, v = x . w^T + bias with w [(nq + 2 nkv) * hd, K]; q and k heads rotated; q to q_out [T, nq * hd], k and v into the paged
// pools.  Head sizes that are multiples of 64.  The sums lie where the epilogue's own registers do not reach them, so the
// largest blocks rotate too.
int gemm_bf16_quad_rope(hipStream_t s, const void* x, const void* w, int bias_dtype, const void* bias, void* q_out,
                        const int32_t* positions, const float* inv_freq, const int32_t* slot_mapping, void* k_pool,
                        void* v_pool, int T, int K, int nq, int nkv, int hd, int page_size, const float* table) {
  const RopeArgs rope = {positions, inv_freq, slot_mapping, (uint16_t*)k_pool, (uint16_t*)v_pool, nq, nkv, hd, page_size,
                         reinterpret_cast<const float2*>(table)};
  return quad_run<kRope>(s, kQuadRotating, x, w, bias, bias_dtype, q_out, T, (nq + 2 * nkv) * hd, K, rope);
}

}  // namespace sprout
