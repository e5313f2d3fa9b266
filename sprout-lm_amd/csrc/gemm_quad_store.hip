// The four-wave tiled product that stores its result, bfloat16 (one output, or two: see RopeArgs) or float32.
#include "gemm_quad.h"

namespace sprout {

int gemm_bf16_quad_store(hipStream_t s, const void* x, const void* w, int bias_dtype, const void* bias, bool f32, void* out, int T, int N, int K,
                         const RopeArgs& epilogue) {
  if (f32) return quad_run<kStoreF32>(s, kQuadStore, x, w, bias, bias_dtype, out, T, N, K);
  return quad_run<kStore>(s, kQuadStore, x, w, bias, bias_dtype, out, T, N, K, epilogue);
}

// The sums of every part of K, side by side (the plan is quad_parts').
int gemm_bf16_quad_parts(hipStream_t s, const void* x, const void* w, float* out, int T, int N, int K) {
  RopeArgs epilogue = {};
  epilogue.parts = 1;
  return quad_run<kStoreF32>(s, kQuadParts, x, w, nullptr, kF32, out, T, N, K, epilogue);
}

}  // namespace sprout
