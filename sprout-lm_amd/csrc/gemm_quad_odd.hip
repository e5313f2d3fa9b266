// The four-wave gated product on blocks of an odd number of tile columns a wave.
//
// A block of the other shapes pairs tiles of gate rows with tiles of up rows, so its columns are a multiple of 64, and where a round of
// blocks does not come out even, an eighth to a third of the CUs have none or one more: 37,888 rows of 3,584 are 198 blocks of 192 or 296 of 128 on
// 256 CUs.  Here a tile holds both, two gate rows and then the two up rows that go with them, and blocks have 160 or 224 columns (237 or
// 170 blocks of those).  37,888 rows of 3,584, us before and now on one machine (single products, others differ by up to 5 %): 320 tokens 100 and 82
// (320 x 160 for 160 x 192), 512 135 and 127, 640 160 and 151, 1,024 255 and 232; 55,296 rows of 5,120: 264 tokens 186 and 149 (288 x 224), 640 341 and 312.  72
// products that the rule takes, of nine matrices, drawn at random: 0.87 to 1.00 of the time.  At 264 tokens of the former 288 x 160 is no faster than 288 x 192 (84 us,
// 3.2 TB/s of weights, which eight tokens read at 5.3: not what the memory gives; what bounds either is not known).  (Stored and added products, and parts
// side by side, gain nothing: K cut along fills the CUs.)
#include "gemm_quad.h"

namespace sprout {

int gemm_bf16_quad_odd_silu(int shape, hipStream_t s, const void* x, const void* w, void* out, int T, int I, int K, const RopeArgs& epilogue) {
  switch (shape) {
#define SPROUT_QUAD_CASE(INDEX, WM, WN, NA) \
    case INDEX: return launch_quad<WM, WN, NA, kSilu>(s, 1, (const uint16_t*)x, (const uint16_t*)w, nullptr, kF32, out, T, I, K, epilogue);
    SPROUT_QUAD_ODD_SHAPES(SPROUT_QUAD_CASE)
#undef SPROUT_QUAD_CASE
  }
  set_error("sp_gate_up_silu (four waves): no shape for %d tokens, %d inner columns, K = %d", T, I, K);
  return 1;
}

}  // namespace sprout
