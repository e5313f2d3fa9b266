// bfloat16 attention of steps that hold prompts and one-query sequences: one launch for both kinds of blocks, one for their merges.
#include "attention_mfma.h"

namespace sprout {

template <int DT, int HPB, int WPT, bool AHEAD, bool PAIRED>
static int launch(hipStream_t s, const uint16_t* q, int q_stride, const uint16_t* k_pool, const uint16_t* v_pool,
                  const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* ctx_len, uint16_t* out, int nq, int nkv,
                  int num_pages, const ScoreStage& st, float scale2, const PromptPart& p, const DecodePart& d) {
  constexpr int UNITS = WPT * HPB / 4;
  const int units = d.n_splits * d.sets * d.n;
  attention_mixed_kernel<DT, HPB, WPT, AHEAD, PAIRED><<<p.nx * p.ny * p.nz + (units + UNITS - 1) / UNITS, 64 * WPT * HPB, 0, s>>>(
      q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, ctx_len, out, nq, nkv, num_pages, st, scale2, p, d);
  if (check_launch("sp_attention (prompts and one-query sequences)")) return 1;
  const int pairs = p.nz > 1 ? p.n_tiles * 32 * nq : 0, per_block = 256 / (16 * DT / 4), prompt_blocks = (pairs + per_block - 1) / per_block;
  const int merges = d.n_splits > 1 ? d.n * nq : 0;
  if (prompt_blocks + merges == 0) return 0;
  if (d.n_splits <= 16)
    attention_mixed_merge_kernel<DT, 1><<<prompt_blocks + (merges + 3) / 4, 256, 0, s>>>(q_start, out, nq, st, p, d, pairs, prompt_blocks);
  else
    attention_mixed_merge_kernel<DT, 4><<<prompt_blocks + merges, 256, 0, s>>>(q_start, out, nq, st, p, d, pairs, prompt_blocks);
  return check_launch("sp_attention (both merges)");
}

// The shapes of staged_shape() and staged_paired() of up to eight waves.
template <int DT>
static int launch_shape(hipStream_t s, int hpb, int wpt, bool paired, const uint16_t* q, int q_stride, const uint16_t* k_pool,
                        const uint16_t* v_pool, const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* ctx_len,
                        uint16_t* out, int nq, int nkv, int num_pages, const ScoreStage& st, float scale2, const PromptPart& p,
                        const DecodePart& d) {
#define SP_MIXED(HPB, WPT, AHEAD, PAIRED)                                                                                              \
  return launch<DT, HPB, WPT, AHEAD, PAIRED>(s, q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, ctx_len, out, nq, nkv, \
                                             num_pages, st, scale2, p, d)
  if (paired) {
    if (hpb == 1) SP_MIXED(1, 4, false, true);
    if (hpb == 2) SP_MIXED(2, 4, true, true);
    if constexpr (DT > 4) SP_MIXED(4, 2, false, true);
  } else {
    if (hpb == 1) SP_MIXED(1, 4, false, false);
    if (hpb == 2) SP_MIXED(2, 4, (DT > 4), false);
    if constexpr (DT > 4) SP_MIXED(4, 2, false, false);
  }
#undef SP_MIXED
  set_error("sp_attention: no mixed kernel of %d heads on %d waves each", hpb, wpt);
  return 1;
}

int launch_mixed(hipStream_t s, int dt, int hpb, int wpt, bool paired, const uint16_t* q, int q_stride, const uint16_t* k_pool,
                 const uint16_t* v_pool, const int32_t* block_tables, int max_blocks, const int32_t* q_start, const int32_t* ctx_len,
                 uint16_t* out, int nq, int nkv, int num_pages, const ScoreStage& st, float scale2, const PromptPart& p, const DecodePart& d) {
#define SP_MFMA(DT)                                                                                                                       \
  case DT:                                                                                                                                \
    return launch_shape<DT>(s, hpb, wpt, paired, q, q_stride, k_pool, v_pool, block_tables, max_blocks, q_start, ctx_len, out, nq, nkv,   \
                            num_pages, st, scale2, p, d)
  switch (dt) { SP_MFMA(1); SP_MFMA(2); SP_MFMA(3); SP_MFMA(4); SP_MFMA(5); SP_MFMA(6); SP_MFMA(8); }
#undef SP_MFMA
  set_error("sp_attention: no mixed kernel for head size %d", 16 * dt);
  return 1;
}

}  // namespace sprout
