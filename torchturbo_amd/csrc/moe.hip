// The experts' forward of a small batch in one call (no gradients): routing
// index, fc1 with the token rows gathered, activation and probabilities, fc2,
// and the sum of each token's rows; for decode and short prefill, where the
// host's work per launch is what a call costs. Every kernel is the one that
// the separate entry points run, on the same values: the same results.
#include "gemm.h"

namespace {

constexpr size_t kAlign = 256;
size_t aligned(size_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

// Scratch of one call, in order: the routing index's rows, tokens, packed
// probabilities and workspace, fc1's output, the activations, and the permuted
// rows (where fc1 does not gather them), which fc2's output replaces.
struct Scratch {
  size_t rows, tokens, probs, index, wide, act, rows_in, total;
  Scratch(int64_t T, int k, int E, int64_t H, int64_t F) {
    const size_t M = (size_t)T * k;
    rows = 0;
    tokens = rows + aligned(M * 4);
    probs = tokens + aligned(M * 4);
    index = probs + aligned(M * 4);
    wide = index + aligned(tt_route_index_workspace(T, E));
    act = wide + aligned(M * 2 * (size_t)(2 * F));
    rows_in = act + aligned(M * 2 * (size_t)F);
    total = rows_in + aligned(M * 2 * (size_t)H);
  }
};

}  // namespace

extern "C" size_t tt_moe_experts_workspace(int64_t num_tokens, int32_t topk, int32_t num_experts,
                                           int64_t hidden, int64_t ffn) {
  if (num_tokens <= 0 || topk <= 0 || num_experts <= 0 || hidden <= 0 || ffn <= 0) return 0;
  return Scratch(num_tokens, topk, num_experts, hidden, ffn).total;
}

extern "C" int tt_moe_experts_fwd(const void* x, int dtype, int64_t num_tokens, int64_t hidden,
                                  const int64_t* expert_indices, const void* probs,
                                  int probs_dtype, int32_t topk, int32_t num_experts,
                                  const void* w1, const void* w2, const void* scale1,
                                  const void* scale2, int scale_dtype, int64_t ffn, int act,
                                  float limit, int clamp_after, int64_t* tokens_per_expert,
                                  void* out, void* workspace, size_t workspace_bytes,
                                  void* stream) {
  TT_REQUIRE(dtype == TT_BF16 || dtype == TT_F16, "moe_experts: tokens must be bf16 or f16");
  TT_REQUIRE(num_tokens >= 0 && hidden > 0 && ffn > 0 && topk > 0 && num_experts > 0,
             "moe_experts: bad sizes");
  TT_REQUIRE((scale1 == nullptr) == (scale2 == nullptr), "moe_experts: both scales or none");
  TT_REQUIRE(scale1 == nullptr || dtype == TT_BF16, "moe_experts: FP8 experts take bf16 tokens");
  TT_REQUIRE(scale1 == nullptr || scale_dtype == TT_BF16 || scale_dtype == TT_F32,
             "moe_experts: scales must be bf16 or f32");
  TT_REQUIRE(probs != nullptr && tt_elem_size(probs_dtype) <= 4 && tt_elem_size(probs_dtype) >= 2,
             "moe_experts: probabilities must be f32, bf16 or f16");
  if (num_tokens == 0) return TT_OK;
  const Scratch off(num_tokens, topk, num_experts, hidden, ffn);
  TT_REQUIRE(workspace_bytes >= off.total, "moe_experts: workspace too small");
  TT_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
             "moe_experts: the workspace must be 16-byte aligned");
  char* const ws = static_cast<char*>(workspace);
  int32_t* const rows = reinterpret_cast<int32_t*>(ws + off.rows);
  int32_t* const tokens = reinterpret_cast<int32_t*>(ws + off.tokens);
  const int64_t M = num_tokens * topk;
  const bool fp8 = scale1 != nullptr;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  int rc = tt_route_index(expert_indices, num_tokens, topk, num_experts, probs, probs_dtype, rows,
                          tokens, ws + off.probs, tokens_per_expert, ws + off.index,
                          off.wide - off.index, stream);
  if (rc != TT_OK) return rc;
  const int took = tt_gmm_rows_fwd(x, num_tokens, tokens, w1, scale1, scale_dtype, dtype, M, hidden,
                                   2 * ffn, num_experts, tokens_per_expert, ws + off.wide, s);
  if (took < 0) return took;
  char* y = ws + off.rows_in;
  if (took == 0) {
    rc = tt_permute_scatter(x, dtype, num_tokens, hidden, topk, rows, ws + off.rows_in, stream);
    if (rc != TT_OK) return rc;
    rc = fp8 ? tt_gmm_fp8_fwd(ws + off.rows_in, static_cast<const uint8_t*>(w1), scale1,
                              scale_dtype, M, hidden, 2 * ffn, num_experts, tokens_per_expert,
                              ws + off.wide, stream)
             : tt_gmm_fwd(ws + off.rows_in, w1, dtype, M, hidden, 2 * ffn, num_experts, 0,
                          tokens_per_expert, ws + off.wide, stream);
    if (rc != TT_OK) return rc;
  }
  rc = act < 0 ? tt_swiglu_fwd(ws + off.wide, dtype, M, ffn, ws + off.probs, probs_dtype,
                               ws + off.act, stream)
               : tt_gated_act_fwd(ws + off.wide, dtype, M, ffn, act, limit, clamp_after,
                                  ws + off.probs, probs_dtype, ws + off.act, stream);
  if (rc != TT_OK) return rc;
  rc = fp8 ? tt_gmm_fp8_fwd(ws + off.act, static_cast<const uint8_t*>(w2), scale2, scale_dtype, M,
                            ffn, hidden, num_experts, tokens_per_expert, y, stream)
           : tt_gmm_fwd(ws + off.act, w2, dtype, M, ffn, hidden, num_experts, 0,
                        tokens_per_expert, y, stream);
  if (rc != TT_OK) return rc;
  return tt_unpermute_gather(y, dtype, num_tokens, hidden, topk, rows, nullptr, nullptr, 0,
                             num_experts, out, stream);
}
