// The dense FFN half of a decoder layer (crates/strata-core/src/qwen35.rs:
// 112-129) on the device, for n_tok tokens:
//   mixed = rms_norm_into(x, post_norm, eps)            (ops.rs:59-69)
//   g = gate . mixed, u = up . mixed                     (ops::gemv)
//   h = g / (1 + exp(-g)) * u                            (qwen35.rs:120-124, f32)
//   out = x + down . h                                   (qwen35.rs:127-129, f32)
// One token with the three matrices of one quantized type takes three
// launches: rms_norm, gate and up in one matvec launch (x staged once), and
// down with silu(g) * u formed while its x is staged and the residual added
// as its sums are written. More than 8 tokens with gate and up of one quantized
// type and a quantized down run on tok_mm.hip: rms_norm, the conversion of
// the tokens, gate and up in one launch, silu(g) * u converted, down, and the
// sum of down's shares with the residual (six launches for any number of
// tokens; the weights are read once per 96 tokens instead of once per 8:
// Q4_K gate and up, Q6_K down at 4096 / 12288, 9 tokens 139 -> 60 us, 24
// tokens 327 -> 63, 77 tokens 1015 -> 118, 512 tokens 6631 -> 527). Otherwise
// each step is its own launch (matvecs 8 tokens at a time; at 2 tokens that
// is still the faster form, 55 against 57 us).
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace sh {

static size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// [mixed: n_tok x n_embd][gu: n_tok x 2 n_ff][h: n_tok x n_ff][m: n_tok x n_embd]
static size_t ffn_step_bytes(int64_t n_tok, int64_t n_embd, int64_t n_ff) {
  const size_t T = size_t(n_tok);
  return align256(sizeof(float) * T * n_embd) + align256(sizeof(float) * T * 2 * n_ff) +
         align256(sizeof(float) * T * n_ff) + align256(sizeof(float) * T * n_embd);
}

// The many-token form's plans and workspace: the A fragments of x, then of h
// (x's are dead by then), and one area that holds mixed, then gate and up's
// shares, then down's (each dead when the next is written).
struct FfnTok {
  TokPlan gu, dn;
  size_t o_part, bytes;
};
static FfnTok ffn_tok_plan(int64_t n_tok, int64_t n_embd, int64_t n_ff, int cu, int gu_split, int dn_split) {
  FfnTok p{};
  p.gu = tok_plan(n_ff, 2, n_embd, int(n_tok), cu, gu_split);
  p.dn = tok_plan(n_embd, 1, n_ff, int(n_tok), cu, dn_split);
  const size_t T = size_t(n_tok) * sizeof(float);
  p.o_part = align256(std::max(tok_image_bytes(p.gu), tok_image_bytes(p.dn)));
  p.bytes = p.o_part + align256(std::max({T * n_embd, T * 2 * n_ff * p.gu.nsplit, T * n_embd * p.dn.nsplit}));
  return p;
}
constexpr int kFfnMaxSplit = 8;

// Small calls keep the size of the step-by-step form, which the fixed
// scratch of the allocation-free entry point holds; the many-token form then
// takes as many shares as fit, of each product by itself (17 tokens at 4096 /
// 12288: one share of gate and up fills what is left, but eight of down do not;
// with one of each the call took 190 us, so 78). Larger ones have room for all it asks for.
size_t ffn_workspace_min(int64_t n_tok, int64_t n_embd, int64_t n_ff) { return ffn_step_bytes(n_tok, n_embd, n_ff); }

size_t ffn_workspace_bytes(int64_t n_tok, int64_t n_embd, int64_t n_ff) {
  const size_t steps = ffn_step_bytes(n_tok, n_embd, n_ff);
  if (n_tok <= 8 || n_tok > kFfnMaxTokTokens) return steps;
  const size_t tok = ffn_tok_plan(n_tok, n_embd, n_ff, kChipCus, kFfnMaxSplit, kFfnMaxSplit).bytes;
  return std::max(steps, steps <= kFfnFixedScratch ? std::min(tok, kFfnFixedScratch) : tok);
}

static hipError_t gemv_rows(uint32_t quant, const void* w, int64_t rows, int64_t cols, const float* x, float* y,
                            int n_tok, int q6s, hipStream_t s) {
  for (int t0 = 0; t0 < n_tok; t0 += 8) {
    const int nb = n_tok - t0 < 8 ? n_tok - t0 : 8;
    const hipError_t e = launch_gemv(quant, w, rows, cols, x + int64_t(t0) * cols, y + int64_t(t0) * rows, nb,
                                     q6s, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_ffn(uint32_t q_gate, uint32_t q_up, uint32_t q_down, const void* gate, const void* up,
                      const void* down, int q6g, int q6u, int q6d, int64_t n_embd, int64_t n_ff, int n_tok,
                      const float* x, const float* post_norm, double eps, float* out, void* workspace,
                      size_t workspace_bytes, hipStream_t s) {
  if (workspace_bytes < ffn_workspace_min(n_tok, n_embd, n_ff)) return hipErrorInvalidValue;
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  const size_t T = size_t(n_tok);
  float* mixed = reinterpret_cast<float*>(ws);
  float* gu = reinterpret_cast<float*>(ws + align256(sizeof(float) * T * n_embd));
  float* h = gu + align256(sizeof(float) * T * 2 * n_ff) / sizeof(float);
  float* m = h + align256(sizeof(float) * T * n_ff) / sizeof(float);
  hipError_t e;
  const bool same = q_gate == q_up && q_up == q_down && q6g == q6u && q6u == q6d;
  if (n_tok == 1 && same && ffn_fused_ok(q_gate, n_embd, n_ff)) {
    if ((e = launch_rms_norm(x, post_norm, mixed, n_tok, n_embd, eps, s)) != hipSuccess) return e;
    return launch_ffn_one(q_gate, gate, up, down, n_embd, n_ff, mixed, gu, x, out, q6g, s);
  }
  if (n_tok > 8 && n_tok <= kFfnMaxTokTokens && q_gate == q_up && q6g == q6u && tok_ok(q_gate, n_ff, n_embd) &&
      tok_ok(q_down, n_embd, n_ff)) {
    // no more than the reported size is used, so results do not depend on
    // how much more than that a caller has
    const size_t room = std::min(workspace_bytes, ffn_workspace_bytes(n_tok, n_embd, n_ff));
    int gu_split = kFfnMaxSplit, dn_split = kFfnMaxSplit;
    const int cu = cu_count();
    FfnTok p = ffn_tok_plan(n_tok, n_embd, n_ff, cu, gu_split, 1);
    while (p.bytes > room && gu_split > 1) p = ffn_tok_plan(n_tok, n_embd, n_ff, cu, --gu_split, 1);
    p = ffn_tok_plan(n_tok, n_embd, n_ff, cu, gu_split, dn_split);
    while (p.bytes > room && dn_split > 1) p = ffn_tok_plan(n_tok, n_embd, n_ff, cu, gu_split, --dn_split);
    if (p.bytes <= room) {
      float* part = reinterpret_cast<float*>(ws + p.o_part);
      const int64_t nx = int64_t(T) * n_embd, ng = int64_t(T) * 2 * n_ff;
      if ((e = launch_rms_norm(x, post_norm, part, n_tok, n_embd, eps, s)) != hipSuccess) return e;
      if ((e = launch_tok_prep(p.gu, q_gate, part, n_embd, int(n_embd), n_tok, ws, s)) != hipSuccess) return e;
      if ((e = launch_tok_mm(p.gu, q_gate, gate, up, n_ff, n_embd, ws, part, 2 * n_ff, ng, n_tok, q6g, s)) != hipSuccess)
        return e;
      if ((e = launch_tok_prep_silu(p.dn, q_down, part, 2 * n_ff, ng, p.gu.nsplit, int(n_ff), n_tok, ws, s)) !=
          hipSuccess)
        return e;
      if ((e = launch_tok_mm(p.dn, q_down, down, nullptr, n_embd, n_ff, ws, part, n_embd, nx, n_tok, q6d, s)) !=
          hipSuccess)
        return e;
      return launch_tok_sum(part, nx, p.dn.nsplit, x, out, nx, s);
    }
  }
  // general path: g in gu[t][0, n_ff), u in gu[t][n_ff, 2 n_ff) as [2][T][n_ff]
  float* g = gu;
  float* u = gu + T * n_ff;
  if ((e = launch_rms_norm(x, post_norm, mixed, n_tok, n_embd, eps, s)) != hipSuccess) return e;
  if ((e = gemv_rows(q_gate, gate, n_ff, n_embd, mixed, g, n_tok, q6g, s)) != hipSuccess) return e;
  if ((e = gemv_rows(q_up, up, n_ff, n_embd, mixed, u, n_tok, q6u, s)) != hipSuccess) return e;
  if ((e = launch_silu_mul(g, u, h, int64_t(T) * n_ff, s)) != hipSuccess) return e;
  if ((e = gemv_rows(q_down, down, n_embd, n_ff, h, m, n_tok, q6d, s)) != hipSuccess) return e;
  return launch_add_out(out, x, m, int64_t(T) * n_embd, s);
}

}  // namespace sh
