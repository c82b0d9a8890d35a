// The routed MoE FFN over out-major expert stacks for many tokens
// (crates/strata-core/src/moe.rs:108-127 after the routing): an expert's
// tokens share one pass over its weights on MFMA (tok_mm.hip), where the
// matvecs of moe_om.hip read and decode them once per two tokens.
//
//   route    as moe.hip's, an expert's pairs `tok` to a work item;
//   prep     the pairs' x to A fragments, item by item;
//   gate/up  tok_mm, an item a token group against its expert's rows:
//            h and p of every pair whole;
//   prep     silu(h) * p of the pairs to A fragments (over x's);
//   down     tok_mm again: d of every pair;
//   combine  out[t] = sum over t's experts in ascending id of w * d.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace sh {

static TokPlan moe_tok_plan(const MoePlan& p, int rows, int mats, int cols) {
  TokPlan t{};
  t.tok = p.tok;
  t.groups = p.z_max;
  t.nsb = t.sb_per = (cols + 255) / 256;
  t.nsplit = 1;
  t.tiles = (rows + 127) / 128 * mats;
  return t;
}

// Pairs per work item, by an expert's average (a group past it reads the
// weights again, from L2 at best; fragments of 16 leave the LDS for one or two
// workgroups a CU beside the weights: 96 tokens of 128 experts, average 6, take
// 169 us in groups of 8, 217 of 16, 191 of 32; 256 tokens, average 16, 299, 302
// and 214), or 0: moe_om.hip's launches, three fewer and one pass over the
// weights per two pairs, stay the faster form for few pairs of small experts.
// Where that ends depends on the types: the two-token form costs the more the
// more a weight's decode does, and its limb dots of Q8_0 rows cost least. Both
// measured over seven shapes from 12 to 130 M of pairs x n_embd x n_ff, all 25
// pairs of types, this form's time over the two-token form's:
//   32 x 1024 x 512 top-2, 24 tokens (25 M)  Q4_K / Q6_K 0.96, Q5_K / Q6_K
//     1.00, Q6_K / Q6_K 1.07, Q8_0 / Q4_K 1.05; 31 tokens (33 M) 0.80, 0.82,
//     0.87, 0.87
//   64 x 1536 x 1024 top-4, 8 tokens (50 M)  Q4_K / Q6_K 0.85, IQ4_XS / IQ4_XS
//     0.96, Q8_0 / Q5_K 1.02, Q8_0 / Q8_0 1.10; 6 tokens (38 M) 0.88, 1.04,
//     1.07, 1.14
// and, Q8_0 matrices only, on how many pairs an expert has:
//   0.31 pairs an expert (128 experts, 5 tokens x 8)  Q5_K / Q8_0 1.03, Q6_K /
//     Q8_0 1.06, Q8_0 / Q6_K 1.02, Q8_0 / Q8_0 1.15; 0.5 (8 tokens) 0.92,
//     0.99, 1.02, 1.16; 0.69 (64 experts, 11 x 4) 0.72, 0.92, 0.84, 1.05;
//     0.94 (15 x 4) 0.64, 0.85, 0.86, 0.99; 1.9 (32 experts, 15 x 4, 55 M)
//     Q8_0 / Q4_K 0.83, Q8_0 / Q6_K 0.89
// Far above the line, 128 x 2048 x 768 top-8 Q4_K / Q6_K, us: 16 tokens 176 /
// 97, 96 640 / 183, 256 1465 / 214.
int moe_tok_group(const MoePlan& p, uint32_t qa, uint32_t qb) {
  if (!tok_ok(qa, p.n_ff, p.n_embd) || !tok_ok(qb, p.n_embd, p.n_ff)) return 0;
  const int64_t pairs = int64_t(p.n_tok) * p.top_k, work = pairs * p.n_embd * p.n_ff;
  const int64_t least = p.n_tok < 16 ? (qa == kQ8_0 && pairs < p.n_expert ? 60 : 50)
                        : qa == kQ6_K || qa == kQ8_0 ? 30
                        : qa == kQ4_K || qb == kQ4_K ? 20
                                                     : 24;
  if (p.n_tok <= 4 || work < least * 1000000) return 0;
  // eighths of a pair an expert
  const int shared = qa == kQ8_0 ? (qb == kQ8_0 ? 6 : qb == kQ4_K || qb == kQ5_K ? 0 : 5)
                     : qb == kQ8_0 ? (qa == kQ4_K ? 0 : qa == kQ6_K ? 5 : 3)
                                   : 0;
  if (8 * pairs < int64_t(shared) * p.n_expert) return 0;
  const int64_t avg = (pairs + p.s_max - 1) / p.s_max;
  return avg <= 8 ? 8 : avg <= 32 ? 32 : avg <= 64 ? 64 : 96;
}

size_t moe_tok_image_bytes(const MoePlan& p) {
  return std::max(tok_image_bytes(moe_tok_plan(p, p.n_ff, 2, p.n_embd)),
                  tok_image_bytes(moe_tok_plan(p, p.n_embd, 1, p.n_ff)));
}

// 4 columns of one token a thread: its experts' rows in ascending id order,
// out += w * d, skipping w == 0 (moe.rs:112-126), then the shared expert's
// sigmoid(s) * d (moe.rs:139-142). Rows are requested eight at a time, ahead
// of their sums.
__global__ void __launch_bounds__(256) moe_tok_combine_kernel(MoePlan plan, const uint8_t* ws, float* __restrict__ out,
                                                              const float* __restrict__ sh_d,
                                                              const float* __restrict__ sh_s) {
  typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));  // out of any float alignment
  const int per_tok = plan.n_embd / 4;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= plan.n_tok * per_tok) return;
  const int t = i / per_tok, c = 4 * (i - t * per_tok);
  const int* tp = reinterpret_cast<const int*>(ws + plan.o_tokpair) + t * plan.top_k;
  const float* wt = reinterpret_cast<const float*>(ws + plan.o_wts) + t * plan.top_k;
  const float* part = reinterpret_cast<const float*>(ws + plan.o_part_b) + c;
  f32x4 sd = {0.f, 0.f, 0.f, 0.f};
  float gate = 0.f;
  if (sh_d) {
    sd = *reinterpret_cast<const f32x4*>(sh_d + int64_t(t) * plan.n_embd + c);
    gate = 1.f / (1.f + expf(-sh_s[t]));
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int a0 = 0; a0 < plan.top_k; a0 += 8) {
    f32x4 d[8];
    float w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int a = min(a0 + k, plan.top_k - 1);
      w[k] = a0 + k < plan.top_k ? wt[a] : 0.f;
      d[k] = *reinterpret_cast<const f32x4*>(part + int64_t(tp[a]) * plan.n_embd);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (w[k] != 0.f) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __fadd_rn(acc[j], __fmul_rn(w[k], d[k][j]));
      }
  }
  if (sh_d) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = __fadd_rn(acc[j], __fmul_rn(gate, sd[j]));
  }
  *reinterpret_cast<f32x4a4*>(out + int64_t(t) * plan.n_embd + c) = acc;
}

hipError_t launch_moe_tok(const MoePlan& p, uint32_t qg, uint32_t qd, const void* gate, const void* up,
                          const void* down, int q6g, int q6u, int q6d, const float* x, float* out, void* workspace,
                          hipStream_t s, const MoeShared* shared) {
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  auto ints = [&](size_t o) { return reinterpret_cast<const int*>(ws + o); };
  float* pa = reinterpret_cast<float*>(ws + p.o_part_a);  // [pair][h | p]
  float* pb = reinterpret_cast<float*>(ws + p.o_part_b);  // [pair][d]
  const int pairs = p.n_tok * p.top_k;
  const TokPlan gu = moe_tok_plan(p, p.n_ff, 2, p.n_embd), dn = moe_tok_plan(p, p.n_embd, 1, p.n_ff);
  TokItems it{ints(p.o_item_e), ints(p.o_item_off), ints(p.o_item_cnt), ints(p.o_meta), p.n_ff * p.rb_a};
  hipError_t e;
  if ((e = launch_tok_prep(gu, qg, x, p.n_embd, p.n_embd, pairs, ws + p.o_img, s, ints(p.o_pairtok),
                           ints(p.o_pairslot))) != hipSuccess)
    return e;
  if (q6g == q6u) {
    e = launch_tok_mm(gu, qg, gate, up, p.n_ff, p.n_embd, ws + p.o_img, pa, 2 * p.n_ff, 0, pairs, q6g, s, &it);
  } else {  // Q6_K in two readings: a launch each
    const TokPlan one = moe_tok_plan(p, p.n_ff, 1, p.n_embd);
    e = launch_tok_mm(one, qg, gate, nullptr, p.n_ff, p.n_embd, ws + p.o_img, pa, 2 * p.n_ff, 0, pairs, q6g, s, &it);
    if (e == hipSuccess)
      e = launch_tok_mm(one, qg, up, nullptr, p.n_ff, p.n_embd, ws + p.o_img, pa + p.n_ff, 2 * p.n_ff, 0, pairs, q6u, s,
                        &it);
  }
  if (e != hipSuccess) return e;
  if ((e = launch_tok_prep_silu(dn, qd, pa, 2 * p.n_ff, 0, 1, p.n_ff, pairs, ws + p.o_img, s, ints(p.o_pairslot))) !=
      hipSuccess)
    return e;
  it.stride = p.n_embd * p.rb_b;
  if ((e = launch_tok_mm(dn, qd, down, nullptr, p.n_embd, p.n_ff, ws + p.o_img, pb, p.n_embd, 0, pairs, q6d, s, &it)) !=
      hipSuccess)
    return e;
  if (shared && shared->join && (e = hipStreamWaitEvent(s, shared->join, 0)) != hipSuccess) return e;
  hipLaunchKernelGGL(moe_tok_combine_kernel, dim3(unsigned((int64_t(p.n_tok) * (p.n_embd / 4) + 255) / 256)), dim3(256),
                     0, s, p, ws, out, shared ? shared->d : nullptr, shared ? shared->s : nullptr);
  return hipGetLastError();
}

}  // namespace sh
