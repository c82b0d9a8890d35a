"""The MoE entry points take any workspace that the two-token form fills
(moe_om.hip's buffers, and around them the layer's): without room for the
many-token forms' fragments and partial sums a call runs without them. Bars:
conftest.check_parity's against the oracle, a token at a time, at every size;
a byte less than the two-token form's is refused.
"""
import numpy as np
import pytest

import strata_hip as H
from conftest import check_parity
from strata_hip import synth as S
from test_gpu_moe_om import OM, layer_om_tensors, om_tensors, oracle_om

pytestmark = pytest.mark.gpu
Q4_K, Q5_K, Q6_K = 12, 13, 14


def al(nbytes):
    return (nbytes + 255) // 256 * 256


def two_token_bytes(n_tok, top_k, n_expert, n_embd, n_ff):
    """ids, weights, meta, the items' expert, first pair, count and tokens,
    the pairs' places, [h | p] and d of every pair."""
    pairs = n_tok * top_k
    items = (pairs + min(pairs, n_expert)) // 2
    return (2 * al(4 * pairs) + 256 + 3 * al(4 * items) + al(8 * items) + al(4 * pairs) + al(8 * pairs * n_ff) +
            al(4 * pairs * n_embd))


def layer_bytes(n_tok, n_expert, n_embd, n_sh):
    """logits, bf16(x), g and u (twice: one launch or two), h, d, the gate."""
    return (al(4 * n_tok * n_expert) + 2 * al(4 * n_tok * n_embd) + al(8 * n_tok * n_sh) + 2 * al(4 * n_tok * n_sh) +
            al(4 * n_tok))


def test_moe_ffn_small_workspace(oracle):
    import torch
    n_expert, n_embd, n_ff, top_k, n_tok = 16, 768, 512, 6, 40
    print("[case] moe workspace", flush=True)
    mats = om_tensors(n_expert, n_embd, n_ff, Q4_K, Q6_K, 300)
    logits = S.router_logits(301, n_tok, n_expert)
    x = S.normal_f32(302, n_tok * n_embd).reshape(n_tok, n_embd)
    want = oracle_om(oracle, Q4_K, Q6_K, n_expert, n_embd, n_ff, *mats, logits, x, top_k)
    dev = [torch.from_numpy(np.ascontiguousarray(m)).cuda() for m in mats]
    tl, tx = torch.from_numpy(logits).cuda(), torch.from_numpy(x).cuda()
    small = two_token_bytes(n_tok, top_k, n_expert, n_embd, n_ff)

    def call(size):
        out = torch.full((n_tok, n_embd), float("nan"), device="cuda")
        ws = torch.full((size,), 0xFF, dtype=torch.uint8, device="cuda")
        H.moe_ffn_dev(*[(q, OM, t.data_ptr()) for q, t in zip((Q4_K, Q4_K, Q6_K), dev)], n_expert, n_embd, n_ff,
                      tl.data_ptr(), n_tok, top_k, tx.data_ptr(), out.data_ptr(), ws.data_ptr(), size,
                      torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    for size in (H.moe_workspace_bytes(n_tok, top_k, n_expert, n_embd, n_ff, Q4_K, Q6_K), small):
        got = call(size)
        for t in range(n_tok):
            check_parity(got[t], want[t], f"{size} bytes, token {t}")
    with pytest.raises(H.BackendError):
        call(small - 1)


@pytest.mark.parametrize("out_major", [True, False])
def test_moe_layer_small_workspace(oracle, out_major):
    import torch
    n_expert, n_embd, n_ff, n_sh, top_k, n_tok = 16, 768, 512, 256, 6, 40
    print("[case] moe layer workspace", out_major, flush=True)
    q, t = layer_om_tensors(n_expert, n_embd, n_ff, n_sh, 310)
    if not out_major:  # [n_expert][in][out]
        t[1:4] = [S.matrix(Q4_K, 311, n_expert * n_embd, n_ff), S.matrix(Q4_K, 312, n_expert * n_embd, n_ff),
                  S.matrix(Q6_K, 313, n_expert * n_ff, n_embd)]
    x = S.normal_f32(314, n_tok * n_embd).reshape(n_tok, n_embd)
    want = [oracle.moe_layer(q, t, n_expert, n_embd, n_ff, n_sh, x[i], top_k, out_major=out_major)
            for i in range(n_tok)]
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in t]
    om = OM if out_major else 0
    tensors = [(q[i], om if 1 <= i <= 3 else 0, dev[i].data_ptr()) for i in range(8)]
    tx = torch.from_numpy(x).cuda()
    # a shared expert of two types has no many-token form: the size without it
    steps = H.moe_layer_workspace_bytes(n_tok, top_k, n_expert, n_embd, n_ff, n_sh, q[:5] + [Q5_K] + q[6:])
    full = H.moe_layer_workspace_bytes(n_tok, top_k, n_expert, n_embd, n_ff, n_sh, q)
    assert full > steps
    sizes = [full, steps]
    if out_major:
        sizes.append(two_token_bytes(n_tok, top_k, n_expert, n_embd, n_ff) + layer_bytes(n_tok, n_expert, n_embd, n_sh))

    def call(size):
        out = torch.full((n_tok, n_embd), float("nan"), device="cuda")
        ws = torch.full((size,), 0xFF, dtype=torch.uint8, device="cuda")
        H.moe_layer_dev(tensors, n_expert, n_embd, n_ff, n_sh, n_tok, top_k, tx.data_ptr(), out.data_ptr(),
                        ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    for size in sizes:
        got = call(size)
        for i in range(n_tok):
            check_parity(got[i], want[i], f"{size} bytes, token {i}")
    with pytest.raises(H.BackendError):
        call(sizes[-1] - 1)
