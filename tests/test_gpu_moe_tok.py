"""The MoE of many tokens over out-major expert stacks (moe_tok.hip) vs the
oracle's out-major composition, at the sizes where it ends: every group size
(8, 32, 64 and 96 tokens of an expert), groups that run over, all tokens
on the same experts, rows that are no multiple of the 128-row tiles, every
type, both routing forms (above and at 16 tokens), the shared expert in the
whole layer, gate and up in two Q6_K readings, and x at float alignment.

Bars: conftest.check_parity's, a token at a time, as the two-token form's.
"""
import numpy as np
import pytest

import strata_hip as H
from conftest import check_parity
from strata_hip import synth as S
from test_gpu_moe_om import OM, om_tensors, om_views, oracle_om, layer_om_tensors
from test_gpu_moe_ws import two_token_bytes

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS = 8, 12, 13, 14, 23


def moe_dev(quants, flags, mats, n_expert, n_embd, n_ff, logits, x, top_k, offset=0, nb=None):
    """offset: floats between x's start and a 256-byte boundary."""
    import torch
    n_tok = x.shape[0]
    dev = [torch.from_numpy(np.ascontiguousarray(m)).cuda() for m in mats]
    tl = torch.from_numpy(logits).cuda()
    xb = torch.zeros(x.size + offset, device="cuda")
    xb[offset:] = torch.from_numpy(x.reshape(-1)).cuda()
    out = torch.full((n_tok, n_embd), float("nan"), device="cuda")
    nb = nb or H.moe_workspace_bytes(n_tok, top_k, n_expert, n_embd, n_ff, quants[0], quants[2])
    ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device="cuda")
    H.moe_ffn_dev(*[(q, OM | f, t.data_ptr()) for q, f, t in zip(quants, flags, dev)], n_expert, n_embd, n_ff,
                  tl.data_ptr(), n_tok, top_k, xb.data_ptr() + 4 * offset, out.data_ptr(), ws.data_ptr(), nb,
                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def group(n_expert, top_k, n_tok):
    """Tokens of an expert that share a pass over its weights (moe_tok_group)."""
    pairs = n_tok * top_k
    avg = -(-pairs // min(pairs, n_expert))
    return next(g for g, most in ((8, 8), (32, 32), (64, 64), (96, pairs)) if avg <= most)


@pytest.mark.parametrize("qg,qd,n_expert,n_embd,n_ff,top_k,n_tok,tokens", [
    (Q4_K, Q6_K, 64, 512, 512, 4, 20, 8),
    (Q5_K, Q4_K, 16, 512, 768, 6, 20, 8),     # most groups full
    (Q6_K, Q8_0, 8, 1024, 256, 3, 40, 32),
    (Q8_0, Q5_K, 4, 512, 768, 2, 60, 32),     # run over
    (Q4_K, Q6_K, 3, 768, 512, 2, 90, 64),
    (Q5_K, Q8_0, 3, 768, 512, 2, 110, 96),
    (Q6_K, Q4_K, 2, 512, 768, 2, 110, 96),    # run over: 110 pairs an expert
    (IQ4_XS, IQ4_XS, 2, 512, 768, 2, 97, 96),
    (Q8_0, Q8_0, 3, 1088, 320, 2, 130, 96),   # rows of 34 and 10 blocks
    (Q8_0, Q8_0, 24, 1088, 320, 4, 24, 8),
    (IQ4_XS, Q4_K, 12, 256, 1024, 5, 17, 8),
    (Q6_K, Q6_K, 32, 768, 2304, 2, 15, 8),
    (Q4_K, Q6_K, 32, 768, 1024, 4, 16, 8),    # one routing launch
    (Q8_0, Q8_0, 24, 1088, 320, 4, 16, 0),    # stays with the two-token form
])
def test_moe_many_tokens(oracle, qg, qd, n_expert, n_embd, n_ff, top_k, n_tok, tokens):
    assert tokens in (0, group(n_expert, top_k, n_tok))
    print("[case] moe tokens", qg, qd, n_expert, n_embd, n_ff, top_k, n_tok, flush=True)
    mats = om_tensors(n_expert, n_embd, n_ff, qg, qd, 60 + n_tok)
    logits = S.router_logits(61 + n_tok, n_tok, n_expert)
    x = S.normal_f32(62 + n_tok, n_tok * n_embd).reshape(n_tok, n_embd)
    x[1] *= 50.0
    x[3] = 0.0
    got = moe_dev((qg, qg, qd), (0, 0, 0), mats, n_expert, n_embd, n_ff, logits, x, top_k)
    want = oracle_om(oracle, qg, qd, n_expert, n_embd, n_ff, *mats, logits, x, top_k)
    for t in range(n_tok):
        check_parity(got[t], want[t], f"token {t}")
    shifted = moe_dev((qg, qg, qd), (0, 0, 0), mats, n_expert, n_embd, n_ff, logits, x, top_k, offset=1)
    assert np.array_equal(got, shifted)
    # the form that ran: a workspace of the two-token form's size runs that one
    two = moe_dev((qg, qg, qd), (0, 0, 0), mats, n_expert, n_embd, n_ff, logits, x, top_k,
                  nb=two_token_bytes(n_tok, top_k, n_expert, n_embd, n_ff))
    assert np.array_equal(got, two) == (tokens == 0)


# the many-token form is taken where it is the faster one: pairs x n_embd x
# n_ff below and above the line of each kind of types, Q8_0 matrices with fewer
# and with more pairs an expert
@pytest.mark.parametrize("qg,qd,n_expert,n_embd,n_ff,top_k,n_tok,tokens", [
    (Q4_K, Q6_K, 32, 512, 1024, 2, 18, False), (Q4_K, Q6_K, 32, 512, 1024, 2, 20, True),
    (Q5_K, Q5_K, 32, 512, 1024, 2, 20, False), (Q5_K, Q5_K, 32, 512, 1024, 2, 24, True),
    (Q6_K, Q6_K, 32, 512, 1024, 2, 24, False), (Q6_K, Q6_K, 32, 512, 1024, 2, 29, True),
    (Q8_0, Q4_K, 32, 512, 1024, 2, 24, False), (Q8_0, Q4_K, 32, 512, 1024, 2, 29, True),
    (IQ4_XS, IQ4_XS, 16, 1536, 1024, 4, 7, False), (IQ4_XS, IQ4_XS, 16, 1536, 1024, 4, 8, True),
    (Q8_0, Q5_K, 40, 1536, 1024, 4, 9, False), (Q8_0, Q5_K, 40, 1536, 1024, 4, 10, True),
    (Q8_0, Q5_K, 16, 1536, 1024, 4, 8, True),
    (Q8_0, Q8_0, 96, 1024, 1024, 8, 8, False), (Q8_0, Q8_0, 80, 1024, 1024, 8, 8, True),
    (Q8_0, Q6_K, 112, 1024, 1024, 8, 8, False), (Q8_0, Q6_K, 96, 1024, 1024, 8, 8, True),
    (Q6_K, Q8_0, 112, 1024, 1024, 8, 8, False), (Q6_K, Q8_0, 96, 1024, 1024, 8, 8, True),
    (Q5_K, Q8_0, 96, 1536, 1024, 4, 8, False), (Q5_K, Q8_0, 80, 1536, 1024, 4, 8, True),
])
def test_moe_many_tokens_rule(qg, qd, n_expert, n_embd, n_ff, top_k, n_tok, tokens):
    """A workspace of the two-token form's size always runs that form: the
    call gives its bits with all of the workspace where the rule keeps it, and
    other roundings where it does not."""
    print("[case] moe tokens, rule", qg, qd, n_expert, n_embd, n_ff, top_k, n_tok, flush=True)
    mats = om_tensors(n_expert, n_embd, n_ff, qg, qd, 65)
    logits = S.router_logits(66, n_tok, n_expert)
    x = S.normal_f32(67, n_tok * n_embd).reshape(n_tok, n_embd)
    args = ((qg, qg, qd), (0, 0, 0), mats, n_expert, n_embd, n_ff, logits, x, top_k)
    assert np.array_equal(moe_dev(*args), moe_dev(*args, nb=two_token_bytes(n_tok, top_k, n_expert, n_embd, n_ff))) != tokens


def test_moe_all_tokens_on_the_same_experts(oracle):
    """Every token picks experts 0 and 1: groups of 8 run over twelve times."""
    print("[case] moe tokens, two experts", flush=True)
    n_expert, n_embd, n_ff, top_k, n_tok = 32, 512, 256, 2, 100
    mats = om_tensors(n_expert, n_embd, n_ff, Q4_K, Q6_K, 70)
    logits = np.zeros((n_tok, n_expert), np.float32)
    x = S.normal_f32(71, n_tok * n_embd).reshape(n_tok, n_embd)
    got = moe_dev((Q4_K, Q4_K, Q6_K), (0, 0, 0), mats, n_expert, n_embd, n_ff, logits, x, top_k)
    want = oracle_om(oracle, Q4_K, Q6_K, n_expert, n_embd, n_ff, *mats, logits, x, top_k)
    for t in range(n_tok):
        check_parity(got[t], want[t], f"token {t}")


@pytest.mark.parametrize("quant,flags", [(Q6_K, (H.FLAG_Q6K_SIGNED_SCALES, 0, H.FLAG_Q6K_SIGNED_SCALES)),
                                         (Q6_K, (0, H.FLAG_Q6K_SIGNED_SCALES, 0)),
                                         (IQ4_XS, (H.FLAG_IQ4XS_GGML,) * 3)])
def test_moe_many_tokens_readings(oracle, quant, flags):
    """The flagged readings (gate's and up's may differ for Q6_K)."""
    print("[case] moe tokens, readings", quant, flags, flush=True)
    n_expert, n_embd, n_ff, top_k, n_tok = 16, 512, 512, 4, 40
    mats = om_tensors(n_expert, n_embd, n_ff, quant, quant, 80)
    logits = S.router_logits(81, n_tok, n_expert)
    x = S.normal_f32(82, n_tok * n_embd).reshape(n_tok, n_embd)
    got = moe_dev((quant,) * 3, flags, mats, n_expert, n_embd, n_ff, logits, x, top_k)
    flagged = oracle.SCALE_I8 if quant == Q6_K else oracle.IQ4XS_GGML
    modes = tuple(flagged if f else 0 for f in flags)
    for t in range(n_tok):
        ids, w = oracle.moe_route(logits[t], top_k)
        want = oracle.moe_routed(quant, quant, quant, n_expert, n_embd, n_ff, *mats, ids, w, x[t], out_major=True,
                                 modes=modes)
        check_parity(got[t], want, f"token {t}")


@pytest.mark.parametrize("n_sh,n_tok", [(256, 9), (768, 33), (512, 100)])
def test_moe_layer_many_tokens(oracle, n_sh, n_tok):
    """The whole layer (router and shared expert of many tokens in one set
    of launches); replayed from a graph, eager calls of four tokens between."""
    import torch
    print("[case] moe layer tokens", n_sh, n_tok, flush=True)
    n_expert, n_embd, n_ff, top_k = 16, 768, 512, 6
    q, t = layer_om_tensors(n_expert, n_embd, n_ff, n_sh, 90)
    x = S.normal_f32(91, n_tok * n_embd).reshape(n_tok, n_embd)
    bufs = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in t]
    flags = [0, OM, OM, OM, 0, 0, 0, 0]
    tensors = [(q[i], flags[i], bufs[i].data_ptr()) for i in range(8)]
    tx = torch.from_numpy(x).cuda()
    out = torch.full((n_tok, n_embd), float("nan"), device="cuda")
    nb = H.moe_layer_workspace_bytes(n_tok, top_k, n_expert, n_embd, n_ff, n_sh, q)
    ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device="cuda")

    def call(t0, n, o):
        H.moe_layer_dev(tensors, n_expert, n_embd, n_ff, n_sh, n, top_k, tx.data_ptr() + 4 * t0 * n_embd, o.data_ptr(),
                        ws.data_ptr(), nb, torch.cuda.current_stream().cuda_stream)

    call(0, n_tok, out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    few = torch.empty((4, n_embd), device="cuda")
    for i in range(n_tok):
        want = oracle.moe_layer(q, t, n_expert, n_embd, n_ff, n_sh, x[i], top_k, out_major=True)
        check_parity(got[i], want, f"token {i}")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        call(0, n_tok, out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(0, n_tok, out)
    for rep in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), got), rep
        call(0, 4, few)
        torch.cuda.synchronize()


@pytest.mark.parametrize("plain,n_expert,n_embd,n_sh,q_sh", [
    (0, 5, 768, 256, Q4_K), (0, 16, 4096, 768, Q5_K), (1, 7, 512, 4608, Q8_0), (30, 12, 2304, 256, Q6_K)])
def test_moe_layer_one_token_front(oracle, plain, n_expert, n_embd, n_sh, q_sh):
    """One token: router, gate input and the shared expert's gate and up in
    one launch (odd and even row counts, every plain type and a row pair per
    wave or several), and two tokens, which take them apart."""
    import torch
    print("[case] moe layer front", plain, n_expert, n_embd, n_sh, q_sh, flush=True)
    n_ff, top_k = 256, 4
    q, t = layer_om_tensors(n_expert, n_embd, n_ff, n_sh, 190 + n_expert)
    q, t = list(q), list(t)
    for i in (0, 7):
        q[i] = plain
        f = torch.from_numpy(t[i].view(np.float32).copy())
        t[i] = (f if plain == 0 else f.to(torch.float16 if plain == 1 else torch.bfloat16)).view(torch.uint8).numpy()
    for i, (r, c) in ((4, (n_sh, n_embd)), (5, (n_sh, n_embd))):
        q[i], t[i] = q_sh, S.matrix(q_sh, 200 + i, r, c)
    x = S.normal_f32(191, 2 * n_embd).reshape(2, n_embd)
    bufs = [torch.from_numpy(np.ascontiguousarray(a).reshape(-1)).cuda() for a in t]
    flags = [0, OM, OM, OM, 0, 0, 0, 0]
    tx = torch.from_numpy(x).cuda()
    want = [oracle.moe_layer(q, t, n_expert, n_embd, n_ff, n_sh, x[i], top_k, out_major=True) for i in range(2)]
    for n in (1, 2):
        out = torch.full((n, n_embd), float("nan"), device="cuda")
        nb = H.moe_layer_workspace_bytes(n, top_k, n_expert, n_embd, n_ff, n_sh, q)
        ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device="cuda")
        H.moe_layer_dev([(q[i], flags[i], bufs[i].data_ptr()) for i in range(8)], n_expert, n_embd, n_ff, n_sh, n, top_k,
                        tx.data_ptr(), out.data_ptr(), ws.data_ptr(), nb, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        for i in range(n):
            check_parity(got[i], want[i], f"{n} tokens, token {i}")
