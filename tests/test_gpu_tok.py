"""Many tokens through the dense FFN (sh_ffn_dev above 8 tokens: tok_mm.hip)
vs the oracle's sho_dense_ffn, at the sizes where the kernels' tiles end:
token groups of 16, 32, 64 and 96 and one more than each, row counts that are
no multiple of the 128-row tiles, columns of one and of several shares, Q8_0
rows that end inside a 256-column step (odd block counts included), weights
at 2-byte alignment, every format in each of its readings.

Tolerance: the matvec bars (conftest.check_parity) on out - x. The
activations are held to 23 bits and every sum is f32, so the result is within
a few f32 roundings of the oracle's, as the 8-token matvecs are.
"""
import numpy as np
import pytest

import strata_hip as H
from conftest import check_parity
from strata_hip import synth as S

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS = 8, 12, 13, 14, 23


def ffn(quants, flags, mats, n_embd, n_ff, x, norm, offset=0):
    """offset: bytes between the weights' start and a 256-byte boundary."""
    import torch
    dev = []
    for m in mats:
        t = torch.zeros(m.nbytes + offset, dtype=torch.uint8, device="cuda")
        t[offset:] = torch.from_numpy(np.ascontiguousarray(m)).cuda()
        dev.append(t)
    xd, nd = torch.from_numpy(np.ascontiguousarray(x)).cuda(), torch.from_numpy(norm).cuda()
    out = torch.full_like(xd, float("nan"))
    nb = H.ffn_workspace_bytes(x.shape[0], n_embd, n_ff)
    ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device="cuda")  # NaNs wherever it is read unwritten
    H.ffn_dev([(q, f, t.data_ptr() + offset) for q, f, t in zip(quants, flags, dev)], n_embd, n_ff, x.shape[0],
              xd.data_ptr(), nd.data_ptr(), 1e-6, out.data_ptr(), ws.data_ptr(), nb,
              torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("quants,n_embd,n_ff,n_tok,offset", [
    ((Q4_K, Q4_K, Q6_K), 512, 768, 9, 0),
    ((Q4_K, Q4_K, Q6_K), 768, 1280, 16, 2),
    ((Q5_K, Q5_K, Q4_K), 768, 1280, 17, 2),
    ((Q6_K, Q6_K, Q5_K), 1024, 512, 33, 2),
    ((Q4_K, Q4_K, Q4_K), 256, 256, 64, 0),
    ((Q8_0, Q8_0, Q6_K), 768, 1280, 65, 0),
    ((Q6_K, Q6_K, Q6_K), 512, 2816, 96, 0),
    ((Q4_K, Q4_K, Q8_0), 1024, 768, 97, 0),
    ((Q5_K, Q5_K, Q5_K), 512, 512, 200, 0),
    ((Q8_0, Q8_0, Q8_0), 1056, 2080, 13, 0),   # 33 and 65 blocks a row
    ((Q8_0, Q8_0, Q8_0), 288, 96, 70, 4),
    ((IQ4_XS, IQ4_XS, Q8_0), 512, 768, 21, 0),
])
def test_ffn_many_tokens(oracle, quants, n_embd, n_ff, n_tok, offset):
    print("[case] ffn tokens", quants, n_embd, n_ff, n_tok, offset, flush=True)
    mats = [S.matrix(quants[0], 91, n_ff, n_embd), S.matrix(quants[1], 92, n_ff, n_embd),
            S.matrix(quants[2], 93, n_embd, n_ff)]
    x = S.normal_f32(94 + n_tok, n_tok * n_embd).reshape(n_tok, n_embd)
    x[n_tok // 2] *= 100.0     # scales of its own
    x[1, :32] *= 1e-7          # a block far below the rest of its super-block
    x[2] = 0.0
    norm = S.normal_f32(95, n_embd)
    got = ffn(quants, (0, 0, 0), mats, n_embd, n_ff, x, norm, offset)
    want = oracle.dense_ffn(quants, mats, n_embd, n_ff, x, norm, 1e-6)
    for t in range(n_tok):  # a token at a time: each has its own magnitude
        check_parity(got[t].astype(np.float64) - x[t], want[t].astype(np.float64) - x[t], f"token {t}",
                     strict_tol=None)
    rest = [t for t in range(n_tok) if t != n_tok // 2]
    check_parity(got[rest].astype(np.float64) - x[rest], want[rest].astype(np.float64) - x[rest], "ffn out - x")


@pytest.mark.parametrize("quant,flag", [(Q6_K, H.FLAG_Q6K_SIGNED_SCALES), (IQ4_XS, H.FLAG_IQ4XS_GGML)])
def test_ffn_many_tokens_other_reading(oracle, quant, flag):
    """The flagged readings, against the oracle on the dequantized rows."""
    print("[case] ffn tokens, reading", quant, flag, flush=True)
    n_embd, n_ff, n_tok = 512, 768, 40
    mats = [S.matrix(quant, 96, n_ff, n_embd), S.matrix(quant, 97, n_ff, n_embd), S.matrix(quant, 98, n_embd, n_ff)]
    x = S.normal_f32(99, n_tok * n_embd).reshape(n_tok, n_embd)
    norm = S.normal_f32(100, n_embd)
    mode = oracle.SCALE_I8 if quant == Q6_K else oracle.IQ4XS_GGML
    f32 = [oracle.dequantize_row(quant, m, r * c, mode) for m, (r, c) in
           zip(mats, ((n_ff, n_embd), (n_ff, n_embd), (n_embd, n_ff)))]
    got = ffn((quant,) * 3, (flag,) * 3, mats, n_embd, n_ff, x, norm)
    want = oracle.dense_ffn((0, 0, 0), [w.view(np.uint8) for w in f32], n_embd, n_ff, x, norm, 1e-6)
    check_parity(got.astype(np.float64) - x, want.astype(np.float64) - x, "ffn out - x")


@pytest.mark.parametrize("n_tok", [12, 30, 60, 96])
@pytest.mark.parametrize("quant", [Q8_0, Q6_K])
def test_ffn_small_elements_beside_large_ones(oracle, quant, n_tok):
    """Every element keeps its own bits: one column of each super-block is
    2^28 times the others (its norm weight) and meets weights of 0, so the
    outputs are the other columns'. They are held to 2^-22 of themselves there
    (2^-50 of the maximum), through two products and f32 sums: 1e-5 of the
    largest output (1.2e-6 and less where the sums are exact to f32; limbs that
    end 2^-39 below the maximum give 1e-4)."""
    print("[case] ffn tokens, small beside large", quant, n_tok, flush=True)
    n_embd, n_ff = 768, 512
    mats = [S.matrix(quant, 21, n_ff, n_embd), S.matrix(quant, 22, n_ff, n_embd), S.matrix(quant, 23, n_embd, n_ff)]
    big = np.arange(3) * 256 + 5
    for i in (0, 1):
        if quant == Q8_0:  # block 0 of each eight: [d][32 codes]
            b = mats[i].reshape(n_ff, n_embd // 256, 8, 34)
            b[:, :, 0, 2 + 5] = 0
        else:  # [ql 128][qh 64][sc 16][d]: code 32 in element 5
            b = mats[i].reshape(n_ff, n_embd // 256, 210)
            b[:, :, 5] &= 0xF0
            b[:, :, 128 + 5] = (b[:, :, 128 + 5] & 0xFC) | 2
    x = S.normal_f32(24 + n_tok, n_tok * n_embd).reshape(n_tok, n_embd)
    norm = S.normal_f32(25, n_embd)
    norm[big] = 2.0 ** 28
    got = ffn((quant,) * 3, (0, 0, 0), mats, n_embd, n_ff, x, norm)
    want = oracle.dense_ffn((quant,) * 3, mats, n_embd, n_ff, x, norm, 1e-6)
    check_parity(got.astype(np.float64) - x, want.astype(np.float64) - x, "ffn out - x", norm_tol=1e-5, strict_tol=None)


def test_ffn_workspace_of_more_tokens(oracle):
    """A workspace reported for n tokens is taken for fewer, and one of the
    step-by-step form's size (mixed, g and u, h, m) always is."""
    import torch
    print("[case] ffn workspace", flush=True)
    n_embd, n_ff, quants = 512, 768, (Q4_K, Q4_K, Q6_K)
    mats = [S.matrix(quants[0], 31, n_ff, n_embd), S.matrix(quants[1], 32, n_ff, n_embd),
            S.matrix(quants[2], 33, n_embd, n_ff)]
    dev = [torch.from_numpy(m).cuda() for m in mats]
    norm = S.normal_f32(34, n_embd)
    nd = torch.from_numpy(norm).cuda()
    for n_tok, size in ((200, H.ffn_workspace_bytes(201, n_embd, n_ff)), (200, 4 * 200 * (2 * n_embd + 3 * n_ff))):
        x = S.normal_f32(35, n_tok * n_embd).reshape(n_tok, n_embd)
        xd = torch.from_numpy(x).cuda()
        out = torch.full_like(xd, float("nan"))
        ws = torch.full((size,), 0xFF, dtype=torch.uint8, device="cuda")
        H.ffn_dev([(q, 0, t.data_ptr()) for q, t in zip(quants, dev)], n_embd, n_ff, n_tok, xd.data_ptr(),
                  nd.data_ptr(), 1e-6, out.data_ptr(), ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        want = oracle.dense_ffn(quants, mats, n_embd, n_ff, x, norm, 1e-6)
        check_parity(out.cpu().numpy().astype(np.float64) - x, want.astype(np.float64) - x, "ffn out - x")
