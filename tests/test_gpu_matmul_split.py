"""The prefill matmul's tile heights (128 and 256 tokens) and column shares
(sh_matmul_dev) vs the oracle, at the sizes where they end: one token, one
more than a tile, row counts that are no multiple of the 96-row tiles, widths
whose last share is short, and a workspace that holds the activations alone
(one share). Few tiles take 128 tokens; test_matmul_tall_tiles has the shapes
for which the rule takes 256, each format with one share and with several.

Reference and bars as test_gpu_matmul.py's: the same operands rounded as the
mode rounds them, 1e-3 normwise and the strict per-element bar (three times
that over the many outputs of the tall tiles); the shares are f32 sums added
in f32, which is within those as any order of the sum is.
"""
import numpy as np
import pytest

import strata_hip as H
from conftest import STRICT_TOL, check_parity
from strata_hip import synth as S

pytestmark = pytest.mark.gpu
Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS = 8, 12, 13, 14, 23


def matmul(quant, rows, cols, w, x, mode, nbytes, flags=0):
    import torch
    m = x.shape[0]
    tw, tx = torch.from_numpy(w).cuda(), torch.from_numpy(np.ascontiguousarray(x)).cuda()
    y = torch.full((m, rows), float("nan"), device="cuda")
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device="cuda")
    H.matmul_dev(quant, tw.data_ptr(), rows, cols, tx.data_ptr(), m, y.data_ptr(), mode, ws.data_ptr(), nbytes,
                 torch.cuda.current_stream().cuda_stream, flags=flags)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("mode", [H.MATMUL_BF16, H.MATMUL_Q8])
@pytest.mark.parametrize("quant,rows,cols,m", [
    (Q4_K, 130, 2304, 9),      # 2 row tiles, 9 super-blocks in shares
    (Q4_K, 97, 4096, 129),     # one token past a 128-token tile
    (Q5_K, 96, 1280, 257),
    (Q5_K, 700, 1792, 1),
    (Q6_K, 95, 3328, 128),
    (Q6_K, 300, 768, 200),
    (Q8_0, 193, 2112, 40),     # 33 chunks: the last share holds one
    (Q8_0, 64, 832, 300),
    (IQ4_XS, 200, 2560, 70),
])
def test_matmul_shares(oracle, quant, rows, cols, m, mode):
    print("[case] matmul shares", quant, rows, cols, m, mode, flush=True)
    w = S.matrix(quant, 41 + rows, rows, cols)
    x = S.normal_f32(42 + m, m * cols).reshape(m, cols)
    if mode == H.MATMUL_BF16:
        wb = oracle.bf16_round_array(oracle.dequantize(quant, w, rows, cols, 0)).astype(np.float64)
        want = (oracle.bf16_round_array(x).astype(np.float64) @ wb.T).astype(np.float32)
    else:
        want = oracle.matmul(quant, rows, cols, w, oracle.q8_activations_for(mode, x), threads=8)
    nb = H.matmul_workspace_bytes(quant, rows, cols, m, mode)
    alone = H.matmul_workspace_bytes(quant, 96 * 1024, cols, m, mode)  # enough tiles for the chip: one share
    assert nb > alone, "shares expected at these shapes"
    for size in (nb, alone):
        got = matmul(quant, rows, cols, w, x, mode, size)
        for t in range(m):
            check_parity(got[t], want[t], f"{size} bytes, row {t}", strict_tol=STRICT_TOL)
    with pytest.raises(H.BackendError):
        matmul(quant, rows, cols, w, x, mode, alone - 256)


def rule(quant, rows, cols, m, mode, cu=256):
    """matmul.hip's choice of (tokens per workgroup, shares), by its model of
    the rounds of workgroups; the shares are checked against the size that the
    library reports, which is planned for 256 CUs."""
    chunks, row_tiles, best = cols // 64, -(-rows // 96), None
    for bm in (256, 128):
        tiles = row_tiles * -(-m // bm)
        for s in range(1, 17):
            per = -(-(-(-chunks // s)) // 4) * 4
            if -(-chunks // per) != s:
                continue
            full = bm == 256 or tiles * s > cu
            chunk = (0.8, 0.5) if mode == H.MATMUL_BF16 else (2.8, 2.1) if quant == Q6_K else (1.3, 0.9)
            t = -(-tiles * s // (cu if bm == 256 else 2 * cu)) * (per + 6) * chunk[0 if full else 1]
            if s > 1:
                t += 3.0 + s * m * rows * 8.0 / 4e6
            if best is None or t < best[0]:
                best = (t, bm, s)
    return best[1:]


@pytest.mark.parametrize("rows,cols,m,mode,shares", [
    (12318, 256, 129, H.MATMUL_BF16, 1), (8244, 256, 257, H.MATMUL_BF16, 1), (6207, 3072, 129, H.MATMUL_BF16, 3),
    (12318, 256, 129, H.MATMUL_Q8, 1), (8244, 256, 257, H.MATMUL_Q8, 1), (2036, 2304, 390, H.MATMUL_Q8, 5),
])
@pytest.mark.parametrize("quant", [Q4_K, Q5_K, Q6_K, Q8_0, IQ4_XS])
def test_matmul_tall_tiles(oracle, quant, rows, cols, m, mode, shares):
    """256-token workgroups, the last partly filled in tokens and in rows."""
    import torch
    print("[case] matmul tall tiles", quant, rows, cols, m, mode, flush=True)
    if quant == Q6_K and mode == H.MATMUL_Q8 and shares > 1:
        cols = 1280  # its own kernel, of other figures
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    assert rule(quant, rows, cols, m, mode) == (256, shares)
    nb = H.matmul_workspace_bytes(quant, rows, cols, m, mode)
    alone = H.matmul_workspace_bytes(quant, 96 * 1024, cols, m, mode)
    assert nb - alone == (4 * rows * m * shares if shares > 1 else 0)
    w = S.matrix(quant, 51, rows, cols)
    x = S.normal_f32(52 + m, m * cols).reshape(m, cols)
    if mode == H.MATMUL_BF16:
        wb = oracle.bf16_round_array(oracle.dequantize(quant, w, rows, cols, 0)).astype(np.float64)
        want = (oracle.bf16_round_array(x).astype(np.float64) @ wb.T).astype(np.float32)
    else:
        want = oracle.matmul(quant, rows, cols, w, oracle.q8_activations_for(mode, x), threads=8)
    got = matmul(quant, rows, cols, w, x, mode, nb)
    # the per-element bar is three times what f32 arithmetic scores at a shape:
    # over these million outputs, many near zero, a plain f32 product of the
    # same operands scores 0.9e-3 to 2.0e-3 of f64 (12318 x 256, 129 tokens)
    for t in range(m):
        check_parity(got[t], want[t], f"row {t}", strict_tol=3 * STRICT_TOL)
