"""The prefill matmul's tile heights (128 and 256 tokens) and column shares
(sh_matmul_dev) vs the oracle, at the sizes where they end: one token, one
more than a tile, row counts that are no multiple of the 96-row tiles, widths
whose last share is short, and a workspace that holds the activations alone
(one share).

Reference and bars as test_gpu_matmul.py's: the same operands rounded as the
mode rounds them, 1e-3 normwise and the strict per-element bar; the shares
are f32 sums added in f32, which is within those as any order of the sum is.
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
