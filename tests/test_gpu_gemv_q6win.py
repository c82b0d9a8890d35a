"""Batched Q6_K matvecs by windows (gemv_q6win_kernel) vs the oracle: one and
an odd number of rows, half windows, several windows, both wave counts, every
batch (slices of 2 to 4 vectors), both readings, and the calls beside its
rule (columns or weights off it) at the same bars.
"""
import numpy as np
import pytest

import strata_hip as H
from conftest import check_parity
from strata_hip import synth as S

pytestmark = pytest.mark.gpu
Q6_K = 14


@pytest.mark.parametrize("rows,cols,batch,offset", [
    (1, 2048, 2, 0), (17, 4096, 3, 0), (33, 6144, 4, 0), (40, 12288, 5, 0), (255, 2048, 6, 0), (64, 4096, 7, 0),
    (13000, 2048, 8, 0),           # 12 waves a workgroup, rows past one round
    (31, 4096, 4, 2), (31, 4352, 4, 0),  # weights off 16 bytes, columns off 2048
])
@pytest.mark.parametrize("flags", [0, H.FLAG_Q6K_SIGNED_SCALES])
def test_gemv_q6_windows(oracle, rows, cols, batch, offset, flags):
    import torch
    print("[case] q6 windows", rows, cols, batch, offset, flags, flush=True)
    w = S.matrix(Q6_K, 11 + rows, rows, cols)
    x = S.normal_f32(12 + cols, batch * cols).reshape(batch, cols)
    x[0, :16] *= 100.0
    tw = torch.zeros(w.nbytes + offset, dtype=torch.uint8, device="cuda")
    tw[offset:] = torch.from_numpy(w.reshape(-1)).cuda()
    tx = torch.from_numpy(x).cuda()
    y = torch.full((batch, rows), float("nan"), device="cuda")
    H.gemv_dev(Q6_K, tw.data_ptr() + offset, rows, cols, tx.data_ptr(), y.data_ptr(), batch, flags=flags,
               stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    mode = oracle.SCALE_I8 if flags else 0
    want = oracle.matmul(Q6_K, rows, cols, w, x, threads=8, mode=mode)
    for b in range(batch):
        check_parity(got[b], want[b], f"vector {b}")
