"""Batched Q6_K matvecs by windows (gemv_q6win_kernel) vs the oracle: odd row
counts a little past a round of gemv_kernel's waves, half windows, several
windows, both wave counts, every batch (slices of 2 to 4 vectors), both
readings, and the calls beside its rule (few rows, columns or weights off it)
at the same bars; and the rule itself: where gemv_kernel is the faster form,
the call still takes it.
"""
import numpy as np
import pytest

import strata_hip as H
from conftest import check_parity
from strata_hip import synth as S

pytestmark = pytest.mark.gpu
Q6_K = 14


@pytest.mark.parametrize("rows,cols,batch,offset", [
    (2049, 2048, 2, 0), (2307, 4096, 3, 0), (3001, 6144, 4, 0), (2306, 12288, 6, 0), (2305, 6144, 7, 0),
    (13000, 2048, 8, 0),           # 12 waves a workgroup, rows past one round
    # gemv_kernel: one round of rows, weights off 16 bytes, columns off 2048
    (1, 2048, 2, 0), (17, 4096, 3, 0), (33, 6144, 4, 0), (40, 12288, 5, 0), (255, 2048, 6, 0), (64, 4096, 7, 0),
    (31, 4096, 4, 2), (31, 4352, 4, 0),
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


# rows in rounds of gemv_kernel's waves (8 a CU, a row each): the windowed form
# is taken where it is the faster one (rows a quarter round under the count)
@pytest.mark.parametrize("rounds,cols,batch,windowed", [
    (1, 2048, 2, False), (1, 4096, 4, False), (1, 12288, 2, False),  # one round of either
    (3, 6144, 2, False), (3, 2048, 4, True),                        # two rounds against three
    (2, 2048, 5, False), (4, 4096, 6, False), (2, 8192, 4, False),  # a launch more
    (5, 4096, 8, False), (4, 8192, 5, False),                       # half a round left over; a vector by itself
    (2, 2048, 2, True), (2, 4096, 4, True), (2, 8192, 3, True), (2, 6144, 6, True), (6, 2048, 8, True),
    (2, 2048, 8, True), (9, 2048, 7, True),
])
def test_gemv_q6_windows_rule(rounds, cols, batch, windowed):
    """gemv_kernel computes a row the same way wherever its weights start, and
    the windowed form needs them on 16 bytes: from 2 bytes past that the same
    matrix gives the same bits where the rule keeps gemv_kernel, and other
    roundings where it does not."""
    import torch
    print("[case] q6 windows, rule", rounds, cols, batch, flush=True)
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    rows = 8 * cu * rounds - (2 * cu if rounds > 1 else 0)
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    nb = rows * (cols // 256)
    b = torch.randint(0, 256, (nb, 210), generator=g, device="cuda", dtype=torch.uint8)
    d = (1e-4 * torch.rand(nb, generator=g, device="cuda")).to(torch.float16)
    b[:, 208:210] = d.view(torch.uint8).reshape(nb, 2)
    x = torch.randn(batch, cols, generator=g, device="cuda")
    ys = []
    for offset in (0, 2):
        tw = torch.zeros(b.numel() + offset, dtype=torch.uint8, device="cuda")
        tw[offset:] = b.reshape(-1)
        y = torch.full((batch, rows), float("nan"), device="cuda")
        H.gemv_dev(Q6_K, tw.data_ptr() + offset, rows, cols, x.data_ptr(), y.data_ptr(), batch,
                   stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        ys.append(y.cpu().numpy())
    assert np.array_equal(*ys) != windowed
