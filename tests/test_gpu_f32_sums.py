"""The fixed-order sums behind the fp32 filter and bias gradients, at the sizes where their
split of the work changes: one, four or sixteen threads per element, runs of parts that do not
divide evenly, bias-gradient runs of 256 positions with a short last one, channel counts off
the 64 of a workgroup.  Small-integer inputs: every partial sum is an integer below 2^24, exact
in fp32 in any order, so a dropped, repeated or misplaced part shows as a wrong value."""
import numpy as np
import pytest
import torch

import my_own_cnn_amd as M
import oracle

pytestmark = pytest.mark.gpu

# (n, h, w, c, k, r, s): few elements and many splits, more elements, more than 2^16 and 2^18
CASES = [(3, 41, 29, 4, 8, 3, 3), (8, 56, 56, 16, 16, 1, 1), (2, 30, 31, 64, 36, 3, 3), (1, 20, 23, 128, 64, 3, 3),
         (2, 13, 11, 256, 128, 3, 3), (1, 3, 5, 8, 4, 3, 3)]


@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_grad_sums_every_part_once(device, case):
    n, h, w, c, k, r, s = case
    rng = np.random.default_rng(sum(case))
    x = rng.integers(-3, 4, size=(n, h, w, c)).astype(np.float32)
    conv = (r // 2, s // 2, 1, 1, 1, 1, 1)
    dy = rng.integers(-3, 4, size=(n, h, w, k)).astype(np.float32)
    want = oracle.grad_f32(x, dy, (k, r, s, c), conv)
    dw = torch.full((k, r, s, c), 7.0, dtype=torch.float32, device=device)
    M.launch_grad_nhwc(torch.from_numpy(x).to(device), torch.from_numpy(dy).to(device), dw, n, h, w, c, r, s, k, conv)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(dw.cpu().numpy().view(np.uint32), (want + 0.0).view(np.uint32))


@pytest.mark.parametrize("case", [(2, 12, 20, 7, 2, 2), (5, 34, 22, 64, 2, 2), (1, 48, 64, 70, 3, 2), (3, 4, 4, 130, 1, 4)],
                         ids=str)
def test_block_dbias_runs(device, case):
    n, h, w, k, by, bx = case
    rng = np.random.default_rng(sum(case))
    dy = rng.standard_normal((n, h, w, k)).astype(np.float32)
    x = np.ones((n, h, w, 4), np.float32)
    p = M.BlockConv2DParams(M.Conv2DParams(0, 0, 1, 1, 1, 1, 1), by, bx)
    dw = torch.empty((k, by, bx, 1, 1, 4), dtype=torch.float32, device=device)
    for mode in (0, 1):
        db = torch.full((k * by * bx,), 7.0, dtype=torch.float32, device=device)
        M.launch_block_grad_nhwc(torch.from_numpy(x).to(device), torch.from_numpy(dy).to(device), dw, n, h, w, 4, 1, 1,
                                 k, p, db, mode)
        torch.cuda.synchronize()
        want = oracle.block_dbias_f32(dy, by, bx, mode)
        np.testing.assert_array_equal(db.cpu().numpy().view(np.uint32), np.asarray(want).reshape(-1).view(np.uint32))
