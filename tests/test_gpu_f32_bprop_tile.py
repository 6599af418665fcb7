"""The tiled direct dx: cpu_bprop_nhwc's bits at the edges of its pixel groups, phases, channel
blocks and filter slices (the oracle's loop, one multiply and one add per term)."""
import numpy as np
import pytest
import torch

import my_own_cnn_amd as M
import oracle

pytestmark = pytest.mark.gpu

# (n, h, w, c, k, r, s, conv): pixel groups that end inside a row, phases without taps, strides and
# dilations that do not meet, several filter slices, 1, 2, 4 and 8 channel quads a block
CASES = [
    (1, 9, 11, 4, 4, 3, 3, (1, 1, 2, 2, 1, 1, 1)),
    (2, 16, 17, 32, 32, 3, 3, (1, 1, 2, 2, 1, 1, 1)),
    (1, 13, 10, 24, 36, 1, 1, (0, 0, 2, 3, 1, 1, 1)),
    (2, 12, 14, 16, 132, 3, 5, (2, 0, 3, 2, 1, 2, 1)),
    (1, 15, 15, 40, 24, 7, 7, (3, 3, 2, 2, 1, 1, 2)),
    (1, 8, 8, 64, 264, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    (1, 6, 9, 32, 8, 3, 3, (1, 1, 4, 4, 2, 2, 1)),
    (3, 5, 3, 12, 16, 2, 2, (4, 3, 2, 1, 3, 1, 1)),
    # on both sides of the rule for strides and dilations with a common factor (the one-pixel kernel
    # below 8 quads a block or 8 output channels), and for one tap on 4 channels
    (2, 12, 14, 16, 132, 3, 5, (2, 0, 3, 3, 1, 2, 1)),
    (2, 11, 13, 16, 16, 3, 3, (2, 2, 2, 2, 2, 2, 1)),
    (2, 11, 13, 64, 4, 3, 3, (2, 2, 2, 2, 2, 2, 1)),
    (1, 14, 9, 32, 12, 3, 1, (2, 0, 4, 1, 2, 1, 1)),
    (1, 14, 9, 20, 64, 1, 1, (0, 0, 2, 2, 1, 1, 1)),
    (1, 14, 9, 20, 60, 1, 1, (0, 0, 2, 2, 1, 1, 1)),
]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_bits_of_the_reference_loop(device, case):
    n, h, w, c, k, r, s, conv = case
    rng = np.random.default_rng(60 + CASES.index(case))
    ho, wo = oracle.conv_output_shape(n, h, w, c, r, s, k, conv)
    wt = rng.uniform(-1, 1, size=(k, r, s, c // conv[6])).astype(np.float32)
    dy = rng.uniform(-1, 1, size=(n, ho, wo, k)).astype(np.float32)
    for special in (False, True):
        if special:  # a tap outside the image multiplies nothing, not zero by infinity
            wt[0, 0, 0, 0], wt[1, r - 1, s - 1, 1] = np.inf, np.nan
        dx = torch.full((n, h, w, c), 7.0, device=device)
        M.launch_bprop_nhwc(torch.from_numpy(dy).to(device), torch.from_numpy(wt).to(device), dx, n, h, w, c, r, s, k,
                            conv, algo="direct")
        torch.cuda.synchronize()
        want = oracle.bprop_f32(dy, wt, (n, h, w, c), conv)
        got = dx.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        m = ~np.isnan(want)
        np.testing.assert_array_equal(got[m].view(np.uint32), want[m].view(np.uint32))
