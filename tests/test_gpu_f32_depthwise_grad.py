"""Depthwise fp32 filter gradient at the edges of its workgroup (128 pixels in 8 runs of 16, 128
channels, 9 or 16 taps held in registers).  Small whole numbers: every product and every partial
sum is exact below 2^24, so the result equals the 64-bit sum whatever the order.  The first pixel
of each image is infinite: a tap outside the image must not bring it in."""
import pytest
import torch

import my_own_cnn_amd as M
from my_own_cnn_amd.conv import Conv2DParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c,r,s,stride", [
    (1, 1, 1, 4, 3, 3, 1),       # one pixel, one quad
    (1, 3, 5, 124, 3, 3, 1),     # 15 pixels, a dead quad
    (1, 1, 17, 128, 1, 1, 1),    # one pixel into the second run
    (1, 8, 16, 132, 3, 3, 1),    # one whole workgroup of pixels, one quad in the second of channels
    (1, 3, 43, 128, 2, 5, 1),    # 129 output pixels, 10 taps
    (3, 9, 13, 36, 4, 4, 1),     # 16 taps
    (2, 15, 17, 64, 3, 3, 2),    # strided
])
def test_depthwise_grad_edges(n, h, w, c, r, s, stride):
    p = Conv2DParams(r // 2, s // 2, stride, stride, 1, 1, c)
    ho, wo = M.infer_conv_shape(n, h, w, c, r, s, c, p)
    gen = torch.Generator().manual_seed(7)
    x = torch.randint(-4, 5, (n, h, w, c), generator=gen).float()
    x[:, 0, 0] = float("inf")
    dy = torch.randint(1, 6, (n, ho, wo, c), generator=gen).float()
    xp = torch.nn.functional.pad(x.double(), (0, 0, s // 2, s // 2, r // 2, r // 2))
    ref = torch.empty(c, r, s, 1)
    for i in range(r):
        for j in range(s):
            win = xp[:, i:i + (ho - 1) * stride + 1:stride, j:j + (wo - 1) * stride + 1:stride]
            ref[:, i, j, 0] = (win * dy.double()).sum(dim=(0, 1, 2)).float()
    dw = torch.full((c, r, s, 1), float("nan"), device="cuda")
    M.launch_grad_nhwc(x.cuda(), dy.cuda(), dw, n, h, w, c, r, s, c, p)
    assert torch.equal(dw.cpu(), ref)
