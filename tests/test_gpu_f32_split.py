"""The fp32 convolution on split bf16 operands: sizes at the edges of its tiles, channel octets,
stages and chunks, and the inputs that it hands back to the fp32 instructions.

Bound against 64 bits: a K-block of 32 reduction values is summed with a few fp32 roundings of
its own (of up to 2^-23 each, the matrix core rounds down) and added with one of 2^-24 more, and the
dropped products are at most 2^-24 of each term, so every output is within (K / 32 + 16) 2^-23 of the
sum of |x w|: K / 32 times 2^-24 for the additions, and less than 16 times 2^-23 for a K-block's own
roundings, the dropped products and the scale (a factor two in hand)."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import my_own_cnn_amd as M

pytestmark = pytest.mark.gpu

# (n, h, w, c, k, r, s, (ph, pw, sh, sw, dh, dw, groups))
CASES = [
    (1, 5, 4, 4, 33, 5, 5, (2, 2, 1, 1, 1, 1, 1)),       # one half octet, a channel past the tile
    (2, 17, 19, 12, 40, 3, 3, (1, 1, 1, 1, 1, 1, 1)),    # octet tail
    (3, 33, 29, 20, 48, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    (5, 7, 7, 72, 65, 3, 3, (1, 1, 1, 1, 1, 1, 1)),      # several images per tile, an uneven chunk
    (37, 3, 3, 64, 36, 3, 3, (1, 1, 1, 1, 1, 1, 1)),     # images past the last tile
    (2, 30, 57, 64, 64, 3, 3, (0, 2, 1, 1, 1, 1, 1)),
    (1, 23, 21, 96, 66, 5, 3, (2, 1, 1, 1, 2, 3, 1)),    # dilation, K not a multiple of 4
    (2, 25, 31, 32, 96, 3, 3, (1, 1, 2, 2, 1, 1, 1)),    # stride
    (1, 40, 18, 24, 64, 7, 7, (3, 3, 2, 1, 1, 1, 1)),
    (2, 14, 15, 80, 64, 3, 3, (1, 1, 1, 1, 1, 1, 4)),    # groups
    (1, 1, 3, 256, 300, 1, 1, (0, 0, 1, 1, 1, 1, 1)),    # one tap
    (1, 9, 130, 264, 32, 1, 1, (0, 0, 1, 1, 1, 1, 1)),
    (1, 6, 6, 16, 32, 3, 3, (3, 3, 1, 1, 1, 1, 1)),      # padding past the filter's reach
    (24, 28, 28, 64, 96, 3, 3, (1, 1, 1, 1, 1, 1, 1)),   # enough tiles for the larger ones
    (32, 14, 14, 64, 256, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    (40, 30, 26, 32, 32, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    (32, 25, 20, 8, 36, 2, 3, (1, 1, 1, 1, 1, 1, 1)),    # one octet
    (32, 66, 4, 96, 8, 2, 3, (1, 1, 1, 1, 1, 1, 1)),
    (64, 23, 3, 64, 8, 3, 3, (1, 1, 1, 1, 2, 2, 1)),     # dx in the largest tile
]
LAYOUTS = {(1, 4, 2), (2, 2, 2), (4, 2, 2), (4, 4, 1), (4, 4, 2)}  # segments, rows and columns of waves


def conv64(x, w, conv):
    ph, pw, sh, sw, dh, dw, g = conv
    y = F.conv2d(x.double().permute(0, 3, 1, 2), w.double().permute(0, 3, 1, 2), padding=(ph, pw), stride=(sh, sw),
                 dilation=(dh, dw), groups=g)
    return y.permute(0, 2, 3, 1)


def data(case, seed):
    n, h, w, c, k, r, s, conv = case
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn((n, h, w, c), generator=gen), torch.randn((k, r, s, c // conv[6]), generator=gen))


def check(got, want, mag, kdim):
    err = (got.double() - want).abs()
    assert bool((err <= (kdim / 32 + 16) * 2.0 ** -23 * mag + 1e-300).all()), float((err / mag.clamp(min=1e-300)).max())


def layout(op, n, h, w, c, k, r, s, conv, by=1, bx=1):
    """The wave layout in which the pass computes on split operands, None where it does not."""
    tile = M.plan_f32_split(op, n, h, w, c, r, s, k, M.BlockConv2DParams(M.Conv2DParams(*conv), by, bx))
    return tile and tile[:3]


def test_cases_reach_every_layout():
    assert {layout("fprop", *c) for c in CASES} - {None} == LAYOUTS
    assert {layout("bprop", *c) for c in CASES} - {None} == LAYOUTS
    assert {layout("bprop", *c) for c in BLOCKED_DX} - {None} == LAYOUTS - {(1, 4, 2)}
    assert [layout("bprop", *c) is None for c in BLOCKED_DX if c[5] * c[6] == 1] == [True, False]
    assert len({c[1:] for c in GRADS_SPLIT}) == 8  # four layouts, one or two tiles in LDS


@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_forward_and_dx(device, case):
    n, h, w, c, k, r, s, conv = case
    x, wt = data(case, 7 + CASES.index(case))
    y = M.conv2d_nhwc_f32(x.to(device), wt.to(device), padding=conv[:2], stride=conv[2:4], dilation=conv[4:6], groups=conv[6])
    check(y.cpu(), conv64(x, wt, conv), conv64(x.abs(), wt.abs(), conv), wt[0].numel())
    if conv[2] != 1 or conv[3] != 1 or (k // conv[6]) % 4:
        return
    xg = x.double().requires_grad_()
    dy = torch.randn(y.shape, generator=torch.Generator().manual_seed(1))
    want, = torch.autograd.grad(conv64(xg, wt, conv), xg, dy.double())
    mag, = torch.autograd.grad(conv64(xg, wt.abs(), conv), xg, dy.double().abs())
    dx = torch.full(x.shape, 7.0, device=device)
    M.launch_bprop_nhwc(dy.to(device), wt.to(device), dx, n, h, w, c, r, s, k, conv)
    check(dx.cpu(), want, mag, r * s * k // conv[6])


@pytest.mark.parametrize("taps", [3, 5])
def test_empty_reductions_are_zero(device, taps):
    y = M.conv2d_nhwc_f32(torch.empty((1, 8, 8, 0), device=device), torch.empty((40, taps, taps, 0), device=device))
    assert float(y.abs().max()) == 0.0
    dx = torch.full((1, 8, 8, 16), 7.0, device=device)
    M.launch_bprop_nhwc(torch.empty((1, 8, 8, 0), device=device), torch.empty((0, taps, taps, 16), device=device), dx,
                        1, 8, 8, 16, taps, taps, 0, (taps // 2, taps // 2, 1, 1, 1, 1, 1))
    assert float(dx.abs().max()) == 0.0


@pytest.mark.parametrize("grid", [(2, 3), (4, 2)])
def test_blocked_forward(device, grid):
    n, h, w, c, k = 3, 16, 18, 40, 70
    by, bx = grid
    assert layout("fprop", n, h, w, c, k, 3, 3, (1, 1, 1, 1, 1, 1, 1), by, bx)
    gen = torch.Generator().manual_seed(3)
    x, wt = torch.randn((n, h, w, c), generator=gen), torch.randn((k, by, bx, 3, 3, c), generator=gen)
    conv = (1, 1, 1, 1, 1, 1, 1)
    y = torch.empty((n, h, w, k), device=device)
    M.launch_block_fprop_nhwc(x.to(device), wt.to(device), y, n, h, w, c, 3, 3, k,
                              M.BlockConv2DParams(M.Conv2DParams(*conv), by, bx))
    for i in range(by):
        for j in range(bx):
            rows, cols = slice(i * h // by, (i + 1) * h // by), slice(j * w // bx, (j + 1) * w // bx)
            f = wt[:, i, j].contiguous()
            check(y[:, rows, cols].cpu(), conv64(x, f, conv)[:, rows, cols], conv64(x.abs(), f.abs(), conv)[:, rows, cols], 9 * c)


def blocked_dx(dy, wt, xshape, conv):
    """dx of a blocked convolution and the sum of its terms' magnitudes, in 64 bits."""
    by, bx = wt.shape[1:3]
    h, w = dy.shape[1:3]
    x = torch.zeros(xshape, dtype=torch.float64, requires_grad=True)
    out = [0, 0]
    for i in range(by):
        for j in range(bx):
            d = torch.zeros_like(dy)
            rows, cols = slice(i * h // by, (i + 1) * h // by), slice(j * w // bx, (j + 1) * w // bx)
            d[:, rows, cols] = dy[:, rows, cols]
            f = wt[:, i, j].contiguous()
            for a, fn in enumerate((lambda v: v, torch.abs)):
                out[a] = out[a] + torch.autograd.grad(conv64(x, fn(f), conv), x, fn(d).double())[0]
    return out


# (n, h, w, c, k, r, s, conv, by, bx): images above and below a segment's 16, blocks of a few
# positions, taps that reach past a neighbour block, clipped regions, groups, 32 channels a group
BLOCKED_DX = [
    (3, 16, 18, 40, 72, 3, 3, (1, 1, 1, 1, 1, 1, 1), 2, 3),
    (20, 12, 14, 36, 24, 3, 3, (1, 1, 1, 1, 1, 1, 1), 4, 2),
    (17, 12, 12, 24, 16, 5, 5, (2, 2, 1, 1, 1, 1, 1), 6, 4),
    (2, 14, 15, 48, 40, 3, 3, (2, 0, 1, 1, 2, 1, 1), 2, 1),
    (16, 10, 9, 64, 128, 3, 2, (0, 1, 1, 1, 1, 1, 2), 4, 2),
    (33, 8, 8, 40, 160, 1, 1, (0, 0, 1, 1, 1, 1, 1), 2, 2),  # one tap: the fp32 implicit GEMM
    (2, 8, 8, 40, 160, 1, 1, (0, 0, 1, 1, 1, 1, 1), 2, 2),   # but for at most 32 positions a block
    (20, 10, 6, 48, 16, 1, 3, (0, 1, 1, 1, 1, 1, 1), 1, 2),
]


@pytest.mark.parametrize("case", BLOCKED_DX, ids=str)
def test_blocked_dx(device, case):
    n, h, w, c, k, r, s, conv, by, bx = case
    gen = torch.Generator().manual_seed(12)
    p = M.BlockConv2DParams(M.Conv2DParams(*conv), by, bx)
    ho, wo = M.infer_block_conv_shape(n, h, w, c, r, s, k, p)[:2]
    wt = torch.randn((k, by, bx, r, s, c // conv[6]), generator=gen)
    dy = torch.randn((n, ho, wo, k), generator=gen)
    dx = torch.full((n, h, w, c), 7.0, device=device)
    for special in (False, True):
        if special:  # one value past the scaled range sends its tiles through the fp32 instructions
            dy[0, ho // 2, wo // 2, 1] = 2.0 ** 112
        M.launch_block_bprop_nhwc(dy.to(device), wt.to(device), dx, n, h, w, c, r, s, k, p)
        want, mag = blocked_dx(dy, wt, (n, h, w, c), conv)
        check(dx.cpu(), want, mag, r * s * k // conv[6])


def test_infinite_and_nan_inputs(device):
    x, wt = data((2, 20, 20, 32, 40, 3, 3, (1, 1, 1, 1, 1, 1, 1)), 5)
    x[0, 3, 4, 5], x[0, 10, 12, 7], x[1, 19, 19, 31], x[1, 0, 0, 0] = float("inf"), float("nan"), float("-inf"), 3.4e38
    y = M.conv2d_nhwc_f32(x.to(device), wt.to(device), padding=1).cpu()
    # image by tap: a tap outside the image multiplies by nothing
    want = conv64(torch.nan_to_num(x, nan=0.0, posinf=0.0, neginf=0.0), wt, (1, 1, 1, 1, 1, 1, 1))
    for im, r, c, ch, v in ((0, 3, 4, 5, float("inf")), (0, 10, 12, 7, float("nan")), (1, 19, 19, 31, float("-inf"))):
        for i in range(3):
            for j in range(3):
                hh, ww = r - i + 1, c - j + 1
                if 0 <= hh < 20 and 0 <= ww < 20:
                    want[im, hh, ww] += v * wt[:, i, j, ch].double()
    over = want.abs() > 3.4028235677973366e38
    want = torch.where(over & want.isfinite(), torch.sign(want) * float("inf"), want)
    assert torch.equal(y.isnan(), want.isnan())
    fin = want.isfinite()
    assert torch.equal(y[~fin & ~want.isnan()].double(), want[~fin & ~want.isnan()])
    assert bool(((y[fin].double() - want[fin]).abs() <= 1e-4 + 1e-5 * want[fin].abs()).all())


@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -112, 2.0 ** -126, 2.0 ** -140])
def test_small_inputs(device, scale):
    case = (1, 12, 12, 32, 36, 3, 3, (1, 1, 1, 1, 1, 1, 1))
    x, wt = data(case, 6)
    x, wt = x * scale, wt * 2.0 ** 30
    y = M.conv2d_nhwc_f32(x.to(device), wt.to(device), padding=1).cpu()
    check(y, conv64(x, wt, case[7]), conv64(x.abs(), wt.abs(), case[7]), 9 * 32)
    dx = torch.empty_like(x, device=device)
    dy = torch.randn((1, 12, 12, 36), generator=torch.Generator().manual_seed(2)) * scale
    M.launch_bprop_nhwc(dy.to(device), wt.to(device), dx, 1, 12, 12, 32, 3, 3, 36, case[7])
    xg = x.double().requires_grad_()
    want, = torch.autograd.grad(conv64(xg, wt, case[7]), xg, dy.double())
    mag, = torch.autograd.grad(conv64(xg, wt.abs(), case[7]), xg, dy.double().abs())
    check(dx.cpu(), want, mag, 9 * 36)


@pytest.mark.parametrize("tiny", [1e-35, 1e-40, 2.0 ** -149])
def test_a_tiny_value_leaves_the_other_results(device, tiny):
    """Every fp32 value is carried by the split: a tile that holds a tiny one keeps the bits of the
    results that the value does not reach."""
    n, h, w, c, k = 2, 20, 20, 40, 72
    conv = (1, 1, 1, 1, 1, 1, 1)
    bp = M.BlockConv2DParams(M.Conv2DParams(*conv), 2, 2)
    kd = 28  # output channels of dw: few enough for the split kernel at this size
    assert layout("fprop", n, h, w, c, k, 3, 3, conv) and layout("bprop", n, h, w, c, k, 3, 3, conv)
    assert layout("bprop", n, h, w, c, k, 3, 3, conv, 2, 2) and layout("grad", n, h, w, c, kd, 3, 3, conv)
    gen = torch.Generator().manual_seed(14)
    x, wt = torch.randn((n, h, w, c), generator=gen), torch.randn((k, 3, 3, c), generator=gen)
    dy, wb = torch.randn((n, h, w, k), generator=gen), torch.randn((k, 2, 2, 3, 3, c), generator=gen)

    def outputs(x, wt, dy):
        x, wt, dy = x.to(device), wt.to(device), dy.to(device)
        y, dx, dxb, dw = torch.empty_like(dy), torch.empty_like(x), torch.empty_like(x), torch.empty_like(wt[:kd])
        M.launch_fprop_nhwc(x, wt, y, n, h, w, c, 3, 3, k, conv)
        M.launch_bprop_nhwc(dy, wt, dx, n, h, w, c, 3, 3, k, conv)
        M.launch_block_bprop_nhwc(dy, wb.to(device), dxb, n, h, w, c, 3, 3, k, bp)
        M.launch_grad_nhwc(x, dy[..., :kd].contiguous(), dw, n, h, w, c, 3, 3, kd, conv)
        return y.cpu(), dx.cpu(), dxb.cpu(), dw.cpu()

    def put(t, at, v):
        t = t.clone()
        t[at] = v
        return t

    at, near = (1, 8, 9, 5), (1, slice(7, 10), slice(8, 11))
    zero, got = (outputs(put(x, at, v), wt, dy) for v in (0.0, tiny))
    for a, b, skip in ((zero[0], got[0], near), (zero[3], got[3], (slice(None), slice(None), slice(None), 5))):
        assert torch.equal(put(a, skip, 0.0), put(b, skip, 0.0))
    zero, got = (outputs(x, wt, put(dy, at, v)) for v in (0.0, tiny))
    for i, skip in ((1, near), (2, near), (3, 5)):
        assert torch.equal(put(zero[i], skip, 0.0), put(got[i], skip, 0.0)), i
    zero, got = (outputs(x, put(wt, (7, 0, 2, 3), v), dy) for v in (0.0, tiny))
    for i in (0, 1):
        assert torch.equal(put(zero[i], (..., 7 if i == 0 else 3), 0.0), put(got[i], (..., 7 if i == 0 else 3), 0.0)), i


@pytest.mark.parametrize("exp", [-55, -60, -63, -65, -70])
def test_subnormal_products(device, exp):
    """Both operands small: products and results reach the subnormal range, where each result (of
    dw: each of its partial sums) is rounded to a multiple of 2^-149 once."""
    n, h, w, c, k = 2, 24, 24, 32, 64
    conv = (1, 1, 1, 1, 1, 1, 1)
    x, wt = data((n, h, w, c, k, 3, 3, conv), 16)
    dy = torch.randn((n, h, w, k), generator=torch.Generator().manual_seed(17))
    x, wt, dy = x * 2.0 ** exp, wt * 2.0 ** exp, dy * 2.0 ** exp
    kd = 32  # output channels of dw: few enough for the split kernel at this size
    dyd = dy[..., :kd].contiguous()
    assert layout("fprop", n, h, w, c, k, 3, 3, conv) and layout("bprop", n, h, w, c, k, 3, 3, conv)
    assert layout("grad", n, h, w, c, kd, 3, 3, conv)
    y, dx, dw = (torch.full(t.shape, 7.0, device=device) for t in (dy, x, wt[:kd]))
    dims = (n, h, w, c, 3, 3)
    M.launch_fprop_nhwc(x.to(device), wt.to(device), y, *dims, k, conv)
    M.launch_bprop_nhwc(dy.to(device), wt.to(device), dx, *dims, k, conv)
    M.launch_grad_nhwc(x.to(device), dyd.to(device), dw, *dims, kd, conv)
    xg = x.double().requires_grad_()
    want_dx, = torch.autograd.grad(conv64(xg, wt, conv), xg, dy.double())
    mag_dx, = torch.autograd.grad(conv64(xg, wt.abs(), conv), xg, dy.double().abs())
    parts = n * h * w // 64 + 1  # at most one partial sum per tile of positions
    for got, want, mag, kdim, roundings in (
            (y, conv64(x, wt, conv), conv64(x.abs(), wt.abs(), conv), 9 * c, 1),
            (dx, want_dx, mag_dx, 9 * k, 1),
            (dw, grad_want(x, dyd, dw.shape, conv), grad_want(x, dyd, dw.shape, conv, torch.abs), n * h * w + 512, parts)):
        err = (got.cpu().double() - want).abs()
        assert bool((err <= (kdim / 32 + 16) * 2.0 ** -23 * mag + roundings * 2.0 ** -150).all()), float(err.max())


@pytest.mark.parametrize("signs", [False, True])
def test_operands_with_the_largest_dropped_products(device, signs):
    """1 + 2^-8 - 2^-17 splits into 1, 2^-8 and -2^-17: the dropped products of every term are 2^-24.01
    of it, all one way.  Every result is within 2^-24 of the sum of |x w| for them and as much for the
    roundings, which are few: the terms are equal, so that short sums of them are nearly exact."""
    n, h, w, c, k = 2, 24, 24, 32, 64
    conv = (1, 1, 1, 1, 1, 1, 1)
    value = 1 + 2.0 ** -8 - 2.0 ** -17
    gen = torch.Generator().manual_seed(19)

    def fill(*shape):
        return value * (torch.randint(0, 2, shape, generator=gen) * 2.0 - 1 if signs else torch.ones(shape))

    x, wt, dy = fill(n, h, w, c), fill(k, 3, 3, c), fill(n, h, w, k)
    kd = 32  # output channels of dw: few enough for the split kernel at this size
    dyd = dy[..., :kd].contiguous()
    assert layout("fprop", n, h, w, c, k, 3, 3, conv) and layout("bprop", n, h, w, c, k, 3, 3, conv)
    assert layout("grad", n, h, w, c, kd, 3, 3, conv)
    y, dx, dw = (torch.full(t.shape, 7.0, device=device) for t in (dy, x, wt[:kd]))
    dims = (n, h, w, c, 3, 3)
    M.launch_fprop_nhwc(x.to(device), wt.to(device), y, *dims, k, conv)
    M.launch_bprop_nhwc(dy.to(device), wt.to(device), dx, *dims, k, conv)
    M.launch_grad_nhwc(x.to(device), dyd.to(device), dw, *dims, kd, conv)
    xg = x.double().requires_grad_()
    want_dx, = torch.autograd.grad(conv64(xg, wt, conv), xg, dy.double())
    mag_dx, = torch.autograd.grad(conv64(xg, wt.abs(), conv), xg, dy.double().abs())
    for got, want, mag in ((y, conv64(x, wt, conv), conv64(x.abs(), wt.abs(), conv)), (dx, want_dx, mag_dx),
                           (dw, grad_want(x, dyd, dw.shape, conv), grad_want(x, dyd, dw.shape, conv, torch.abs))):
        err = (got.cpu().double() - want).abs()
        assert bool((err <= 2.0 ** -23 * mag).all()), float((err / mag).max())


# filter gradients of small layers, most of which the fp32 GEMM takes: (n, h, w, c, k, r, s, conv)
GRADS = [
    (2, 9, 11, 4, 8, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    (3, 19, 17, 36, 68, 3, 3, (1, 1, 1, 1, 1, 1, 1)),     # channels past the tiles
    (9, 7, 7, 64, 96, 3, 3, (1, 1, 1, 1, 1, 1, 1)),       # several images per tile
    (2, 31, 29, 32, 32, 3, 3, (1, 1, 2, 2, 1, 1, 1)),     # stride
    (1, 26, 40, 68, 28, 3, 3, (2, 0, 1, 2, 2, 1, 1)),     # dilation
    (2, 21, 18, 20, 72, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    (2, 15, 14, 128, 64, 1, 1, (0, 0, 1, 1, 1, 1, 1)),    # one tap, two channel tiles per wave
    (2, 13, 15, 16, 40, 2, 3, (1, 1, 1, 1, 1, 1, 1)),     # fewer taps than a workgroup takes
    (1, 20, 22, 64, 64, 5, 5, (2, 2, 1, 1, 1, 1, 1)),     # more
    (2, 16, 16, 96, 64, 3, 3, (1, 1, 1, 1, 1, 1, 2)),     # groups
    (1, 56, 56, 64, 64, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
]


# filter gradients on split operands: the case, its wave layout (32-channel rows, columns of input
# channels, wave groups that share a tile's positions) and the tiles in flight in LDS
GRADS_SPLIT = [
    ((1, 14, 21, 68, 36, 1, 1, (0, 0, 1, 1, 1, 1, 1)), (2, 4, 1), 2),      # one tap, two channel tiles per wave
    ((3, 71, 26, 36, 68, 3, 3, (0, 1, 1, 1, 1, 1, 1)), (2, 4, 1), 2),
    ((3, 114, 63, 36, 68, 3, 3, (1, 1, 2, 2, 1, 1, 1)), (2, 4, 1), 2),     # stride
    ((5, 71, 68, 36, 68, 3, 3, (1, 1, 2, 2, 2, 3, 1)), (2, 4, 1), 1),      # stride and dilation
    ((9, 40, 29, 36, 68, 3, 4, (1, 2, 1, 2, 2, 3, 1)), (2, 4, 1), 1),      # 12 taps: two workgroups' worth
    ((1, 52, 50, 64, 64, 5, 5, (2, 2, 1, 1, 1, 1, 1)), (2, 4, 1), 2),
    ((1, 17, 23, 20, 40, 1, 1, (0, 0, 1, 1, 1, 1, 1)), (2, 2, 2), 2),      # one tap, one channel tile
    ((5, 84, 45, 20, 40, 3, 3, (0, 1, 1, 1, 2, 3, 1)), (2, 2, 2), 2),
    ((2, 78, 111, 40, 80, 3, 3, (1, 1, 1, 2, 2, 3, 2)), (2, 2, 2), 2),     # groups
    ((5, 125, 114, 20, 40, 3, 3, (1, 1, 2, 2, 1, 1, 1)), (2, 2, 2), 1),
    ((9, 23, 50, 20, 40, 5, 5, (0, 2, 1, 1, 1, 1, 1)), (2, 2, 2), 1),
    ((2, 114, 44, 68, 28, 1, 1, (0, 0, 1, 2, 1, 1, 1)), (1, 4, 2), 1),
    ((1, 9, 38, 40, 12, 3, 3, (1, 1, 1, 1, 1, 1, 1)), (1, 4, 2), 2),
    ((2, 89, 48, 40, 12, 3, 3, (1, 1, 2, 1, 2, 1, 1)), (1, 4, 2), 1),
    ((5, 23, 11, 68, 28, 2, 3, (0, 1, 1, 1, 1, 1, 1)), (1, 4, 2), 1),      # fewer taps than a workgroup takes
    ((1, 35, 9, 20, 28, 3, 3, (0, 1, 1, 1, 2, 3, 1)), (1, 2, 4), 2),
    ((2, 96, 94, 32, 32, 3, 3, (1, 1, 2, 2, 1, 1, 1)), (1, 2, 4), 2),
    ((2, 51, 82, 16, 24, 3, 3, (1, 1, 2, 1, 2, 1, 1)), (1, 2, 4), 1),
    ((1, 128, 10, 16, 24, 2, 3, (0, 1, 1, 1, 2, 3, 1)), (1, 2, 4), 1),
]


def grad_want(x, dy, wshape, conv, f=lambda v: v):
    w = torch.zeros(wshape, dtype=torch.float64, requires_grad=True)
    return torch.autograd.grad(conv64(f(x), w, conv), w, f(dy).double())[0]


@pytest.mark.parametrize("case", GRADS + GRADS_SPLIT, ids=str)
def test_filter_gradient(device, case):
    seed = 31 + (GRADS + GRADS_SPLIT).index(case)
    if len(case) == 3:
        case, waves, tiles = case
        plan = M.plan_f32_split("grad", *case[:4], *case[5:7], case[4], case[7])
        assert plan and (plan[:3], plan[6]) == (waves, tiles), plan
    n, h, w, c, k, r, s, conv = case
    x, wt = data(case, seed)
    dy = torch.randn(conv64(x, wt, conv).shape, generator=torch.Generator().manual_seed(4))
    dw = torch.full(wt.shape, 7.0, device=device)
    M.launch_grad_nhwc(x.to(device), dy.to(device), dw, n, h, w, c, r, s, k, conv)
    # K-blocks of 32 positions, then the splits
    check(dw.cpu(), grad_want(x, dy, wt.shape, conv), grad_want(x, dy, wt.shape, conv, torch.abs), dy[..., 0].numel() + 512)


@pytest.mark.parametrize("shape", [(8, 40, 40, 64, 64), (8, 40, 40, 32, 32), (4, 40, 40, 96, 40)])
def test_errors_do_not_lean(device, shape):
    """The errors of a result's elements cancel: their mean is a small part of their rms.  The sums of
    the matrix core alone lean one way (means of 0.3 rms forward, 0.8 in the filter gradient).  Over
    N = 36,864 elements and more, independent errors give a mean of N^-1/2 = 0.005 rms; a step left over
    from an odd count of them leans by a ninth of the 0.3."""
    n, h, w, c, k = shape
    conv = (1, 1, 1, 1, 1, 1, 1)
    gen = torch.Generator().manual_seed(18)
    x, wt = torch.randn((n, h, w, c), generator=gen).clamp(min=0), torch.randn((k, 3, 3, c), generator=gen)
    dy, wb = torch.randn((n, h, w, k), generator=gen), torch.randn((k, 2, 2, 3, 3, c), generator=gen)
    dims = (n, h, w, c, 3, 3, k)
    for op, b in (("fprop", 1), ("bprop", 1), ("bprop", 2), ("grad", 1)):
        assert layout(op, n, h, w, c, k, 3, 3, conv, b, b), op
    y, dx, dxb, dw = (torch.empty(t.shape, device=device) for t in (dy, x, x, wt))
    M.launch_fprop_nhwc(x.to(device), wt.to(device), y, *dims, conv)
    M.launch_bprop_nhwc(dy.to(device), wt.to(device), dx, *dims, conv)
    M.launch_block_bprop_nhwc(dy.to(device), wb.to(device), dxb, *dims, M.BlockConv2DParams(M.Conv2DParams(*conv), 2, 2))
    M.launch_grad_nhwc(x.to(device), dy.to(device), dw, *dims, conv)
    xg = x.double().requires_grad_()
    want_dx, = torch.autograd.grad(conv64(xg, wt, conv), xg, dy.double())
    for name, got, want in (("y", y, conv64(x, wt, conv)), ("dx", dx, want_dx), ("blocked dx", dxb, blocked_dx(dy, wb, x.shape, conv)[0]),
                            ("dw", dw, grad_want(x, dy, wt.shape, conv))):
        err = got.cpu().double() - want
        assert abs(float(err.mean())) <= 0.1 * float(err.square().mean().sqrt()), name


@pytest.mark.parametrize("grid", [(2, 3), (4, 1)])
def test_blocked_filter_gradient(device, grid):
    n, h, w, c, k = 21, 16, 18, 40, 70
    by, bx = grid
    gen = torch.Generator().manual_seed(8)
    x, dy = torch.randn((n, h, w, c), generator=gen), torch.randn((n, h, w, k + 2), generator=gen)
    k += 2
    conv = (1, 1, 1, 1, 1, 1, 1)
    assert layout("grad", n, h, w, c, k, 3, 3, conv, by, bx)
    dw = torch.empty((k, by, bx, 3, 3, c), device=device)
    M.launch_block_grad_nhwc(x.to(device), dy.to(device), dw, n, h, w, c, 3, 3, k,
                             M.BlockConv2DParams(M.Conv2DParams(*conv), by, bx))
    got = dw.cpu()
    for i in range(by):
        for j in range(bx):
            d = torch.zeros_like(dy)
            rows, cols = slice(i * h // by, (i + 1) * h // by), slice(j * w // bx, (j + 1) * w // bx)
            d[:, rows, cols] = dy[:, rows, cols]
            check(got[:, i, j], grad_want(x, d, (k, 3, 3, c), conv), grad_want(x, d, (k, 3, 3, c), conv, torch.abs), n * h * w)


@pytest.mark.parametrize("shape", [(12, 24, 24, 64, 64), (2, 24, 24, 32, 32)])
def test_filter_gradient_of_special_values(device, shape):
    n, h, w, c, k = shape
    conv = (1, 1, 1, 1, 1, 1, 1)
    assert layout("grad", n, h, w, c, k, 3, 3, conv)
    gen = torch.Generator().manual_seed(9)
    x, dy = torch.randn((n, h, w, c), generator=gen), torch.randn((n, h, w, k), generator=gen)
    args = (n, h, w, c, 3, 3, k, conv)
    dw = torch.empty((k, 3, 3, c), device=device)
    M.launch_grad_nhwc((x * 2.0 ** -130).to(device), (dy * 2.0 ** 20).to(device), dw, *args)
    xs, ds = x * 2.0 ** -130, dy * 2.0 ** 20
    check(dw.cpu(), grad_want(xs, ds, (k, 3, 3, c), conv), grad_want(xs, ds, (k, 3, 3, c), conv, torch.abs), n * h * w + 512)
    x[0, 5, 6, 3], x[1, 9, 9, 9] = float("inf"), float("nan")
    M.launch_grad_nhwc(x.to(device), dy.to(device), dw, *args)
    got = dw.cpu()
    clean = torch.nan_to_num(x, nan=0.0, posinf=0.0)
    want = grad_want(clean, dy, (k, 3, 3, c), conv)
    for i in range(3):
        for j in range(3):
            want[:, i, j, 3] += float("inf") * dy[0, 5 - i + 1, 6 - j + 1].double()
            want[:, i, j, 9] = float("nan")
    assert torch.equal(got.isnan(), want.isnan())
    fin = want.isfinite()
    assert torch.equal(got[~fin & ~want.isnan()].double(), want[~fin & ~want.isnan()])
    mag = grad_want(clean, dy, (k, 3, 3, c), conv, torch.abs)
    assert bool(((got.double() - want).abs()[fin] <= (n * h * w) * 2.0 ** -23 * mag[fin]).all())
