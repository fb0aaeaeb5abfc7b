"""Depthwise 3x3 filter gradients walked down columns (depthwise_wgrad3x3_columns_kernel), against torch in 64 bits."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from test_split_gemm import _geometry, _kernels

# (channels, filters per channel, stride, pad, batch, h, w)
CASES = [(1, 1, 1, 1, 1, 1, 1), (3, 1, 1, 0, 2, 3, 5), (33, 1, 1, 1, 3, 9, 7), (5, 3, 1, 2, 4, 17, 30), (700, 1, 1, 1, 2, 8, 8), (40, 1, 2, 1, 5, 15, 13), (6, 2, 2, 0, 3, 8, 9),
         (24, 1, (1, 2), 1, 3, 21, 16), (24, 1, (2, 1), (0, 1), 3, 21, 16), (16, 1, 1, 1, 70, 14, 14)]


@pytest.mark.gpu
@pytest.mark.parametrize("c", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_depthwise_wgrad_columns(c):
    ch, mult, s, p, b, h, w = c
    gen = torch.Generator().manual_seed(ch + h)
    x = torch.randn((b, ch, h, w), generator=gen)
    f = (ch * mult, 1, 3, 3)
    st = dlp.Conv2DSettings(ch, ch * mult, 3, s, 1, p, ch, tuple(x.shape))
    dy = torch.randn(dlp.conv2d_output_shape(st, x.shape), generator=gen)
    old = torch.randn(f, generator=gen)
    op = dlp.Conv2DBackwardFilter.create(st)
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    grad = lambda x, dy: torch.nn.grad.conv2d_weight(x.double(), f, dy.double(), s, p, 1, ch)
    n = dy.numel() // dy.shape[1]
    for factor in (0.0, 0.5):
        dw = old.cuda() if factor else torch.full(f, float("nan"), device="cuda:0")
        (name,) = _kernels(lambda: op.enqueue(x.cuda(), dw, dy.cuda(), work, factor), "wgrad_depthwise")
        assert name.startswith("depthwise_wgrad3x3_columns_kernel<"), name
        assert ((dw.cpu().double() - grad(x, dy) - factor * old).abs() <= (grad(x.abs(), dy.abs()) + old.abs()) * ((n + 4) * 2.0 ** -24)).all()
    x[0, 0, 0, 0] = float("inf")  # reaches the filters of its channel only, and only taps that meet it
    dw = torch.full(f, float("nan"), device="cuda:0")
    op.enqueue(x.cuda(), dw, dy.abs().cuda() + 0.5, work)
    assert torch.equal(torch.isfinite(dw.cpu()), torch.isfinite(grad(x, dy.abs() + 0.5)))


@pytest.mark.gpu
@pytest.mark.parametrize("c, rows", [((40, 1, 1, 1, 26, 16, 16), 1), ((40, 1, 1, 1, 26, 16, 17), 8), ((40, 1, 1, 1, 27, 16, 16), 8), ((40, 1, 2, 1, 26, 31, 32), 1), ((40, 1, 2, 1, 26, 33, 31), 4),
                                     ((1, 2, 2, 0, 1, 3, 3), 1)], ids=str)
def test_gpu_depthwise_wgrad_rows_of_a_lane(c, rows):
    """one pixel a lane up to 256 of one image a workgroup, more down a column: whole numbers, exact in any order"""
    ch, mult, s, p, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f = torch.randint(-3, 4, (b, ch, h, w), generator=gen).float(), (ch * mult, 1, 3, 3)
    st = dlp.Conv2DSettings(ch, ch * mult, 3, s, 1, p, ch, tuple(x.shape))
    dy = torch.randint(-3, 4, dlp.conv2d_output_shape(st, x.shape), generator=gen).float()
    op = dlp.Conv2DBackwardFilter.create(st)
    work, dw = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0"), torch.full(f, float("nan"), device="cuda:0")
    (name,) = _kernels(lambda: op.enqueue(x.cuda(), dw, dy.cuda(), work), "wgrad_depthwise")
    assert name == "depthwise_wgrad3x3_columns_kernel<%d, %d>" % (s, rows), name
    assert torch.equal(dw.cpu().double(), torch.nn.grad.conv2d_weight(x.double(), f, dy.double(), s, p, 1, ch))
