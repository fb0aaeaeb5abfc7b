"""Small bf16 convolutions in tiles of 32x32 and 16x16, their reduction dealt to the wavefronts of a workgroup (conv_wave_bf16_kernel),
against torch in 64 bits on the same bf16 operands."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from dlprimitives_amd.capi import BFLOAT16_DATA
from test_split_gemm import _geometry, _kernels

# (cin, cout, k, stride, pad, dilate, groups, batch, h, w): tile, wavefronts a tile
CASES = {
    (32, 8, 1, 1, 0, 1, 1, 1, 1, 1): (32, 4),            # one K tile, one pixel: three wavefronts without work
    (64, 72, 1, 1, 0, 1, 1, 2, 9, 7): (32, 4),           # rows and pixels off the tile
    (96, 40, 3, 1, 1, 1, 1, 1, 13, 11): (16, 8),         # 27 K tiles over eight wavefronts
    (512, 24, 1, 2, 0, 1, 1, 3, 9, 5): (16, 4),          # 16 K tiles, strided
    (512, 512, 3, 1, 1, 1, 1, 1, 7, 7): (16, 8),
    (128, 136, 3, 2, 1, 1, 1, 8, 29, 27): (32, 4),
    (128, 64, 3, 1, 2, 2, 1, 2, 40, 41): (32, 8),        # dilated
    (128, 48, 3, 1, 1, 1, 2, 6, 30, 30): (32, 4),        # groups of 64 channels, filters off the tile
    (64, 64, 1, 1, 0, 1, 1, 5, 56, 56): (32, 2),
    (64, 32, 5, 1, 2, 1, 1, 5, 33, 31): (32, 8),
}


@pytest.mark.gpu
@pytest.mark.parametrize("ycl", [True, False])
@pytest.mark.parametrize("c", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_wave_conv(c, ycl):
    cin, cout, k, s, p, d, g, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    x, f, old = (torch.randn(n, generator=gen).bfloat16() for n in (xs, ws, ys))
    bias = torch.randn(cout, generator=gen)
    conv = lambda x, f: torch.nn.functional.conv2d(x.double(), f.double(), None, s, p, d, g)
    want = conv(x, f) + bias.double().view(1, -1, 1, 1)
    # sums in fp32, one rounding a product at most, then the rounding to bf16
    slack = (conv(x.abs(), f.abs()) + 8) * ((cin // g * k * k + 8) * 2.0 ** -24)
    store = lambda t: t.permute(0, 2, 3, 1).contiguous().cuda() if ycl else t.cuda()
    xd, fd, bd = x.permute(0, 2, 3, 1).contiguous().cuda(), f.cuda(), bias.cuda()
    for act, first in (("relu", False), ("identity", True)):
        op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs, dtype=BFLOAT16_DATA), True, act, "gemm")
        op.accumulate_before_activation(first)
        op.channels_last(True, ycl)
        work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
        packed = torch.empty(max(op.packed_size(), 1), dtype=torch.uint8, device="cuda:0")
        op.pack(fd, packed)
        for raw in (False, True):
            y = store(old if first else torch.full(ys, float("nan"), dtype=torch.bfloat16))
            factor = 0.5 if first else 0.0
            (name,) = _kernels(lambda: op.enqueue(xd, fd, bd, y, work, factor) if raw else op.enqueue_packed(xd, fd, packed, bd, y, work, factor))
            assert name.startswith("conv_wave_bf16_kernel<%d, %d, " % CASES[c]), name
            res = want + factor * old.double() if first else want.relu()
            got = (y.permute(0, 3, 1, 2) if ycl else y).cpu().double()
            assert ((got - res).abs() <= res.abs() * 2.0 ** -8 + slack).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c, wave", [((448, 200, 7, 31, 31), False), ((448, 200, 5, 31, 31), True), ((352, 144, 38, 19, 14), False), ((256, 320, 18, 15, 15), True),
                                     ((320, 80, 35, 22, 22), False), ((352, 32, 8, 78, 78), True), ((512, 200, 16, 31, 31), True)], ids=str)
def test_gpu_wave_conv_lines(c, wave):
    """1x1 of 8 to 15 K tiles: up to 1300 tiles (1600 of up to 64 filters) and 17000 K tiles; whole numbers, their sums exact in any order before the one rounding"""
    cin, cout, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f = torch.randint(-3, 4, (b, h, w, cin), generator=gen).bfloat16().cuda(), torch.randint(-3, 4, (cout, cin, 1, 1), generator=gen).bfloat16().cuda()
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, 1, 1, 1, 0, 1, (b, cin, h, w), dtype=BFLOAT16_DATA), False, "identity", "gemm")
    op.channels_last(True, True)
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    packed = torch.empty(max(op.packed_size(), 1), dtype=torch.uint8, device="cuda:0")
    op.pack(f, packed)
    y = torch.full((b, h, w, cout), float("nan"), dtype=torch.bfloat16, device="cuda:0")
    (name,) = _kernels(lambda: op.enqueue_packed(x, f, packed, None, y, work))
    assert name.startswith("conv_wave_bf16_kernel<") == wave, name
    want = torch.matmul(x.view(-1, cin).float().cpu(), f.view(cout, cin).float().cpu().t().contiguous())
    assert torch.equal(y.view(-1, cout).cpu(), want.bfloat16())
