"""1x1 convolutions of few input channels and many filters over large images (conv_expand_f32_kernel), against torch in 64 bits."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from test_split_gemm import _kernels


@pytest.mark.gpu
# channels one, odd and at the edges of the two instances; filters off 32; pixels off the tile of 512; many and few filter blocks per wavefront
@pytest.mark.parametrize("c", [(1, 33, 3, 330, 338), (7, 100, 40, 50, 52), (16, 65, 41, 63, 64), (17, 96, 9, 110, 110), (23, 144, 30, 55, 56), (24, 400, 11, 52, 47)],
                         ids=lambda c: "x".join(map(str, c)))
def test_gpu_expand(c):
    cin, cout, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f, bias = torch.randn((b, cin, h, w), generator=gen), torch.randn((cout, cin, 1, 1), generator=gen), torch.randn(cout, generator=gen)
    xd, fd, bd = x.cuda(), f.cuda(), bias.cuda()
    prod = lambda x, f: torch.matmul(f.view(cout, cin).double(), x.view(b, cin, h * w).double()).view(b, cout, h, w)
    want, bound = prod(xd, fd) + bd.double().view(1, -1, 1, 1), prod(xd.abs(), fd.abs()) + bd.double().abs().view(1, -1, 1, 1)
    for act, res in (("relu6", want.clamp(0, 6)), ("identity", want)):
        op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, 1, 1, 1, 0, 1, (b, cin, h, w)), True, act)
        work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
        packed = torch.empty(max(op.packed_size(), 1), dtype=torch.uint8, device="cuda:0")
        op.pack(fd, packed)
        for call in (lambda y: op.enqueue(xd, fd, bd, y, work), lambda y: op.enqueue_packed(xd, fd, packed, bd, y, work)):
            y = torch.full((b, cout, h, w), float("nan"), device="cuda:0")
            (name,) = _kernels(lambda: call(y))
            assert name.startswith("conv_expand_f32_kernel<%d>" % (8 if cin <= 16 else 12)), name
            assert ((y.double() - res).abs() <= bound * ((cin + 4) * 2.0 ** -24)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c, expand", [((24, 128, 18, 68, 68), False), ((24, 128, 88, 68, 68), True), ((8, 128, 19, 68, 68), True), ((8, 256, 40, 68, 68), False),
                                       ((24, 124, 19, 68, 68), True)], ids=str)
def test_gpu_expand_lines(c, expand):
    """filters in whole tiles of 64: outputs of 190 MB and more, of 40 with few channels; whole numbers, exact in any order"""
    cin, cout, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f = torch.randint(-4, 5, (b, cin, h, w), generator=gen).float(), torch.randint(-4, 5, (cout, cin, 1, 1), generator=gen).float()
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, 1, 1, 1, 0, 1, (b, cin, h, w)), False)
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    packed = torch.empty(max(op.packed_size(), 1), dtype=torch.uint8, device="cuda:0")
    xd, fd = x.cuda(), f.cuda()
    op.pack(fd, packed)
    want = torch.matmul(fd.view(cout, cin).double(), xd.view(b, cin, h * w).double()).view(b, cout, h, w)
    for call in (lambda y: op.enqueue(xd, fd, None, y, work), lambda y: op.enqueue_packed(xd, fd, packed, None, y, work)):
        y = torch.full((b, cout, h, w), float("nan"), device="cuda:0")
        (name,) = _kernels(lambda: call(y))
        assert name.startswith("conv_expand_f32_kernel<") == expand, name
        assert torch.equal(y.double(), want)
