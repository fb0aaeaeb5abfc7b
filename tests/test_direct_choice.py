"""Operators whose algorithm was left open and is Winograd by size: large batches run directly in tiles of the bf16 matrix instruction, with
filters raw and packed, smaller ones through the transform; gradients alike."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from test_split_gemm import _kernels


@pytest.mark.gpu
@pytest.mark.parametrize("cin", [64, 40])
def test_gpu_automatic_choice_by_batch(cin):
    gen = torch.Generator().manual_seed(cin)
    h, cout, hint = 40, 64, 48  # 600 tiles of 64 filters x 128 pixels at 48 images, 450 at 36
    f, bias = torch.randn((cout, cin, 3, 3), generator=gen), torch.randn(cout, generator=gen)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, 3, 1, 1, 1, 1, (hint, cin, h, h)), True, "relu")
    back = dlp.Conv2DBackwardData.create(dlp.Conv2DSettings(64, 64, 3, 1, 1, 1, 1, (hint, cout, h, h)))
    assert cin != 64 or op.algo() == "winograd"
    fd, bd = f.cuda(), bias.cuda()
    work = torch.empty(max(op.workspace(), back.workspace()), dtype=torch.uint8, device="cuda:0")
    packed = torch.full((op.packed_size(),), 255, dtype=torch.uint8, device="cuda:0")
    op.pack(fd, packed)
    for batch in (48, 36, 2):
        x = torch.randn((batch, cin, h, h), generator=gen)
        xd = x.cuda()
        ref = torch.nn.functional.conv2d(x[-2:].double(), f.double(), bias.double(), 1, 1).relu()
        scale = torch.nn.functional.conv2d(x[-2:].double().abs(), f.double().abs(), bias.double().abs(), 1, 1)
        for call in (lambda y: op.enqueue(xd, fd, bd, y, work), lambda y: op.enqueue_packed(xd, fd, packed, bd, y, work)):
            y = torch.full((batch, cout, h, h), float("nan"), device="cuda:0")
            names = _kernels(lambda: call(y))
            if cin == 64:
                start = {48: ["conv_split_f32_kernel<64, 128,"], 36: [], 2: ["conv_wave_f32_kernel<"]}[batch]
                assert len(names) == len(start) and all(n.startswith(t) for n, t in zip(names, start)), names
            # Winograd's transforms round at the size of sixteen products
            assert ((y[-2:].cpu().double() - ref).abs() <= scale * ((cin * 9 + 16) * 2.0 ** -24)).all()
    if cin == 64:
        dy, dx = torch.randn((hint, 64, h, h), generator=gen), torch.full((hint, 64, h, h), float("nan"), device="cuda:0")
        (name,) = _kernels(lambda: back.enqueue(dx, fd, dy.cuda(), work))
        assert name.startswith("conv_split_f32_kernel<64, 128,"), name
        want = torch.nn.functional.conv_transpose2d(dy[-2:].double(), f.double(), None, 1, 1)
        scale = torch.nn.functional.conv_transpose2d(dy[-2:].double().abs(), f.double().abs(), None, 1, 1)
        assert ((dx[-2:].cpu().double() - want).abs() <= scale * ((64 * 9 + 16) * 2.0 ** -24)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("batch, start", [(16, "conv_split_f32_kernel<64, 64,"), (21, "conv_patch_f32_kernel<")])
def test_gpu_tiles_of_64_or_patch_by_rounds(batch, start):
    """144 K tiles a tile: 196 tiles of 64x64 are cut to fill 256 CUs, 260 would leave four of them a round of their own."""
    gen = torch.Generator().manual_seed(batch)
    x, f = torch.randn((batch, 256, 14, 14), generator=gen), torch.randn((256, 256, 3, 3), generator=gen)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(256, 256, 3, 1, 1, 1, 1, (batch, 256, 14, 14)), False, "identity", algo="gemm")
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    packed = torch.full((op.packed_size(),), 255, dtype=torch.uint8, device="cuda:0")
    xd, fd, y = x.cuda(), f.cuda(), torch.full((batch, 256, 14, 14), float("nan"), device="cuda:0")
    op.pack(fd, packed)
    (name,) = _kernels(lambda: op.enqueue_packed(xd, fd, packed, None, y, work))
    assert name.startswith(start), name
    pick = slice(batch - 2, batch)
    want = torch.nn.functional.conv2d(x[pick].double(), f.double(), None, 1, 1)
    scale = torch.nn.functional.conv2d(x[pick].double().abs(), f.double().abs(), None, 1, 1)
    assert ((y[pick].cpu().double() - want).abs() <= scale * (256 * 9 * 2.0 ** -24)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c, start", [
    ((912, 64, 5, 1, 5, 12, 12), "conv_gemm_f32_kernel<"),         # 12 tiles of 1425 K tiles: eight slices leave most CUs without work
    ((336, 448, 5, 2, 15, 8, 8), "conv_gemm_f32_kernel<"),         # 28 of 525
    ((176, 512, 5, 2, 2, 22, 30), "conv_split_f32_kernel<64, 64,"),  # 48 of 275
    ((96, 64, 5, 1, 13, 21, 21), "conv_split_f32_kernel<64, 64,"),   # 90 of 150
], ids=str)
def test_gpu_tiles_of_64_by_slices(c, start):
    """both sides of the line where K slices of 64x64 tiles no longer fill the chip"""
    cin, cout, k, s, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f = torch.randn((b, cin, h, w), generator=gen), torch.randn((cout, cin, k, k), generator=gen)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, 1, k // 2, 1, tuple(x.shape)), False, "identity", "gemm")
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    packed = torch.full((op.packed_size(),), 255, dtype=torch.uint8, device="cuda:0")
    xd, fd = x.cuda(), f.cuda()
    op.pack(fd, packed)
    want = torch.nn.functional.conv2d(x.double(), f.double(), None, s, k // 2)
    scale = torch.nn.functional.conv2d(x.double().abs(), f.double().abs(), None, s, k // 2)
    for call in (lambda y: op.enqueue(xd, fd, None, y, work), lambda y: op.enqueue_packed(xd, fd, packed, None, y, work)):
        y = torch.full(tuple(want.shape), float("nan"), device="cuda:0")
        (name,) = _kernels(lambda: call(y))
        assert name.startswith(start), name
        # a rounding per product
        assert ((y.cpu().double() - want).abs() <= scale * ((cin * k * k + 8) * 2.0 ** -24)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c, direct", [
    ((96, 64, 19, 83, 76), False),    # 937 tiles of 54 K tiles, a second round of workgroups
    ((96, 64, 12, 83, 76), True),     # 592
    ((64, 64, 13, 83, 76), True),     # 641 of 36
    ((208, 256, 55, 23, 23), False),  # rows of 128: 912 of 117
    ((208, 256, 40, 23, 23), True),   # 664
], ids=str)
def test_gpu_automatic_choice_by_length_of_sums(c, direct):
    """both sides of the lines between Winograd and the direct kernel for long sums, filters packed"""
    cin, cout, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f = torch.randn((b, cin, h, w), generator=gen), torch.randn((cout, cin, 3, 3), generator=gen)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, 3, 1, 1, 1, 1, tuple(x.shape)), False)
    assert op.algo() == "winograd"
    work = torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
    packed = torch.full((op.packed_size(),), 255, dtype=torch.uint8, device="cuda:0")
    xd, fd, y = x.cuda(), f.cuda(), torch.full((b, cout, h, w), float("nan"), device="cuda:0")
    op.pack(fd, packed)
    names = _kernels(lambda: op.enqueue_packed(xd, fd, packed, None, y, work))
    assert [n.startswith("conv_split_f32_kernel<") for n in names] == [True] * direct, names
    want = torch.nn.functional.conv2d(x[-2:].double(), f.double(), None, 1, 1)
    scale = torch.nn.functional.conv2d(x[-2:].double().abs(), f.double().abs(), None, 1, 1)
    # Winograd's transforms round at the size of sixteen products
    assert ((y[-2:].cpu().double() - want).abs() <= scale * ((cin * 9 + 16) * 2.0 ** -24)).all()
