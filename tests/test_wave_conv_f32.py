"""Small float convolutions in tiles of 32x32 and 16x16 on the weight tensor as it lies (conv_wave_f32_kernel), against torch in 64 bits."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from test_split_gemm import _geometry, _kernels

# (cin, cout, k, stride, pad, dilate, groups, batch, h, w): tile, wavefronts a tile
CASES = {
    (224, 8, 1, 1, 0, 1, 1, 1, 1, 1): (16, 8),           # one pixel, 14 K tiles
    (237, 58, 1, 1, 0, 1, 1, 2, 9, 7): (16, 8),          # a last K tile of 13, rows of the weights off 16 bytes
    (256, 120, 1, 2, 0, 1, 1, 4, 41, 27): (32, 8),
    (300, 30, 1, 1, 1, 1, 1, 18, 17, 15): (32, 8),       # 1x1 with padding
    (17, 24, 3, 1, 1, 1, 1, 1, 13, 11): (16, 8),
    (215, 489, 3, 1, 1, 1, 1, 1, 7, 8): (16, 8),
    (512, 64, 3, 1, 1, 1, 1, 1, 7, 7): (16, 8),
    (26, 48, 3, 1, 1, 1, 1, 11, 33, 33): (32, 4),
    (96, 72, 3, 2, 1, 1, 1, 4, 29, 57): (32, 8),
    (64, 40, 3, 1, 2, 2, 1, 2, 40, 41): (32, 8),         # dilated
    (60, 46, 3, 1, 1, 1, 2, 6, 30, 30): (32, 8),         # groups, everything off the tiles
    (20, 40, 5, 1, 2, 1, 1, 3, 33, 31): (32, 8),
    (455, 256, 3, 1, 1, 1, 1, 4, 14, 14): (32, 8),       # 4095 and 6125 k: all of the 64 KB of LDS
    (245, 64, 5, 1, 2, 1, 1, 1, 7, 7): (16, 8),
}


def _tensors(c):
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    return gen, xs, ws, ys


@pytest.mark.gpu
@pytest.mark.parametrize("c", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_wave_conv_f32(c):
    cin, cout, k, s, p, d, g, b, h, w = c
    gen, xs, ws, ys = _tensors(c)
    x, f, old, bias = (torch.randn(n, generator=gen) for n in (xs, ws, ys, (cout,)))
    conv = lambda x, f: torch.nn.functional.conv2d(x.double(), f.double(), None, s, p, d, g)
    chan = bias.double().view(1, -1, 1, 1)
    # as for the other kernels on bf16 parts: a rounding per four products, and a few behind
    bound = (conv(x.abs(), f.abs()) + chan.abs() + old.double().abs() + 1) * ((cin // g * k * k / 4 + 12) * 2.0 ** -24)
    for act, first, factor in (("relu6", False, 0.0), ("identity", True, 0.5), ("tanh", False, -2.0)):
        op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), True, act, "gemm")
        op.accumulate_before_activation(first)
        work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
        y = old.cuda() if factor else torch.full(ys, float("nan"), device="cuda:0")
        (name,) = _kernels(lambda: op.enqueue(x.cuda(), f.cuda(), bias.cuda(), y, work, factor))
        assert name.startswith("conv_wave_f32_kernel<%d, %d, " % CASES[c]), name
        v = conv(x, f) + chan
        res = {"relu6": lambda: v.clamp(0, 6), "identity": lambda: v + factor * old.double(), "tanh": lambda: v.tanh() + factor * old.double()}[act]()
        assert ((y.cpu().double() - res).abs() <= bound + (4e-7 if act == "tanh" else 0)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(456, 256, 3, 1, 1, 1, 1, 4, 14, 14), (246, 64, 5, 1, 2, 1, 1, 1, 7, 7), (256, 256, 5, 1, 2, 1, 1, 1, 10, 10)],
                         ids=lambda c: "x".join(map(str, c)))
def test_gpu_wave_conv_f32_longer_reductions(c):
    """more k than the table has room for: the other kernels"""
    cin, cout, k, s, p, d, g, b, h, w = c
    gen, xs, ws, ys = _tensors(c)
    x, f = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), False, "identity", "gemm")
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    y = torch.full(ys, float("nan"), device="cuda:0")
    names = _kernels(lambda: op.enqueue(x.cuda(), f.cuda(), None, y, work))
    assert names and not any(n.startswith("conv_wave_f32_kernel") for n in names), names
    conv = lambda x, f: torch.nn.functional.conv2d(x.double(), f.double(), None, s, p, d, g)
    # a rounding per product
    assert ((y.cpu().double() - conv(x, f)).abs() <= conv(x.abs(), f.abs()) * ((cin * k * k + 8) * 2.0 ** -24)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c, packed, wave", [
    ((18, 128, 3, 1, 1, 1, 1, 4, 56, 56), True, False),     # 1568 tiles of 11 K tiles
    ((18, 128, 3, 1, 1, 1, 1, 2, 56, 56), True, True),
    ((25, 192, 3, 1, 1, 1, 1, 16, 14, 71), False, False),   # 2982 of 15
    ((154, 256, 3, 2, 1, 1, 1, 16, 68, 8), False, False),   # strided
    ((1024, 256, 1, 2, 0, 1, 1, 6, 28, 28), False, False),
    ((1024, 256, 1, 2, 0, 1, 1, 2, 28, 28), False, True),
], ids=str)
def test_gpu_wave_conv_f32_lines(c, packed, wave):
    """calls on either side of the lines to the other kernels"""
    cin, cout, k, s, p, d, g, b, h, w = c
    gen, xs, ws, ys = _tensors(c)
    x, f = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), False, "identity", "gemm")
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    y, xd, fd = torch.full(ys, float("nan"), device="cuda:0"), x.cuda(), f.cuda()
    buf = torch.empty(op.packed_size(), dtype=torch.uint8, device="cuda:0")
    op.pack(fd, buf)
    names = _kernels(lambda: op.enqueue_packed(xd, fd, buf, None, y, work) if packed else op.enqueue(xd, fd, None, y, work))
    assert len(names) == 1 and names[0].startswith("conv_wave_f32_kernel") == wave, names
    conv = lambda x, f: torch.nn.functional.conv2d(x.double(), f.double(), None, s, p, d, g)
    # a rounding per product
    assert ((y.cpu().double() - conv(x, f)).abs() <= conv(x.abs(), f.abs()) * ((cin * k * k + 8) * 2.0 ** -24)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c, packed, algo, wave", [
    ((16, 64, 3, 1, 1, 1, 1, 2, 140, 140), False, "gemm", False),  # 2450 tiles
    ((16, 64, 3, 1, 1, 1, 1, 1, 140, 140), False, "gemm", True),
    ((16, 48, 3, 1, 1, 1, 1, 1, 160, 160), False, "gemm", False),  # 1600
    ((16, 64, 3, 1, 1, 1, 1, 2, 140, 140), False, "", True),       # Winograd otherwise
    ((16, 48, 3, 1, 1, 1, 1, 2, 81, 81), True, "gemm", False),     # 822
    ((16, 48, 3, 1, 1, 1, 1, 1, 81, 81), True, "gemm", True),
    ((16, 48, 3, 1, 1, 1, 1, 4, 56, 56), True, "gemm", True),      # the LDS-patch kernel otherwise
], ids=str)
def test_gpu_wave_conv_f32_wide_images(c, packed, algo, wave):
    """3x3 of 16 channels: both sides of the lines to the gathering kernel, whole numbers, exact in any order"""
    cin, cout, k, s, p, d, g, b, h, w = c
    gen, xs, ws, ys = _tensors(c)
    x, f = torch.randint(-3, 4, xs, generator=gen).float(), torch.randint(-3, 4, ws, generator=gen).float()
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), False, "identity", algo)
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    y, xd, fd = torch.full(ys, float("nan"), device="cuda:0"), x.cuda(), f.cuda()
    buf = torch.empty(op.packed_size(), dtype=torch.uint8, device="cuda:0")
    op.pack(fd, buf)
    (name,) = _kernels(lambda: op.enqueue_packed(xd, fd, buf, None, y, work) if packed else op.enqueue(xd, fd, None, y, work))
    assert name.startswith("conv_wave_f32_kernel") == wave, name
    assert torch.equal(y.cpu(), torch.nn.functional.conv2d(x, f, None, s, p))


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(237, 58, 1, 1, 0, 1, 1, 2, 9, 7), (26, 48, 3, 1, 1, 1, 1, 11, 33, 33)], ids=lambda c: "x".join(map(str, c)))
def test_gpu_wave_conv_f32_special_values(c):
    """infinities, NaN, operands near the ends of the range: what the fp32 sum of the products is"""
    cin, cout, k, s, p, d, g, b, h, w = c
    gen, xs, ws, ys = _tensors(c)
    x0, f0 = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), False, "identity", "gemm")
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    conv = lambda x, f: torch.nn.functional.conv2d(x.double(), f.double(), None, s, p, d, g)

    def run(x, f):
        y = torch.full(ys, 5.0, device="cuda:0")
        op.enqueue(x.cuda(), f.cuda(), None, y, work)
        return y.cpu().double()

    one_x, one_f = x0.clone(), f0.clone()
    one_x[:, :, h // 2] *= 2.0 ** -120
    one_f[3] *= 2.0 ** -120
    for x, f in [(x0 * 2.0 ** -120, f0 * 2.0 ** 60), (x0 * 2.0 ** 60, f0 * 2.0 ** -120), (x0 * 2.0 ** 55, f0 * 2.0 ** 55), (one_x, f0), (x0, one_f)]:
        want, got = conv(x, f), run(x, f)
        assert ((got - want).abs() <= conv(x.abs(), f.abs()) * ((cin // g * k * k + 8) * 2.0 ** -24)).all()
        assert (got[:, 3] - want[:, 3]).norm() <= want[:, 3].norm() * 2.0 ** -20
    f = f0.abs() + 0.5
    for value in (float("inf"), float("-inf"), float("nan"), 3.4e38):
        x = x0.clone()
        x[0, 1, 0, 0] = x[1, cin - 1, h // 2, w // 2] = value
        want, got = conv(x, f).float().double(), run(x, f)
        for test in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(test(got), test(want)), value
        assert torch.equal(run(x * 0, f), conv(x * 0, f).float().double()) or value != 3.4e38


@pytest.mark.gpu
def test_gpu_wave_conv_f32_automatic_choice():
    """an operator whose algorithm was left open runs small batches directly, also with its weights transformed ahead; one asked for by name does not"""
    xs, ws = (1, 64, 32, 32), (64, 64, 3, 3)
    gen = torch.Generator().manual_seed(1)
    x, f = torch.randint(-4, 5, xs, generator=gen).float(), torch.randint(-4, 5, ws, generator=gen).float()
    want = torch.nn.functional.conv2d(x, f, None, 1, 1)
    for algo, batch, section in (("", 64, "conv_gemm"), ("winograd", 64, "winograd_fused")):
        op = dlp.Conv2DForward.create(dlp.Conv2DSettings(64, 64, 3, 1, 1, 1, 1, (batch,) + xs[1:]), False, "identity", algo)
        assert op.algo() == "winograd"
        work = torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
        packed = torch.empty(op.packed_size(), dtype=torch.uint8, device="cuda:0")
        op.pack(f.cuda(), packed)
        for call in (lambda y: op.enqueue(x.cuda(), f.cuda(), None, y, work), lambda y: op.enqueue_packed(x.cuda(), f.cuda(), packed, None, y, work)):
            y = torch.full(xs, float("nan"), device="cuda:0")
            assert len(_kernels(lambda: call(y), section)) == 1
            assert (y.cpu() - want).abs().max() <= 2e-3 and (algo or torch.equal(y.cpu(), want))


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(512, 512, 3, 1, 1, 1, 1, 1, 7, 7), (60, 46, 3, 1, 1, 1, 2, 6, 30, 30), (256, 120, 1, 2, 0, 1, 1, 4, 41, 27)],
                         ids=lambda c: "x".join(map(str, c)))
def test_gpu_wave_conv_f32_large_operands(c):
    """operands above 2^16 in every tile: the fp32 sums, in little more time than others take (the tile again on the fp32 instruction; one thread an
    output, a product at a time, took 11 to 34 times as long)"""
    cin, cout, k, s, p, d, g, b, h, w = c
    gen, xs, ws, ys = _tensors(c)
    x, f = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
    large = x.clone()
    large[:, 1::2] *= 2.0 ** 17
    conv = lambda x, f: torch.nn.functional.conv2d(x.double(), f.double(), None, s, p, d, g)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), False, "identity", "gemm")
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    y, fd, times = torch.full(ys, float("nan"), device="cuda:0"), f.cuda(), []
    for v in (x, large):
        vd = v.cuda()
        (name,) = _kernels(lambda: op.enqueue(vd, fd, None, y, work))
        assert name.startswith("conv_wave_f32_kernel"), name
        # a rounding per product
        assert ((y.cpu().double() - conv(v, f)).abs() <= conv(v.abs(), f.abs()) * ((cin // g * k * k + 8) * 2.0 ** -24)).all()
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        for _ in range(50):
            op.enqueue(vd, fd, None, y, work)
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end))
    assert times[1] <= 8 * times[0], times
