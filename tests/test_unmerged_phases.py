"""Stride phases that run one by one (an activation that the one launch of all phases does not have): which kernels serve them, and the sums."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from test_split_gemm import _kernels


# (cin, cout, k, pad, output pad, batch, h): phases on the small-tile kernel
CASES = {
    (128, 64, 3, 1, 1, 16, 28): 0,  # 32, 16, 16 and 8 K tiles a phase
    (64, 32, 6, 2, 0, 16, 32): 4,   # four of 36
    (256, 40, 1, 0, 1, 4, 14): 1,   # one phase of one tap
}


@pytest.mark.gpu
@pytest.mark.parametrize("c", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_phases_one_by_one(c):
    cin, cout, k, p, extra, b, h = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f, bias = torch.randn((b, cin, h, h), generator=gen), torch.randn((cin, cout, k, k), generator=gen), torch.randn(cout, generator=gen)
    x, bias = x / (cin * k * k / 4) ** 0.5, bias / 4
    op = dlp.TransposedConv2DForward.create(dlp.Conv2DSettings(cin, cout, k, 2, 1, p, 1, tuple(x.shape)), (extra, extra), True, "tanh")
    y = torch.full(op.output_shape(tuple(x.shape)), float("nan"), device="cuda:0")
    work = torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
    names = _kernels(lambda: op.enqueue(x.cuda(), f.cuda(), bias.cuda(), y, work))
    assert sum(n.startswith("conv_wave_f32_kernel") for n in names) == CASES[c], names
    back = lambda x, f: torch.nn.functional.conv_transpose2d(x.double(), f.double(), None, 2, p, extra)
    chan = bias.double().view(1, -1, 1, 1)
    # a rounding per product ahead of tanh, which shrinks every difference, and a few of its own
    bound = (back(x.abs(), f.abs()) + chan.abs()) * ((cin * k * k + 8) * 2.0 ** -24) + 4e-7
    assert ((y.cpu().double() - (back(x, f) + chan).tanh()).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c, merged", [((8, 128, 6, 2, 64, 56), False), ((8, 128, 6, 2, 32, 56), True), ((32, 128, 5, 2, 136, 56), False), ((33, 128, 6, 2, 64, 56), True)], ids=str)
def test_gpu_few_rows(c, merged):
    """at most 32 rows leave half of a tile of the one launch empty, which large calls do not take: whole numbers, exact in any order (Winograd's: rounded)"""
    cin, cout, k, p, b, h = c
    gen = torch.Generator().manual_seed(sum(c))
    oh = (h + 2 * p - k) // 2 + 1
    f, dy = (torch.randint(-2, 3, n, generator=gen).float() for n in ((cout, cin, k, k), (b, cout, oh, oh)))
    op = dlp.Conv2DBackwardData.create(dlp.Conv2DSettings(cin, cout, k, 2, 1, p, 1, (b, cin, h, h)))
    dx, work = torch.full((b, cin, h, h), float("nan"), device="cuda:0"), torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
    dlp.timing_enable(True)
    dlp.timing_reset()
    try:
        op.enqueue(dx, f.cuda(), dy.cuda(), work)
        sections = [s for s, _ in dlp.timing_records()]
    finally:
        dlp.timing_enable(False)
        dlp.timing_reset()
    assert ("bwd_data_interleave" not in sections) == merged, sections
    pick = slice(b - 2, b)
    extra = h - ((oh - 1) * 2 - 2 * p + k)
    want = torch.nn.functional.conv_transpose2d(dy[pick], f, None, 2, p, extra)
    # Winograd's transforms: values of up to four times the operands', in sums of every channel
    bound = 0.0 if merged else cout * 4 * 9 * 2.0 ** -20
    assert (dx[pick].cpu() - want).abs().max() <= bound


@pytest.mark.gpu
@pytest.mark.parametrize("c, merged", [((176, 8, 4, 1, 0, 48, 43, 30), False), ((176, 8, 4, 1, 0, 24, 43, 30), True), ((192, 24, 5, 2, 1, 13, 64, 64), False), ((192, 24, 5, 2, 1, 9, 64, 64), True),
                                       ((32, 3, 4, 1, 0, 44, 92, 92), False)], ids=str)
def test_gpu_few_filters(c, merged):
    """... and up to 16 rows leave three quarters of it empty: whole numbers, exact in any order"""
    cin, cout, k, p, extra, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    x, f = torch.randint(-2, 3, (b, cin, h, w), generator=gen).float(), torch.randint(-2, 3, (cin, cout, k, k), generator=gen).float()
    op = dlp.TransposedConv2DForward.create(dlp.Conv2DSettings(cin, cout, k, 2, 1, p, 1, tuple(x.shape)), (extra, extra), False, "identity", "gemm")
    y = torch.full(op.output_shape(tuple(x.shape)), float("nan"), device="cuda:0")
    work = torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
    names = _kernels(lambda: op.enqueue(x.cuda(), f.cuda(), None, y, work))
    assert (len(names) == 1) == merged, names
    pick = slice(b - 2, b)
    assert torch.equal(y[pick].cpu(), torch.nn.functional.conv_transpose2d(x[pick], f, None, 2, p, extra))
