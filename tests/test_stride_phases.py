"""All stride phases of a backward-data pass or transposed convolution as one launch (conv_phases_f32_kernel, conv_split_f32_kernel on
PhasesArgs), against torch in 64 bits."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from test_split_gemm import _geometry, _kernels

# (cin, cout, k, stride, pad, dilate, groups, batch, h, w) of the convolution whose data gradient is taken
CASES = [
    (64, 16, 2, 2, 0, 1, 1, 1, 2, 2),       # one pixel and one K tile a phase
    (40, 32, 4, 2, 1, 1, 1, 3, 18, 22),     # rows off the tile
    (33, 48, 3, 2, 1, 1, 1, 2, 15, 13),     # rows off multiples of 8; phases of four extents
    (16, 512, 3, 2, 1, 1, 1, 2, 21, 20),    # K slices
    (65, 256, 5, 2, 2, 1, 1, 1, 9, 30),     # K slices, ragged
    (48, 32, 3, 3, 0, 1, 1, 2, 12, 15),     # nine phases of one tap each
    (24, 32, 5, 3, 2, 1, 2, 2, 17, 19),     # groups
    (32, 64, 3, 2, 2, 3, 1, 2, 17, 19),     # dilated taps
    (129, 32, 4, 2, 1, 1, 1, 32, 56, 54),   # tiles of 64 rows x 128 pixels, ragged
    (200, 48, 4, 2, 1, 1, 1, 32, 56, 54),   # tiles of 128x128
]
MERGED = ("conv_phases_f32_kernel", "conv_split_f32_kernel")


@pytest.mark.gpu
@pytest.mark.parametrize("c", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_phases_in_one_launch(c):
    cin, cout, k, s, p, d, g, b, h, w = c
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    f, dy, bias, old = (torch.randn(n, generator=gen) for n in (ws, ys, (cin,), xs))
    extra = tuple(n - ((o - 1) * s - 2 * p + d * (k - 1) + 1) for n, o in zip(xs[2:], ys[2:]))
    back = lambda y, v: torch.nn.functional.conv_transpose2d(y.double(), v.double(), None, s, p, extra, g, d)
    chan = bias.double().view(1, -1, 1, 1)
    want = back(dy, f)
    bound = (back(dy.abs(), f.abs()) + chan.abs() + 2 * old.double().abs()) * ((cout // g * k * k / 4 + 10) * 2.0 ** -24)
    op = dlp.Conv2DBackwardData.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), "gemm")
    tr = dlp.TransposedConv2DForward.create(dlp.Conv2DSettings(cout, cin, k, s, d, p, g, ys), extra, True, "relu6", "gemm")
    full = op.workspace()
    work = torch.full((full,), 255, dtype=torch.uint8, device="cuda:0")
    for factor in (0.0, 2.0):
        dx = old.cuda() if factor else torch.full(xs, float("nan"), device="cuda:0")
        names = _kernels(lambda: op.enqueue(dx, f.cuda(), dy.cuda(), work, factor))
        assert len(names) == 1 and names[0].startswith(MERGED), names
        assert ((dx.cpu().double() - want - factor * old.double()).abs() <= bound).all()
    y = torch.full(xs, float("nan"), device="cuda:0")
    tr.enqueue(dy.cuda(), f.cuda(), bias.cuda(), y, torch.empty(tr.workspace(), dtype=torch.uint8, device="cuda:0"))
    assert ((y.cpu().double() - (want + chan).clamp(0, 6)).abs() <= bound).all()
    # an infinity: its tiles are computed again, the others keep their values
    dy[0, 0, 0, 0] = float("inf")
    op.enqueue(dx, f.cuda(), dy.cuda(), work, 0.0)
    got, want = dx.cpu().double(), back(dy, f.abs())
    reached = ~torch.isfinite(want)
    assert (~torch.isfinite(got)[reached]).all() and torch.isfinite(got)[~reached].all()


@pytest.mark.gpu
def test_gpu_phases_with_a_small_workspace_and_in_a_graph():
    """whole numbers, exact in any order: as many K slices as there is room for; replays of a capture repeat the result"""
    c = (64, 256, 4, 2, 1, 1, 1, 2, 18, 18)
    gen = torch.Generator().manual_seed(5)
    xs, ws, ys = _geometry(c)
    f, dy = (torch.randint(-3, 4, n, generator=gen).float() for n in (ws, ys))
    want = torch.nn.functional.conv_transpose2d(dy.double(), f.double(), None, 2, 1)
    op = dlp.Conv2DBackwardData.create(dlp.Conv2DSettings(64, 256, 4, 2, 1, 1, 1, xs), "gemm")
    fd, dyd = f.cuda(), dy.cuda()
    sizes = [op.workspace(), op.workspace() - 256]
    for room in sizes + [op.workspace() * 3 // 4, op.workspace() // 2]:
        dx = torch.full(xs, float("nan"), device="cuda:0")
        try:
            op.enqueue(dx, fd, dyd, torch.empty(room, dtype=torch.uint8, device="cuda:0"))
        except dlp.ValidationError:
            assert room not in sizes
            continue
        assert torch.equal(dx.cpu().double(), want), room
    work = torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        op.enqueue(dx, fd, dyd, work)
    for _ in range(3):
        dx.fill_(float("nan"))
        work.fill_(171)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(dx.cpu().double(), want)
