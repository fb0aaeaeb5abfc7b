"""fp32 convolutions on the bf16 matrix instruction (conv_split_f32_kernel: three bf16 parts per operand) at the sizes where its tiles,
K slices and masks can go wrong, against torch in 64 bits."""
import pytest
import torch

import dlprimitives_amd as dlp


def _geometry(c):
    cin, cout, k, s, p, d, g, b, h, w = c
    oh, ow = ((n + 2 * p - d * (k - 1) - 1) // s + 1 for n in (h, w))
    return (b, cin, h, w), (cout, cin // g, k, k), (b, cout, oh, ow)


def _run(c, x, w, bias, packed, act="identity", factor=0.0, y0=None, shift=0, hint=None, first=False, room=None):
    cin, cout, k, s, p, d, g, b, h, wd = c
    xs, ws_, ys = _geometry(c)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, ((hint or b),) + xs[1:]), bias is not None, act, "gemm")
    if first:
        op.accumulate_before_activation(True)
    wbuf = torch.empty(w.numel() + shift, device="cuda:0")  # shift: a weight tensor off its 16-byte boundary
    wbuf[shift:].copy_(w.reshape(-1))
    wdev = wbuf[shift:].view(ws_)
    y = torch.full(ys, float("nan"), device="cuda:0") if y0 is None else y0.float().cuda()
    ws = torch.empty(max(op.workspace(), 1) if room is None else room, dtype=torch.uint8, device="cuda:0")
    bd = None if bias is None else bias.float().cuda()
    if packed:
        buf = torch.empty(max(op.packed_size(), 1), dtype=torch.uint8, device="cuda:0")
        op.pack(wdev, buf)
        op.enqueue_packed(x.float().cuda(), wdev, buf, bd, y, ws, factor)
    else:
        op.enqueue(x.float().cuda(), wdev, bd, y, ws, factor)
    torch.cuda.synchronize()
    return y.cpu().double()


def _conv64(c, x, w, bias):
    cin, cout, k, s, p, d, g, b, h, wd = c
    return torch.nn.functional.conv2d(x.double(), w.double(), None if bias is None else bias.double(), s, p, d, g)


def _kernels(f, section="conv_gemm"):
    """names of the kernels that f launches in a section of the timing records"""
    dlp.timing_enable(True)
    dlp.timing_reset()
    try:
        f()
        return [k for s, _, k in dlp.timing_records(kernels=True) if s == section]
    finally:
        dlp.timing_enable(False)
        dlp.timing_reset()


def _tile(names):
    """rows of the tiles of the one launch, which is one of conv_split_f32_kernel<rows, pixels, wavefronts, weights in place, ..>"""
    (name,) = names
    assert name.startswith("conv_split_f32_kernel<"), name
    args = name[name.index("<") + 1:].split(", ")
    return int(args[0]), args[4] == "true"


# every one large enough for these kernels: 350 tiles of 64 filters x 128 pixels, or 20000 K tiles in all
# (cin, cout, k, stride, pad, dilate, groups, batch, h, w)
CASES = [
    (16, 64, 1, 1, 0, 1, 1, 32, 38, 38),     # one K tile, 64x128 tiles
    (16, 33, 1, 1, 0, 1, 1, 47, 31, 33),     # rows and pixels off the tile
    (32, 80, 1, 2, 0, 1, 1, 90, 31, 33),     # two tiles of 64 rows, the second mostly empty; strided
    (48, 128, 1, 1, 0, 1, 1, 32, 38, 38),    # 128x128 tiles, three K tiles
    (16, 200, 3, 1, 1, 1, 1, 20, 31, 30),    # rows off 64, taps outside the image
    (16, 97, 3, 2, 1, 1, 1, 64, 39, 41),
    (64, 64, 3, 1, 1, 1, 1, 16, 53, 53),     # a last round of few tiles, cut into K slices
    (192, 96, 3, 1, 1, 1, 1, 5, 61, 43),     # K slices throughout
    (640, 128, 3, 1, 1, 1, 1, 5, 27, 27),
    (32, 48, 5, 1, 4, 2, 1, 40, 31, 33),     # dilation
    (64, 320, 3, 1, 1, 1, 4, 9, 33, 31),     # groups
    (16, 40, 5, 3, 0, 1, 1, 81, 75, 75),
    (64, 128, 3, 1, 1, 1, 1, 16, 53, 53),    # 128x128 tiles: filter taps outside the image
    (32, 200, 3, 1, 1, 1, 1, 25, 31, 30),    # ... rows off 128
    (256, 96, 3, 1, 1, 1, 1, 10, 37, 37),    # ... K slices, rows off 128
    (128, 512, 1, 1, 0, 1, 4, 16, 33, 33),   # ... groups
    (64, 160, 1, 1, 0, 1, 2, 21, 33, 33),    # ... groups whose rows are off 128
]
ROWS = {c: 128 for c in CASES[-5:]}
ROWS[(48, 128, 1, 1, 0, 1, 1, 32, 38, 38)] = 128
SLICES = {(64, 64, 3, 1, 1, 1, 1, 16, 53, 53), (64, 128, 3, 1, 1, 1, 1, 16, 53, 53), (32, 48, 5, 1, 4, 2, 1, 40, 31, 33), (192, 96, 3, 1, 1, 1, 1, 5, 61, 43),
          (640, 128, 3, 1, 1, 1, 1, 5, 27, 27), (256, 96, 3, 1, 1, 1, 1, 10, 37, 37)}


def _bounds(want, scale, k):
    """elementwise and in the 2-norm"""
    # a product is off by 2^-23 at most; the sums, none above sum |x||w|, round by 2^-24 of themselves once per four k and a few times behind
    each = scale * ((k / 4 + 8) * 2.0 ** -24)
    # roundings of either sign add up as their squares: sqrt(K / 4) of them, each a third of 2^-24 or so of a sum that has grown to sqrt(K)
    # products, stay below 2^-22 of the result up to K = 6000; a piece too few would show as 2^-17, a lost small product as 2^-17 to 2^-9
    return each, want.norm() * 2.0 ** -22


def _parts(t):
    """a float as three bf16 numbers, as the kernels cut it"""
    out = []
    rest = t.float()
    for _ in range(3):
        out.append(rest.bfloat16().float())
        rest = rest - out[-1]
    assert not rest.any()
    return [p.double() for p in out]


def test_bounds_see_a_lost_product():
    """the parity bounds hold for the six products of the kernels and for no five of them, nor with two parts exchanged"""
    gen = torch.Generator().manual_seed(1)
    kept = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]
    for k in (16, 144, 1728):
        a, b = torch.randn((96, k), generator=gen), torch.randn((k, 80), generator=gen)
        pa, pb = _parts(a), _parts(b)
        want, scale = a.double() @ b.double(), a.double().abs() @ b.double().abs()
        each, norm = _bounds(want, scale, k)
        holds = lambda pairs: bool(((sum(pa[i] @ pb[j] for i, j in pairs) - want).abs() <= each).all()) and (sum(pa[i] @ pb[j] for i, j in pairs) - want).norm() <= norm
        assert holds(kept)
        for lost in kept:
            assert not holds([p for p in kept if p != lost])
        assert not holds([(0, 0), (0, 2), (1, 0), (1, 2), (0, 1), (2, 0)])  # second and third part of b in each other's place


def test_parts_of_small_floats():
    """three bf16 numbers hold a float from 2^-110 on, below it they lose bits"""
    gen = torch.Generator().manual_seed(2)
    t = (torch.rand(4096, generator=gen) + 1) * torch.where(torch.rand(4096, generator=gen) < 0.5, -1.0, 1.0)
    for e in (-110, -100, 0, 126):
        x = t * 2.0 ** e
        assert torch.equal(sum(_parts(x)), x.double())
    lost = 0
    rest = t * 2.0 ** -111
    for _ in range(3):
        rest = rest - rest.bfloat16().float()
    assert rest.any()


@pytest.mark.gpu
@pytest.mark.parametrize("mode,c", [(m, c) for m in ("packed", "raw", "in_place") for c in CASES if m != "in_place" or c[2] == 1],  # 1x1: read in place
                         ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_gpu_split_parity(mode, c):
    packed, shift = mode == "packed", int(mode == "raw")
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    x, w, bias = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen), torch.randn(c[1], generator=gen)
    want = _conv64(c, x, w, bias)
    got = []
    names = _kernels(lambda: got.append(_run(c, x, w, bias, packed, shift=shift)))
    assert _tile(names) == (ROWS.get(c, 64), mode == "in_place")
    got = got[0]
    scale = _conv64(c, x.abs(), w.abs(), bias.abs())
    each, norm = _bounds(want, scale, w[0].numel())
    assert ((got - want).abs() <= each).all()
    assert (got - want).norm() <= norm
    if packed:  # without a workspace there is one slice: other bits where there are more
        assert torch.equal(_run(c, x, w, bias, True, room=0), got) == (c not in SLICES)
    old = torch.randn(ys, generator=gen)
    for first in (False, True):
        got = _run(c, x, w, None, packed, "relu", 0.5, old, shift=shift, first=first)
        want = _conv64(c, x, w, None)
        want = (want + 0.5 * old.double()).relu() if first else want.relu() + 0.5 * old.double()
        assert ((got - want).abs() <= each + old.abs() * 2.0 ** -22).all()


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["identity", "relu", "relu6"])
@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("c", [(16, 64, 1, 1, 0, 1, 1, 32, 38, 38), (48, 248, 1, 1, 0, 1, 1, 32, 38, 38), (16, 33, 1, 1, 0, 1, 1, 47, 31, 33), (64, 500, 1, 1, 0, 1, 2, 33, 38, 38),
                               (32, 100, 3, 1, 1, 1, 1, 3, 9, 11)], ids=lambda c: "x".join(map(str, c)))
def test_gpu_residual_sums(c, first, act):
    """factor * y before and behind the activation: rows in whole eights and not, tiles of 64 and 128 rows, the fp32 instruction (last)"""
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    x, w, bias = torch.randint(-3, 4, xs, generator=gen).float(), torch.randint(-3, 4, ws, generator=gen).float(), torch.randint(-9, 10, (c[1],), generator=gen).float()
    old = torch.randint(-9, 10, ys, generator=gen).float()
    f = {"identity": lambda t: t, "relu": torch.relu, "relu6": lambda t: t.clamp(0, 6)}[act]
    conv = _conv64(c, x, w, bias)
    want = f(conv - 2 * old.double()) if first else f(conv) - 2 * old.double()
    assert torch.equal(_run(c, x, w, bias, True, act, -2.0, old, first=first), want)  # whole numbers are exact


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("c", [(32, 64, 1, 1, 0, 1, 1, 32, 38, 38), (48, 128, 1, 1, 0, 1, 1, 32, 38, 38), (192, 96, 3, 1, 1, 1, 1, 5, 61, 43),
                               (256, 96, 3, 1, 1, 1, 1, 10, 37, 37)], ids=["64x128", "128x128", "slices", "128x128 slices"])
def test_gpu_split_not_finite(c, packed):
    """infinities, NaN and values next to the largest float come out as the definition has them"""
    gen = torch.Generator().manual_seed(5)
    xs, ws, ys = _geometry(c)
    x, w = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
    x[0, 3, 4, 5], x[0, 7, 20, 9], x[1, 1, 30, 30], x[2, 2, 11, 3] = float("inf"), float("-inf"), float("nan"), 3.4e38
    w[:, 2] *= 1e-3  # the products with 3.4e38 stay finite
    want = _conv64(c, x, w, None)
    got = _run(c, x, w, None, packed)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isposinf(got), torch.isposinf(want))
    assert torch.equal(torch.isneginf(got), torch.isneginf(want))
    scale = _conv64(c, torch.nan_to_num(x, 0.0, 0.0, 0.0).abs(), w.abs(), None)
    ok = torch.isfinite(want)
    assert ((got - want).abs()[ok] <= scale[ok] * 2.0 ** -18).all()  # an fp32 sum of K terms where the tile is computed again
    w[3, 1], w[5, 2], w[9, 0] = float("inf"), float("nan"), 3.4e38
    x = torch.rand(xs, generator=gen) * 1e-3 + 1e-3
    want = _conv64(c, x, w, None)
    got = _run(c, x, w, None, packed)
    inside = (slice(None), slice(None), slice(1, -1), slice(1, -1))  # (infinity times the padding's zeros is left to either)
    for f in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(f(got[inside]), f(want[inside]))


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["packed", "raw", "in_place"])
@pytest.mark.parametrize("c", [(32, 64, 1, 1, 0, 1, 1, 32, 38, 38), (48, 128, 1, 1, 0, 1, 1, 32, 38, 38), (192, 96, 3, 1, 1, 1, 1, 5, 61, 43)],
                         ids=["64x128", "128x128", "slices"])
def test_gpu_split_small_operands(c, mode):
    """operands too small for three bf16 parts (a float below 2^-110 is no multiple of the smallest bf16 number, 2^-133) lose nothing"""
    gen = torch.Generator().manual_seed(11)
    xs, ws, ys = _geometry(c)
    x0, w0 = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
    k = w0[0].numel()

    def check(x, w):
        got, want = _run(c, x, w, None, mode == "packed", shift=int(mode == "raw")), _conv64(c, x, w, None)
        scale = _conv64(c, x.abs(), w.abs(), None)
        # the fp32 instruction rounds once per product; the last bits of 2^-120 lost would show as 2^-15
        assert ((got - want).abs() <= scale * ((k + 8) * 2.0 ** -24)).all()
        assert (got - want).norm() <= want.norm() * 2.0 ** -19

    check(x0 * 2.0 ** -120, w0 * 2.0 ** 60)
    check(x0 * 2.0 ** 60, w0 * 2.0 ** -120)
    x, w = x0.clone(), w0.clone()
    x[:, 3] *= 2.0 ** -120  # one channel of the input, as large in the sums as the others
    w[:, 3] *= 2.0 ** 120
    check(x, w)
    x, w = x0.clone(), w0.clone()
    x[:, 5] *= 2.0 ** 120
    w[:, 5] *= 2.0 ** -120
    w[7] *= 2.0 ** -115  # and a filter that is small throughout
    check(x, w)
    x = x0.clone()
    x[1, 2, 3, 4] = 2.0 ** -149  # one operand of one tile: the tile is computed again, its neighbours are not
    check(x, w0)


@pytest.mark.gpu
def test_gpu_split_other_batches():
    """weights packed at the batch of the settings stay valid at others"""
    c = (192, 96, 3, 1, 1, 1, 1, 5, 61, 43)
    gen = torch.Generator().manual_seed(6)
    for batch in (1, 4, 9):
        cb = c[:7] + (batch,) + c[8:]
        xs, ws, _ = _geometry(cb)
        x, w = torch.randint(-4, 5, xs, generator=gen).float(), torch.randint(-4, 5, ws, generator=gen).float()
        for packed in (False, True):
            assert torch.equal(_run(cb, x, w, None, packed, hint=5), _conv64(cb, x, w, None))  # whole numbers are exact


# (cin, cout, k, stride, pad, h, batch of the settings, batch of the call): on either side of the lines between the kernels at the
# call's batch, weights packed for 128 rows run in tiles of 64 and in fp32 tiles (of 64 and of 32 rows, stream and slices)
OTHER = [(128, 128, 3, 1, 1, 28, 64, 64), (128, 128, 3, 1, 1, 28, 64, 20), (128, 128, 3, 1, 1, 28, 64, 5), (512, 512, 3, 1, 1, 7, 64, 33),
         (128, 200, 3, 2, 1, 28, 64, 40), (128, 200, 3, 2, 1, 28, 64, 3), (64, 256, 1, 1, 0, 56, 32, 8), (64, 256, 1, 1, 0, 56, 32, 1),
         (256, 96, 1, 1, 0, 28, 64, 60), (256, 96, 1, 1, 0, 28, 64, 2), (48, 80, 5, 1, 2, 35, 9, 9), (48, 80, 5, 1, 2, 35, 9, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("c", OTHER, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("packed", [False, True])
def test_gpu_kernel_of_the_call_s_batch(c, packed):
    """an operator runs the kernel at any batch that one created for that batch runs, on weights packed once"""
    cin, cout, k, s, p, h, hint, batch = c
    cb = (cin, cout, k, s, p, 1, 1, batch, h, h)
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, _ = _geometry(cb)
    x, w, bias = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen), torch.randn(cout, generator=gen)
    out = {}
    names = {n: _kernels(lambda: out.update({n: _run(cb, x, w, bias, packed, shift=1, hint=n)})) for n in (hint, batch)}
    assert names[hint] == names[batch] and len(names[hint]) == 1
    want, scale = _conv64(cb, x, w, bias), _conv64(cb, x.abs(), w.abs(), bias.abs())
    for n in (hint, batch):
        # fp32 sums of K products, one rounding each
        assert ((out[n] - want).abs() <= scale * ((w[0].numel() + 8) * 2.0 ** -24)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("c", [(512, 512, 3, 1, 1, 7, 64), (128, 128, 3, 1, 1, 28, 64), (64, 128, 3, 2, 1, 56, 64), (256, 512, 3, 2, 1, 14, 64), (1024, 256, 1, 1, 0, 14, 64),
                               (48, 80, 5, 1, 2, 21, 33)], ids=lambda c: "x".join(map(str, c)))
def test_gpu_slices_of_the_call_s_batch(c, packed):
    """a workspace sized for the batch of the settings has room for the K slices of every smaller one: the same bits as from an operator
    created for that batch (another cut adds up in another order)"""
    cin, cout, k, s, p, h, hint = c
    gen = torch.Generator().manual_seed(sum(c))
    for batch in sorted({1, 2, 3, 5, 8, 12, 16, 21, hint // 2, hint - 9, hint - 1}):
        cb = (cin, cout, k, s, p, 1, 1, batch, h, h)
        xs, ws, _ = _geometry(cb)
        x, w = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
        assert torch.equal(_run(cb, x, w, None, packed, hint=hint), _run(cb, x, w, None, packed)), batch


@pytest.mark.gpu
def test_gpu_split_small_workspaces():
    """as many K slices as there is room for, fp32 tiles where the split ones find none, an error below that"""
    c = (192, 96, 3, 1, 1, 1, 1, 5, 61, 43)
    gen = torch.Generator().manual_seed(3)
    xs, ws, ys = _geometry(c)
    x, w = torch.randint(-4, 5, xs, generator=gen).float(), torch.randint(-4, 5, ws, generator=gen).float()
    want = _conv64(c, x, w, None)
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(192, 96, 3, 1, 1, 1, 1, xs), False, "identity", "gemm")
    floats, split = 2 * 108 * 16 * 64 * 4, 2 * 108 * 64 * 96  # two row tiles of 108 K tiles
    for size in (op.workspace(), op.workspace() - 256, split + (op.workspace() - split) // 2, split + 200000, split, split - 256, floats):
        y = torch.full(ys, float("nan"), device="cuda:0")
        op.enqueue(x.cuda(), w.cuda(), None, y, torch.empty(size, dtype=torch.uint8, device="cuda:0"))
        assert torch.equal(y.cpu().double(), want), size  # whole numbers are exact
    with pytest.raises(dlp.DlprimError):
        op.enqueue(x.cuda(), w.cuda(), None, y, torch.empty(floats - 256, dtype=torch.uint8, device="cuda:0"))


# the kernels that the phases run on: float tiles, split tiles of 64 and 128 rows
PHASES = {
    (48, 64, 3, 2, 1, 1, 1, 24, 79, 81): {0}, (40, 32, 4, 2, 1, 1, 1, 3, 18, 22): {0}, (64, 48, 3, 1, 1, 1, 2, 33, 40, 40): set(),  # (24 channels a group are not packed)
    (20, 16, 5, 3, 2, 1, 1, 2, 17, 19): {0}, (36, 64, 3, 2, 1, 1, 2, 4, 18, 18): {0},  # groups
    (128, 48, 4, 2, 1, 1, 1, 32, 56, 56): {64}, (96, 64, 3, 2, 1, 1, 1, 33, 55, 57): {64}, (128, 64, 4, 2, 1, 1, 2, 32, 56, 56): {64},
    (200, 32, 4, 2, 1, 1, 1, 32, 56, 54): {128}, (160, 64, 2, 2, 0, 1, 2, 64, 56, 56): {128}, (72, 32, 3, 1, 1, 1, 1, 40, 38, 38): {128},
}


@pytest.mark.gpu
@pytest.mark.parametrize("c", PHASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_backward_data_phase_packing(c):
    """filters of all stride phases packed by one launch, in float and in split tiles; bias and activation behind the interleaving"""
    cin, cout, k, s, p, d, g, b, h, wd = c
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    w, dy, bias = torch.randn(ws, generator=gen), torch.randn(ys, generator=gen), torch.randn(cin, generator=gen)
    extra = tuple(n - ((o - 1) * s - 2 * p + d * (k - 1) + 1) for n, o in zip(xs[2:], ys[2:]))
    want = torch.nn.functional.conv_transpose2d(dy.double(), w.double(), None, s, p, extra, g, d)
    scale = torch.nn.functional.conv_transpose2d(dy.double().abs(), w.double().abs(), None, s, p, extra, g, d) + bias.double().abs().view(1, -1, 1, 1)
    bound = (cout // g * k * k + 8) * 2.0 ** -24  # one rounding per product and a few behind
    op = dlp.Conv2DBackwardData.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs), "gemm")
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    dx = torch.full(xs, float("nan"), device="cuda:0")
    names = _kernels(lambda: op.enqueue(dx, w.cuda(), dy.cuda(), work))
    if PHASES[c]:
        assert {_tile([n])[0] if n.startswith("conv_split") else 0 for n in names} == PHASES[c]
    if 0 not in PHASES[c]:
        bound = (cout // g * k * k / 4 + 8) * 2.0 ** -24  # (_bounds)
    assert ((dx.cpu().double() - want).abs() <= scale * bound).all()
    tr = dlp.TransposedConv2DForward.create(dlp.Conv2DSettings(cout, cin, k, s, d, p, g, ys), extra, True, "relu", "gemm")
    work = torch.empty(max(tr.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    y = torch.full(xs, float("nan"), device="cuda:0")
    tr.enqueue(dy.cuda(), w.cuda(), bias.cuda(), y, work)
    assert ((y.cpu().double() - (want + bias.double().view(1, -1, 1, 1)).relu()).abs() <= scale * bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(32, 80, 3, 1, 1, 1, 1, 3, 12, 12), (33, 130, 3, 2, 1, 1, 1, 2, 15, 13), (48, 70, 5, 1, 2, 1, 1, 1, 9, 7), (16, 65, 7, 1, 3, 1, 1, 2, 10, 8),
                               (256, 144, 1, 1, 0, 1, 2, 5, 8, 8), (128, 128, 1, 1, 0, 1, 1, 1, 1, 1), (20, 200, 8, 1, 4, 1, 1, 2, 9, 9)], ids=lambda c: "x".join(map(str, c)))
def test_gpu_split_filter_gradient(c):
    """filter gradients in tiles of 128x128 (more than 64 filters and 64 columns): remainders in rows, columns and pixels, planes of whole
    16-byte pieces and others, one and two words of tap mask and none; then infinities and NaN"""
    cin, cout, k, s, p, d, g, b, h, wd = c
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    x, dy = torch.randn(xs, generator=gen), torch.randn(ys, generator=gen)
    op = dlp.Conv2DBackwardFilter.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs))
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")

    def got(x):
        dw = torch.full(ws, float("nan"), device="cuda:0")
        op.enqueue(x.cuda(), dw, dy.cuda(), work)
        return dw.cpu().double()

    (name,) = _kernels(lambda: got(x), "wgrad")
    assert name.startswith("conv_wgrad_f32_kernel<128, 128,") and name.endswith(", true>") == (ys[0] * ys[2] * ys[3] >= 3), name
    grad = lambda x, dy: torch.nn.grad.conv2d_weight(x.double(), ws, dy.double(), s, p, d, g)
    want, scale = grad(x, dy), grad(x.abs(), dy.abs())
    n = ys[0] * ys[2] * ys[3]
    err = (got(x) - want).abs()
    assert (err <= scale * (n / 4 + 8) * 2.0 ** -24).all()  # as for the forward pass
    dy = dy.abs() + 0.5  # no product of infinity and zero inside the image
    for values in [(float("inf"), float("nan")), (float("-inf"), 3.4e38), (float("nan"), float("inf"))]:
        # the first pixel that a tap meets, and one in the middle
        x[0, 1, 0, 0], x[0, 3, xs[2] // 2, xs[3] // 2] = values
        mine, want = got(x), grad(x, dy)
        for f in (torch.isnan, torch.isposinf, torch.isneginf):
            # (a sum that the fp32 instruction rounds to infinity is finite in 64 bits)
            assert torch.equal(f(mine), f(want.float().double()))
        ok = torch.isfinite(mine)
        scale = grad(torch.nan_to_num(x, 0.0, 0.0, 0.0).abs(), dy)
        # the tile is computed again: one rounding per product
        assert ((mine - want).abs()[ok] <= scale[ok] * (n + 8) * 2.0 ** -24).all()


@pytest.mark.gpu
@pytest.mark.parametrize("c", [(32, 80, 3, 1, 1, 1, 1, 3, 12, 12), (33, 130, 3, 2, 1, 1, 1, 2, 15, 13), (256, 144, 1, 1, 0, 1, 2, 5, 8, 8)], ids=lambda c: "x".join(map(str, c)))
def test_gpu_split_filter_gradient_small_operands(c):
    cin, cout, k, s, p, d, g, b, h, wd = c
    gen = torch.Generator().manual_seed(sum(c))
    xs, ws, ys = _geometry(c)
    x0, dy0 = torch.randn(xs, generator=gen), torch.randn(ys, generator=gen)
    op = dlp.Conv2DBackwardFilter.create(dlp.Conv2DSettings(cin, cout, k, s, d, p, g, xs))
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    one_x, one_dy = x0.clone(), dy0.clone()
    one_x[:, :, h // 2] *= 2.0 ** -120  # one row of the image
    one_dy[:, 3] *= 2.0 ** -120
    for x, dy in [(x0 * 2.0 ** -120, dy0 * 2.0 ** 60), (x0 * 2.0 ** 60, dy0 * 2.0 ** -120), (one_x, dy0), (x0, one_dy)]:
        dw = torch.full(ws, float("nan"), device="cuda:0")
        op.enqueue(x.cuda(), dw, dy.cuda(), work)
        grad = lambda x, dy: torch.nn.grad.conv2d_weight(x.double(), ws, dy.double(), s, p, d, g)
        want, scale = grad(x, dy), grad(x.abs(), dy.abs())
        err = (dw.cpu().double() - want).abs()
        assert (err <= scale * ((ys[0] * ys[2] * ys[3] + 8) * 2.0 ** -24)).all()
        assert (err.norm() <= want.norm() * 2.0 ** -20) and (err[3].norm() <= want[3].norm() * 2.0 ** -20)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 2])
def test_gpu_filter_gradient_of_single_products(batch):
    """one product is rounded once, two at most three times, as on the fp32 instruction"""
    gen = torch.Generator().manual_seed(batch)
    x, dy = torch.randn((batch, 160, 1, 1), generator=gen), torch.randn((batch, 144, 1, 1), generator=gen)
    x = torch.cat([x] * 2, 1)[:, :256]
    op = dlp.Conv2DBackwardFilter.create(dlp.Conv2DSettings(256, 144, 1, 1, 1, 0, 1, tuple(x.shape)))
    work = torch.empty(max(op.workspace(), 1), dtype=torch.uint8, device="cuda:0")
    dw = torch.full((144, 256, 1, 1), float("nan"), device="cuda:0")
    op.enqueue(x.cuda(), dw, dy.cuda(), work)
    got, terms = dw.cpu().double()[:, :, 0, 0], dy.double()[:, :, 0, 0].unsqueeze(2) * x.double()[:, :, 0, 0].unsqueeze(1)
    assert ((got - terms.sum(0)).abs() <= terms.abs().sum(0) * (2 * batch - 1) * 2.0 ** -24).all()


# (cin, cout, k, stride, pad, create batch, call batch, h, w): gradients and transposed convolutions whose kernel reads the filter as it is
# from 131072 pixels and at most 32 rows on, and packed tiles below
@pytest.mark.gpu
@pytest.mark.parametrize("c", [(32, 16, 1, 1, 0, 2, 42, 56, 56), (24, 32, 1, 1, 0, 1, 140, 32, 32), (32, 16, 2, 2, 0, 2, 170, 56, 56), (16, 48, 3, 2, 1, 1, 44, 111, 111)],
                         ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("grow", [False, True])
def test_gpu_backward_data_batch_other_than_created(c, grow):
    """created at a small batch and called at a large one, and the other way round"""
    cin, cout, k, s, p, small, large, h, w = c
    create, batch = (small, large) if grow else (large, small)
    gen = torch.Generator().manual_seed(sum(c))
    f = torch.randint(-4, 5, (cout, cin, k, k), generator=gen).float()
    oh, ow = ((n + 2 * p - k) // s + 1 for n in (h, w))
    dy = torch.randint(-4, 5, (batch, cout, oh, ow), generator=gen).float()
    extra = tuple(n - ((o - 1) * s - 2 * p + k) for n, o in zip((h, w), (oh, ow)))
    want = torch.nn.functional.conv_transpose2d(dy, f, None, s, p, extra)  # whole numbers: exact in any order
    op = dlp.Conv2DBackwardData.create(dlp.Conv2DSettings(cin, cout, k, s, 1, p, 1, (create, cin, h, w)), "gemm")
    # the part for phase outputs grows with the batch
    work = torch.empty(max(op.workspace(), 1) * max(1, -(-batch // create)), dtype=torch.uint8, device="cuda:0")
    dx = torch.full((batch, cin, h, w), float("nan"), device="cuda:0")
    op.enqueue(dx, f.cuda(), dy.cuda(), work)
    assert torch.equal(dx.cpu(), want)
    tr = dlp.TransposedConv2DForward.create(dlp.Conv2DSettings(cout, cin, k, s, 1, p, 1, (create, cout, oh, ow)), extra, False, "identity", "gemm")
    work = torch.empty(max(tr.workspace(), 1) * max(1, -(-batch // create)), dtype=torch.uint8, device="cuda:0")
    y = torch.full((batch, cin, h, w), float("nan"), device="cuda:0")
    tr.enqueue(dy.cuda(), f.cuda(), None, y, work)
    assert torch.equal(y.cpu(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
def test_gpu_first_call_of_a_smaller_batch_in_a_capture(packed):
    """an operator's first call may sit in a capture at any batch up to the settings' one: nothing is allocated, replays repeat"""
    gen = torch.Generator().manual_seed(4)
    w = torch.randint(-4, 5, (128, 128, 3, 3), generator=gen).float()
    for batch in (64, 20, 3):
        op = dlp.Conv2DForward.create(dlp.Conv2DSettings(128, 128, 3, 1, 1, 1, 1, (64, 128, 14, 14)), False, "identity", "gemm")
        x, wd = torch.randint(-4, 5, (batch, 128, 14, 14), generator=gen).float().cuda(), w.cuda()
        y = torch.empty_like(x)
        ws = torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
        buf = torch.empty(op.packed_size(), dtype=torch.uint8, device="cuda:0")
        op.pack(wd, buf)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            if packed:
                op.enqueue_packed(x, wd, buf, None, y, ws)
            else:
                op.enqueue(x, wd, None, y, ws)
        for _ in range(3):
            x.copy_(torch.randint(-4, 5, x.shape, generator=gen).float())
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y.cpu().double(), torch.nn.functional.conv2d(x.cpu().double(), w.double(), None, 1, 1))


@pytest.mark.gpu
def test_gpu_rows_of_128_in_tiles_of_64_computed_again():
    """weights packed for 128-row tiles, a call in 64-row ones: infinities, NaN, and weights that are kept whole"""
    c = (128, 200, 3, 1, 1, 1, 1, 14, 28, 28)
    gen = torch.Generator().manual_seed(8)
    xs, ws, _ = _geometry(c)
    x, w = torch.randn(xs, generator=gen), torch.randn(ws, generator=gen)
    x[0, 3, 4, 5], x[5, 7, 20, 9] = float("inf"), float("nan")
    w[70] *= 2.0 ** -118  # second tile of 64, in the first packed one
    w[150, 5] *= 2.0 ** 40  # first tile of the second
    w[199, 2] = float("inf")
    got = []
    names = _kernels(lambda: got.append(_run(c, x, w, None, True, hint=64)))
    assert _tile(names) == (64, False)
    want = _conv64(c, x, w, None)
    inside = (slice(None), slice(None), slice(1, -1), slice(1, -1))  # (infinity times the padding's zeros is left to either)
    for f in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(f(got[0][inside]), f(want[inside]))
    scale = _conv64(c, torch.nan_to_num(x, 0.0, 0.0, 0.0).abs(), torch.nan_to_num(w, 0.0, 0.0, 0.0).abs(), None)
    ok = torch.isfinite(want)
    assert ((got[0] - want).abs()[ok] <= scale[ok] * ((128 * 9 + 8) * 2.0 ** -24)).all()  # one rounding per product
