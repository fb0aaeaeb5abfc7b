"""Packed float weights stand for the filter: it may have been given back, and its memory to others, by the time of a call."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from test_split_gemm import _kernels

# (cin, cout, k, stride, batch of the settings, of the call, h, algorithm): start of the kernel's name
CASES = {
    (64, 64, 3, 1, 1, 1, 32, "gemm"): "conv_wave_f32_kernel",
    (237, 58, 1, 1, 2, 2, 9, "gemm"): "conv_wave_f32_kernel",
    (64, 64, 3, 1, 64, 1, 32, ""): "conv_wave_f32_kernel",      # Winograd by size, small calls directly
    (256, 256, 3, 1, 64, 1, 14, "gemm"): "conv_wave_f32_kernel",  # ... of an operator whose own batch is in bf16 parts
    (24, 96, 1, 1, 2, 48, 56, "gemm"): "conv_expand_f32_kernel",  # a batch above the settings'
    (256, 256, 3, 1, 64, 64, 14, "gemm"): "conv_split_f32_kernel",
}


@pytest.mark.gpu
@pytest.mark.parametrize("c", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_packed_weights_hold_the_filter(c):
    cin, cout, k, s, hint, b, h, algo = c
    gen = torch.Generator().manual_seed(sum(c[:7]))
    x, f = torch.randint(-3, 4, (b, cin, h, h), generator=gen).float(), torch.randint(-3, 4, (cout, cin, k, k), generator=gen).float()
    op = dlp.Conv2DForward.create(dlp.Conv2DSettings(cin, cout, k, s, 1, k // 2, 1, (hint, cin, h, h)), False, "identity", algo)
    work = torch.empty(op.workspace(), dtype=torch.uint8, device="cuda:0")
    size = op.packed_size()
    buf = torch.full((size + 256,), 171, dtype=torch.uint8, device="cuda:0")
    fd, y = f.cuda(), torch.full((b, cout, h, h), float("nan"), device="cuda:0")
    op.pack(fd, buf[:size])
    fd.fill_(float("nan"))
    (name,) = _kernels(lambda: op.enqueue_packed(x.cuda(), fd, buf[:size], None, y, work))
    assert name.startswith(CASES[c]), name
    assert torch.equal(y.cpu(), torch.nn.functional.conv2d(x, f, None, s, k // 2))
    assert (buf[size:] == 171).all()
