"""Inner products in tiles of 16 outputs x 16 batch rows (ip_stream_kernel_16x16) and on either side of the line to ip_stream_kernel, against torch
in 64 bits on the same operands."""
import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp
from dlprimitives_amd.capi import BFLOAT16_DATA, FLOAT_DATA
from test_split_gemm import _kernels

# batch, inputs, outputs: whether the tiles are 16x16
CASES = {
    (1, 8, 1): True,          # a piece of a K tile, fifteen wavefronts without work
    (16, 64, 16): True,       # one whole K tile
    (15, 4104, 1000): True,   # a last K tile of eight, outputs and batch off the tile
    (16, 1000, 8200): True,   # more tiles than CUs
    (17, 520, 4096): True,    # 512 tiles
    (17, 520, 4112): False,
    (33, 8192, 1360): True,   # 255 tiles of long rows
    (49, 8192, 1040): False,
    (4, 240, 8192): True,     # short rows: two tiles a CU
    (4, 240, 8208): False,
    (2, 8192, 4112): False,   # a tile more than CUs
    (16, 20000, 2000): True,  # rows of 80 KB (40 in bf16): enough tiles
    (1, 24576, 32): False,    # ... and too few
}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("c", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gpu_ip_tiles(c, dtype):
    batch, inputs, outputs = c
    gen = torch.Generator().manual_seed(sum(c))
    x, w = torch.randn(batch, inputs, generator=gen).to(dtype), torch.randn(outputs, inputs, generator=gen).to(dtype)
    bias = torch.randn(outputs, generator=gen)
    op = dlp.IPForward.create(dlp.IPSettings(inputs, outputs, batch, dtype=BFLOAT16_DATA if dtype == torch.bfloat16 else FLOAT_DATA), True, "relu")
    y = torch.full((batch, outputs), float("nan"), dtype=dtype, device="cuda:0")
    (name,) = _kernels(lambda: op.enqueue(x.cuda(), w.cuda(), bias.cuda(), y), "ip_direct")
    assert name.startswith("ip_stream_kernel_16x16<") == CASES[c], name
    want = (x.double() @ w.double().t() + bias.double()).relu()
    # one rounding a product, a few behind, and that to the storage type
    bound = (x.double().abs() @ w.double().abs().t() + bias.double().abs()) * ((inputs + 8) * 2.0 ** -24) + (want * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
    assert ((y.cpu().double() - want).abs() <= bound).all()
