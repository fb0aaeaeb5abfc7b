"""Plans of convolutions called at another batch than they were created with (tests/cpp/plans.cpp: the library's own plan functions, no GPU), and
the calls themselves on whole numbers, exact in any order of the sums."""
import os
import subprocess

import pytest

torch = pytest.importorskip("torch")

import dlprimitives_amd as dlp

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "bin", "plans")


@pytest.mark.parametrize("part", ["packed", "tiles", "lds"])
def test_plans(part):
    if not os.path.exists(BIN):
        pytest.fail("tests/bin/plans is not built: run `make -C tests/cpp` (or __graft_entry__.build())")
    r = subprocess.run([BIN, part], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("algo", ["gemm", ""])
@pytest.mark.parametrize("channels, size, hint, batches", [(256, 14, 21, (15, 16, 20, 21)), (384, 7, 28, (25, 27)), (192, 14, 30, (26,))])
def test_gpu_batch_below_the_settings(channels, size, hint, batches, algo):
    """Batches that an operator of their own would run in 64x64 tiles of bf16 parts, on one created where the LDS-patch kernel is the better one."""
    gen = torch.Generator().manual_seed(channels + hint)
    x, f = (torch.randint(-3, 4, n, generator=gen).float() for n in ((hint, channels, size, size), (channels, channels, 3, 3)))
    settings = dlp.Conv2DSettings(channels, channels, 3, 1, 1, 1, 1, tuple(x.shape))
    op = dlp.Conv2DForward.create(settings, False, "identity", algo)
    back = dlp.Conv2DBackwardData.create(settings, algo)
    xd, fd = x.cuda(), f.cuda()
    work = torch.empty(max(op.workspace(), back.workspace()), dtype=torch.uint8, device="cuda:0")
    packed = torch.full((op.packed_size(),), 255, dtype=torch.uint8, device="cuda:0")
    op.pack(fd, packed)
    # (Winograd's transforms round, at the size of the sum)
    bound = 0.0 if op.algo() == "gemm" else channels * 9 * 9 * 2.0 ** -20
    for batch in batches:
        shape = (batch,) + tuple(x.shape[1:])
        want = torch.nn.functional.conv2d(x[:batch], f, None, 1, 1)
        grad = torch.nn.functional.conv_transpose2d(x[:batch], f, None, 1, 1)
        part = xd[:batch].contiguous()
        for call, ref in ((lambda y: op.enqueue(part, fd, None, y, work), want), (lambda y: op.enqueue_packed(part, fd, packed, None, y, work), want),
                          (lambda y: back.enqueue(y, fd, part, work), grad)):
            y = torch.full(shape, float("nan"), device="cuda:0")
            call(y)
            assert (y.cpu() - ref).abs().max() <= bound, batch
