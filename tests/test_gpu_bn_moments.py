"""BatchNorm batch statistics: chunk moments by row group and their merge over few and many chunks, against float64."""

import pytest
import torch

from robolearn_amd import kernels as K

pytestmark = pytest.mark.gpu


# rows at the edges of the 16 row groups, of the 256-row chunks, of the batches of 4 chunks and of the 8 chunks that an
# apply pass merges itself; channels at the edges of the 64 that a workgroup takes
@pytest.mark.parametrize("rows", [2, 15, 16, 17, 255, 256, 257, 1024, 1030, 1290, 2047, 2048, 2049])
@pytest.mark.parametrize("channels", [4, 64, 68])
@pytest.mark.parametrize("bf16", [False, True])
def test_batch_statistics(gpu, rows, channels, bf16):
    """Bound: each of the at most 16 + 16 + 9 roundings of a chunk's, a group's and a merge's mean is 2^-24 of a value
    below 4 sigma + |mean|, and each term of the variance takes twice the relative error of its difference."""
    print(f"case statistics rows={rows} channels={channels} bf16={bf16}", flush=True)
    g = torch.Generator().manual_seed(rows + channels)
    x = torch.randn(2, rows, channels, generator=g) * 1.5 + torch.randn(2, 1, channels, generator=g)
    x = x.to(torch.bfloat16) if bf16 else x
    xd, ones = x.to(gpu), torch.ones(2, channels, device=gpu)
    zeros, dy = torch.zeros(2, channels, device=gpu), torch.randn(2, rows, channels, generator=g).to(gpu)
    mean, var, rm, rv = (torch.full((2, channels), v, device=gpu) for v in (7.0, 7.0, 0.0, 1.0))
    partial = torch.empty(4 * K.chunks(rows) * channels, device=gpu)
    y, dx = torch.empty(2, rows, channels, device=gpu), torch.empty(2, rows, channels, device=gpu)
    K.bn_forward(xd, ones, zeros, rm, rv, mean, var, partial, y, rows=rows, channels=channels, ensemble=2)
    x64 = x.double()
    mu, variance = x64.mean(1), x64.var(1, unbiased=False)
    spread = x64.abs().amax(1)
    assert ((mean.cpu().double() - mu).abs() <= 41 * 2.0**-24 * spread).all()
    assert ((var.cpu().double() - variance).abs() <= 4 * 41 * 2.0**-24 * spread**2).all()
    sums, dw, db = torch.empty(4 * channels, device=gpu), torch.empty_like(mean), torch.empty_like(mean)
    K.bn_backward(xd, dy, None, ones, mean, var, partial, sums, dx, dw, db, rows=rows, channels=channels,
                  ensemble=2)
    dy64 = dy.cpu().double()
    unit = (x64 - mu[:, None]) * torch.rsqrt(variance + 1e-5)[:, None]
    slack = 64 * 2.0**-24  # the sums' 16 + 16 + 9 roundings and those of the unit input
    assert ((db.cpu().double() - dy64.sum(1)).abs() <= slack * dy64.abs().sum(1)).all()
    scale = (spread * torch.rsqrt(variance + 1e-5))[:, None]
    # the mean's error moves the unit input by `scale`, the variance's by its square
    dw_slack = slack * (dy64.abs() * (unit.abs() * (1 + 2 * scale**2) + scale)).sum(1)
    assert ((dw.cpu().double() - (dy64 * unit).sum(1)).abs() <= dw_slack).all()
