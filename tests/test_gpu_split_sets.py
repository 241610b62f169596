"""fp32-accurate products (mode 2) whose K steps are dealt to two or four sets of waves per tile, against float64."""

import math

import pytest
import torch

from robolearn_amd import kernels as K

pytestmark = pytest.mark.gpu

# (m, n, k, splits, batch): one set (k < 256, or more than 256 tiles), two sets (k from 256) and four (k from 512),
# with every remainder of the 32-deep steps over the sets, short last steps, and splits whose last one is shorter
SHAPES = [(1, 1, 255, 1, 1), (1, 1, 256, 1, 1), (65, 63, 257, 1, 2), (64, 64, 289, 1, 1), (130, 70, 511, 1, 1),
          (64, 128, 512, 1, 2), (63, 65, 513, 1, 1), (100, 37, 545, 1, 2), (64, 1, 577, 1, 1), (33, 64, 609, 1, 1),
          (1024, 1024, 520, 1, 1), (1040, 1024, 520, 1, 1), (200, 101, 1100, 2, 1), (64, 70, 1030, 4, 2)]


@pytest.mark.parametrize("a_kcontig,b_kcontig", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("m,n,k,splits,batch", SHAPES)
def test_products_of_several_sets(gpu, m, n, k, splits, batch, a_kcontig, b_kcontig):
    """Row pitches past the row, a bias with ReLU, and a row with an infinity that must reach no other row.

    Bound per element: each of the 6 ceil(k / 16) accumulations and each sum of sets or splits rounds once at 2^-23
    (the matrix instruction may truncate) of sums that Cauchy-Schwarz bounds by the row's times the column's norm;
    the dropped products are below 2^-26 each, and the bias adds one rounding."""
    print(f"case sets m={m} n={n} k={k} splits={splits} batch={batch} ak={a_kcontig} bk={b_kcontig}", flush=True)
    g = torch.Generator().manual_seed(m + 3 * n + 7 * k)
    a, b = torch.randn(batch, m, k, generator=g), torch.randn(batch, n, k, generator=g)
    bias = torch.randn(batch, n, generator=g)
    bad = m // 2 if m > 1 else m
    if bad < m:
        a[:, bad, k - 1] = float("inf")

    def laid_out(t, kcontig, pad):  # rows of the operand with a pitch `pad` values past them
        t = t if kcontig else t.transpose(1, 2)
        out = torch.full((batch, t.shape[1], t.shape[2] + pad), float("nan"))
        out[:, :, : t.shape[2]] = t
        return out.to(gpu)

    ad, bd = laid_out(a, a_kcontig, 3), laid_out(b, b_kcontig, 1)
    d = torch.full((batch, m, n + 2), 7.0, device=gpu)
    workspace = torch.empty(splits * batch * m * n * 4, dtype=torch.uint8, device=gpu) if splits > 1 else None
    K.gemm(ad, bd, d, m=m, n=n, k=k, batch=batch, a_kcontig=a_kcontig, b_kcontig=b_kcontig, lda=ad.shape[2],
           ldb=bd.shape[2], ldd=n + 2, stride_a=ad[0].numel(), stride_b=bd[0].numel(), stride_d=m * (n + 2),
           bias=bias.to(gpu), stride_bias=n, epilogue="relu", mode=K.FP32_SPLIT, splits=splits, workspace=workspace)
    got = d.cpu().double()
    assert (got[:, :, n:] == 7.0).all()
    rows = torch.arange(m) != bad
    a64, b64 = a.double()[:, rows], b.double()
    expected = torch.relu(a64 @ b64.transpose(1, 2) + bias.double()[:, None])
    norms = a64.norm(dim=2)[:, :, None] * b64.norm(dim=2)[:, None]
    bound = norms * (4 + 2 * 6 * math.ceil(k / 16) + 2 * (splits + 4)) * 2.0**-24
    bound += (norms + bias.double().abs()[:, None]) * 2.0**-24
    error = (got[:, rows, :n] - expected).abs()
    assert (error <= bound).all(), float((error / bound).max())
