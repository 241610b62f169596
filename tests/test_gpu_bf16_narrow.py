"""bf16 products on 64 x 64 tiles against float64, and bit for bit against the 256 x 128 tiles."""

import math

import pytest
import torch

from robolearn_amd import kernels as K

pytestmark = pytest.mark.gpu

# (m, n, k, splits, batch): one value, edges of the 64-wide tiles and of the 64-deep steps, odd row lengths
SHAPES = [(1, 1, 1, 1, 1), (1, 130, 39, 1, 2), (63, 65, 64, 1, 1), (64, 128, 65, 1, 2), (130, 101, 32, 1, 2),
          (2, 3, 200, 4, 1), (300, 77, 123, 2, 2), (1000, 512, 39, 1, 2), (101, 514, 1000, 8, 2)]


@pytest.mark.parametrize("a_kcontig,b_kcontig", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("pad", [0, 1, 6])
@pytest.mark.parametrize("m,n,k,splits,batch", SHAPES)
def test_narrow_products(gpu, m, n, k, splits, batch, pad, a_kcontig, b_kcontig):
    """Row pitches with pads of 0, 1 and 6 values (rows at any even address; the pad holds NaN), with bias, ReLU, beta
    C and the bf16 copy when unsplit.  The same operands stored as float32 run the 256 x 128 tiles, whose products
    and sums are the same; against float64 each of ceil(k / 16) accumulations, the splits and the epilogue may round
    once at 2^-23 of a sum bounded by the row's times the column's norm."""
    print(f"case narrow m={m} n={n} k={k} splits={splits} batch={batch} pad={pad} ak={a_kcontig} bk={b_kcontig}", flush=True)
    g = torch.Generator().manual_seed(m + 3 * n + 7 * k)
    a = torch.randn(batch, m, k, generator=g).bfloat16()
    b = torch.randn(batch, n, k, generator=g).bfloat16()
    bias, c = torch.randn(batch, n, generator=g).to(gpu), torch.randn(batch, m, n, generator=g).to(gpu)

    def stored(x, kcontig, dtype):
        x = x if kcontig else x.transpose(1, 2)
        out = torch.full((batch, x.shape[1], x.shape[2] + pad), float("nan"), dtype=dtype)
        out[..., : x.shape[2]] = x
        return out.to(gpu), out.shape[2], out.shape[1] * out.shape[2]

    results = []
    for dtype in (torch.bfloat16, torch.float32):
        (ad, lda, sa), (bd, ldb, sb) = stored(a, a_kcontig, dtype), stored(b, b_kcontig, dtype)
        d = torch.full((batch, m, n), 7.0, device=gpu)
        half = torch.full((batch, m, n), 7.0, device=gpu, dtype=torch.bfloat16)
        workspace = torch.empty(splits * batch * (m * n + m) * 4, dtype=torch.uint8, device=gpu) if splits > 1 else None
        K.gemm(ad, bd, d, m=m, n=n, k=k, batch=batch, a_kcontig=a_kcontig, b_kcontig=b_kcontig, lda=lda, ldb=ldb,
               ldd=n, stride_a=sa, stride_b=sb, stride_d=m * n, c=c, beta=0.5, bias=bias, stride_bias=n,
               epilogue="relu", mode=K.BF16, splits=splits, workspace=workspace, d_bf16=half)
        results.append((d.cpu(), half.cpu()))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    a64, b64 = a.double(), b.double()
    exact = torch.stack([x @ y.t() for x, y in zip(a64, b64)]) + bias.cpu().double()[:, None, :]
    exact = torch.relu(exact) + 0.5 * c.cpu().double()
    scale = a64.norm(dim=2)[:, :, None] * b64.norm(dim=2)[:, None, :] + 10.0
    bound = scale * (4 + 2 * math.ceil(k / 16) + splits) * 2.0**-24
    assert ((results[0][0].double() - exact).abs() <= bound).all()
    assert torch.equal(results[0][1], results[0][0].bfloat16())


# just past the line from which products on operands of 16-byte rows take 256 x 128 tiles (in one launch, in two splits, as
# twins, with output rows of odd length) and just below it (k 104); ragged rows, columns and K, and pitches of 16-byte
# rows (pads of 0 and 8 values)
@pytest.mark.parametrize("a_kcontig,b_kcontig", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("pad", [0, 8])
@pytest.mark.parametrize("m,n,k,splits,batch", [(2040, 4216, 1416, 1, 1), (2040, 4216, 104, 1, 1), (1016, 4216, 2832, 2, 1),
                                                (1016, 4216, 1416, 1, 2), (1001, 8101, 552, 1, 2)])
def test_products_at_the_line_between_tiles(gpu, m, n, k, splits, batch, pad, a_kcontig, b_kcontig):
    test_narrow_products(gpu, m, n, k, splits, batch, pad, a_kcontig, b_kcontig)


# rows too far apart for the small tiles' offsets run the 256 x 128 tiles, rows of 16 bytes (2^22) and others alike
@pytest.mark.parametrize("a_kcontig,b_kcontig", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("pitch", [(1 << 22) - 1, 1 << 22, (1 << 22) + 1])
@pytest.mark.parametrize("far", [0, 1])
def test_far_rows_give_the_same_bits(gpu, far, pitch, a_kcontig, b_kcontig):
    print(f"case far bf16 operand={far} pitch={pitch} ak={a_kcontig} bk={b_kcontig}", flush=True)
    m, n, k = 70, 133, 41
    g = torch.Generator(device=gpu).manual_seed(pitch)
    shapes = ((m, k) if a_kcontig else (k, m), (n, k) if b_kcontig else (k, n))
    values = [torch.randn(s, generator=g, device=gpu).bfloat16() for s in shapes]
    results = []
    for apart in (False, True):
        ops = list(values)
        if apart:
            rows, cols = shapes[far]
            store = torch.empty((rows - 1) * pitch + cols, dtype=torch.bfloat16, device=gpu)
            ops[far] = store.as_strided((rows, cols), (pitch, 1)).copy_(values[far])
        d = torch.full((m, n), 7.0, device=gpu)
        K.gemm(ops[0], ops[1], d, m=m, n=n, k=k, a_kcontig=a_kcontig, b_kcontig=b_kcontig, lda=ops[0].stride(0),
               ldb=ops[1].stride(0), ldd=n, mode=K.BF16)
        results.append(d)
    assert torch.equal(*results)
