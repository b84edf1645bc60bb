"""Short bf16 products (csrc/kernels/mix_rank.hip) against 64-bit sums: rows and columns around the
tiles, column slices of wider rows, the forms that stay with the library, infinities, derivatives."""
import pytest
import torch

from replisense_rfq_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(x, w, out_dtype):
    y = ops.matmul_nt(x, w, out_dtype)
    assert y.dtype == (out_dtype or torch.bfloat16) and y.is_contiguous()
    xd, wd = x.double().cpu(), w.double().cpu()
    want, size = xd @ wd.t(), xd.abs() @ wd.abs().t()
    # products of bf16 are exact in fp32, each of K sums rounds a part of `size` to 2^-24; bf16: half
    # a step of 2^-8 of the value more
    tol = x.shape[1] * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if y.dtype == torch.bfloat16 else 0)
    assert bool(((y.double().cpu() - want).abs() <= tol).all())


# 512 x 4,096 is the largest, one row more stays with the library
@pytest.mark.parametrize("M,N", [(1, 4), (15, 60), (16, 64), (17, 260), (64, 2048), (129, 68), (512, 4096), (513, 4096)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 40])          # 40: the library
@pytest.mark.parametrize("out_dtype", [None, torch.float32])
def test_short_products(M, N, K, out_dtype):
    g = torch.Generator().manual_seed(M + K)
    wide, w = torch.randn(M, K + 16, generator=g).to(DEV, torch.bfloat16), torch.randn(N, K, generator=g).to(DEV, torch.bfloat16)
    _check(wide[:, 8:8 + K], w, out_dtype)
    _check(wide[:, 3:3 + K], w, out_dtype)                    # rows that begin at odd addresses
    if N % 4 == 0 and N > 4:
        _check(wide[:, :K], w[:N - 1], out_dtype)             # columns that are no multiple of four


def test_infinities_stay_in_their_row_and_column():
    x, w = torch.ones(20, 64, device=DEV, dtype=torch.bfloat16), torch.ones(72, 64, device=DEV, dtype=torch.bfloat16)
    x[3, 5], w[70, 9] = float("inf"), float("nan")
    y = ops.matmul_nt(x, w, torch.float32)
    want = torch.full((20, 72), 64.0)
    want[3], want[:, 70] = float("inf"), float("nan")
    torch.testing.assert_close(y.cpu(), want, atol=0, rtol=0, equal_nan=True)


def test_derivatives_are_the_library_products():
    x, w = (torch.randn(n, 64, device=DEV, dtype=torch.bfloat16) for n in (8, 12))
    x.requires_grad_()
    ops.matmul_nt(x, w).sum().backward()
    torch.testing.assert_close(x.grad, w.sum(0, keepdim=True).expand(8, 64), atol=0.05, rtol=0.02)
    with torch.no_grad():
        assert ops.matmul_nt(x, w).shape == (8, 12)


def _check_f32(x, w):
    y = ops.matmul_nt(x, w)
    assert y.dtype == torch.float32 and y.is_contiguous()
    xd, wd = x.double().cpu(), w.double().cpu()
    # each of K sums rounds a part of the sum of sizes to 2^-24; what the parts leave out is less than 2^-24 of every product
    tol = (x.shape[1] + 1) * 2.0 ** -24 * (xd.abs() @ wd.abs().t())
    assert bool(((y.double().cpu() - xd @ wd.t()).abs() <= tol).all())


# a wave with 16, 32 (from 2,048 tiles of 16 x 16 on) and 64 columns (9,216), one block of rows (64 x 2,048) to sixteen
# (300,000 x 4), fewer columns than a wave takes otherwise (20, 36), more than a round of them beside each other (70,000); tiles
# that are cut, columns slices of wider rows, rows at odd addresses (there the library, or a copy)
@pytest.mark.parametrize("M,N", [(1, 4), (17, 60), (64, 2048), (129, 68), (645, 1028), (1540, 1030 * 2), (2100, 2052), (9000, 1024),
                                 (40000, 20), (20000, 36), (300000, 4), (33, 70000)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 40])
def test_short_fp32_products(M, N, K):
    g = torch.Generator().manual_seed(M + K)
    wide, w = torch.randn(M, K + 12, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV)
    _check_f32(wide[:, 4:4 + K], w)
    if M < 200:
        _check_f32(wide[:, 3:3 + K], w)
        _check_f32(torch.frombuffer(bytearray(4 * M * K + 4), dtype=torch.float32)[1:].view(M, K).to(DEV), w[:N - 1])


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38, 1e-38])
def test_fp32_products_at_the_ends_of_the_range(value):
    x, w = torch.full((40, 64), 0.25, device=DEV), torch.full((72, 64), 0.5, device=DEV)
    w[:, 7] = -0.5
    x[3, 5], w[70, 9] = value, value
    y = ops.matmul_nt(x, w)
    want = x.cpu() @ w.cpu().t()
    torch.testing.assert_close(y.cpu(), want, atol=0, rtol=1e-6, equal_nan=True)


@pytest.mark.parametrize("M,N,K", [(40, 72, 64), (2100, 2052, 64), (64, 512, 128)])
def test_fp32_products_that_end_just_below_the_range(M, N, K):
    """(2^64 - 2^55)^2 is a number of fp32; the square of what it rounds to in bf16 is not."""
    x, w = torch.zeros(M, K, device=DEV), torch.zeros(N, K, device=DEV)
    x[::3, 5] = w[::2, 5] = 2.0 ** 64 - 2.0 ** 55
    _check_f32(x, w)
    x[::2, 7], w[::2, 7] = 2.0 ** 63, -(2.0 ** 63)           # finite sums of both signs
    _check_f32(x, w)


@pytest.mark.parametrize("a,b", [(1e-36, 1.0), (1.0, 1e-36), (1e10, 1e-36), (1e-33, 1e-4)])
@pytest.mark.parametrize("M,N,K", [(40, 72, 64), (2100, 2052, 32), (64, 512, 128)])
def test_fp32_products_of_small_operands(M, N, K, a, b):
    """Entries whose third part bf16 does not hold, of all rows and of every third, keep the precision that others have."""
    g = torch.Generator().manual_seed(M)
    x, w = (torch.randn(n, K, generator=g).to(DEV) for n in (M, N))
    _check_f32(x * a, w * b)
    x[1::3] *= a
    w[::3] *= b
    x[5] = 0.0
    _check_f32(x, w)


def test_fp32_products_keep_autocast_and_derivatives():
    x, w = (torch.randn(n, 64, device=DEV) for n in (8, 12))
    with torch.autocast("cuda", torch.bfloat16):
        assert ops.matmul_nt(x, w).dtype == torch.bfloat16
    x.requires_grad_()
    ops.matmul_nt(x, w).sum().backward()
    torch.testing.assert_close(x.grad, w.sum(0, keepdim=True).expand(8, 64), atol=1e-4, rtol=1e-4)
    y = torch.func.vmap(lambda a: ops.matmul_nt(a, w))(torch.ones(3, 5, 64, device=DEV))
    torch.testing.assert_close(y, w.sum(1).expand(3, 5, 12), atol=1e-4, rtol=1e-4)


# rows and columns around a wave's tile, slices of wider rows on all sides, results of rows in either order; what stays with
# the library: 2^20 results and one row of 128 terms, columns that are no whole tiles, 40 terms, a result in memory of an operand
@pytest.mark.parametrize("B,M,N", [(1, 1, 64), (3, 17, 320), (32, 64, 512), (32, 65, 512), (2, 5, 72)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 40])
@pytest.mark.parametrize("rows_first", [False, True])
def test_batches_of_short_products(B, M, N, K, rows_first):
    g = torch.Generator().manual_seed(B * M + K)
    x = torch.randn(M, B, K + 24, generator=g).to(DEV, torch.bfloat16)[:, :, 8:8 + K].transpose(0, 1)
    w = torch.randn(B, K, N + 8, generator=g).to(DEV, torch.bfloat16)[:, :, :N]
    wide = torch.full((M, B, N + 64) if rows_first else (B, M, N + 64), 7.0, device=DEV)
    out = wide[:, :, :N].transpose(0, 1) if rows_first else wide[:, :, :N]
    assert ops.bmm_f32(x, w, out=out) is out
    xd, wd = x.double().cpu(), w.double().cpu()
    tol = K * 2.0 ** -24 * (xd.abs() @ wd.abs())             # as above
    assert bool(((out.double().cpu() - xd @ wd).abs() <= tol).all()) and bool((wide[:, :, N:] == 7.0).all())


# more than 2^20 results: workgroups of one, three and eight waves, several columns' workgroups, rows that blocks do not divide,
# more blocks than workgroups and fewer, results past the caches; 128 terms and fewer than 500 rows, or up to 2^23 results, stay
# with the library
@pytest.mark.parametrize("B,M,N,K", [(70, 501, 64, 128), (9, 500, 576, 96), (9, 499, 576, 128), (2, 2100, 512, 128), (1, 600, 4096, 32),
                                     (300, 65, 128, 64), (32, 130, 512, 32), (5, 4097, 128, 64),
                                     (3, 21899, 512, 32), (33, 501, 576, 128), (70, 1999, 64, 128), (3, 2100, 1536, 128)])
@pytest.mark.parametrize("rows_first", [False, True])
def test_batches_of_many_rows(B, M, N, K, rows_first):
    test_batches_of_short_products(B, M, N, K, rows_first)


def test_batches_that_the_kernel_leaves_alone():
    x, w = torch.randn(2, 4, 64, device=DEV).bfloat16(), torch.randn(2, 64, 64, device=DEV).bfloat16()
    out = torch.empty(2, 4, 64, device=DEV)
    ok = lambda *a: ops._short_batch(*a)  # noqa: E731
    assert ok(x, w, out) and not ok(x, w, out.bfloat16()) and not ok(x[:, :, 1:33], w[:, :32], out)
    assert not ok(x, w.transpose(1, 2), out) and not ok(x, w, out[:, :1].expand(2, 4, 64)) and not ok(x, w[:1], out)
    assert not ok(x[:, :0], w, out[:, :0]) and not ok(x, w, torch.empty(2, 5, 64, device=DEV))
    # a result beside an operand in the same memory, operands at odd addresses, and shapes alone
    both = torch.zeros(2, 4, 96 + 64, device=DEV)
    a = both.view(torch.bfloat16)[:, :, :64].copy_(x)
    ops.bmm_f32(a, w, out=both[:, :, 96:])
    torch.testing.assert_close(both[:, :, 96:], x.float() @ w.float(), atol=1e-4, rtol=1e-4)
    assert torch.equal(both.view(torch.bfloat16)[:, :, :64], x)
    odd = torch.zeros(2 * 4 * 64 + 1, device=DEV, dtype=torch.bfloat16)[1:].view(2, 4, 64).copy_(x)
    torch.testing.assert_close(ops.bmm_f32(odd, w, out=out), x.float() @ w.float(), atol=1e-4, rtol=1e-4)
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        fake = [torch.empty(2, 4, 64, device=DEV, dtype=torch.bfloat16), torch.empty(2, 64, 64, device=DEV, dtype=torch.bfloat16)]
        assert ops.bmm_f32(*fake, out=torch.empty(2, 4, 64, device=DEV)).shape == (2, 4, 64)
        assert ops.matmul_nt(torch.empty(4, 64, device=DEV), torch.empty(8, 64, device=DEV)).shape == (4, 8)
    y = torch.func.vmap(lambda a: ops.bmm_f32(a, w))(torch.stack([x, x]))
    torch.testing.assert_close(y[1], x.float() @ w.float(), atol=1e-3, rtol=1e-4)
